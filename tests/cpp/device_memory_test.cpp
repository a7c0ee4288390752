// Host test of device_memory.hip: the runtime's entry points are stood in for, with two
// devices of a fixed room.  Prints "ok".
#include "../../m3lb_amd/csrc/device_memory.hpp"

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>

namespace {
int g_current = 0;
size_t g_room[2] = {100, 100};
std::map<void*, std::pair<int, size_t>> g_live;
uintptr_t g_next = 16;
int g_other_error = 0;
#define REQUIRE(x)                                \
  do {                                            \
    if (!(x)) {                                   \
      std::printf("line %d: %s\n", __LINE__, #x); \
      std::exit(1);                               \
    }                                             \
  } while (0)

struct Handle {
  int device = 0;
  void* spare = nullptr;
  int asked = 0;
};
bool give_back(void* owner) {
  Handle* h = static_cast<Handle*>(owner);
  ++h->asked;
  if (!h->spare) return false;
  REQUIRE(hipFree(h->spare) == hipSuccess);
  h->spare = nullptr;
  return true;
}
}  // namespace

extern "C" {
hipError_t hipGetDevice(int* d) { *d = g_current; return hipSuccess; }
hipError_t hipSetDevice(int d) {
  if (d < 0 || d > 1) return hipErrorInvalidDevice;
  g_current = d;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipExtGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
  if (g_other_error) return hipErrorUnknown;
  if (n > g_room[g_current]) return hipErrorOutOfMemory;
  g_room[g_current] -= n;
  *p = reinterpret_cast<void*>(g_next += 16);
  g_live[*p] = {g_current, n};
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  const auto it = g_live.find(p);
  if (it == g_live.end()) return hipErrorInvalidValue;
  g_room[it->second.first] += it->second.second;
  g_live.erase(it);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = g_room[g_current];
  *t = 100;
  return hipSuccess;
}
}

int main() {
  using namespace m3lb;
  Handle a, b, c;
  c.device = 1;
  for (Handle* h : {&a, &b, &c}) {
    REQUIRE(device_alloc_plain(h->device, &h->spare, 30) == hipSuccess);
    REQUIRE(g_live[h->spare].first == h->device);  // whatever device is current
    spare_register({h->device, h, give_back});
  }
  REQUIRE(g_current == 0 && device_free_bytes(0) == 40 && device_free_bytes(1) == 70);
  void* p = nullptr;
  // room without the spares: nobody is asked
  REQUIRE(device_alloc(0, &p, 40) == hipSuccess && a.asked + b.asked + c.asked == 0);
  // one spare is enough; those of another device stay
  void* q = nullptr;
  REQUIRE(device_alloc(0, &q, 25) == hipSuccess && !a.spare && b.spare && c.spare);
  REQUIRE(g_live[q].first == 0 && c.asked == 0);
  // the same without asking: refused, and the pointer says so
  void* r = &a;
  REQUIRE(device_alloc_plain(0, &r, 25) == hipErrorOutOfMemory && r == nullptr && b.spare);
  // more than the spares hold: all are taken, and it fails
  REQUIRE(device_alloc(0, &r, 90) == hipErrorOutOfMemory && r == nullptr && !b.spare && c.spare);
  // another device's memory, the current device unchanged
  REQUIRE(device_alloc(1, &r, 95) == hipSuccess && !c.spare && g_live[r].first == 1 && g_current == 0);
  // another error is no reason to ask
  REQUIRE(hipFree(p) == hipSuccess);
  REQUIRE(device_alloc_plain(0, &a.spare, 30) == hipSuccess);
  const int asked = a.asked;
  g_other_error = 1;
  REQUIRE(device_alloc(0, &p, 5) == hipErrorUnknown && a.asked == asked && a.spare);
  g_other_error = 0;
  // a handle that is gone is not asked
  spare_unregister(&a);
  REQUIRE(device_alloc(0, &p, 90) == hipErrorOutOfMemory && a.asked == asked && a.spare);
  REQUIRE(device_alloc(7, &p, 1) == hipErrorInvalidDevice && device_free_bytes(7) == 0);
  std::printf("ok\n");
  return 0;
}
