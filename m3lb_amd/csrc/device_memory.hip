// device_memory.hip -- allocations of device_memory.hpp.
#include "device_memory.hpp"

#include <algorithm>
#include <mutex>
#include <vector>

namespace m3lb {
namespace {

struct Registry {
  std::mutex mu;
  std::vector<Spare> spares;
};
Registry& registry() {
  static Registry* r = new Registry;  // never destroyed: handles may outlive static destructors
  return *r;
}

// Makes `device` current for a scope.
struct OnDevice {
  int before = -1;
  bool ok = true;
  explicit OnDevice(int device) {
    ok = hipGetDevice(&before) == hipSuccess;
    if (ok && before != device) ok = hipSetDevice(device) == hipSuccess;
    else before = -1;
  }
  ~OnDevice() {
    if (before >= 0) (void)hipSetDevice(before);
  }
};

}  // namespace

void spare_register(const Spare& s) {
  Registry& r = registry();
  std::lock_guard<std::mutex> l(r.mu);
  r.spares.push_back(s);
}

void spare_unregister(void* owner) {
  Registry& r = registry();
  std::lock_guard<std::mutex> l(r.mu);
  r.spares.erase(std::remove_if(r.spares.begin(), r.spares.end(),
                                [&](const Spare& s) { return s.owner == owner; }),
                 r.spares.end());
}

hipError_t device_alloc_plain(int device, void** p, size_t bytes) {
  *p = nullptr;
  const OnDevice on(device);
  if (!on.ok) return hipErrorInvalidDevice;
  const hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();  // the caller has it
  }
  return e;
}

hipError_t device_alloc(int device, void** p, size_t bytes) {
  hipError_t e = device_alloc_plain(device, p, bytes);
  if (e != hipErrorOutOfMemory) return e;
  Registry& r = registry();
  std::lock_guard<std::mutex> l(r.mu);  // a handle is not destroyed meanwhile
  for (const Spare& s : r.spares) {
    if (s.device != device || !s.give_back(s.owner)) continue;
    e = device_alloc_plain(device, p, bytes);
    if (e != hipErrorOutOfMemory) return e;
  }
  return e;
}

size_t device_free_bytes(int device) {
  const OnDevice on(device);
  size_t free_b = 0, total_b = 0;
  if (!on.ok || hipMemGetInfo(&free_b, &total_b) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return free_b;
}

}  // namespace m3lb
