// Host test of transfer.hip without a device: the runtime's entry points are stood in
// for below, "kernels" run on the calling thread.  A range of memory counts as in
// flight from its launch until the wait for it or for its stream.  Prints "ok".
#include "../../m3lb_amd/csrc/transfer.hpp"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <thread>
#include <vector>

namespace {
std::mutex g_mu;
std::map<char*, size_t> g_pinned;       // live pinned ranges
std::set<char*> g_in_flight;            // pinned ranges that the device may still write
std::map<hipEvent_t, char*> g_event_of; // what the event's last record waits for
thread_local char* t_last = nullptr;    // range of this thread's last launch
std::atomic<int> g_fail_records{0}, g_fail_syncs{0}, g_fail_mallocs{0};
std::atomic<int> g_peak{0}, g_mallocs{0}, g_incoherent{0}, g_device_events{0}, g_reused{0};
thread_local std::string t_msg;

char* range_of(const void* p) {
  auto it = g_pinned.upper_bound(const_cast<char*>(static_cast<const char*>(p)));
  if (it == g_pinned.begin()) std::abort();
  --it;
  if (static_cast<const char*>(p) >= it->first + it->second) std::abort();
  return it->first;
}
void launched_into(const void* p) {
  std::lock_guard<std::mutex> l(g_mu);
  char* r = range_of(p);
  if (!g_in_flight.insert(r).second) ++g_reused;  // the device still writes an older result there
  t_last = r;
}
#define REQUIRE(x)                                             \
  do {                                                         \
    if (!(x)) {                                                \
      std::printf("line %d: %s\n", __LINE__, #x);              \
      std::exit(1);                                            \
    }                                                          \
  } while (0)
}  // namespace

extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipExtGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "failed by the test"; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
  if (g_fail_mallocs > 0) { --g_fail_mallocs; return hipErrorOutOfMemory; }
  *p = std::malloc(n);
  std::lock_guard<std::mutex> l(g_mu);
  g_pinned[static_cast<char*>(*p)] = n;
  ++g_mallocs;
  if (!(flags & hipHostMallocCoherent)) ++g_incoherent;
  if (int(g_pinned.size()) > g_peak) g_peak = int(g_pinned.size());
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> l(g_mu);
  REQUIRE(g_in_flight.count(static_cast<char*>(p)) == 0);  // never freed while written
  REQUIRE(g_pinned.erase(static_cast<char*>(p)) == 1);
  std::free(p);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags) {
  if (!(flags & hipEventReleaseToSystem)) ++g_device_events;
  *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  if (g_fail_records > 0) { --g_fail_records; return hipErrorUnknown; }
  std::lock_guard<std::mutex> l(g_mu);
  g_event_of[e] = t_last;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  std::lock_guard<std::mutex> l(g_mu);
  g_in_flight.erase(g_event_of[e]);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  if (g_fail_syncs > 0) { --g_fail_syncs; return hipErrorUnknown; }
  std::lock_guard<std::mutex> l(g_mu);
  g_in_flight.clear();
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t) {
  launched_into(kind == hipMemcpyHostToDevice ? src : dst);
  std::memcpy(dst, src, n);
  return hipSuccess;
}
const char* m3lb_last_error(void) { return t_msg.c_str(); }
}
namespace m3lb {
int set_error(int code, const char* msg) { t_msg = msg; return code; }
}

namespace {
void macro(const m3lb::ReadArgs& a, hipStream_t) {
  launched_into(a.out2[0]);
  for (int k = 0; k < 4; ++k)
    for (int n = a.n0; n < a.n1; ++n)
      static_cast<float*>(a.out2[k])[n - a.n0] = float(n % 1000) + 0.25f * float(k);
}
void rows(const m3lb::ReadArgs& a, hipStream_t) {
  launched_into(a.out);
  for (int n = a.n0; n < a.n1; ++n)
    for (int q = 0; q < 9; ++q)
      static_cast<double*>(a.out)[size_t(n - a.n0) * 9 + size_t(q)] = n * 10.0 + q;
}
m3lb::KernelSet kernels(int real_bytes) {
  m3lb::KernelSet k;
  std::memset(&k, 0, sizeof k);
  k.macro = macro;
  k.gather = k.storage = rows;
  k.real_bytes = real_bytes;
  return k;
}
int fields(int np, bool check = true) {
  const m3lb::KernelSet ks = kernels(4);
  m3lb::ReadArgs a;
  std::memset(&a, 0, sizeof a);
  a.d.np = np;
  std::vector<double> out[4];
  double* dst[4];
  for (int k = 0; k < 4; ++k) {
    out[k].assign(size_t(np), -1.0);
    dst[k] = out[k].data();
  }
  const int rc = m3lb::read_macroscopic(&ks, a, 0, nullptr, dst);
  if (rc == 0 && check)
    for (int k = 0; k < 4; ++k)
      for (int n = 0; n < np; ++n) REQUIRE(out[k][size_t(n)] == double(n % 1000) + 0.25 * k);
  return rc;
}
int populations(int np) {
  const m3lb::KernelSet ks = kernels(8);
  m3lb::ReadArgs a;
  std::memset(&a, 0, sizeof a);
  a.d.np = np;
  std::vector<double> out(size_t(np) * 9, -1.0);
  const int rc = m3lb::read_populations(&ks, a, 9, true, 0, nullptr, out.data());
  if (rc == 0)
    for (int n = 0; n < np; ++n)
      for (int q = 0; q < 9; ++q) REQUIRE(out[size_t(n) * 9 + size_t(q)] == n * 10.0 + q);
  return rc;
}
int upload(size_t n) {
  std::vector<double> src(n);
  for (size_t k = 0; k < n; ++k) src[k] = double(k) * 0.5;
  std::vector<float> dst(n);
  const int rc = m3lb::upload_real(dst.data(), src.data(), n, 4, 0, nullptr);
  if (rc == 0)
    for (size_t k = 0; k < n; ++k) REQUIRE(dst[k] == float(src[k]));
  return rc;
}
}  // namespace

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  m3lb::staging_acquire();
  if (what == "visible") {
    REQUIRE(fields(100) == M3LB_OK && fields(1500000) == M3LB_OK);
    // the host sees what kernels wrote after the wait: coherent memory, or events
    // that release to the system
    REQUIRE(g_incoherent == 0 || g_device_events == 0);
  } else if (what == "failed_wait") {
    // one wait of several fails: none of the slots is used again before the work
    // in flight has ended
    for (int np : {100, 1500000}) {
      g_fail_records = 1;
      REQUIRE(fields(np) == M3LB_EDEVICE);
      REQUIRE(fields(np) == M3LB_OK && populations(np) == M3LB_OK && upload(size_t(np)) == M3LB_OK);
    }
    REQUIRE(g_reused == 0);
    // the stream cannot be waited for either: the slots are given up, and calls go on
    for (int k = 0; k < 20; ++k) {
      g_fail_records = 1;
      g_fail_syncs = 1;
      REQUIRE(fields(1500000) == M3LB_EDEVICE);
    }
    REQUIRE(fields(1500000) == M3LB_OK);
    REQUIRE(g_reused == 0);
  } else if (what == "threads") {
    std::vector<std::thread> t;
    for (int k = 0; k < 8; ++k)
      t.emplace_back([k] {
        for (int rep = 0; rep < 6; ++rep) {
          REQUIRE(fields(k % 2 ? 900000 : 2000) == M3LB_OK);
          REQUIRE(populations(k % 3 ? 50 : 200000) == M3LB_OK);
          REQUIRE(upload(k % 2 ? 3000000 : 77) == M3LB_OK);
        }
      });
    for (std::thread& x : t) x.join();
    REQUIRE(g_peak <= m3lb::kSlots);
    REQUIRE(g_reused == 0 && g_in_flight.empty());
  } else if (what == "no_memory") {
    g_fail_mallocs = 100;
    REQUIRE(fields(100) == M3LB_ENOMEM && fields(1500000) == M3LB_ENOMEM);
    g_fail_mallocs = 0;
    REQUIRE(fields(1500000) == M3LB_OK);
  } else {
    return 2;
  }
  m3lb::staging_release();
  if (what != "failed_wait") REQUIRE(g_pinned.empty());  // all given back with the last user
  std::printf("ok\n");
  return 0;
}
