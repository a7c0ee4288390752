// transfer.hip -- staged transfers of transfer.hpp.
#include "transfer.hpp"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <string>
#include <system_error>
#include <thread>
#include <vector>

#include <sched.h>

namespace m3lb {
namespace {

int err(int code, const std::string& m) { return set_error(code, m.c_str()); }

struct Slot {
  int device = -1;
  size_t bytes = 0;
  void* host = nullptr;  // pinned, written and read by the device in place
  hipEvent_t done = nullptr;
};

class Pool {
 public:
  void acquire_user() {
    std::lock_guard<std::mutex> l(mu_);
    ++users_;
  }
  void release_user() {
    std::lock_guard<std::mutex> l(mu_);
    if (--users_ > 0) return;
    // no handle is left, so no call is in progress and every slot is free
    for (Slot& s : free_) drop(s);
    free_.clear();
    total_ = 0;
  }
  // Up to `want` slots of `device` and at least `bytes`; at least one, waiting
  // while other calls hold them all.  Empty with *rc set when not even one can be
  // had.
  std::vector<Slot> take(int device, int want, size_t bytes, int* rc) {
    std::unique_lock<std::mutex> l(mu_);
    std::vector<Slot> got;
    *rc = M3LB_OK;
    for (;;) {
      for (size_t k = 0; k < free_.size() && int(got.size()) < want;) {
        if (free_[k].device == device && free_[k].bytes >= bytes) {
          got.push_back(free_[k]);
          free_.erase(free_.begin() + std::ptrdiff_t(k));
        } else {
          ++k;
        }
      }
      while (int(got.size()) < want && total_ < kSlots) {
        Slot s;
        if (!make(device, bytes, s)) break;
        ++total_;
        got.push_back(s);
      }
      if (!got.empty()) return got;
      if (!free_.empty()) {  // all free ones are too small or another device's
        drop(free_.back());
        free_.pop_back();
        --total_;
        continue;
      }
      if (total_ == 0) {
        *rc = M3LB_ENOMEM;
        return got;
      }
      cv_.wait(l);
    }
  }
  void give(const std::vector<Slot>& slots) {
    {
      std::lock_guard<std::mutex> l(mu_);
      for (const Slot& s : slots) free_.push_back(s);
    }
    cv_.notify_all();
  }
  // Slots that the device may still write, for good: not used again and not freed.
  void forget(size_t n) {
    {
      std::lock_guard<std::mutex> l(mu_);
      total_ -= int(n);
    }
    cv_.notify_all();
  }

 private:
  static bool make(int device, size_t bytes, Slot& s) {
    int cur = device;
    (void)hipGetDevice(&cur);
    if (cur != device && hipSetDevice(device) != hipSuccess) return false;
    s.device = device;
    s.bytes = bytes;
    // The host reads a slot after a wait for this event alone, which need not
    // release to the system: so the memory is coherent by itself, whatever the
    // process's default is.  (An event that releases costs 1 us a readout.)
    bool ok = hipHostMalloc(&s.host, bytes, hipHostMallocCoherent) == hipSuccess;
    ok = ok && hipEventCreateWithFlags(&s.done, hipEventDisableTiming) == hipSuccess;
    if (!ok) {
      (void)hipGetLastError();
      drop(s);
    }
    if (cur != device) (void)hipSetDevice(cur);
    return ok;
  }
  static void drop(Slot& s) {
    if (s.done) (void)hipEventDestroy(s.done);
    if (s.host) (void)hipHostFree(s.host);
    s.done = nullptr;
    s.host = nullptr;
  }
  std::mutex mu_;
  std::condition_variable cv_;
  std::vector<Slot> free_;
  int total_ = 0, users_ = 0;
};

Pool& pool() {
  static Pool* p = new Pool;  // never destroyed: handles may outlive static destructors
  return *p;
}

int cpus() {
  cpu_set_t set;
  CPU_ZERO(&set);
  if (sched_getaffinity(0, sizeof set, &set) == 0) return std::max(1, CPU_COUNT(&set));
  return 1;
}

// Runs fn(chunk, slot) for every chunk, each thread with a slot of its own;
// the caller is one of the threads.  fn returns an M3LB code; the first
// failure stops the rest.  After a failure work that fn queued on `st` may still
// read or write a slot, so the slots go back only once the stream has been waited
// for.  `bytes` is what one chunk takes: pinning a whole slot
// is 0.1 ms, which a program of small boxes would notice, so a call that
// needs less than a small slot asks for no more.
template <class Fn>
int each_chunk(size_t chunks, size_t bytes, int device, hipStream_t st, Fn&& fn) {
  if (chunks == 0) return M3LB_OK;
  static const int most = std::max(1, std::min(kSlots - 4, cpus() - 2));
  int rc = M3LB_OK;
  std::vector<Slot> slots = pool().take(device, int(std::min<size_t>(chunks, size_t(most))),
                                       bytes <= kSmallSlotBytes ? kSmallSlotBytes : kSlotBytes, &rc);
  if (rc) return err(rc, "pinned staging memory");
  std::atomic<size_t> next{0};
  std::atomic<int> first_rc{M3LB_OK};
  std::mutex msg_mu;
  std::string msg;
  auto body = [&](const Slot& s, bool own_thread) {
    if (own_thread && hipSetDevice(device) != hipSuccess) {
      first_rc = M3LB_EDEVICE;
      return;
    }
    for (;;) {
      const size_t c = next.fetch_add(1);
      if (c >= chunks || first_rc.load() != M3LB_OK) return;
      const int r = fn(c, s);
      if (r) {
        int ok = M3LB_OK;
        if (first_rc.compare_exchange_strong(ok, r)) {
          std::lock_guard<std::mutex> l(msg_mu);
          msg = m3lb_last_error();  // this thread's message, for the caller's thread
        }
        return;
      }
    }
  };
  std::vector<std::thread> threads;
  threads.reserve(slots.size());
  for (size_t t = 1; t < slots.size(); ++t) {
    try {
      threads.emplace_back(body, std::cref(slots[t]), true);
    } catch (const std::system_error&) {
      break;  // fewer threads do the same work
    }
  }
  body(slots[0], false);
  for (std::thread& t : threads) t.join();
  if (first_rc.load() == M3LB_OK || hipStreamSynchronize(st) == hipSuccess) pool().give(slots);
  else pool().forget(slots.size());
  if (first_rc.load()) return err(first_rc.load(), msg.empty() ? "staged transfer failed" : msg);
  return M3LB_OK;
}

int wait_for(const Slot& s, hipStream_t st) {
  hipError_t e = hipEventRecord(s.done, st);
  if (e == hipSuccess) e = hipEventSynchronize(s.done);
  if (e != hipSuccess) return err(M3LB_EDEVICE, std::string("readout: ") + hipGetErrorString(e));
  return M3LB_OK;
}

int launched() {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return err(M3LB_EDEVICE, std::string("kernel launch: ") + hipGetErrorString(e));
  return M3LB_OK;
}

void widen(double* dst, const void* src, size_t n, int real_bytes) {
  if (real_bytes == 8) {
    std::memcpy(dst, src, n * sizeof(double));
  } else {
    const float* f = static_cast<const float*>(src);
    for (size_t k = 0; k < n; ++k) dst[k] = double(f[k]);
  }
}

}  // namespace

void staging_acquire() { pool().acquire_user(); }
void staging_release() { pool().release_user(); }

int read_macroscopic(const KernelSet* ks, ReadArgs a, int device, hipStream_t st,
                     double* const dst[4]) {
  const size_t np = size_t(a.d.np), rb = size_t(ks->real_bytes);
  // whole multiples of 64 nodes, so that every plane of a slot starts aligned
  const size_t per = std::min(kSlotBytes / (4 * rb) / 64 * 64, (np + 63) / 64 * 64);
  return each_chunk((np + per - 1) / per, per * 4 * rb, device, st, [&](size_t c, const Slot& s) -> int {
    ReadArgs r = a;
    r.n0 = int(c * per);
    r.n1 = int(std::min(np, (c + 1) * per));
    const size_t n = size_t(r.n1 - r.n0);
    char* h = static_cast<char*>(s.host);
    for (size_t k = 0; k < 4; ++k) r.out2[k] = dst[k] ? h + k * per * rb : nullptr;
    ks->macro(r, st);
    int rc = launched();
    if (!rc) rc = wait_for(s, st);
    if (rc) return rc;
    for (size_t k = 0; k < 4; ++k)
      if (dst[k]) widen(dst[k] + r.n0, h + k * per * rb, n, int(rb));
    return M3LB_OK;
  });
}

int read_populations(const KernelSet* ks, ReadArgs a, int q, bool logical, int device,
                     hipStream_t st, double* dst) {
  const size_t np = size_t(a.d.np), rb = size_t(ks->real_bytes), row = size_t(q);
  const size_t per = kSlotBytes / (row * rb) / kBlock * kBlock;
  return each_chunk((np + per - 1) / per, std::min(np, per) * row * rb, device, st, [&](size_t c, const Slot& s) -> int {
    ReadArgs r = a;
    r.n0 = int(c * per);
    r.n1 = int(std::min(np, (c + 1) * per));
    r.out = s.host;
    if (logical) ks->gather(r, st);
    else ks->storage(r, st);
    int rc = launched();
    if (!rc) rc = wait_for(s, st);
    if (rc) return rc;
    widen(dst + size_t(r.n0) * row, s.host, size_t(r.n1 - r.n0) * row, int(rb));
    return M3LB_OK;
  });
}

int upload_real(void* dst, const double* src, size_t n, int real_bytes, int device, hipStream_t st) {
  const size_t rb = size_t(real_bytes), per = kSlotBytes / rb;
  return each_chunk((n + per - 1) / per, std::min(n, per) * rb, device, st, [&](size_t c, const Slot& s) -> int {
    const size_t k0 = c * per, k1 = std::min(n, k0 + per);
    if (real_bytes == 8) {
      std::memcpy(s.host, src + k0, (k1 - k0) * rb);
    } else {
      float* f = static_cast<float*>(s.host);
      for (size_t k = k0; k < k1; ++k) f[k - k0] = float(src[k]);
    }
    if (hipMemcpyAsync(static_cast<char*>(dst) + k0 * rb, s.host, (k1 - k0) * rb,
                       hipMemcpyHostToDevice, st) != hipSuccess)
      return err(M3LB_EDEVICE, "upload failed");
    return wait_for(s, st);
  });
}

int upload_bytes(void* dst, const void* src, size_t n, int device, hipStream_t st) {
  return each_chunk((n + kSlotBytes - 1) / kSlotBytes, std::min(n, kSlotBytes), device, st, [&](size_t c, const Slot& s) -> int {
    const size_t k0 = c * kSlotBytes, m = std::min(n - k0, kSlotBytes);
    std::memcpy(s.host, static_cast<const char*>(src) + k0, m);
    if (hipMemcpyAsync(static_cast<char*>(dst) + k0, s.host, m, hipMemcpyHostToDevice, st) !=
        hipSuccess)
      return err(M3LB_EDEVICE, "upload failed");
    return wait_for(s, st);
  });
}

int read_column_sums(const double* partial_d, unsigned grid, int cols, int device, hipStream_t st,
                     double* out) {
  const size_t bytes = size_t(grid) * size_t(cols) * sizeof(double);
  if (bytes > kSlotBytes) return err(M3LB_EINVAL, "too many reduction partials");
  return each_chunk(1, bytes, device, st, [&](size_t, const Slot& s) -> int {
    if (hipMemcpyAsync(s.host, partial_d, bytes, hipMemcpyDeviceToHost, st) != hipSuccess)
      return err(M3LB_EDEVICE, "partials download failed");
    const int rc = wait_for(s, st);
    if (rc) return rc;
    const double* h = static_cast<const double*>(s.host);
    for (int k = 0; k < cols; ++k) out[k] = 0;
    for (unsigned b = 0; b < grid; ++b)
      for (int k = 0; k < cols; ++k) out[k] += h[size_t(b) * size_t(cols) + size_t(k)];
    return M3LB_OK;
  });
}

}  // namespace m3lb
