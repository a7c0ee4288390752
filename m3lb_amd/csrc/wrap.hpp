// wrap.hpp -- periodic coordinates, for any axis an int32 node index allows.
// Plain C++ on the host, so that the CPU tests can check it.
#pragma once

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define M3LB_WRAP_HD __host__ __device__ __forceinline__
#else
#define M3LB_WRAP_HD inline
#endif

namespace m3lb {

// Coordinate v of a margin beside an axis of s nodes that wraps.  One period is all
// that is to be added but on axes shorter than the margin; no product with s,
// which would not fit an int.
M3LB_WRAP_HD int wrapped(int v, int s) {
  if (v < 0) v += s;
  else if (v >= s) v -= s;
  if (v < 0 || v >= s) {
    v %= s;
    if (v < 0) v += s;
  }
  return v;
}

}  // namespace m3lb
