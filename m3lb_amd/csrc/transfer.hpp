// transfer.hpp -- fields between device and caller's arrays.
//
// The caller's arrays are ordinary memory, often not touched yet.  A copy into
// them by the runtime runs at 9 GB/s here (one thread copies out of a staging
// buffer and takes the page faults); PCIe carries 57 GB/s.  So: the readout
// kernels write compute-type values (half the bytes of the FP64 arrays for
// every form but F64) straight into pinned staging slots, a range of nodes at
// a time, and a few threads convert the slots into the caller's arrays while
// later ranges are on their way.  Uploads go the other way.  Fields of a box to the
// caller, before and now: FP32 512^3 (4.3 GB of FP64 arrays) 485 and 46 ms, 256^3
// 60 and 8.6, 128^3 6.9 and 2.0; FP64 64^3 0.77 and 0.47; populations of 64^3 FP64
// 5.7 and 1.6 ms.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "launch.hpp"

namespace m3lb {

// Pinned slots shared by every handle of a device: taken for the length of one
// call, at most kSlots of them (the calls of several threads wait for each
// other beyond that), allocated when first needed and given back when the last
// handle is destroyed.
constexpr size_t kSlotBytes = 4u << 20;
constexpr size_t kSmallSlotBytes = 512u << 10;
constexpr int kSlots = 16;

// One reference per live solver or server.
void staging_acquire();
void staging_release();

// rho, ux, uy, uz of every padded node (entries of dst may be null).  Ordered
// after the work on `st`; returns when the arrays are written.  `a` is a
// filled ReadArgs.
int read_macroscopic(const KernelSet* ks, ReadArgs a, int device, hipStream_t st, double* const dst[4]);

// (node, direction) populations: logical (gather) or the slot image (storage).
int read_populations(const KernelSet* ks, ReadArgs a, int q, bool logical, int device,
                     hipStream_t st, double* dst);

// n caller doubles to `dst` on the device as the compute type (real_bytes 4 or 8).
int upload_real(void* dst, const double* src, size_t n, int real_bytes, int device, hipStream_t st);

// n bytes as they are.
int upload_bytes(void* dst, const void* src, size_t n, int device, hipStream_t st);

// Device partials (grid rows of `cols` doubles) summed in row order.
int read_column_sums(const double* partial_d, unsigned grid, int cols, int device, hipStream_t st,
                     double* out);

}  // namespace m3lb
