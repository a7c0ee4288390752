// device_memory.hpp -- device allocations, and arrays that a handle can do without.
//
// A solver whose passes write a second population array (plane.hpp, march.hpp)
// holds it from the first pass on.  It can step without: so an allocation of
// any handle that finds no memory takes such arrays back first, and fails only
// if there is none to take.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace m3lb {

// A handle that may hold a spare array on `device`.  give_back(owner) frees what is
// idle and returns whether it freed anything; it is called from any thread, with no
// other call on the spares in progress, and must not allocate through
// device_alloc.  Registered for the life of the handle.
struct Spare {
  int device;
  void* owner;
  bool (*give_back)(void* owner);
};
void spare_register(const Spare& s);
void spare_unregister(void* owner);

// hipMalloc on `device`, the calling thread's current device unchanged.  Not to be
// called by a thread that holds what a give_back waits for.
hipError_t device_alloc(int device, void** p, size_t bytes);
template <class T>
hipError_t device_alloc(int device, T** p, size_t bytes) {
  return device_alloc(device, reinterpret_cast<void**>(p), bytes);
}

// The same without taking spares back.
hipError_t device_alloc_plain(int device, void** p, size_t bytes);

// Free bytes of `device` by the runtime's count; 0 when it cannot be had.
size_t device_free_bytes(int device);

}  // namespace m3lb
