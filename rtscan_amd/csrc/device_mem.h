// device_mem.h -- device memory of the library (device_pool.cpp).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace rts {

// Device memory of index arrays and of call workspaces (device_pool.cpp): blocks on the
// current device, kept for later calls when freed.  pool_free: `idle` says that no queued
// work uses the block any more (the caller has waited for it); otherwise it goes back to the
// device, which waits.  pool_trim gives every kept block of a device back, pool_kept is their
// bytes.
hipError_t pool_alloc(void **ptr, size_t bytes);
void pool_free(void *ptr, bool idle);
void pool_trim(int dev);
size_t pool_kept(int dev);
template <class T>
inline hipError_t pool_alloc(T **ptr, size_t bytes) {
  return pool_alloc(reinterpret_cast<void **>(ptr), bytes);
}

// Waits for all work of the current device, as a hipFree of the memory would; false where that
// is refused (a capture in progress that forbids hipFree, no memory).  hipDeviceSynchronize will
// not do: it ends the stream captures of all threads, in the relaxed mode too.
bool device_wait();

// hipMalloc, tried again with the pool's kept blocks given back when the device is out of
// memory.
hipError_t device_malloc(void **ptr, size_t bytes);

}  // namespace rts
