// device_ptr.h -- address spaces and scalar registers for pointers read from descriptors.
#pragma once

#include "common.h"

namespace rts {

// Device memory reached through pointers that a kernel reads from its descriptors (columns,
// filter vectors, list entries and directories, result bitmaps) is global memory.  Saying so turns
// the generic (flat) accesses the compiler would emit for such pointers into global ones:
// flat accesses also count against the LDS wait counter, so every LDS wait in the kernel
// would wait for outstanding loads and result stores as well.
#define RTS_GLOBAL __attribute__((address_space(1)))
template <class T>
__device__ __forceinline__ const RTS_GLOBAL T *gmem(const T *p) {
  return (const RTS_GLOBAL T *)p;
}
template <class T>
__device__ __forceinline__ RTS_GLOBAL T *gmem(T *p) {
  return (RTS_GLOBAL T *)p;
}
// Memory that no kernel writes while a batch runs (the lists' tile directories), read
// through the constant address space: a wave-uniform address then becomes a scalar load,
// whose wait does not also wait for the wave's outstanding result stores.
#define RTS_CONST __attribute__((address_space(4)))
template <class T>
__device__ __forceinline__ const RTS_CONST T *cmem(const T *p) {
  return (const RTS_CONST T *)p;
}

// A value that is the same in every lane, moved to a scalar register (the builtin takes and
// returns 32-bit values: a pointer goes one half at a time).
__device__ __forceinline__ uint32_t uniform_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}
__device__ __forceinline__ uint64_t uniform_u64(uint64_t v) {
  return ((uint64_t)uniform_u32((uint32_t)(v >> 32)) << 32) | uniform_u32((uint32_t)v);
}
template <class T>
__device__ __forceinline__ T *uniform_ptr(T *p) {
  const uint64_t a = (uint64_t)p;
  return (T *)(((uint64_t)uniform_u32((uint32_t)(a >> 32)) << 32) | uniform_u32((uint32_t)a));
}

}  // namespace rts
