// transpose.h -- 32 x 32 bit transpose in one lane's registers.
#pragma once

#include "common.h"

namespace rts {

// out[p] bit 31 - r = in[r] bit p, in place (word 31 - p holds predicate p afterwards).
__device__ __forceinline__ void transpose32(uint32_t (&a)[32]) {
#pragma unroll
  for (int k = 0; k < 16; k++) {
    const uint32_t x = a[k], y = a[k + 16];
    a[k] = __builtin_amdgcn_perm(x, y, 0x07060302);       // the upper halves
    a[k + 16] = __builtin_amdgcn_perm(x, y, 0x05040100);  // the lower halves
  }
#pragma unroll
  for (int b = 0; b < 32; b += 16)
#pragma unroll
    for (int k = b; k < b + 8; k++) {
      const uint32_t x = a[k], y = a[k + 8];
      a[k] = __builtin_amdgcn_perm(x, y, 0x07030501);      // bytes 3 and 1 of each
      a[k + 8] = __builtin_amdgcn_perm(x, y, 0x06020400);  // bytes 2 and 0 of each
    }
#pragma unroll
  for (int j = 4, s = 0; s < 3; j >>= 1, s++) {
    const uint32_t m = j == 4 ? 0x0F0F0F0Fu : j == 2 ? 0x33333333u : 0x55555555u;
#pragma unroll
    for (int k = 0; k < 32; k++) {
      if (k & j) continue;
      const uint32_t x = a[k], y = a[k + j];
      a[k] = (x & ~m) | ((y >> j) & m);
      a[k + j] = ((x << j) & ~m) | (y & m);
    }
  }
}

}  // namespace rts
