// A real number as two bfloat16 (hi = bf16(x), lo = bf16(x - hi)), and complex numbers
// packed for the bf16 MFMA (k_zgemm_bf3 says how).
#pragma once
#include <hip/hip_runtime.h>

namespace ccgpu {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void bf3_split(float x, float y, unsigned &hi, unsigned &lo) {
  const __bf16 xh = (__bf16)x, yh = (__bf16)y;
  const __bf16 xl = (__bf16)(x - (float)xh), yl = (__bf16)(y - (float)yh);
  hi = __builtin_bit_cast(unsigned, (bf16x2){xh, yh});
  lo = __builtin_bit_cast(unsigned, (bf16x2){xl, yl});
}
// (br, -bi) -> (bi, br): swap the halves, then flip the sign of the new low half
__device__ __forceinline__ u32x4 bf3_im_pairs(u32x4 v) {
  u32x4 r;
#pragma unroll
  for (int q = 0; q < 4; ++q) r[q] = ((v[q] >> 16) | (v[q] << 16)) ^ 0x8000u;
  return r;
}

}  // namespace ccgpu
