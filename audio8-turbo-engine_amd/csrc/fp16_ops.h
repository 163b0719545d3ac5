// fp16 arithmetic shared by the vocoder's convolution kernels (conv.hip, conv_tile.hip).
#pragma once
#include "a8_common.h"

namespace a8 {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x4 mfma16x16x32_f16(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                 0);
}
// fp16 word <-> fp32 (exact), two fp32 -> one dword of two fp16 (round to nearest even)
__device__ __forceinline__ float h_lo(uint32_t w) { return (float)__builtin_bit_cast(f16x2, w)[0]; }
__device__ __forceinline__ float h_hi(uint32_t w) { return (float)__builtin_bit_cast(f16x2, w)[1]; }
__device__ __forceinline__ uint32_t pack_f16x2(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, f16x2{(_Float16)lo, (_Float16)hi});
}
// sin(x) on the hardware sine (v_sin_f32 takes revolutions): x / 2 pi reduced to [-1/2, 1/2] by its nearest
// integer, so the unit sees its most accurate range; absolute error ~1e-6 for the snake's |a x| < 100, far
// below the fp16 rounding of the result
__device__ __forceinline__ float sin_hw(float x) {
  float r = x * 0.15915494309189535f;
  r -= __builtin_rintf(r);
  return __builtin_amdgcn_sinf(r);
}
__device__ __forceinline__ u32x2 ld8(const void *p) { return *reinterpret_cast<const u32x2 *>(p); }
// the snake x + ib sin(a x)^2 on 2, 4 and 8 channels (fp32, one rounding to fp16). No contraction: left free, the compiler
// fuses the last add and the fp16 conversion into one v_fma_mix at some call sites and not at others (one
// rounding against two), and the same row would get different bits in snake_cat, the conv loads and the state.
__device__ __forceinline__ uint32_t snake2(uint32_t v, float a0, float ib0, float a1, float ib1) {
#pragma clang fp contract(off)
  const float x0 = h_lo(v), x1 = h_hi(v);
  const float s0 = sin_hw(x0 * a0), s1 = sin_hw(x1 * a1);
  return pack_f16x2(x0 + ib0 * s0 * s0, x1 + ib1 * s1 * s1);
}
__device__ __forceinline__ u32x2 snake4(u32x2 v, const float *a, const float *ib) {
  return u32x2{snake2(v[0], a[0], ib[0], a[1], ib[1]), snake2(v[1], a[2], ib[2], a[3], ib[3])};
}
__device__ __forceinline__ u32x4 snake8(u32x4 v, const float *a, const float *ib) {
  u32x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = snake2(v[j], a[2 * j], ib[2 * j], a[2 * j + 1], ib[2 * j + 1]);
  return o;
}

// D = A(32x16) * B(16x32) + C, fp16 in, fp32 accumulate. Lane l supplies A[l%32][8*(l/32)+j] and B[8*(l/32)+j][l%32]
// (j = 0..7) and receives D[8*(r/4) + 4*(l/32) + r%4][l%32] (r = 0..15).
__device__ __forceinline__ f32x16 mfma32x32x16_f16(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                 0);
}

}  // namespace a8
