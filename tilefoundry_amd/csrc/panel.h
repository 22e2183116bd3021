// Panel order: the activations of a prompt pass.  The rows are cut into panels
// of 32, each panel in the skinny GEMMs' operand order over its K values (32 x K
// bf16, 1 KiB blocks of 16 rows x 32 k): panel p starts at p * 32 * K.
#pragma once

#include "decode_common.h"

namespace tfd {

__device__ __forceinline__ int64_t panel_off(int64_t m, int k, int K) {
  const int r = (int)(m & 31);
  return (m >> 5) * 32 * K +
         ((int64_t)((k >> 5) * 2 + (r >> 4)) * 64 + (r & 15) + 16 * ((k >> 3) & 3)) * 8 + (k & 7);
}

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr float kPanelNegInf = -__builtin_huge_valf();

// D[i][j] += sum_k A[i][k] B[j][k]: lane l holds A[l % 16] and B[l % 16] at k = 8 (l / 16)
// .. +7 and gets D[4 (l / 16) .. +3][l % 16].
__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// Eight e4m3fn codes as bf16 values (gfx950's scaled conversion at scale 1.0 is exact).
__device__ __forceinline__ u32x4 fp8x8_to_bf16(u32x2 r) {
  const bf16x2_t a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(r.x, 1.0f, false);
  const bf16x2_t b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(r.x, 1.0f, true);
  const bf16x2_t c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(r.y, 1.0f, false);
  const bf16x2_t d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(r.y, 1.0f, true);
  return u32x4{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
               __builtin_bit_cast(uint32_t, c), __builtin_bit_cast(uint32_t, d)};
}

// The sum of a value's K slices, in slice order, rounded once.
__device__ __forceinline__ float slice_sum(const float* p, int64_t stride, int slices) {
  float a = p[0];
  for (int s = 1; s < slices; ++s) a += p[s * stride];
  return rbf(a);
}
// The same for four neighbours, not rounded (slices 0: zeros).
__device__ __forceinline__ f32x4 slice_sum4(const float* p, int64_t stride, int slices) {
  f32x4 a = {0.f, 0.f, 0.f, 0.f};
  if (slices > 0) a = *reinterpret_cast<const f32x4*>(p);
  for (int s = 1; s < slices; ++s) a += *reinterpret_cast<const f32x4*>(p + s * stride);
  return a;
}

}  // namespace tfd
