// Pieces shared by the kernels that multiply affine group-64 codes: a lane's 16 codes of a tile-group
// as bf16 MFMA operands, and the gated epilogues' activations.
#pragma once

#include "common.h"

namespace dsk {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// a lane's 16 codes of one tile-group, as stored
template <int BITS> struct WeightChunk;
template <> struct WeightChunk<8> { using type = u32x4; };
template <> struct WeightChunk<4> { using type = u32x2; };

// u8 x 16 -> two bf16 x 8 (exact: q <= 255 needs 8 significant bits, the fp32 from
// v_cvt_f32_ubyteN is truncated to its top half).
__device__ __forceinline__ void u8x16_to_bf16(const u32x4 w, bf16x8& lo, bf16x8& hi) {
  uint32_t r[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t v = w[i];
    const float f0 = (float)(v & 0xffu), f1 = (float)((v >> 8) & 0xffu);
    const float f2 = (float)((v >> 16) & 0xffu), f3 = (float)(v >> 24);
    r[2 * i] = __builtin_amdgcn_perm(f32_bits(f1), f32_bits(f0), 0x07060302u);
    r[2 * i + 1] = __builtin_amdgcn_perm(f32_bits(f3), f32_bits(f2), 0x07060302u);
  }
  lo = __builtin_bit_cast(bf16x8, (u32x4{r[0], r[1], r[2], r[3]}));
  hi = __builtin_bit_cast(bf16x8, (u32x4{r[4], r[5], r[6], r[7]}));
}

__device__ __forceinline__ float silu_f(float g) { return g / (1.0f + expf(-g)); }
__device__ __forceinline__ float gelu_tanh_f(float x) {
  const float c = 0.7978845608028654f;  // sqrt(2/pi)
  return 0.5f * x * (1.0f + tanhf(c * (x + 0.044715f * x * x * x)));
}

}  // namespace dsk
