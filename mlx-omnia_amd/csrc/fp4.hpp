// The FP4 formats' codes and scales, as every kernel over MXFP4 and NVFP4 stacks reads them.
#pragma once

#include "common.hpp"

namespace omnia {

// The e8m0 group scale as the reference applies it: the fp32 with exponent field `byte`.
__device__ __forceinline__ float e8m0(uint32_t byte) { return __uint_as_float(byte << 23); }

// The e4m3 group scale as mlx decodes it: sign, 4 exponent bits (bias 7), 3 mantissa bits;
// exponent 0 is subnormal (m / 8 * 2^-6) and the all-ones codes are +-480. A normal code's
// 7 magnitude bits shifted to the top of an fp32's exponent and mantissa, with the
// exponent rebased by 127 - 7, give 2^(e - 7) (1 + m / 8) exactly.
__device__ __forceinline__ float e4m3(uint32_t byte) {
  const uint32_t mag = byte & 0x7Fu;
  const float normal = __uint_as_float((mag << 20) + (120u << 23));
  const float subnormal = static_cast<float>(mag) * 0x1p-9f;
  const float v = mag < 8u ? subnormal : normal;
  return __uint_as_float(__float_as_uint(v) | ((byte & 0x80u) << 24));
}

// The e2m1 codes of byte B of a word as a bf16 pair, low nibble first.
template <int B>
__device__ __forceinline__ uint32_t fp4_pair(uint32_t word) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, 1.0f, B));
}

}  // namespace omnia
