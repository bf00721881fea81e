// Device pieces of the block-32 MX quantisation (OCP Microscaling Formats v1.0, E4M3 elements with
// an E8M0 shared scale) used by the attention epilogues and by the standalone kernel. Device code
// only: include from .hip files.
//
//   shared_exp = floor(log2(max |v|)) - 8, clamped to [-127, 127];  scale code = shared_exp + 127
//   code_i     = e4m3(v_i * 2^-shared_exp), round to nearest even, saturating at +-448
//   a block of zeros: scale code 0, zero elements; a block with Inf/NaN: scale 0xff, NaN elements
#pragma once

#include <hip/hip_runtime.h>

namespace mlakv {

struct MxScale {
  unsigned code;  // E8M0
  float inverse;  // 2^-shared_exp, a normal fp32 for every bf16 input
  bool nan;
};

// The input is bf16, so the largest magnitude of a block is the largest 15-bit pattern, and its
// floor(log2) is the exponent field (a subnormal or zero maximum clamps to the smallest scale).
__device__ __forceinline__ MxScale MxScaleFromMaxBits(unsigned max_magnitude_bits) {
  const unsigned exponent = max_magnitude_bits >> 7;
  MxScale s;
  s.nan = exponent == 255u;
  s.code = s.nan ? 0xffu : (exponent > 8u ? exponent - 8u : 0u);
  s.inverse = __builtin_bit_cast(float, (254u - (s.nan ? 127u : s.code)) << 23);
  return s;
}

__device__ __forceinline__ unsigned MxMagnitudeMax(unsigned word, unsigned running) {
  const unsigned lo = word & 0x7fffu, hi = (word >> 16) & 0x7fffu;
  return max(running, max(lo, hi));
}

// Four bf16 values (two dwords, low halves first) -> their four codes.
// v_cvt_pk_fp8_f32 rounds to nearest even onto the E4M3 grid for |v| < 464 and returns NaN beyond,
// so the clamp (one median of three per value) supplies the saturation; a block with a NaN does not
// get there. The second conversion writes the upper half of the first one's destination.
__device__ __forceinline__ unsigned MxEncodeFour(unsigned first, unsigned second, const MxScale& s) {
  if (s.nan) {
    return ((first >> 8) & 0x80u) | ((first >> 16) & 0x8000u) | ((second << 8) & 0x800000u) | (second & 0x80000000u) | 0x7f7f7f7fu;
  }
  const auto scaled = [&](unsigned bits) __attribute__((always_inline)) {
    return __builtin_amdgcn_fmed3f(__builtin_bit_cast(float, bits) * s.inverse, -448.0f, 448.0f);
  };
  const int low = __builtin_amdgcn_cvt_pk_fp8_f32(scaled(first << 16), scaled(first & 0xffff0000u), 0, false);
  return static_cast<unsigned>(__builtin_amdgcn_cvt_pk_fp8_f32(scaled(second << 16), scaled(second & 0xffff0000u), low, true));
}

}  // namespace mlakv
