// Exact sums of FP32 products in 64-bit fixed point, for LDS integer atomics.
#pragma once

#include "common.hpp"

namespace spmspv {

// Fixed-point row sums. A product v = m * 2^(ef - 150), with m its 24-bit
// significand and ef = max(exponent field, 1), enters row r's sum as the
// integer q = m * 2^(ef - E + 22) (rounded to nearest when the shift is to
// the right), where E is the largest ef among the products of r that
// are summed together: |q| < 2^46, so at most 2^14 of them sum exactly in 64
// bits, in any order, and the row's value is the sum times 2^(E - 172), rounded
// to FP64 and from there to FP32. Each product's error is at most 2^-46 of the row's
// largest |product|. Integer LDS atomics (max for E, add for the sum) run
// about 15 times faster on gfx950 than FP32 LDS atomic adds.
__device__ __forceinline__ unsigned prod_ef(float v) {
  const unsigned e = (__float_as_uint(v) >> 23) & 0xFFu;
  return e ? e : 1u;
}

__device__ __forceinline__ long long prod_fixed(float v, unsigned E) {
  const unsigned b = __float_as_uint(v);
  const unsigned ef = (b >> 23) & 0xFFu;
  const unsigned long long m = (b & 0x7FFFFFu) | (ef ? 0x800000u : 0u);
  const int d = (int)E - (int)(ef ? ef : 1u);
  unsigned long long q;
  if (d <= 22) q = m << (22 - d);
  else if (d - 22 <= 24) q = (m + (1ull << (d - 23))) >> (d - 22);
  else q = 0;
  return (b >> 31) ? -(long long)q : (long long)q;
}

__device__ __forceinline__ float fixed_value(long long sum, unsigned E) {
  return (float)ldexp((double)sum, (int)E - 172);
}

// A sum with an Inf or NaN among its terms, in any order: the kinds of its
// terms (1: +Inf, 2: -Inf, 4: NaN, 0: finite) ORed, and its value from them.
__device__ __forceinline__ unsigned special_kind(float v) {
  const unsigned b = __float_as_uint(v);
  if ((b & 0x7F800000u) != 0x7F800000u) return 0u;
  return (b & 0x7FFFFFu) ? 4u : 1u << (b >> 31);
}

__device__ __forceinline__ float special_value(unsigned kinds) {
  return __uint_as_float(kinds == 1u ? 0x7F800000u : kinds == 2u ? 0xFF800000u : 0x7FC00000u);
}

}  // namespace spmspv
