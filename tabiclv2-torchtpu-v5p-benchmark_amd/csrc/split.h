// Exact splits of fp32 values into three bf16 values, the operands of fp32-accurate products on the bf16
// matrix units. gfx950 multiplies fp32 matrices at 1/16 of its bf16 rate. x = h + m + l (8 significant bits
// each, round to nearest; the residuals are exact in fp32), so a product of fp32 values is nine bf16 products;
// six of them (h h, h m, m h, m m, h l, l h) leave out m l + l m + l l: at most 2^-24 of the product (2^-27 rms, of either
// sign), as much as one rounding of it to fp32. An infinite (or, above 2^128 - 2^119, rounded to infinite)
// x gives NaN in m and l.
#pragma once
#include "common.h"

struct Split8 { bf16x8 h, m, l; };

// Two values: packed pairs h, m, l (11 VALU).
__device__ __forceinline__ void split2(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x0, x1}, bf16x2));
  const float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xffff0000u);
  m = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{r0, r1}, bf16x2));
  const float q0 = r0 - __uint_as_float(m << 16), q1 = r1 - __uint_as_float(m & 0xffff0000u);
  l = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{q0, q1}, bf16x2));
}

__device__ __forceinline__ Split8 split8(f32x4 a, f32x4 b) {
  uint32_t h[4], m[4], l[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    split2(a[2 * i], a[2 * i + 1], h[i], m[i], l[i]);
    split2(b[2 * i], b[2 * i + 1], h[2 + i], m[2 + i], l[2 + i]);
  }
  return {__builtin_bit_cast(bf16x8, uint4{h[0], h[1], h[2], h[3]}), __builtin_bit_cast(bf16x8, uint4{m[0], m[1], m[2], m[3]}),
          __builtin_bit_cast(bf16x8, uint4{l[0], l[1], l[2], l[3]})};
}
