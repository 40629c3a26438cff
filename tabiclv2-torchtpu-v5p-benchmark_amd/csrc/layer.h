// Pieces shared by the encoder-layer kernels (layer.hip, icl_layer.hip): products Y^T = W X^T by 32x32 MFMA tiles,
// A = weight rows in the order el_perm, B = activations, so that a result's lane holds one row's features in
// runs of eight.
#pragma once
#include "common.h"

// Tile row m -> feature within the tile's 32: result register r of lane half h is feature
// 16 (r / 8) + 8 h + r % 8.
__device__ __forceinline__ int el_perm(int m) {
  return ((m >> 4) << 4) | (((m >> 2) & 1) << 3) | (((m >> 3) & 1) << 2) | (m & 3);
}

// GELU (erf form): gelu(x) = max(x, 0) - a erfc(a / sqrt 2) / 2, a = |x|: no cancellation on either side.
// fp32: erfc(a / sqrt 2) / 2 = exp(-a^2 / 2) R(a), R a degree-12 polynomial fitted here to erfcx on [0, 6.5]
// under the weight exp(-a^2 / 2). With the coefficients rounded as they stand here the largest error of the product is
// 1.3e-8, of a times it (what gelu subtracts) 2.4e-8, near a = 5.5; past 6.5 a times it is below 5e-9.
// Against float64 on N(0, 1) inputs: rms error 2.0e-8, largest 2.5e-7; 0.5 x (1 + erff(x / sqrt 2)) gives
// 2.4e-8 and 2.8e-7 at twice the instructions (erff runs both of its branches in a mixed wave).
// bf16: erfc(z) = (a1 t + .. + a5 t^5) exp(-z^2), t = 1 / (1 + 0.3275911 z) (Abramowitz & Stegun 7.1.26,
// |error| <= 1.5e-7).
template <typename T> __device__ __forceinline__ float el_gelu(float x) {
  const float t0 = 0.5f * x, relu = t0 + __builtin_fabsf(t0);  // -inf and NaN give NaN, as x (1 + erf) does
  if constexpr (sizeof(T) == 4) {
    const float a = __builtin_fminf(__builtin_fabsf(x), 16.f);
    const float e = __builtin_amdgcn_exp2f(a * a * (-0.5f * TA_LOG2E));
    float q = 5.853344831052709e-08f;
    q = __builtin_fmaf(q, a, -1.6036694887588965e-06f);
    q = __builtin_fmaf(q, a, 1.989309566852171e-05f);
    q = __builtin_fmaf(q, a, -0.0001497915800428018f);
    q = __builtin_fmaf(q, a, 0.0007796756108291447f);
    q = __builtin_fmaf(q, a, -0.0030553529504686594f);
    q = __builtin_fmaf(q, a, 0.009659801609814167f);
    q = __builtin_fmaf(q, a, -0.026069175451993942f);
    q = __builtin_fmaf(q, a, 0.062262386083602905f);
    q = __builtin_fmaf(q, a, -0.1329168975353241f);
    q = __builtin_fmaf(q, a, 0.24999110400676727f);
    q = __builtin_fmaf(q, a, -0.3989417850971222f);
    q = __builtin_fmaf(q, a, 0.5f);
    return __builtin_fmaf(-a, e * q, relu);
  } else {
    const float a = __builtin_fminf(__builtin_fabsf(x), 1e18f), z = a * 0.70710678118654752440f;
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.3275911f, z, 1.0f));
    float q = __builtin_fmaf(1.061405429f, t, -1.453152027f);
    q = __builtin_fmaf(q, t, 1.421413741f);
    q = __builtin_fmaf(q, t, -0.284496736f);
    q = __builtin_fmaf(q, t, 0.254829592f);
    return __builtin_fmaf(-0.5f * a, __builtin_amdgcn_exp2f(z * z * -TA_LOG2E) * (q * t), relu);
  }
}

// v(o) + .. + v(o + N - 1) in pairs: exact for equal values, so that a constant row's LayerNorm is its bias. (Summed one
// after the other, 128 values of 12345.678 have a mean 1e-3 off, which 1 / sqrt(0 + eps) makes a normalised 0.3.)
template <int N, typename V> __device__ __forceinline__ float el_sum(V v, int o) {
  if constexpr (N == 1) return v(o);
  else return el_sum<N / 2>(v, o) + el_sum<N / 2>(v, o + N / 2);
}

__device__ __forceinline__ bf16x8 el_pack8(f32x4 a, f32x4 b) {
  const uint2 lo = __builtin_bit_cast(uint2, cvt_bf16x4(a)), hi = __builtin_bit_cast(uint2, cvt_bf16x4(b));
  return __builtin_bit_cast(bf16x8, uint4{lo.x, lo.y, hi.x, hi.y});
}
