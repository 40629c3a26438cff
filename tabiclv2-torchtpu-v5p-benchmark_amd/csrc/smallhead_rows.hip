// bf16 small-head attention (8 heads x 16 dims) with RoPE or a key mask over keys that fit in LDS: the row stage's
// self-attention beyond 128 tokens (tables of more than 124 features), partial-rotary forms at any length, and masks
// that are not prefix masks.
//
// Workgroup = HPW heads of one batch element and a run of 16-query blocks, 8 waves; the waves of a head share its
// operands and take query blocks in turn. Per 32 keys and head LDS holds 2 KB: K (four dims of key 16 g + lane % 16, 8
// bytes a lane) and V^T (this lane's dim of the eight keys whose probabilities it holds, 16 bytes). K is rotated and
// rounded once per workgroup, in the fill. Per 32 keys and block: 2 + 1 + 1 products (scores of q' = bf16(rope(q) scale),
// O^T += V^T P^T, row sums by a ones operand), 8 fp32 fmas (s log2e - m), 8 exponentials, 4 packed converts: bound by
// the exponentials. m is the maximum of the first 64 keys (of the first 64 with a live key); a row sum outside [2^-64, 2^64] or a non-finite O sends the
// block through the exact online softmax.
//
// Precision: the scores are smallhead_fwd_kernel's, the weights bf16 as there, with the largest of the first 64 keys
// exactly 1; the row sum is that of the bf16 weights that multiply V, so that their roundings cancel in part. Relative
// error against float64 (N(0, 1) inputs, RoPE), smallhead_fwd_kernel / here, 1e-3: 129 tokens 3.438 / 3.417, 260 3.614
// / 3.598, 768 3.771 / 3.763, 28 (partial rotary) 2.538 / 2.519; 260 tokens with queries 4 times larger 6.159 / 6.085.
// (Without a reference, no weight exact, 3.483 at 129 tokens; unrounded row sums, 3.438.)
//
// Against smallhead_fwd_kernel (all heads per wave, online maximum, a key tile at a time), self-attention with RoPE, us:
// 5000 x 129 tokens 1340 -> 422, 4000 x 180 1130 -> 398, 3000 x 237 1190 -> 441 (with a mask of padded tokens 456), 2500 x
// 260 1420 -> 442, 300 x 768 905 -> 272; a mask term on every key, 3000 x 237 817 -> 407. (With a branch on the mask
// inside the loop, which cuts its body into blocks, 497 at 260 tokens; with the masked pairs in a loop of their own, 442.)
#include "common.h"
#include "launch.h"

namespace {

constexpr int SW_H = 8, SW_D = 16, SW_E = 128;
constexpr int SW_PAIR = 2048;  // LDS bytes of 32 keys of a head: K of both 16-key groups, V^T
constexpr float SW_BIAS_FLOOR = -1e37f, SW_SHUT = -1e29f;  // a mask term; from here down the key is shut out
constexpr float SW_L_LO = 0x1p-64f, SW_L_HI = 0x1p64f;
typedef uint32_t u32v2 __attribute__((ext_vector_type(2)));

struct SwParams {
  const bf16 *q, *k, *v;
  bf16* o;
  int64_t q_sb, q_sr, k_sb, k_sr, v_sb, v_sr;  // element strides
  const float* bias;
  int64_t bias_sb;
  const int32_t *valid, *skip;
  int valid_n, skip_n;
  const float *cq, *sq, *ck, *sk;
  int rope, half, rot, tab_sr;
  float scale;
  int B, Lq, Lk, nqb, qbpw, nwg_b;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t sw_rsrc(const bf16* base, int rows, int64_t sr) {
  return __builtin_amdgcn_make_buffer_rsrc((bf16*)base, 0, (rows - 1) * (int)sr * 2 + SW_D * 2, TA_BUF_WORD3);
}
__device__ __forceinline__ u32v2 sw_ld4(__amdgpu_buffer_rsrc_t rs, int off) {
  return __builtin_bit_cast(u32v2, __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0));
}
__device__ __forceinline__ f32x4 sw_f32(u32v2 u) {
  return f32x4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
               __uint_as_float(u.y & 0xffff0000u)};
}
__device__ __forceinline__ u32v2 sw_bf16(f32x4 x) { return __builtin_bit_cast(u32v2, cvt_bf16x4(x)); }

// Four dims d0 .. + 3 of a head row, with RoPE the four at d0 ^ 8 and the position's cos and sin.
struct SwRow { u32v2 y, pt; f32x4 c, s; };
template <bool ROPE>
__device__ __forceinline__ SwRow sw_row(const SwParams& p, __amdgpu_buffer_rsrc_t rs, int off, int d0, const float* c,
                                        const float* s, int64_t tab) {
  SwRow r = {};
  r.y = sw_ld4(rs, off + d0 * 2);
  if constexpr (ROPE) {
    r.pt = sw_ld4(rs, off + (d0 ^ 8) * 2);
    r.c = *(const f32x4*)(c + tab);
    r.s = *(const f32x4*)(s + tab);
  }
  return r;
}
template <bool ROPE>
__device__ __forceinline__ f32x4 sw_rope(const SwParams& p, const SwRow& r, __amdgpu_buffer_rsrc_t rs, int off, int d0) {
  const f32x4 y = sw_f32(r.y);
  if constexpr (!ROPE) return y;
  f32x4 out;
  if (p.rope == 2 && p.half == 8) {
    const f32x4 pt = sw_f32(r.pt);
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = __builtin_fmaf(y[i], r.c[i], (d0 & 8 ? pt[i] : -pt[i]) * r.s[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int pt;
      float sg;
      rope_partner(d0 + i, p.rope, p.half, p.rot, &pt, &sg);
      const float xp = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rs, off + pt * 2, 0, 0) << 16);
      out[i] = __builtin_fmaf(y[i], r.c[i], sg * xp * r.s[i]);
    }
  }
  return out;
}

__device__ __forceinline__ float sw_max(f32x4 a, f32x4 b) {
  return fmaxf(fmaxf(fmaxf(a[0], a[1]), fmaxf(a[2], a[3])), fmaxf(fmaxf(b[0], b[1]), fmaxf(b[2], b[3])));
}

template <bool ROPE, int HPW> __global__ __launch_bounds__(512, 4) void sw_rows_kernel(SwParams p) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr int WPH = 8 / HPW;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, kap = lane >> 4;
  const int hd = wave / WPH, wv = wave % WPH;
  const int work = xcd_remap(blockIdx.x, gridDim.x);
  const int head = (work % (SW_H / HPW)) * HPW + hd, rest = work / (SW_H / HPW);
  const int b = rest / p.nwg_b, qb0 = (rest % p.nwg_b) * p.qbpw;
  if (p.skip && p.skip[p.skip_n == 1 ? 0 : b]) return;
  const int nb = p.nqb - qb0 < p.qbpw ? p.nqb - qb0 : p.qbpw;
  int lk = p.Lk;
  if (p.valid) {
    const int vl = p.valid[p.valid_n == 1 ? 0 : b];
    lk = vl < 0 ? 0 : (vl < lk ? vl : lk);
  }
  const int np = (lk + 31) >> 5, npmax = (p.Lk + 31) >> 5;  // 32-key pairs of groups
  const int d0 = 4 * kap, hc = head * SW_D, tc = (hc & (p.tab_sr - 1)) + d0;
  const int lr = lk > 0 ? lk : 1;  // rows from lk on read as zero
  const __amdgpu_buffer_rsrc_t krs = sw_rsrc(p.k + b * p.k_sb + hc, lr, p.k_sr);
  const __amdgpu_buffer_rsrc_t vrs = sw_rsrc(p.v + b * p.v_sb + hc, lr, p.v_sr);
  const int q0 = qb0 * 16, qrows = p.Lq - q0 < nb * 16 ? p.Lq - q0 : nb * 16;
  const __amdgpu_buffer_rsrc_t qrs = sw_rsrc(p.q + b * p.q_sb + (int64_t)q0 * p.q_sr + hc, qrows, p.q_sr);
  const int ksr = (int)p.k_sr * 2, vsr = (int)p.v_sr * 2, qsr = (int)p.q_sr * 2;
  char* mine = lds + hd * npmax * SW_PAIR;
  float* lb2 = (float*)(lds + HPW * npmax * SW_PAIR);
  auto qrow = [&](int blk) {
    const int qi = q0 + blk * 16 + l16;
    return sw_row<ROPE>(p, qrs, (blk * 16 + l16) * qsr, d0, p.cq, p.sq, (int64_t)(qi < p.Lq ? qi : p.Lq - 1) * p.tab_sr + tc);
  };
  SwRow qr = qrow(wv);
  for (int j = threadIdx.x; j < npmax * 32; j += 512) {
    float b2 = j < lk ? 0.f : TA_NEG_INF;
    if (p.bias && j < lk) b2 = fmaxf(p.bias[b * p.bias_sb + j] * TA_LOG2E, SW_BIAS_FLOOR);
    lb2[j] = b2;
  }
  // fill: this wave's 16-key groups (the pair's half g & 1), the next one's loads in flight
  auto krow = [&](int g) {
    const int key = 16 * g + l16;
    return sw_row<ROPE>(p, krs, key * ksr, d0, p.ck, p.sk, (int64_t)(key < p.Lk ? key : p.Lk - 1) * p.tab_sr + tc);
  };
  auto vrow = [&](int g) {
    uint32_t u[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      u[j] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(vrs, (16 * g + 4 * kap + j) * vsr + l16 * 2, 0, 0);
    return u32v2{u[0] | u[1] << 16, u[2] | u[3] << 16};
  };
  {
    SwRow kr = krow(wv);
    u32v2 v = vrow(wv);
    for (int g = wv; g < 2 * np; g += WPH) {
      const SwRow krn = krow(g + WPH);
      const u32v2 vn = vrow(g + WPH);
      const u32v2 k = ROPE ? sw_bf16(sw_rope<ROPE>(p, kr, krs, (16 * g + l16) * ksr, d0)) : kr.y;
      *(u32v2*)(mine + g * 512 + (g >> 1) * 1024 + lane * 8) = k;
      *(u32v2*)(mine + (g >> 1) * SW_PAIR + 1024 + lane * 16 + (g & 1) * 8) = v;
      kr = krn;
      v = vn;
    }
  }
  __syncthreads();
  // Pairs before `clean` need no mask term (padded features shut out the last keys alone: with the term on every pair
  // 482 us in place of 456 at 237 tokens). Pairs tr and tr + 1 give the softmax reference: the first 64 keys that hold one the
  // mask does not shut out (without a live key among them no weight is exactly 1: 129 tokens, 64 shut out, error 2.29e-3
  // for 2.11e-3).
  int clean = lk >> 5, tr = 0;
  if (p.bias) {
    bool zero = true, shut = true;
    for (int i = 0; i < np && (zero || shut); i += 2) {  // two pairs: a key a lane
      const int j = i * 32 + lane;
      const float b2 = j < npmax * 32 ? lb2[j] : TA_NEG_INF;
      const uint64_t terms = __ballot(b2 != 0.f);
      if (zero && terms) {
        zero = false;
        clean = (uint32_t)terms ? i : i + 1;
      }
      if (shut && wave_any(b2 > SW_SHUT)) {
        shut = false;
        tr = i;
      }
    }
  }
  const bf16x8 ones = {(bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f, (bf16)1.f};
  for (int bi = wv; bi < nb; bi += WPH) {
    f32x4 y = sw_rope<ROPE>(p, qr, qrs, (bi * 16 + l16) * qsr, d0);
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] *= p.scale;
    const bf16x4 q = cvt_bf16x4(y);
    if (bi + WPH < nb) qr = qrow(bi + WPH);
    f32x4 o = {0.f, 0.f, 0.f, 0.f}, l = o, nm = o;  // nm: -m
    auto keys = [&](int g) { return *(const bf16x4*)(mine + g * 512 + (g >> 1) * 1024 + lane * 8); };
    auto score = [&](int g) { return mfma16x16x16(keys(g), q, f32x4{0.f, 0.f, 0.f, 0.f}); };
    struct Pair { f32x4 a, b; };
    auto scores = [&](int t) { return Pair{score(2 * t), score(2 * t + 1)}; };
    // log2 units against the reference, with the mask term where asked
    auto scaled = [&](f32x4 x, int g, bool term) {
      f32x4 c = nm;
      if (term) c += *(const f32x4*)(lb2 + 16 * g + 4 * kap);
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = __builtin_fmaf(x[r], TA_LOG2E, c[r]);
      return x;
    };
    auto accumulate = [&](int t, const Pair& x, bool term) {
      f32x4 x0 = scaled(x.a, 2 * t, term), x1 = scaled(x.b, 2 * t + 1, term);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x0[r] = __builtin_amdgcn_exp2f(x0[r]);
        x1[r] = __builtin_amdgcn_exp2f(x1[r]);
      }
      const u32v2 p0 = sw_bf16(x0), p1 = sw_bf16(x1);
      const bf16x8 pv = __builtin_bit_cast(bf16x8, uint4{p0.x, p0.y, p1.x, p1.y});
      o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(mine + t * SW_PAIR + 1024 + lane * 16), pv, o, 0, 0, 0);
      l = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pv, l, 0, 0, 0);
    };
    if (np > 0) {
      auto top = [&](int t, const Pair& x) { return sw_max(scaled(x.a, 2 * t, true), scaled(x.b, 2 * t + 1, true)); };
      Pair x = scores(0), y = x;
      float m = top(0, x);
      if (np > 1) {
        y = scores(1);
        m = fmaxf(m, top(1, y));
      }
      if (tr) {
        m = top(tr, scores(tr));
        if (tr + 1 < np) m = fmaxf(m, top(tr + 1, scores(tr + 1)));
      }
      m = quad_max(m);
      m = m > -1e4f ? fminf(m, 1e4f) : 0.f;  // every key masked, -inf and NaN: 0
      nm = f32x4{-m, -m, -m, -m};
      if (clean > 0) accumulate(0, x, false);
      else accumulate(0, x, true);
      if (np > 1) {
        int t = 1;  // y: its scores; the next pair's scores ahead of this one's exponentials
        for (; t + 1 < clean && t + 2 < np; t += 2) {
          x = scores(t + 1);
          accumulate(t, y, false);
          y = scores(t + 2);
          accumulate(t + 1, x, false);
        }
        for (; t + 1 < np; ++t) {
          x = scores(t + 1);
          accumulate(t, y, true);
          y = x;
        }
        accumulate(t, y, true);
      }
    }
    float lt = l[0];
    bool bad = !(lt >= SW_L_LO && lt <= SW_L_HI);
#pragma unroll
    for (int r = 0; r < 4; ++r) bad |= !(__builtin_fabsf(o[r]) <= 0x1p127f);
    if (wave_any(bad) && lk > 0) {  // rare: the exact online softmax, one 16-key group at a time
      float m = TA_NEG_INF, ls = 0.f;
      o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int g = 0; 16 * g < lk; ++g) {
        f32x4 x = score(g);
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = fmaf(x[r], TA_LOG2E, lb2[16 * g + 4 * kap + r]);
        // the maximum itself, not one that lags: no weight above 1, so a finite O of values near the largest float
        const float mn = fmaxf(m, quad_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]))));
        if (wave_any(mn > m)) {
          const float alpha = __builtin_amdgcn_exp2f(m - mn);
          ls *= alpha;
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] *= alpha;
          m = mn;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = __builtin_amdgcn_exp2f(x[r] - m);
        const bf16x4 pv = cvt_bf16x4(x);
#pragma unroll
        for (int r = 0; r < 4; ++r) ls += x[r];
        o = mfma16x16x16(*(const bf16x4*)(mine + (g >> 1) * SW_PAIR + 1024 + lane * 16 + (g & 1) * 8), pv, o);
      }
      lt = quad_sum(ls);
    }
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    const int qi = q0 + bi * 16 + l16;
    if (qi < p.Lq) {
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = lk > 0 ? o[r] * inv : 0.f;
      *(bf16x4*)(p.o + ((int64_t)b * p.Lq + qi) * SW_E + hc + d0) = cvt_bf16x4(o);
    }
  }
}

template <bool ROPE, int HPW> int launch_sw_inst(SwParams p, int pairs, hipStream_t stream) {
  const int lds = pairs * (HPW * SW_PAIR + 128);
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute((const void*)sw_rows_kernel<ROPE, HPW>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return (int)e;
  }
  constexpr int WPH = 8 / HPW;
  // runs of query blocks: long ones share the fill, while the grid keeps ~8 workgroups per CU
  int64_t run = (p.B * (int64_t)(SW_H / HPW) * p.nqb + 2047) / 2048;
  run = run < WPH ? WPH : (run > 16 * WPH ? 16 * WPH : (run + WPH - 1) / WPH * WPH);
  p.qbpw = (int)(run > p.nqb ? p.nqb : run);
  p.nwg_b = (p.nqb + p.qbpw - 1) / p.qbpw;
  const int64_t wgs = p.B * (int64_t)(SW_H / HPW) * p.nwg_b;
  if (wgs > (1ll << 31) - 1) return (int)hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((sw_rows_kernel<ROPE, HPW>), dim3((unsigned)wgs), dim3(512), (unsigned)lds, stream, p);
  return (int)hipGetLastError();
}
template <int HPW> int launch_sw(const SwParams& p, int pairs, hipStream_t stream) {
  return p.rope ? launch_sw_inst<true, HPW>(p, pairs, stream) : launch_sw_inst<false, HPW>(p, pairs, stream);
}

}  // namespace

int tabicl_launch_sw(const void* q, int64_t q_sb, int64_t q_sr, const void* k, int64_t k_sb, int64_t k_sr,
                     const void* v, int64_t v_sb, int64_t v_sr, void* o, const float* bias, int64_t bias_sb,
                     const int32_t* valid, int64_t valid_n, const float* cq, const float* sq, const float* ck,
                     const float* sk, int rope, int half, int rot, float scale, int64_t B, int64_t Lq, int64_t Lk,
                     const int32_t* skip, int64_t skip_n, hipStream_t stream) {
  if (Lk > SW_MAX_KEYS || ((q_sr | k_sr | v_sr | q_sb | k_sb | v_sb) & 3) || k_sr <= 0 || v_sr <= 0 || q_sr <= 0 ||
      k_sr >= 512 || v_sr >= 512 || q_sr >= 512)
    return -1;
  if (B > SMALLHEAD_MAX_BATCH) {
    for (int64_t b = 0; b < B; b += SMALLHEAD_MAX_BATCH) {
      const int64_t n = B - b < SMALLHEAD_MAX_BATCH ? B - b : SMALLHEAD_MAX_BATCH;
      const int st = tabicl_launch_sw(
          (const bf16*)q + b * q_sb, q_sb, q_sr, (const bf16*)k + b * k_sb, k_sb, k_sr, (const bf16*)v + b * v_sb, v_sb, v_sr,
          (bf16*)o + b * Lq * SW_E, bias ? bias + b * bias_sb : nullptr, bias_sb, valid && valid_n != 1 ? valid + b : valid,
          valid_n == 1 ? 1 : n, cq, sq, ck, sk, rope, half, rot, scale, n, Lq, Lk, skip && skip_n != 1 ? skip + b : skip,
          skip_n == 1 ? 1 : n, stream);
      if (st) return st;
    }
    return 0;
  }
  SwParams p = {};
  p.q = (const bf16*)q; p.q_sb = q_sb; p.q_sr = q_sr;
  p.k = (const bf16*)k; p.k_sb = k_sb; p.k_sr = k_sr;
  p.v = (const bf16*)v; p.v_sb = v_sb; p.v_sr = v_sr;
  p.o = (bf16*)o;
  p.bias = bias; p.bias_sb = bias_sb;
  p.valid = valid; p.valid_n = (int)valid_n;
  p.skip = skip; p.skip_n = (int)skip_n;
  p.cq = cq; p.sq = sq; p.ck = ck; p.sk = sk;
  p.tab_sr = (rope & TA_ROPE_SHARED) ? SW_D : SW_E;
  p.rope = rope & ~TA_ROPE_SHARED; p.half = half; p.rot = rot;
  p.scale = scale;
  p.B = (int)B; p.Lq = (int)Lq; p.Lk = (int)Lk;
  p.nqb = (p.Lq + 15) / 16;
  const int pairs = (int)((Lk + 31) / 32);
  if (pairs <= 6) return launch_sw<4>(p, pairs, stream);   // 72 KB: two workgroups per CU
  if (pairs <= 12) return launch_sw<2>(p, pairs, stream);
  return launch_sw<1>(p, pairs, stream);
}
