// fp32 small-head attention (8 heads x 16 dims), scores on the bf16 matrix units through exact splits
// (split.h), probabilities and values in fp32. Per 16-key x 16-query tile of a head:
//
//   x = K (q' log2e)       three v_mfma_f32_16x16x32_bf16: the 32-deep contraction holds two of the six
//                          split products of the same 16 dims, each lane four dims of both: [Kh | Kl] [ql | qh],
//                          [Km | Kh] [qm | qm], [Km | Kh] [qh | qh]; 48 cycles where fp32 MFMA takes 128
//   p = exp2(x - m), l += p, O^T += V^T P^T  in fp32 (four v_mfma_f32_16x16x4_f32: splitting every p would cost
//                          more VALU than the matrix cycles it saves)
//
// m is a softmax reference fixed by the first 16 keys (their ceiled maximum); a row sum outside
// [2^-64, 2^96] or a non-finite O (a score far above m, every key masked, NaN or inf in the inputs, which the
// splits turn into NaN) sends the wave's block through the exact online softmax on fp32 MFMA.
// A wave is one head; its operands come straight from global memory (a head's 64 bytes of a row; the waves of a
// row's other heads run beside it and share the cache lines).
//
// sx_resident_kernel: up to 128 keys held in registers (12 per 16 keys), no LDS or barrier; any run of query
//   blocks.
// sx_lds_kernel: 129 to 384 keys (with RoPE to 768) prepared once per workgroup into LDS (3 KB per 16 keys and
//   head): at these lengths registers would leave two waves per SIMD and spill.
// sx_stream_kernel: longer; up to 128 queries held in registers, keys streamed; a workgroup's waves take a part of
//   the keys each and merge at the end.
//
// Bound by issue: per tile 176 matrix cycles and ~25 VALU. Measured against the fp32 MFMA kernel these replace
// (us): 832 x 5000 q over 128 keys 2841 -> 2227; 400 x 128 q over 1024 keys 365 -> 312, 430 x 8029 keys 2459 ->
// 1969, 9 x 27680 keys 986 -> 289; self-attention with RoPE, 20000 x 28 tokens 815 -> 302, 16384 x 104 1542 -> 1330,
// 5000 x 129 1285 -> 708, 3000 x 237 1441 -> 841 (on sx_resident_kernel's scheme 2770).
#include "common.h"
#include "launch.h"
#include "split.h"

namespace {

constexpr int SX_H = 8, SX_D = 16, SX_E = 128;
constexpr int SX_MIN_WAVES = 1024;  // 9 x 128 q x 27680 keys: 4 blocks a workgroup 289 us, 8 blocks 499, 2 blocks 330
constexpr int SX_SEG = 65536;  // groups (1M keys)
constexpr float SX_EMPTY_REF = -32.0f;
constexpr float SX_BIAS_FLOOR = -1e37f;

struct SxParams {
  const float *q, *k, *v;
  float* o;
  int64_t q_sb, q_sr, k_sb, k_sr, v_sb, v_sr;  // element strides
  const float* bias;
  int64_t bias_sb;
  const int32_t* valid;
  int valid_n;
  const float *cq, *sq, *ck, *sk;
  int rope, half, rot, tab_sr;  // tab_sr: 128 ([L, E] tables) or 16 (one head's columns for all heads)
  float scale;
  int B, Lq, Lk, nqb, qbpw, nwg_b;
};

__device__ __forceinline__ int sx_lk(const SxParams& p, int b) {
  int lk = p.Lk;
  if (p.valid) {
    const int vl = p.valid[p.valid_n == 1 ? 0 : b];
    lk = vl < 0 ? 0 : (vl < lk ? vl : lk);
  }
  return lk;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t sx_rsrc(const float* base, int rows, int64_t sr) {
  return __builtin_amdgcn_make_buffer_rsrc((float*)base, 0, (rows - 1) * (int)sr * 4 + SX_D * 4, TA_BUF_WORD3);
}
__device__ __forceinline__ f32x4 sx_ld4(__amdgpu_buffer_rsrc_t rs, int off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
}
__device__ __forceinline__ float sx_ld1(__amdgpu_buffer_rsrc_t rs, int off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
}

// Four dims d0 .. d0 + 3 (d0 = 4 kap) of a head row: the raw values, with RoPE their partner dims (of the
// full-width halves form, one more load of the row's line) and the position's cos and sin.
struct SxRow { f32x4 y, pt; };
struct SxTab { f32x4 c, s; };
__device__ __forceinline__ SxTab sx_tab(const float* c, const float* s, int64_t pos, const SxParams& p, int col) {
  return {*(const f32x4*)(c + pos * p.tab_sr + col), *(const f32x4*)(s + pos * p.tab_sr + col)};
}
template <bool ROPE> __device__ __forceinline__ SxRow sx_row(__amdgpu_buffer_rsrc_t rs, int off, int d0) {
  SxRow r;
  r.y = sx_ld4(rs, off + d0 * 4);
  if constexpr (ROPE) r.pt = sx_ld4(rs, off + (d0 ^ 8) * 4);
  return r;
}
__device__ __forceinline__ f32x4 sx_rope(const SxParams& p, const SxRow& r, const SxTab& t, __amdgpu_buffer_rsrc_t rs, int off,
                                         int d0) {
  f32x4 out;
  if (p.rope == 2 && p.half == 8) {
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = __builtin_fmaf(r.y[i], t.c[i], (d0 & 8 ? r.pt[i] : -r.pt[i]) * t.s[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int pt;
      float sg;
      rope_partner(d0 + i, p.rope, p.half, p.rot, &pt, &sg);
      out[i] = __builtin_fmaf(r.y[i], t.c[i], sg * sx_ld1(rs, off + pt * 4) * t.s[i]);
    }
  }
  return out;
}

__device__ __forceinline__ f32x4 sx_mm(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// A key row's two score operands and a query's three, from this lane's four dims.
struct SxK { bf16x8 mh, hl; };
struct SxQ { bf16x8 hh, mm, lh; };
__device__ __forceinline__ bf16x8 sx_cat(const uint32_t* a, const uint32_t* b) {
  return __builtin_bit_cast(bf16x8, uint4{a[0], a[1], b[0], b[1]});
}
__device__ __forceinline__ SxK sx_kop(f32x4 y) {
  uint32_t h[2], m[2], l[2];
  split2(y[0], y[1], h[0], m[0], l[0]);
  split2(y[2], y[3], h[1], m[1], l[1]);
  return {sx_cat(m, h), sx_cat(h, l)};
}
__device__ __forceinline__ SxQ sx_qop(f32x4 y) {
  uint32_t h[2], m[2], l[2];
  split2(y[0], y[1], h[0], m[0], l[0]);
  split2(y[2], y[3], h[1], m[1], l[1]);
  return {sx_cat(h, h), sx_cat(m, m), sx_cat(l, h)};
}
// K q, summed from zero: started from -m, each of the three sums would be rounded at m's magnitude (the output's
// error against float64 4% above the fp32 MFMA kernel's; subtracted afterwards, below it).
__device__ __forceinline__ f32x4 sx_score(const SxK& k, const SxQ& q) {
  return sx_mm(k.mh, q.hh, sx_mm(k.mh, q.mm, sx_mm(k.hl, q.lh, f32x4{0.f, 0.f, 0.f, 0.f})));
}

// The softmax reference of a block from its first 16 keys' scores (log2 units).
__device__ __forceinline__ float sx_ref(f32x4 x) {
  const float tm = quad_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
  return tm > -1e4f ? fminf(ceilf(tm), 1e4f) : 0.f;  // -inf and NaN: 0
}

// l: the row's whole sum (a lane's part may hold masked keys alone).
__device__ __forceinline__ bool sx_suspect(f32x4 o, float l) {
  bool bad = !(l >= 0x1p-64f && l <= 0x1p96f);
#pragma unroll
  for (int r = 0; r < 4; ++r) bad |= !(__builtin_fabsf(o[r]) <= 0x1p127f);
  return bad;
}

// b2 of keys k0 .. k0 + 3 in log2 units from their mask (zeros without one): -inf from lk on.
__device__ __forceinline__ f32x4 sx_b2(f32x4 bias, int k0, int lk) {
  f32x4 b2;
#pragma unroll
  for (int r = 0; r < 4; ++r) b2[r] = k0 + r < lk ? fmaxf(bias[r] * TA_LOG2E, SX_BIAS_FLOOR) : TA_NEG_INF;
  return b2;
}

// The exact online softmax of one block over groups [kt0, kt1), fp32 MFMA (rare: rolled up, operands loaded
// again). q: q' (unsplit); key(kt) / val(kt): this lane's four dims of key 16 kt + l16, and its dim of keys 16 kt +
// 4 kap .. + 3; b2(kt): those keys' mask.
template <typename FK, typename FV, typename FB>
__device__ __forceinline__ void sx_exact(f32x4 q, int kt0, int kt1, FK key, FV val, FB b2, f32x4& o, float& m, float& l) {
  o = f32x4{0.f, 0.f, 0.f, 0.f};
  m = TA_NEG_INF;
  l = 0.f;
#pragma unroll 1
  for (int kt = kt0; kt < kt1; ++kt) {
    f32x4 x = mfma16x16x16(key(kt), q, f32x4{0.f, 0.f, 0.f, 0.f});
    const f32x4 b = b2(kt);
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = fmaf(x[r], TA_LOG2E, b[r]);
    // the maximum itself, not one that lags: no weight above 1, so a finite O of values near the largest float
    const float m_new = fmaxf(m, quad_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]))));
    if (wave_any(m_new > m)) {
      const float alpha = __builtin_amdgcn_exp2f(m - m_new);
      l *= alpha;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] *= alpha;
      m = m_new;
    }
    f32x4 pv;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      pv[r] = __builtin_amdgcn_exp2f(x[r] - m);
      l += pv[r];
    }
    o = mfma16x16x16(val(kt), pv, o);
  }
}

// NG: 16-key groups held; MF: 0 a mask or per-batch lengths (b2 added to every tile, from LDS), 1 the end of the
// last group may be past Lk. Workgroup = 4 heads of (batch element, run of
// query blocks).
// One query block at a time: two, for twice the independent products, took the registers of a third wave per SIMD
// and ran 7-60% slower.
template <int NG, int MF, bool ROPE>
__global__ __launch_bounds__(256, NG <= 3 ? 4 : NG <= (ROPE ? 6 : 8) ? 3 : 2) void sx_resident_kernel(SxParams p) {
  __shared__ __attribute__((aligned(16))) float lb2[MF == 0 ? NG * 16 : 4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, kap = lane >> 4;
  const int work = xcd_remap(blockIdx.x, gridDim.x);
  const int head = (work & 1) * 4 + wave, rest = work >> 1;
  const int b = rest / p.nwg_b, qb0 = (rest % p.nwg_b) * p.qbpw;
  const int nb = p.nqb - qb0 < p.qbpw ? p.nqb - qb0 : p.qbpw;
  const int lk = MF == 0 ? sx_lk(p, b) : p.Lk;
  const int d0 = 4 * kap, hc = head * SX_D, tc = (hc & (p.tab_sr - 1)) + d0;
  // keys from lk on read as zero (the resource ends at row lk - 1; without keys a row is read and masked)
  const int lr = MF == 0 ? (lk > 0 ? lk : 1) : lk;
  const __amdgpu_buffer_rsrc_t krs = sx_rsrc(p.k + b * p.k_sb + hc, lr, p.k_sr);
  const __amdgpu_buffer_rsrc_t vrs = sx_rsrc(p.v + b * p.v_sb + hc, lr, p.v_sr);
  const int q0 = qb0 * 16, qrows = p.Lq - q0 < nb * 16 ? p.Lq - q0 : nb * 16;
  const __amdgpu_buffer_rsrc_t qrs = sx_rsrc(p.q + b * p.q_sb + (int64_t)q0 * p.q_sr + hc, qrows, p.q_sr);
  const int ksr = (int)p.k_sr * 4, vsr = (int)p.v_sr * 4, qsr = (int)p.q_sr * 4;
  SxRow kr[NG], qr;
  f32x4 va[NG];
#pragma unroll
  for (int kt = 0; kt < NG; ++kt) kr[kt] = sx_row<ROPE>(krs, (16 * kt + l16) * ksr, d0);
  qr = sx_row<ROPE>(qrs, l16 * qsr, d0);
#pragma unroll
  for (int kt = 0; kt < NG; ++kt)
#pragma unroll
    for (int j = 0; j < 4; ++j) va[kt][j] = sx_ld1(vrs, (16 * kt + 4 * kap + j) * vsr + l16 * 4);
  if constexpr (MF == 0) {
    for (int j = threadIdx.x; j < NG * 16; j += 256) {
      float b2 = j < lk ? 0.f : TA_NEG_INF;
      if (p.bias && j < lk) b2 = fmaxf(p.bias[b * p.bias_sb + j] * TA_LOG2E, SX_BIAS_FLOOR);
      lb2[j] = b2;
    }
    __syncthreads();
  }
  SxK kop[NG];
  if constexpr (ROPE) {
    auto tab = [&](int kt) {
      const int key = 16 * kt + l16;
      return sx_tab(p.ck, p.sk, key < p.Lk ? key : p.Lk - 1, p, tc);
    };
    SxTab t = tab(0);
#pragma unroll
    for (int kt = 0; kt < NG; ++kt) {
      const SxTab tn = kt + 1 < NG ? tab(kt + 1) : t;
      kop[kt] = sx_kop(sx_rope(p, kr[kt], t, krs, (16 * kt + l16) * ksr, d0));
      t = tn;
      __builtin_amdgcn_sched_barrier(0);  // one group's tables ahead, not all of them
    }
  } else {
#pragma unroll
    for (int kt = 0; kt < NG; ++kt) kop[kt] = sx_kop(kr[kt].y);
  }
  const float qc = p.scale;
  // q' of a block (zeros past Lq)
  auto qtab = [&](int blk) {
    const int qi = q0 + blk * 16 + l16;
    return sx_tab(p.cq, p.sq, qi < p.Lq ? qi : p.Lq - 1, p, tc);
  };
  auto qprime = [&](const SxRow& r, const SxTab& t, int blk) {
    f32x4 y = r.y;
    if constexpr (ROPE) y = sx_rope(p, r, t, qrs, (blk * 16 + l16) * qsr, d0);
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] *= qc;
    return y;
  };
  auto exact = [&](int blk, f32x4& o, float& m, float& l) {
    sx_exact(
        qprime(sx_row<ROPE>(qrs, (blk * 16 + l16) * qsr, d0), ROPE ? qtab(blk) : SxTab{}, blk), 0, (lk + 15) >> 4,
        [&](int kt) {
          const int key = 16 * kt + l16;
          const SxRow r = sx_row<ROPE>(krs, key * ksr, d0);
          if constexpr (ROPE)
            return sx_rope(p, r, sx_tab(p.ck, p.sk, key < p.Lk ? key : p.Lk - 1, p, tc), krs, key * ksr, d0);
          else return r.y;
        },
        [&](int kt) {
          f32x4 v;
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = sx_ld1(vrs, (16 * kt + 4 * kap + j) * vsr + l16 * 4);
          return v;
        },
        [&](int kt) {
          f32x4 b2;
#pragma unroll
          for (int r = 0; r < 4; ++r)
            b2[r] = MF == 0 ? lb2[MF == 0 ? 16 * kt + 4 * kap + r : 0] : 16 * kt + 4 * kap + r < lk ? 0.f : TA_NEG_INF;
          return b2;
        },
        o, m, l);
  };
  SxTab qt = {};
  if constexpr (ROPE) qt = qtab(0);
  for (int bi = 0; bi < nb; ++bi) {
    f32x4 y = qprime(qr, qt, bi);
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] *= TA_LOG2E;
    const SxQ q = sx_qop(y);
    if (bi + 1 < nb) {
      qr = sx_row<ROPE>(qrs, ((bi + 1) * 16 + l16) * qsr, d0);
      if constexpr (ROPE) qt = qtab(bi + 1);
    }
    auto score = [&](int kt) {
      f32x4 x = sx_score(kop[kt], q);
      if constexpr (MF == 0) {
        x += *(const f32x4*)(lb2 + 16 * kt + 4 * kap);
      } else if (kt == NG - 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = 16 * kt + 4 * kap + r < lk ? x[r] : TA_NEG_INF;
      }
      return x;
    };
    // scores one group ahead of the exponentials and value products
    f32x4 o0 = {0.f, 0.f, 0.f, 0.f}, o1 = o0, x = score(0);
    float l = 0.f, m = sx_ref(x);
#pragma unroll
    for (int kt = 0; kt < NG; ++kt) {
      const f32x4 xn = kt + 1 < NG ? score(kt + 1 < NG ? kt + 1 : kt) : x;
      f32x4 pv;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pv[r] = __builtin_amdgcn_exp2f(x[r] - m);
        l += pv[r];
      }
      if (kt & 1) o1 = mfma16x16x16(va[kt], pv, o1);
      else o0 = mfma16x16x16(va[kt], pv, o0);
      x = xn;
    }
    f32x4 o = o0 + o1;
    float lt = quad_sum(l);
    if (wave_any(sx_suspect(o, lt)) && lk > 0) {
      exact(bi, o, m, l);
      lt = quad_sum(l);
    }
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    const int qi = q0 + bi * 16 + l16;
    if (qi < p.Lq) {
      f32x4 out;
#pragma unroll
      for (int r = 0; r < 4; ++r) out[r] = MF == 0 && lk == 0 ? 0.f : o[r] * inv;
      *(f32x4*)(p.o + ((int64_t)b * p.Lq + qi) * SX_E + hc + d0) = out;
    }
  }
}

// Keys in LDS: HPW heads per workgroup of 8 waves, the waves of a head share its operands (3 KB per 16 keys: the two
// score operands and V, each lane's 16 bytes at 16 lane) and take query blocks in turn. Any key count that fits.
template <bool MASKED, bool ROPE, int HPW>
__global__ __launch_bounds__(512, 4) void sx_lds_kernel(SxParams p) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int WPH = 8 / HPW;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, kap = lane >> 4;
  const int hd = wave / WPH, wv = wave % WPH;
  const int work = xcd_remap(blockIdx.x, gridDim.x);
  const int head = (work % (SX_H / HPW)) * HPW + hd, rest = work / (SX_H / HPW);
  const int b = rest / p.nwg_b, qb0 = (rest % p.nwg_b) * p.qbpw;
  const int nb = p.nqb - qb0 < p.qbpw ? p.nqb - qb0 : p.qbpw;
  const int lk = sx_lk(p, b), ng = (lk + 15) >> 4, ngmax = (p.Lk + 15) >> 4;
  const int d0 = 4 * kap, hc = head * SX_D, tc = (hc & (p.tab_sr - 1)) + d0;
  const int lr = lk > 0 ? lk : 1;  // rows from lk on read as zero
  const __amdgpu_buffer_rsrc_t krs = sx_rsrc(p.k + b * p.k_sb + hc, lr, p.k_sr);
  const __amdgpu_buffer_rsrc_t vrs = sx_rsrc(p.v + b * p.v_sb + hc, lr, p.v_sr);
  const int q0 = qb0 * 16, qrows = p.Lq - q0 < nb * 16 ? p.Lq - q0 : nb * 16;
  const __amdgpu_buffer_rsrc_t qrs = sx_rsrc(p.q + b * p.q_sb + (int64_t)q0 * p.q_sr + hc, qrows, p.q_sr);
  const int ksr = (int)p.k_sr * 4, vsr = (int)p.v_sr * 4, qsr = (int)p.q_sr * 4;
  char* mine = (char*)lds + hd * ngmax * 3072 + lane * 16;
  float* lb2 = lds + HPW * ngmax * 768;
  auto qrow = [&](int blk) { return sx_row<ROPE>(qrs, (blk * 16 + l16) * qsr, d0); };
  auto qtab = [&](int blk) {
    const int qi = q0 + blk * 16 + l16;
    return sx_tab(p.cq, p.sq, qi < p.Lq ? qi : p.Lq - 1, p, tc);
  };
  auto ktab = [&](int kt) {
    const int key = 16 * kt + l16;
    return sx_tab(p.ck, p.sk, key < p.Lk ? key : p.Lk - 1, p, tc);
  };
  auto krow = [&](int kt) { return sx_row<ROPE>(krs, (16 * kt + l16) * ksr, d0); };
  auto vrow = [&](int kt) {
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = sx_ld1(vrs, (16 * kt + 4 * kap + j) * vsr + l16 * 4);
    return v;
  };
  SxRow qr = qrow(wv);
  SxTab qt;
  if constexpr (ROPE) qt = qtab(wv);
  {  // fill: this wave's groups, the next one's loads in flight
    SxRow kr = krow(wv);
    f32x4 v = vrow(wv);
    SxTab t;
    if constexpr (ROPE) t = ktab(wv);
    for (int kt = wv; kt < ng; kt += WPH) {
      const SxRow krn = krow(kt + WPH);
      const f32x4 vn = vrow(kt + WPH);
      SxTab tn;
      if constexpr (ROPE) tn = ktab(kt + WPH);
      SxK k;
      if constexpr (ROPE) k = sx_kop(sx_rope(p, kr, t, krs, (16 * kt + l16) * ksr, d0));
      else k = sx_kop(kr.y);
      *(bf16x8*)(mine + kt * 3072) = k.mh;
      *(bf16x8*)(mine + kt * 3072 + 1024) = k.hl;
      *(f32x4*)(mine + kt * 3072 + 2048) = v;
      kr = krn;
      v = vn;
      if constexpr (ROPE) t = tn;
    }
  }
  if constexpr (MASKED) {
    for (int j = threadIdx.x; j < ngmax * 16; j += 512) {
      float b2 = j < lk ? 0.f : TA_NEG_INF;
      if (p.bias && j < lk) b2 = fmaxf(p.bias[b * p.bias_sb + j] * TA_LOG2E, SX_BIAS_FLOOR);
      lb2[j] = b2;
    }
  }
  __syncthreads();
  for (int bi = wv; bi < nb; bi += WPH) {
    f32x4 y = qr.y;
    if constexpr (ROPE) y = sx_rope(p, qr, qt, qrs, (bi * 16 + l16) * qsr, d0);
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = y[r] * p.scale * TA_LOG2E;
    const SxQ q = sx_qop(y);
    if (bi + WPH < nb) {
      qr = qrow(bi + WPH);
      if constexpr (ROPE) qt = qtab(bi + WPH);
    }
    f32x4 o0 = {0.f, 0.f, 0.f, 0.f}, o1 = o0;
    float l = 0.f, m = 0.f;
    auto score = [&](int kt) {
      const SxK k = {*(const bf16x8*)(mine + kt * 3072), *(const bf16x8*)(mine + kt * 3072 + 1024)};
      f32x4 x = sx_score(k, q);
      if constexpr (MASKED) {
        x += *(const f32x4*)(lb2 + 16 * kt + 4 * kap);
      } else if (kt == ng - 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = 16 * kt + 4 * kap + r < lk ? x[r] : TA_NEG_INF;
      }
      return x;
    };
    auto accumulate = [&](int kt, f32x4 x, f32x4& o) {
      f32x4 pv;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pv[r] = __builtin_amdgcn_exp2f(x[r] - m);
        l += pv[r];
      }
      o = mfma16x16x16(*(const f32x4*)(mine + kt * 3072 + 2048), pv, o);
    };
    if (ng > 0) {
      // scores one group ahead of the exponentials and value products
      f32x4 x = score(0);
      m = sx_ref(x);
      int kt = 0;
      for (; kt + 2 < ng; kt += 2) {
        const f32x4 x1 = score(kt + 1);
        accumulate(kt, x, o0);
        x = score(kt + 2);
        accumulate(kt + 1, x1, o1);
      }
      if (kt + 1 < ng) {
        const f32x4 x1 = score(kt + 1);
        accumulate(kt, x, o0);
        accumulate(kt + 1, x1, o1);
      } else {
        accumulate(kt, x, o0);
      }
    }
    f32x4 o = o0 + o1;
    float lt = quad_sum(l);
    if (wave_any(sx_suspect(o, lt)) && lk > 0) {
      f32x4 qe = sx_row<false>(qrs, (bi * 16 + l16) * qsr, d0).y;
      if constexpr (ROPE) qe = sx_rope(p, qrow(bi), qtab(bi), qrs, (bi * 16 + l16) * qsr, d0);
#pragma unroll
      for (int r = 0; r < 4; ++r) qe[r] *= p.scale;
      sx_exact(
          qe, 0, ng,
          [&](int kt) {
            const SxRow r = krow(kt);
            if constexpr (ROPE) return sx_rope(p, r, ktab(kt), krs, (16 * kt + l16) * ksr, d0);
            else return r.y;
          },
          vrow,
          [&](int kt) {
            f32x4 b2;
#pragma unroll
            for (int r = 0; r < 4; ++r)
              b2[r] = MASKED ? lb2[16 * kt + 4 * kap + r] : 16 * kt + 4 * kap + r < lk ? 0.f : TA_NEG_INF;
            return b2;
          },
          o, m, l);
      lt = quad_sum(l);
    }
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    const int qi = q0 + bi * 16 + l16;
    if (qi < p.Lq) {
      f32x4 out;
#pragma unroll
      for (int r = 0; r < 4; ++r) out[r] = lk > 0 ? o[r] * inv : 0.f;
      *(f32x4*)(p.o + ((int64_t)b * p.Lq + qi) * SX_E + hc + d0) = out;
    }
  }
}

// Wave w of NW takes the w-th part of the keys for the workgroup's NB query blocks of one head; merged in LDS.
template <int NB, int NW, bool BIAS, bool ROPE>
__global__ __launch_bounds__(NW * 64, 2) void sx_stream_kernel(SxParams p) {
  extern __shared__ __attribute__((aligned(16))) float lds[];  // per wave and block: O [4][64], m [64], l [64]
  __shared__ int bad_w[NW];  // per wave: a result that may not be trusted
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, kap = lane >> 4;
  const int work = xcd_remap(blockIdx.x, gridDim.x);
  const int head = work % SX_H, rest = work / SX_H;
  const int b = rest / p.nwg_b, q0 = (rest % p.nwg_b) * NB * 16;
  const int lk = sx_lk(p, b), ng = (lk + 15) >> 4, per = (ng + NW - 1) / NW;
  const int g0 = wave * per < ng ? wave * per : ng, g1 = g0 + per < ng ? g0 + per : ng;
  const int d0 = 4 * kap, hc = head * SX_D, tc = (hc & (p.tab_sr - 1)) + d0;
  SxQ q[NB];
  f32x4 o[NB];
  float m[NB], l[NB];
  const int nrow = p.Lq - q0 < NB * 16 ? p.Lq - q0 : NB * 16;
  const __amdgpu_buffer_rsrc_t qrs = sx_rsrc(p.q + b * p.q_sb + (int64_t)q0 * p.q_sr + hc, nrow, p.q_sr);
  auto qprime = [&](int j) {  // q' of block j, zeros past Lq
    const int off = (16 * j + l16) * (int)p.q_sr * 4, qi = q0 + 16 * j + l16;
    const SxRow r = sx_row<ROPE>(qrs, off, d0);
    f32x4 y = r.y;
    if constexpr (ROPE) y = sx_rope(p, r, sx_tab(p.cq, p.sq, qi < p.Lq ? qi : p.Lq - 1, p, tc), qrs, off, d0);
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] *= p.scale;
    return y;
  };
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    f32x4 y = qprime(j);
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] *= TA_LOG2E;
    q[j] = sx_qop(y);
    o[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    m[j] = TA_NEG_INF;
    l[j] = 0.f;
    __builtin_amdgcn_sched_barrier(0);
  }
  // the part's rows as a resource, SX_SEG groups at a time (32-bit offsets); rows past lk read as zero
  bool first = true;
#pragma unroll 1
  for (int s0 = g0; s0 < g1; s0 += SX_SEG) {
    const int s1 = g1 - s0 < SX_SEG ? g1 : s0 + SX_SEG;
    const int row0 = s0 * 16, rows = lk - row0 < (s1 - s0) * 16 ? lk - row0 : (s1 - s0) * 16;
    const __amdgpu_buffer_rsrc_t krs = sx_rsrc(p.k + b * p.k_sb + (int64_t)row0 * p.k_sr + hc, rows, p.k_sr);
    const __amdgpu_buffer_rsrc_t vrs = sx_rsrc(p.v + b * p.v_sb + (int64_t)row0 * p.v_sr + hc, rows, p.v_sr);
    const int ksr = (int)p.k_sr * 4, vsr = (int)p.v_sr * 4;
    SxRow ky, kz;  // this group's rows and the next one's, in flight
    f32x4 vy, vz;
    SxTab ty, tz;
    f32x4 by = {0.f, 0.f, 0.f, 0.f};  // the next group's mask, in flight (loaded at its use: 339 against 270 us for the same call)
    const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc(
        (float*)(BIAS ? p.bias + b * p.bias_sb + row0 : p.q), 0, BIAS ? rows * 4 : 0, TA_BUF_WORD3);
    auto fetch = [&](int g, SxRow& kk, f32x4& vv, SxTab& tt) {
      kk = sx_row<ROPE>(krs, (16 * g + l16) * ksr, d0);
#pragma unroll
      for (int j = 0; j < 4; ++j) vv[j] = sx_ld1(vrs, (16 * g + 4 * kap + j) * vsr + l16 * 4);
      if constexpr (ROPE) {
        const int key = 16 * (s0 + g) + l16;
        tt = sx_tab(p.ck, p.sk, key < p.Lk ? key : p.Lk - 1, p, tc);
      }
    };
    auto mask = [&](int g) { return sx_ld4(brs, (16 * g + 4 * kap) * 4); };
    fetch(0, ky, vy, ty);
    if constexpr (BIAS) by = mask(0);
    fetch(1, kz, vz, tz);  // past the last group: zeros, unused
#pragma unroll 1
    for (int g = 0; g < s1 - s0; ++g) {
      SxK k;
      if constexpr (ROPE) k = sx_kop(sx_rope(p, ky, ty, krs, (16 * g + l16) * ksr, d0));
      else k = sx_kop(ky.y);
      const f32x4 va = vy, bc = by;
      ky = kz;
      vy = vz;
      ty = tz;
      if constexpr (BIAS) by = mask(g + 1);
      fetch(g + 2, kz, vz, tz);
      const bool tail = 16 * (s0 + g) + 16 > lk;
      f32x4 b2 = {0.f, 0.f, 0.f, 0.f};
      if (BIAS || tail) b2 = sx_b2(bc, 16 * (s0 + g) + 4 * kap, lk);
      if (first) {
        first = false;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          m[j] = sx_ref(sx_score(k, q[j]) + b2);
        }
      }
      // the next block's scores ahead of this one's exponentials and value products
      auto score = [&](int j) {
        f32x4 x = sx_score(k, q[j]);
        if (BIAS || tail) x += b2;
        return x;
      };
      f32x4 x = score(0);
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const f32x4 xn = j + 1 < NB ? score(j + 1 < NB ? j + 1 : 0) : x;
        f32x4 pv;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          pv[r] = __builtin_amdgcn_exp2f(x[r] - m[j]);
          l[j] += pv[r];
        }
        o[j] = mfma16x16x16(va, pv, o[j]);
        x = xn;
      }
    }
  }
  // Trust test. With a mask a part may hold masked keys alone (a prefix mask leaves the last waves nothing): such a
  // part, l = 0 and O = 0 exactly, is left out of the merge (m = -inf). Its scores are below -126 (no key of its first
  // group set a reference, so m = 0); a trusted part's sum is at least 2^(m - 1), or 2^-64 where m = 0. So where the
  // row's largest reference is SX_EMPTY_REF or more, 2^20 keys left out are below 2^-42 of it; where it is lower the
  // row is not trusted. (Judged by itself, a part without live keys sent the workgroup through the exact pass: prefix
  // mask of 300 of 1024 keys, 400 x 128 q, 1969 against 270 us.)
  float* const mine = lds + wave * NB * 384;
  bool bad = false;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    if (g0 < g1) {
      const float lt = quad_sum(l[j]);
      const bool empty = BIAS && lt == 0.f && o[j][0] == 0.f && o[j][1] == 0.f && o[j][2] == 0.f && o[j][3] == 0.f;
      if (empty) m[j] = TA_NEG_INF;
      else bad |= sx_suspect(o[j], lt);
    }
    *(f32x4*)(mine + j * 384 + lane * 4) = o[j];
    mine[j * 384 + 256 + lane] = m[j];
    mine[j * 384 + 320 + lane] = l[j];
  }
  if constexpr (BIAS) {
    __syncthreads();
    for (int j = wave; j < NB; j += NW) {
      float mt = TA_NEG_INF, least = SX_EMPTY_REF;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        if (w * per >= ng) continue;  // no keys in that part
        const float mw = lds[w * NB * 384 + j * 384 + 256 + lane];
        mt = fmaxf(mt, mw);
        least = fminf(least, mw);
      }
      bad |= least == TA_NEG_INF && mt < SX_EMPTY_REF;
    }
  }
  bad = wave_any(bad);
  if (lane == 0) bad_w[wave] = bad;
  __syncthreads();
  int redo = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) redo |= bad_w[w];
  if (redo) {  // rare: every wave redoes its part with the exact online softmax
    if (g0 < g1) {
      float* dst = mine;
      const float* kb = p.k + b * p.k_sb + hc;
      const float* vb = p.v + b * p.v_sb + hc;
#pragma unroll 1
      for (int j = 0; j < NB; ++j, dst += 384) {
        f32x4 oj;
        float mj, lj;
        sx_exact(
            qprime(j), g0, g1,
            [&](int kt) {
              const int key = 16 * kt + l16, kc = key < lk ? key : lk - 1;
              const __amdgpu_buffer_rsrc_t rs =
                  sx_rsrc(kb + (int64_t)(16 * kt) * p.k_sr, lk - 16 * kt < 16 ? lk - 16 * kt : 16, p.k_sr);
              const int off = l16 * (int)p.k_sr * 4;
              const SxRow r = sx_row<ROPE>(rs, off, d0);
              if constexpr (ROPE) return sx_rope(p, r, sx_tab(p.ck, p.sk, kc, p, tc), rs, off, d0);
              else return r.y;
            },
            [&](int kt) {
              const __amdgpu_buffer_rsrc_t rs =
                  sx_rsrc(vb + (int64_t)(16 * kt) * p.v_sr, lk - 16 * kt < 16 ? lk - 16 * kt : 16, p.v_sr);
              f32x4 v;
#pragma unroll
              for (int i = 0; i < 4; ++i) v[i] = sx_ld1(rs, (4 * kap + i) * (int)p.v_sr * 4 + l16 * 4);
              return v;
            },
            [&](int kt) {
              f32x4 bias = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
              for (int r = 0; r < 4; ++r)
                if (BIAS && 16 * kt + 4 * kap + r < lk) bias[r] = p.bias[b * p.bias_sb + 16 * kt + 4 * kap + r];
              return sx_b2(bias, 16 * kt + 4 * kap, lk);
            },
            oj, mj, lj);
        *(f32x4*)(dst + lane * 4) = oj;
        dst[256 + lane] = mj;
        dst[320 + lane] = lj;
      }
    }
    __syncthreads();
  }
  for (int j = wave; j < NB; j += NW) {
    const int qi = q0 + 16 * j + l16;
    float mt = TA_NEG_INF;
#pragma unroll
    for (int w = 0; w < NW; ++w) mt = fmaxf(mt, lds[w * NB * 384 + j * 384 + 256 + lane]);
    f32x4 ot = {0.f, 0.f, 0.f, 0.f};
    float lt = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float* src = lds + w * NB * 384 + j * 384;
      const float mw = src[256 + lane];
      const float f = mw == TA_NEG_INF ? 0.f : __builtin_amdgcn_exp2f(mw - mt);  // no keys in that part
      lt += src[320 + lane] * f;
      const f32x4 ow = *(const f32x4*)(src + lane * 4);
#pragma unroll
      for (int r = 0; r < 4; ++r) ot[r] += ow[r] * f;
    }
    lt = quad_sum(lt);
    if (qi < p.Lq) {
      const float inv = lk > 0 && !(lt <= 0.f) ? 1.f / lt : 0.f;
      f32x4 out;
#pragma unroll
      for (int r = 0; r < 4; ++r) out[r] = lk > 0 ? ot[r] * inv : 0.f;
      *(f32x4*)(p.o + ((int64_t)b * p.Lq + qi) * SX_E + hc + 4 * kap) = out;
    }
  }
}

template <int NG> void launch_sx_resident(const SxParams& p, dim3 grid, hipStream_t stream) {
  const dim3 block(256);
  const bool masked = p.bias || p.valid;
  if (p.rope) {
    if (masked) hipLaunchKernelGGL((sx_resident_kernel<NG, 0, true>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((sx_resident_kernel<NG, 1, true>), grid, block, 0, stream, p);
  } else {
    if (masked) hipLaunchKernelGGL((sx_resident_kernel<NG, 0, false>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((sx_resident_kernel<NG, 1, false>), grid, block, 0, stream, p);
  }
}

template <bool MASKED, bool ROPE, int HPW>
int launch_sx_lds_inst(SxParams p, int lds, hipStream_t stream) {
  if (lds > 65536) {  // above the default limit of dynamic LDS
    const hipError_t e = hipFuncSetAttribute((const void*)sx_lds_kernel<MASKED, ROPE, HPW>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return (int)e;
  }
  constexpr int WPH = 8 / HPW;
  // runs of query blocks: long ones share the key operands, while the grid keeps ~8 workgroups per CU
  int64_t run = (p.B * (int64_t)(SX_H / HPW) * p.nqb + 2047) / 2048;
  run = run < WPH ? WPH : (run > 16 * WPH ? 16 * WPH : (run + WPH - 1) / WPH * WPH);
  p.qbpw = (int)(run > p.nqb ? p.nqb : run);
  p.nwg_b = (p.nqb + p.qbpw - 1) / p.qbpw;
  const int64_t wgs = p.B * (int64_t)(SX_H / HPW) * p.nwg_b;
  if (wgs > (1ll << 31) - 1) return (int)hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((sx_lds_kernel<MASKED, ROPE, HPW>), dim3((unsigned)wgs), dim3(512), (unsigned)lds, stream, p);
  return (int)hipGetLastError();
}
template <int HPW> int launch_sx_lds(const SxParams& p, int groups, hipStream_t stream) {
  const int lds = groups * (HPW * 3072 + 64);
  if (p.bias || p.valid)
    return p.rope ? launch_sx_lds_inst<true, true, HPW>(p, lds, stream) : launch_sx_lds_inst<true, false, HPW>(p, lds, stream);
  return p.rope ? launch_sx_lds_inst<false, true, HPW>(p, lds, stream) : launch_sx_lds_inst<false, false, HPW>(p, lds, stream);
}

template <int NB, int NW, bool BIAS, bool ROPE>
int launch_sx_stream_inst(const SxParams& p, hipStream_t stream) {
  constexpr int LDS = NW * NB * 384 * 4;
  if (LDS > 65536) {  // above the default limit of dynamic LDS
    const hipError_t e = hipFuncSetAttribute((const void*)sx_stream_kernel<NB, NW, BIAS, ROPE>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (e != hipSuccess) return (int)e;
  }
  hipLaunchKernelGGL((sx_stream_kernel<NB, NW, BIAS, ROPE>), dim3((unsigned)((int64_t)p.B * SX_H * p.nwg_b)),
                     dim3(NW * 64), LDS, stream, p);
  return (int)hipGetLastError();
}

template <int NB, int NW>
int launch_sx_stream(const SxParams& p, hipStream_t stream) {
  if constexpr (NB <= 4) {
    if (p.rope)
      return p.bias ? launch_sx_stream_inst<NB, NW, true, true>(p, stream)
                    : launch_sx_stream_inst<NB, NW, false, true>(p, stream);
  }
  return p.bias ? launch_sx_stream_inst<NB, NW, true, false>(p, stream)
                : launch_sx_stream_inst<NB, NW, false, false>(p, stream);
}

}  // namespace

// fp32 small-head attention (arguments as tabicl_launch_smallhead). Element strides must be multiples of 4
// and row strides below 512 (E, 2 E or 3 E here).
int tabicl_launch_sx(const void* q, int64_t q_sb, int64_t q_sr, const void* k, int64_t k_sb, int64_t k_sr,
                     const void* v, int64_t v_sb, int64_t v_sr, void* o, const float* bias, int64_t bias_sb,
                     const int32_t* valid, int64_t valid_n, const float* cq, const float* sq, const float* ck,
                     const float* sk, int rope, int half, int rot, float scale, int64_t B, int64_t Lq, int64_t Lk,
                     hipStream_t stream) {
  if (B > SMALLHEAD_MAX_BATCH) {
    for (int64_t b = 0; b < B; b += SMALLHEAD_MAX_BATCH) {
      const int64_t n = B - b < SMALLHEAD_MAX_BATCH ? B - b : SMALLHEAD_MAX_BATCH;
      const int st = tabicl_launch_sx(
          (const float*)q + b * q_sb, q_sb, q_sr, (const float*)k + b * k_sb, k_sb, k_sr, (const float*)v + b * v_sb, v_sb,
          v_sr, (float*)o + b * Lq * SX_E, bias ? bias + b * bias_sb : nullptr, bias_sb,
          valid && valid_n != 1 ? valid + b : valid, valid_n == 1 ? 1 : n, cq, sq, ck, sk, rope, half, rot, scale, n, Lq, Lk,
          stream);
      if (st) return st;
    }
    return 0;
  }
  SxParams p = {};
  p.q = (const float*)q; p.q_sb = q_sb; p.q_sr = q_sr;
  p.k = (const float*)k; p.k_sb = k_sb; p.k_sr = k_sr;
  p.v = (const float*)v; p.v_sb = v_sb; p.v_sr = v_sr;
  p.o = (float*)o;
  p.bias = bias; p.bias_sb = bias_sb;
  p.valid = valid; p.valid_n = (int)valid_n;
  p.cq = cq; p.sq = sq; p.ck = ck; p.sk = sk;
  p.tab_sr = (rope & TA_ROPE_SHARED) ? SX_D : SX_E;
  p.rope = rope & ~TA_ROPE_SHARED; p.half = half; p.rot = rot;
  p.scale = scale;
  p.B = (int)B; p.Lq = (int)Lq; p.Lk = (int)Lk;
  if (((q_sr | k_sr | v_sr | q_sb | k_sb) & 3) || k_sr <= 0 || v_sr <= 0 || q_sr <= 0 || k_sr >= 512 || v_sr >= 512 ||
      q_sr >= 512)
    return (int)hipErrorInvalidValue;
  p.nqb = (p.Lq + 15) / 16;
  const int64_t lim = (1ll << 31) - 1;
  const int groups = (int)((Lk + 15) / 16);
  if (groups > 8 && (groups <= 24 || (p.rope && groups <= 48))) {
    if (groups <= 12) return launch_sx_lds<2>(p, groups, stream);
    return launch_sx_lds<1>(p, groups, stream);
  }
  if (groups <= 8) {
    // runs of query blocks: the keys' operands are made once per wave (about three blocks' work per 8 groups),
    // so long runs, while the grid keeps 12 workgroups per CU
    int64_t run = (B * 2 * (int64_t)p.nqb + 3071) / 3072;
    run = run < 1 ? 1 : (run > 32 ? 32 : run);
    p.qbpw = (int)(run > p.nqb ? p.nqb : run);
    p.nwg_b = (p.nqb + p.qbpw - 1) / p.qbpw;
    const int64_t wgs = B * 2 * (int64_t)p.nwg_b;
    if (wgs > lim) return (int)hipErrorInvalidConfiguration;
    const dim3 grid((unsigned)wgs);
    switch (groups) {
      case 1: launch_sx_resident<1>(p, grid, stream); break;
      case 2: launch_sx_resident<2>(p, grid, stream); break;
      case 3: launch_sx_resident<3>(p, grid, stream); break;
      case 4: launch_sx_resident<4>(p, grid, stream); break;
      case 5: launch_sx_resident<5>(p, grid, stream); break;
      case 6: launch_sx_resident<6>(p, grid, stream); break;
      case 7: launch_sx_resident<7>(p, grid, stream); break;
      default: launch_sx_resident<8>(p, grid, stream); break;
    }
    return (int)hipGetLastError();
  }
  // 8 blocks of queries per workgroup, fewer for few queries, with RoPE (its tables take registers) and where the
  // grid's waves would not fill the chip twice; the workgroup's 4 or 8 waves split the keys
  int nbk = p.nqb >= 8 && !p.rope ? 8 : p.nqb > 2 ? 4 : p.nqb;
  const int nw = Lk >= 2048 ? 8 : 4;
  auto wgs = [&](int nb) { return B * SX_H * (int64_t)((p.nqb + nb - 1) / nb); };
  while (nbk > 2 && wgs(nbk) * nw < SX_MIN_WAVES) nbk /= 2;
  p.nwg_b = (p.nqb + nbk - 1) / nbk;
  if (wgs(nbk) > lim) return (int)hipErrorInvalidConfiguration;
  const bool wide = nw == 8 && wgs(nbk) < 2048;
  if (nbk == 8) return wide ? launch_sx_stream<8, 8>(p, stream) : launch_sx_stream<8, 4>(p, stream);
  if (nbk == 4) return wide ? launch_sx_stream<4, 8>(p, stream) : launch_sx_stream<4, 4>(p, stream);
  if (nbk == 2) return wide ? launch_sx_stream<2, 8>(p, stream) : launch_sx_stream<2, 4>(p, stream);
  return wide ? launch_sx_stream<1, 8>(p, stream) : launch_sx_stream<1, 4>(p, stream);
}
