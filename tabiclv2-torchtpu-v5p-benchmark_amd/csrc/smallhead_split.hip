// fp32 small-head attention (8 heads x 16 dims), scores on the bf16 matrix units through exact splits
// (split.h), probabilities and values in fp32. Per 16-key x 16-query tile of a head:
//
//   x = K (q' log2e) - m   three v_mfma_f32_16x16x32_bf16: the 32-deep contraction holds two of the six
//                          split products of the same 16 dims: [Kl | Kh] [qh | ql], [Kh | Km] [qm | qm],
//                          [Kh | Km] [qh | qh] (the smallest first); 48 cycles where fp32 MFMA takes 128
//   p = exp2(x), l += p, O^T += V^T P^T  in fp32 (four v_mfma_f32_16x16x4_f32: splitting every p would cost
//                          more VALU than the matrix cycles it saves)
//
// m is a softmax reference fixed by the first 16 keys (their ceiled maximum); a row sum outside
// [2^-64, 2^96] or a non-finite O (a score far above m, every key masked, NaN or inf in the inputs, which the
// splits turn into NaN) sends the wave's block through the exact online softmax on fp32 MFMA.
// A wave is one head; operands come straight from global memory into registers (a head's 64 bytes of a row;
// the waves of a row's other heads run beside it and share the cache lines), no LDS and no barrier in the
// sweep.
//
// sx_resident_kernel: up to 16 NG keys held in registers (12 per 16 keys), any run of query blocks.
// sx_stream_kernel: 16 NB queries held in registers, keys streamed; a workgroup's waves take a part of the
// keys each and merge at the end.
#include <atomic>

#include "common.h"
#include "launch.h"
#include "split.h"

namespace {

constexpr int SX_H = 8, SX_D = 16, SX_E = 128;
constexpr int SX_SEG = 65536;  // groups (1M keys)
constexpr float SX_LAZY = 8.0f;
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

// Eight dims j0 .. j0 + 7 (j0 = 0 or 8) of a head row after RoPE: y the raw dims (the other eight are with lane
// l ^ 16), t the cos and sin of the position at those dims; rs / off: the head row in its resource, for the
// partner dims of the other forms.
struct SxTab { f32x4 c[2], s[2]; };
__device__ __forceinline__ SxTab sx_tab(const float* cs, const float* sn, int j0) {
  SxTab t;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    t.c[i] = *(const f32x4*)(cs + j0 + 4 * i);
    t.s[i] = *(const f32x4*)(sn + j0 + 4 * i);
  }
  return t;
}
__device__ __forceinline__ void sx_rope8(const SxParams& p, f32x4 (&y)[2], const SxTab& t, __amdgpu_buffer_rsrc_t rs,
                                         int off, int j0) {
  f32x4 out[2];
  if (p.rope == 2 && p.half == 8) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float pt = __uint_as_float(__builtin_amdgcn_ds_swizzle(__float_as_uint(y[i][r]), 0x401f));  // lane ^ 16
        out[i][r] = y[i][r] * t.c[i][r] + (j0 ? pt : -pt) * t.s[i][r];
      }
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        int pt;
        float sg;
        rope_partner(j0 + 4 * i + r, p.rope, p.half, p.rot, &pt, &sg);
        out[i][r] = y[i][r] * t.c[i][r] + sg * sx_ld1(rs, off + pt * 4) * t.s[i][r];
      }
  }
  y[0] = out[0];
  y[1] = out[1];
}

__device__ __forceinline__ f32x4 sx_mm(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// A key row's two score operands and a query's three (lo: this lane holds the contraction's first half).
struct SxK { bf16x8 hm, lh; };
struct SxQ { bf16x8 h, m, hl; };
__device__ __forceinline__ SxK sx_kop(const f32x4 (&y)[2], bool lo) {
  const Split8 s = split8(y[0], y[1]);
  return {lo ? s.h : s.m, lo ? s.l : s.h};
}
__device__ __forceinline__ SxQ sx_qop(const f32x4 (&y)[2], bool lo) {
  const Split8 s = split8(y[0], y[1]);
  return {s.h, s.m, lo ? s.h : s.l};
}
__device__ __forceinline__ f32x4 sx_score(const SxK& k, const SxQ& q, f32x4 init) {
  return sx_mm(k.hm, q.h, sx_mm(k.hm, q.m, sx_mm(k.lh, q.hl, init)));
}

// The softmax reference of a block from its first 16 keys' scores (log2 units).
__device__ __forceinline__ float sx_ref(f32x4 x) {
  const float tm = quad_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
  return tm > -1e4f ? fminf(ceilf(tm), 1e4f) : 0.f;  // -inf and NaN: 0
}

__device__ __forceinline__ bool sx_suspect(f32x4 o, float l) {
  bool bad = !(l >= 0x1p-64f && l <= 0x1p96f);
#pragma unroll
  for (int r = 0; r < 4; ++r) bad |= !(__builtin_fabsf(o[r]) <= 0x1p127f);
  return bad;
}

// b2 of keys k0 .. k0 + 3 in log2 units: the mask, -inf from lk on.
__device__ __forceinline__ f32x4 sx_b2(const SxParams& p, int b, int k0, int lk) {
  f32x4 b2;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int key = k0 + r;
    b2[r] = key < lk ? 0.f : TA_NEG_INF;
    if (p.bias && key < lk) b2[r] = fmaxf(p.bias[b * p.bias_sb + key] * TA_LOG2E, SX_BIAS_FLOOR);
  }
  return b2;
}

// q' = rope(q) scale of 4 dims d0.. of a query (fp32 layout of the exact pass); zero past Lq.
__device__ __forceinline__ f32x4 sx_q4(const SxParams& p, int b, int qi, int d0) {
  if (qi >= p.Lq) return f32x4{0.f, 0.f, 0.f, 0.f};
  const float* row = p.q + b * p.q_sb + (int64_t)qi * p.q_sr;
  f32x4 y = p.rope ? rope4<float>(row, p.cq + (int64_t)qi * p.tab_sr, p.sq + (int64_t)qi * p.tab_sr, d0, p.rope,
                                  p.half, p.rot, d0 & (p.tab_sr - 1))
                   : *(const f32x4*)(row + d0);
#pragma unroll
  for (int r = 0; r < 4; ++r) y[r] *= p.scale;
  return y;
}

// The exact online softmax of one block over keys [16 kt0, 16 kt1), fp32 MFMA, operands from memory (rare).
__device__ __forceinline__ void sx_exact(const SxParams& p, int b, int qi, int head, int kt0, int kt1, int lk,
                                                   int l16, int kap, f32x4& o, float& m, float& l) {
  const int d0 = head * SX_D + 4 * kap;
  const f32x4 q = sx_q4(p, b, qi, d0);
  o = f32x4{0.f, 0.f, 0.f, 0.f};
  m = TA_NEG_INF;
  l = 0.f;
#pragma unroll 1
  for (int kt = kt0; kt < kt1; ++kt) {
    const int key = 16 * kt + l16, kc = key < lk ? key : lk - 1;
    const float* krow = p.k + b * p.k_sb + (int64_t)kc * p.k_sr;
    f32x4 a = p.rope ? rope4<float>(krow, p.ck + (int64_t)kc * p.tab_sr, p.sk + (int64_t)kc * p.tab_sr, d0, p.rope,
                                    p.half, p.rot, d0 & (p.tab_sr - 1))
                     : *(const f32x4*)(krow + d0);
    if (key >= lk) a = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 x = mfma16x16x16(a, q, f32x4{0.f, 0.f, 0.f, 0.f}), va;
    const f32x4 b2 = sx_b2(p, b, 16 * kt + 4 * kap, lk);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      x[r] = fmaf(x[r], TA_LOG2E, b2[r]);
      const int vk = 16 * kt + 4 * kap + r;
      va[r] = vk < lk ? p.v[b * p.v_sb + (int64_t)vk * p.v_sr + head * SX_D + l16] : 0.f;
    }
    const float m_new = fmaxf(m, quad_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]))));
    if (wave_any(m_new - m > SX_LAZY)) {
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
    o = mfma16x16x16(va, pv, o);
  }
}

// NG: 16-key groups held (above 8, the last may be wholly past Lk); MF: 0 a mask or per-batch lengths (b2 added
// to every tile, from LDS), 1 the end of the last groups is past Lk. Workgroup = 4 heads of (batch element, run of
// query blocks).
template <int NG, int MF, bool ROPE>
__global__ __launch_bounds__(256, (ROPE || MF == 0) ? (NG <= 1 ? 4 : NG <= 3 ? 3 : 2) : (NG <= 2 ? 4 : NG <= 6 ? 3 : 2)) void sx_resident_kernel(SxParams p) {
  __shared__ __attribute__((aligned(16))) float lb2[MF == 0 ? NG * 16 : 4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, kap = lane >> 4;
  const int work = xcd_remap(blockIdx.x, gridDim.x);
  const int head = (work & 1) * 4 + wave, rest = work >> 1;
  const int b = rest / p.nwg_b, qb0 = (rest % p.nwg_b) * p.qbpw;
  const int nb = p.nqb - qb0 < p.qbpw ? p.nqb - qb0 : p.qbpw;
  const int lk = MF == 0 ? sx_lk(p, b) : p.Lk;
  const int j0 = 8 * (kap & 1), hc = head * SX_D;
  const bool lo = kap < 2;
  const int tc = hc & (p.tab_sr - 1);
  // keys from lk on read as zero (the resource ends at row lk - 1; without keys a row is read and masked)
  const int lr = MF == 0 ? (lk > 0 ? lk : 1) : lk;
  const __amdgpu_buffer_rsrc_t krs = sx_rsrc(p.k + b * p.k_sb + hc, lr, p.k_sr);
  const __amdgpu_buffer_rsrc_t vrs = sx_rsrc(p.v + b * p.v_sb + hc, lr, p.v_sr);
  const int q0 = qb0 * 16, qrows = p.Lq - q0 < nb * 16 ? p.Lq - q0 : nb * 16;
  const __amdgpu_buffer_rsrc_t qrs = sx_rsrc(p.q + b * p.q_sb + (int64_t)q0 * p.q_sr + hc, qrows, p.q_sr);
  const int ksr = (int)p.k_sr * 4, vsr = (int)p.v_sr * 4, qsr = (int)p.q_sr * 4;
  f32x4 qy[2], ky[NG][2], va[NG];
#pragma unroll
  for (int kt = 0; kt < NG; ++kt)
#pragma unroll
    for (int i = 0; i < 2; ++i) ky[kt][i] = sx_ld4(krs, (16 * kt + l16) * ksr + (j0 + 4 * i) * 4);
#pragma unroll
  for (int i = 0; i < 2; ++i) qy[i] = sx_ld4(qrs, l16 * qsr + (j0 + 4 * i) * 4);
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
      const int key = 16 * kt + l16, kc = key < p.Lk ? key : p.Lk - 1;
      return sx_tab(p.ck + (int64_t)kc * p.tab_sr + tc, p.sk + (int64_t)kc * p.tab_sr + tc, j0);
    };
    SxTab t = tab(0);
#pragma unroll
    for (int kt = 0; kt < NG; ++kt) {
      const SxTab tn = kt + 1 < NG ? tab(kt + 1) : t;
      sx_rope8(p, ky[kt], t, krs, (16 * kt + l16) * ksr, j0);
      kop[kt] = sx_kop(ky[kt], lo);
      t = tn;
      __builtin_amdgcn_sched_barrier(0);  // one group's tables ahead, not all of them
    }
  } else {
#pragma unroll
    for (int kt = 0; kt < NG; ++kt) kop[kt] = sx_kop(ky[kt], lo);
  }
  const float qc = p.scale;
  for (int bi = 0; bi < nb; ++bi) {
    const int ql = bi * 16 + l16, qi = q0 + ql;
    f32x4 y[2] = {qy[0], qy[1]};
    if (bi + 1 < nb) {
#pragma unroll
      for (int i = 0; i < 2; ++i) qy[i] = sx_ld4(qrs, (ql + 16) * qsr + (j0 + 4 * i) * 4);
    }
    if constexpr (ROPE) {
      const int qt = qi < p.Lq ? qi : p.Lq - 1;
      const SxTab t = sx_tab(p.cq + (int64_t)qt * p.tab_sr + tc, p.sq + (int64_t)qt * p.tab_sr + tc, j0);
      sx_rope8(p, y, t, qrs, ql * qsr, j0);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) y[i][r] = y[i][r] * qc * TA_LOG2E;
    const SxQ q = sx_qop(y, lo);
    f32x4 o0 = {0.f, 0.f, 0.f, 0.f}, o1 = o0;
    float l = 0.f, m = 0.f;
    auto mask = [&](f32x4 x, int kt) {
      if constexpr (MF == 0) {
        const f32x4 b2 = *(const f32x4*)(lb2 + 16 * kt + 4 * kap);
        x += b2;
      } else if (kt >= NG - (NG > 8 ? 2 : 1)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = 16 * kt + 4 * kap + r < lk ? x[r] : TA_NEG_INF;
      }
      return x;
    };
    // scores one group ahead of the exponentials and value products
    f32x4 x = mask(sx_score(kop[0], q, f32x4{0.f, 0.f, 0.f, 0.f}), 0);
    m = sx_ref(x);
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] -= m;
    const f32x4 minit = {-m, -m, -m, -m};
#pragma unroll
    for (int kt = 0; kt < NG; ++kt) {
      f32x4 xn;
      if (kt + 1 < NG) xn = mask(sx_score(kop[kt + 1 < NG ? kt + 1 : kt], q, minit), kt + 1);
      f32x4 pv;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pv[r] = __builtin_amdgcn_exp2f(x[r]);
        l += pv[r];
      }
      if (kt & 1) o1 = mfma16x16x16(va[kt], pv, o1);
      else o0 = mfma16x16x16(va[kt], pv, o0);
      x = xn;
    }
    f32x4 o = o0 + o1;
    if (wave_any(sx_suspect(o, l)) && lk > 0) sx_exact(p, b, qi, head, 0, (lk + 15) >> 4, lk, l16, kap, o, m, l);
    const float lt = quad_sum(l), inv = lt > 0.f ? 1.f / lt : 0.f;
    if (qi < p.Lq) {
      f32x4 out;
#pragma unroll
      for (int r = 0; r < 4; ++r) out[r] = MF == 0 && lk == 0 ? 0.f : o[r] * inv;
      *(f32x4*)(p.o + ((int64_t)b * p.Lq + qi) * SX_E + hc + 4 * kap) = out;
    }
  }
}

// Wave w of NW takes the w-th part of the keys for the workgroup's NB query blocks of one head; merged in LDS.
template <int NB, int NW, bool BIAS, bool ROPE>
__global__ __launch_bounds__(NW * 64, 2) void sx_stream_kernel(SxParams p) {
  extern __shared__ __attribute__((aligned(16))) float lds[];  // per wave and block: O [4][64], m [64], l [64]
  __shared__ int bad_flag;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, kap = lane >> 4;
  const int work = xcd_remap(blockIdx.x, gridDim.x);
  const int head = work % SX_H, rest = work / SX_H;
  const int b = rest / p.nwg_b, q0 = (rest % p.nwg_b) * NB * 16;
  const int lk = sx_lk(p, b), ng = (lk + 15) >> 4, per = (ng + NW - 1) / NW;
  const int g0 = wave * per < ng ? wave * per : ng, g1 = g0 + per < ng ? g0 + per : ng;
  const int j0 = 8 * (kap & 1), hc = head * SX_D, tc = hc & (p.tab_sr - 1);
  const bool lo = kap < 2;
  SxQ q[NB];
  f32x4 o[NB];
  float m[NB], l[NB];
  const int nrow = p.Lq - q0 < NB * 16 ? p.Lq - q0 : NB * 16;
  const __amdgpu_buffer_rsrc_t qrs = sx_rsrc(p.q + b * p.q_sb + (int64_t)q0 * p.q_sr + hc, nrow, p.q_sr);
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int off = (16 * j + l16) * (int)p.q_sr * 4;  // past Lq: zeros
    f32x4 y[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) y[i] = sx_ld4(qrs, off + (j0 + 4 * i) * 4);
    if constexpr (ROPE) {
      const int qi = q0 + 16 * j + l16, qt = qi < p.Lq ? qi : p.Lq - 1;
      const SxTab t = sx_tab(p.cq + (int64_t)qt * p.tab_sr + tc, p.sq + (int64_t)qt * p.tab_sr + tc, j0);
      sx_rope8(p, y, t, qrs, off, j0);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) y[i][r] = y[i][r] * p.scale * TA_LOG2E;
    q[j] = sx_qop(y, lo);
    o[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    m[j] = TA_NEG_INF;
    l[j] = 0.f;
    __builtin_amdgcn_sched_barrier(0);
  }
  if (threadIdx.x == 0) bad_flag = 0;
  // the part's rows as a resource, SX_SEG groups at a time (32-bit offsets); rows past lk read as zero
  bool first = true;
#pragma unroll 1
  for (int s0 = g0; s0 < g1; s0 += SX_SEG) {
    const int s1 = g1 - s0 < SX_SEG ? g1 : s0 + SX_SEG;
    const int row0 = s0 * 16, rows = lk - row0 < (s1 - s0) * 16 ? lk - row0 : (s1 - s0) * 16;
    const __amdgpu_buffer_rsrc_t krs = sx_rsrc(p.k + b * p.k_sb + (int64_t)row0 * p.k_sr + hc, rows, p.k_sr);
    const __amdgpu_buffer_rsrc_t vrs = sx_rsrc(p.v + b * p.v_sb + (int64_t)row0 * p.v_sr + hc, rows, p.v_sr);
    const int ksr = (int)p.k_sr * 4, vsr = (int)p.v_sr * 4;
    f32x4 ky[2], vy, kz[2], vz;  // this group's rows and the next one's, in flight
    auto fetch = [&](int g, f32x4 (&kk)[2], f32x4& vv) {
#pragma unroll
      for (int i = 0; i < 2; ++i) kk[i] = sx_ld4(krs, (16 * g + l16) * ksr + (j0 + 4 * i) * 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) vv[j] = sx_ld1(vrs, (16 * g + 4 * kap + j) * vsr + l16 * 4);
    };
    auto tab = [&](int g) {
      const int key = 16 * (s0 + g) + l16, kc = key < p.Lk ? key : p.Lk - 1;
      return sx_tab(p.ck + (int64_t)kc * p.tab_sr + tc, p.sk + (int64_t)kc * p.tab_sr + tc, j0);
    };
    SxTab ty, tz;
    fetch(0, ky, vy);
    if constexpr (ROPE) ty = tab(0);
    fetch(1, kz, vz);  // past the last group: zeros, unused
    if constexpr (ROPE) tz = tab(1);
#pragma unroll 1
    for (int g = 0; g < s1 - s0; ++g) {
      if constexpr (ROPE) {
        sx_rope8(p, ky, ty, krs, (16 * g + l16) * ksr, j0);
        ty = tz;
        tz = tab(g + 2);
      }
      const SxK k = sx_kop(ky, lo);
      const f32x4 va = vy;
      ky[0] = kz[0];
      ky[1] = kz[1];
      vy = vz;
      fetch(g + 2, kz, vz);
      const bool tail = 16 * (s0 + g) + 16 > lk;
      f32x4 b2 = {0.f, 0.f, 0.f, 0.f};
      if (BIAS || tail) b2 = sx_b2(p, b, 16 * (s0 + g) + 4 * kap, lk);
      if (first) {
        first = false;
#pragma unroll
        for (int j = 0; j < NB; ++j) m[j] = sx_ref(sx_score(k, q[j], f32x4{0.f, 0.f, 0.f, 0.f}) + b2);
      }
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        f32x4 x = sx_score(k, q[j], f32x4{-m[j], -m[j], -m[j], -m[j]});
        if (BIAS || tail) x += b2;
        f32x4 pv;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          pv[r] = __builtin_amdgcn_exp2f(x[r]);
          l[j] += pv[r];
        }
        o[j] = mfma16x16x16(va, pv, o[j]);
      }
    }
  }
  if (g0 < g1) {
    bool bad = false;
#pragma unroll
    for (int j = 0; j < NB; ++j) bad |= sx_suspect(o[j], l[j]);
    if (wave_any(bad) && lane == 0) bad_flag = 1;
  }
  __syncthreads();
  if (bad_flag && g0 < g1) {  // rare: every wave redoes its part with the exact online softmax
    float* dst = lds + wave * NB * 384;
#pragma unroll 1
    for (int j = 0; j < NB; ++j, dst += 384) {
      f32x4 oj;
      float mj, lj;
      sx_exact(p, b, q0 + 16 * j + l16, head, g0, g1, lk, l16, kap, oj, mj, lj);
      *(f32x4*)(dst + lane * 4) = oj;
      dst[256 + lane] = mj;
      dst[320 + lane] = lj;
    }
  } else {
    float* dst = lds + wave * NB * 384;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      *(f32x4*)(dst + j * 384 + lane * 4) = o[j];
      dst[j * 384 + 256 + lane] = m[j];
      dst[j * 384 + 320 + lane] = l[j];
    }
  }
  __syncthreads();
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

template <int NG>
void launch_sx_resident(const SxParams& p, dim3 grid, hipStream_t stream) {
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
  if (groups <= 12) {
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
      case 8: launch_sx_resident<8>(p, grid, stream); break;
      case 9:
      case 10: launch_sx_resident<10>(p, grid, stream); break;
      default: launch_sx_resident<12>(p, grid, stream); break;
    }
    return (int)hipGetLastError();
  }
  // 8 blocks of queries per workgroup (fewer for few queries, and with RoPE, whose tables take registers); the
  // workgroup's waves split the keys, more of them when there are few workgroups
  const int nbk = p.nqb >= 8 && !p.rope ? 8 : p.nqb > 2 ? 4 : p.nqb;
  p.nwg_b = (p.nqb + nbk - 1) / nbk;
  const int64_t wgs = B * SX_H * (int64_t)p.nwg_b;
  if (wgs > lim) return (int)hipErrorInvalidConfiguration;
  const bool wide = wgs < 1024 && Lk >= 2048;
  if (nbk == 8) return wide ? launch_sx_stream<8, 8>(p, stream) : launch_sx_stream<8, 4>(p, stream);
  if (nbk == 4) return wide ? launch_sx_stream<4, 8>(p, stream) : launch_sx_stream<4, 4>(p, stream);
  if (nbk == 2) return wide ? launch_sx_stream<2, 8>(p, stream) : launch_sx_stream<2, 4>(p, stream);
  return wide ? launch_sx_stream<1, 8>(p, stream) : launch_sx_stream<1, 4>(p, stream);
}
