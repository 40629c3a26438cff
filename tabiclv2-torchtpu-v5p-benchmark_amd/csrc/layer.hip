// Pre-norm encoder layers of width 128 (feed-forward 256, GELU) around the small-head attention: the column
// and row blocks of a cached query. Two kernels hold everything of a layer that is not attention:
//
//   el_proj_kernel   y = LN1(x) W^T + b                       (q, k|v or q|k|v projection)
//   el_tail_kernel   s = x + a Wo^T + bo;  out = s + W2 gelu(W1 LN2(s) + b1) + b2
//
// per row of 128 values, bf16 or fp32 (nothing of fp32 accuracy is rounded below it: fp32 MFMA, or the ex_*
// kernels' exact three-way bf16 splits). In separate launches
// these are GEMMs, LayerNorms, activations and adds that each read and write the [rows, 128] or [rows, 256]
// tensors: 13 passes over memory for the tail in place of three (read a and x, write out).
//
// Layout. A wave owns 32 rows and computes the transposed products Y^T = W X^T with 32x32 MFMA tiles
// (A = weights, B = activations): the result of a product has a row of x on each lane pair (l, l ^ 32) and its
// features in registers, so LayerNorm is a sum over registers and one lane swap, and a product's result is the
// next product's B operand without leaving the lane. W's rows enter the tile in the order el_perm so that lane
// half h holds features 16 s + 8 h + 0..7 of each 16: contiguous 16 / 32-byte pieces of a row of x or out.
//
// Weights stream through LDS in steps of 16 KB (32 fp32 or 64 bf16 output features of a K = 128 product; 128
// bytes of all 128 rows of W2; the ex_* kernels' split image 24 KB), copied by the load unit two steps ahead into a
// ring of three buffers shared by the workgroup's four waves; 16-byte chunks XOR-swizzled by row, so that the 16
// lanes that read together hit all banks. A 128-row workgroup of the tail reads its weights from L2 once: 160 KB in
// bf16, in fp32 the 480 KB of the split image (20 steps).
//
// Measured at 4.16M rows (8 x 104 columns of 5000 rows). fp32: tail 4.1 ms (6.5 ms with fp32 MFMA, 14.6 ms as
// separate launches), projection to 128 features 1.17 ms (1.32, 2.4), to 384 2.64 ms; the tail's matrix cores are
// busy 52% and its VALU about as long (LN, splits, GELU), at 1.78 GHz. bf16: tail 1.39 ms, projections 0.49 and
// 1.00 ms (to 384: 4.3 TB/s). Column stage of that size, fp32: 55.6 -> 27.0 ms.
#include "common.h"
#include "launch.h"
#include "layer.h"
#include "split.h"

namespace {

constexpr int EL_W = 128, EL_FF = 256;
constexpr int EL_NW = 4, EL_ROWS = 32 * EL_NW;
constexpr int EL_STEP = 16384, EL_RING = 3;
constexpr int EL_IPW = EL_STEP / (EL_NW * 1024);  // copies of 1 KB per wave and step

template <typename T> struct El {
  static constexpr int RB = EL_W * (int)sizeof(T);       // bytes of a 128-value row
  static constexpr int OUTS = EL_STEP / RB;              // output features per wide step
  static constexpr int NB = OUTS / 32;                   // 32-feature tiles per wide step
  static constexpr int FFC = 128 / (int)sizeof(T);       // feed-forward features per W2 step (= OUTS)
};

// B operand of a 128-deep (X) or one step's FFC-deep (G) product: fp32 the values, bf16 in eights.
template <typename T> struct ElOp;
template <> struct ElOp<float> { float v[64]; };
template <> struct ElOp<bf16> { bf16x8 v[8]; };

// Copy one step of weights into the ring buffer at LDS address dst: 16 KB of whole 128-value rows ...
template <typename T> __device__ __forceinline__ void el_copy_wide(const void* src, uint32_t dst, int w, int lane) {
  constexpr int CPR = El<T>::RB / 16;
#pragma unroll
  for (int i = 0; i < EL_IPW; ++i) {
    const int c0 = (w * EL_IPW + i) * 64;
    const int p = c0 + lane, row = p / CPR, pos = p % CPR;
    lds_dma16_s((uint32_t)(row * El<T>::RB + ((pos ^ (row & 15)) << 4)), src, dst + c0 * 16);
  }
}
// ... or 128 bytes of each of the 128 rows (stride 256 values) of W2.
__device__ __forceinline__ void el_copy_w2(const void* src, uint32_t dst, int w, int lane) {
#pragma unroll
  for (int i = 0; i < EL_IPW; ++i) {
    const int c0 = (w * EL_IPW + i) * 64;
    const int p = c0 + lane, row = p >> 3, pos = p & 7;
    lds_dma16_s((uint32_t)(row * EL_FF * 2 + ((pos ^ ((row >> 1) & 7)) << 4)), src, dst + c0 * 16);
  }
}

// One 32-feature tile of a K = 128 product: acc += W[tile] X^T; rb = this lane's swizzled row address
// (el_wide_base) plus the tile's offset.
__device__ __forceinline__ void el_mm_wide(f32x16& acc, const char* buf, uint32_t rb, const ElOp<float>& x) {
  // i: the 16 chunks of this lane half (bit 1 of a chunk's index is the half's); weights two reads ahead
  auto rd = [&](int i) { return *(const f32x4*)(buf + (rb ^ ((((i & ~1) << 1) | (i & 1)) << 4))); };
  f32x4 w0 = rd(0), w1 = rd(1);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    f32x4 w2 = w1;
    if (i + 2 < 16) w2 = rd(i + 2);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(w0[j], x.v[4 * i + j], acc, 0, 0, 0);
    w0 = w1;
    w1 = w2;
    __builtin_amdgcn_sched_barrier(0);  // further reads hoisted here would cost registers
  }
}
__device__ __forceinline__ void el_mm_wide(f32x16& acc, const char* buf, uint32_t rb, const ElOp<bf16>& x) {
#pragma unroll
  for (int kk = 0; kk < 8; ++kk)
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(buf + (rb ^ (kk << 5))), x.v[kk], acc, 0, 0, 0);
}
template <typename T> __device__ __forceinline__ uint32_t el_wide_base(int prow, int hh) {
  return (uint32_t)(prow * El<T>::RB + (((hh << (sizeof(T) == 4 ? 1 : 0)) ^ (prow & 15)) << 4));
}

// One 32-feature tile of a W2 step: acc += W2[tile, step's 64 columns] G^T (g: the step's activations).
__device__ __forceinline__ void el_mm_w2(f32x16& acc, const char* buf, uint32_t rb, const ElOp<bf16>& g) {
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(buf + (rb ^ (kk << 5))), g.v[kk], acc, 0, 0, 0);
}
__device__ __forceinline__ uint32_t el_w2_base(int prow, int hh) {
  return (uint32_t)(prow * 128 + ((hh ^ ((prow >> 1) & 7)) << 4));
}

__device__ __forceinline__ float el_pair_sum(float x) {
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Eight consecutive values of a row (byte offset off in the resource; past its end: 0) as fp32.
template <typename T> __device__ __forceinline__ void el_load8(__amdgpu_buffer_rsrc_t rs, int off, float* v) {
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const f32x4 c = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off + 16 * i, 0, 0));
#pragma unroll
      for (int j = 0; j < 4; ++j) v[4 * i + j] = c[j];
    }
  } else {
    const bf16x8 c = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (float)c[j];
  }
}
// Eight consecutive values to a row (dropped past the resource's end: every lane stores, so that the number of
// outstanding memory operations is the same in every wave).
template <typename T> __device__ __forceinline__ void el_store8(__amdgpu_buffer_rsrc_t rs, int off, const float* v) {
  typedef uint32_t u32v4 __attribute__((ext_vector_type(4)));
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_raw_buffer_store_b128(
          __builtin_bit_cast(u32v4, f32x4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]}), rs, off + 16 * i, 0, 0);
  } else {
    const uint2 lo = __builtin_bit_cast(uint2, cvt_bf16x4(f32x4{v[0], v[1], v[2], v[3]}));
    const uint2 hi = __builtin_bit_cast(uint2, cvt_bf16x4(f32x4{v[4], v[5], v[6], v[7]}));
    __builtin_amdgcn_raw_buffer_store_b128(u32v4{lo.x, lo.y, hi.x, hi.y}, rs, off, 0, 0);
  }
}

// LayerNorm of the row held by a lane pair: mean and 1 / sqrt(var + eps) of v (this lane's 64 of the 128 values,
// in two passes), then the normalised values 4 i .. 4 i + 3 (lw / lb: weight and bias in LDS).
struct ElNorm { float mean, rstd; };
template <typename V> __device__ __forceinline__ ElNorm el_stats(V v, float eps) {
  const float mean = el_pair_sum(el_sum<64>(v, 0)) * (1.0f / EL_W);
  float q[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 64; ++i) {
    const float d = v(i) - mean;
    q[i & 3] = __builtin_fmaf(d, d, q[i & 3]);
  }
  return {mean, __builtin_amdgcn_rsqf(el_pair_sum((q[0] + q[1]) + (q[2] + q[3])) * (1.0f / EL_W) + eps)};
}
template <typename V>
__device__ __forceinline__ f32x4 el_normed(V v, int i, ElNorm n, const float* lw, const float* lb, int hh) {
  const int f = 16 * (i >> 1) + 8 * hh + 4 * (i & 1);
  const f32x4 ww = *(const f32x4*)(lw + f), bb = *(const f32x4*)(lb + f);
  f32x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = __builtin_fmaf((v(4 * i + j) - n.mean) * n.rstd, ww[j], bb[j]);
  return o;
}

// The operand from its values 4 i .. 4 i + 3 (x(i), i < 16).
template <typename X> __device__ __forceinline__ void el_operand(X x, ElOp<float>& o) {
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const f32x4 c = x(i);
#pragma unroll
    for (int j = 0; j < 4; ++j) o.v[4 * i + j] = c[j];
  }
}
template <typename X> __device__ __forceinline__ void el_operand(X x, ElOp<bf16>& o) {
#pragma unroll
  for (int k = 0; k < 8; ++k) o.v[k] = el_pack8(x(2 * k), x(2 * k + 1));
}

// acc = the 32-feature tile of a bias vector in LDS, on every row.
__device__ __forceinline__ void el_bias(f32x16& acc, const float* b, int hh) {
#pragma unroll
  for (int i = 0; i < 16; i += 4) {
    const f32x4 bb = *(const f32x4*)(b + 16 * (i >> 3) + 8 * hh + (i & 7));
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i + j] = bb[j];
  }
}

template <typename T> __device__ __forceinline__ float el_param(const T* b, int i) { return b ? (float)b[i] : 0.f; }

// Join the workgroup with at most 4 k (k = 0..3) of this wave's memory operations outstanding.
__device__ __forceinline__ void el_join(int k) {
  if (k >= 3) TA_WAIT_JOIN(12);
  else if (k == 2) TA_WAIT_JOIN(8);
  else if (k == 1) TA_WAIT_JOIN(4);
  else TA_WAIT_JOIN(0);
}

struct ElParams {
  const void *a, *x;                         // attention output and residual stream [rows, 128]
  const float *ln_w, *ln_b;                  // [128] (null: 1 / 0)
  const void *wo, *bo, *w1, *b1, *w2, *b2;   // el_proj: w1 [N, 128], b1 [N]
  void* out;
  int* live;        // per group of group_rows rows: nonzero if a value differs from `skip` (null: not asked)
  uint32_t group_rows;
  float eps, skip;
  int64_t rows;
  int n_out, steps_per_wg;  // el_proj
};

// A tail workgroup's skip rule: keep = this lane's row belongs to a live group; true (uniform) where the tile
// holds nothing but skipped rows, whose output is then written.
template <typename T>
__device__ __forceinline__ bool el_skip_tile(const ElParams& p, int64_t row0, int nrow, int row, __amdgpu_buffer_rsrc_t ors,
                                             int xoff, bool& keep) {
  keep = true;
  if (!p.live) return false;
  keep = p.live[((uint32_t)row0 + (row < nrow ? row : nrow - 1)) / p.group_rows] != 0;
  const uint32_t g0 = (uint32_t)row0 / p.group_rows, g1 = (uint32_t)(row0 + nrow - 1) / p.group_rows;
  for (uint32_t g = g0; g <= g1; ++g)
    if (p.live[g] != 0) return false;
  float o[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = p.skip;
#pragma unroll
  for (int i = 0; i < 8; ++i) el_store8<T>(ors, xoff + i * 16 * (int)sizeof(T), o);
  return true;
}

// The tail's vectors into LDS: bo, LN2 weight and bias, b2, b1.
template <typename T> __device__ __forceinline__ void el_tail_params(const ElParams& p, float* prm) {
  for (int i = threadIdx.x; i < EL_FF; i += EL_NW * 64) {
    if (i < EL_W) {
      prm[i] = el_param((const T*)p.bo, i);
      prm[EL_W + i] = p.ln_w ? p.ln_w[i] : 1.f;
      prm[2 * EL_W + i] = p.ln_b ? p.ln_b[i] : 0.f;
      prm[3 * EL_W + i] = el_param((const T*)p.b2, i);
    }
    prm[4 * EL_W + i] = el_param((const T*)p.b1, i);
  }
}

// grid (row tiles, step groups): workgroup (i, j) projects rows [128 i, 128 i + 128) to its steps' features.
template <typename T> __global__ __launch_bounds__(EL_NW * 64, sizeof(T) == 4 ? 2 : 3) void el_proj_kernel(ElParams p) {
  __shared__ __attribute__((aligned(512))) char ring[EL_RING * EL_STEP];
  __shared__ __attribute__((aligned(16))) float prm[2 * EL_W + 3 * EL_W];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, m = lane & 31, hh = lane >> 5;
  const int64_t row0 = (int64_t)blockIdx.x * EL_ROWS;
  const int nrow = (int)(p.rows - row0 < EL_ROWS ? p.rows - row0 : EL_ROWS);
  const int s0 = blockIdx.y * p.steps_per_wg;
  const int nsteps = p.n_out / El<T>::OUTS;
  const int S = nsteps - s0 < p.steps_per_wg ? nsteps - s0 : p.steps_per_wg;
  const uint32_t ring0 = lds_addr(ring);
  const char* wsrc = (const char*)p.w1 + (int64_t)s0 * EL_STEP;
  el_copy_wide<T>(wsrc, ring0, w, lane);
  if (S > 1) el_copy_wide<T>(wsrc + EL_STEP, ring0 + EL_STEP, w, lane);

  const __amdgpu_buffer_rsrc_t xrs =
      __builtin_amdgcn_make_buffer_rsrc((T*)p.x + row0 * EL_W, 0, nrow * El<T>::RB, TA_BUF_WORD3);
  const int xoff = (w * 32 + m) * El<T>::RB + hh * 8 * (int)sizeof(T);
  float v[64];
#pragma unroll
  for (int i = 0; i < 8; ++i) el_load8<T>(xrs, xoff + i * 16 * (int)sizeof(T), v + 8 * i);
  for (int i = threadIdx.x; i < EL_W; i += EL_NW * 64) {
    prm[i] = p.ln_w ? p.ln_w[i] : 1.f;
    prm[EL_W + i] = p.ln_b ? p.ln_b[i] : 0.f;
  }
  for (int i = threadIdx.x; i < S * El<T>::OUTS; i += EL_NW * 64)
    prm[2 * EL_W + i] = el_param((const T*)p.b1, s0 * El<T>::OUTS + i);
  if (p.live && blockIdx.y == 0) {
    bool diff = false;
#pragma unroll
    for (int i = 0; i < 64; ++i) diff |= !(v[i] == p.skip);
    diff = diff && w * 32 + m < nrow;
    if (diff) p.live[(uint32_t)(row0 + w * 32 + m) / p.group_rows] = 1;
  }
  TA_JOIN_LDS();
  const auto val = [&](int i) { return v[i]; };
  const ElNorm norm = el_stats(val, p.eps);
  ElOp<T> op;
  el_operand([&](int i) { return el_normed(val, i, norm, prm, prm + EL_W, hh); }, op);

  const __amdgpu_buffer_rsrc_t ors = __builtin_amdgcn_make_buffer_rsrc(
      (T*)p.out + row0 * p.n_out, 0, nrow * p.n_out * (int)sizeof(T), TA_BUF_WORD3);
  const int ooff = ((w * 32 + m) * p.n_out + s0 * El<T>::OUTS + hh * 8) * (int)sizeof(T);
  const uint32_t rb = el_wide_base<T>(el_perm(m), hh);
  int slot = 0;
  for (int s = 0; s < S; ++s) {
    // younger than step s's copies: the next step's copies and the last two steps' stores (4 each)
    el_join((s < S - 1) + (s >= 1) + (s >= 2));
    if (s + 2 < S) {
      const int next = slot == 0 ? 2 : slot - 1;
      el_copy_wide<T>(wsrc + (int64_t)(s + 2) * EL_STEP, ring0 + next * EL_STEP, w, lane);
    }
#pragma unroll
    for (int nb = 0; nb < El<T>::NB; ++nb) {
      f32x16 acc = {}, bias;
      el_mm_wide(acc, ring + slot * EL_STEP, rb + nb * 32 * El<T>::RB, op);
      el_bias(bias, prm + 2 * EL_W + s * El<T>::OUTS + nb * 32, hh);
      acc += bias;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        float o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = acc[8 * i + j];
        el_store8<T>(ors, ooff + (s * El<T>::OUTS + nb * 32 + i * 16) * (int)sizeof(T), o);
      }
    }
    slot = slot == 2 ? 0 : slot + 1;
  }
}

// Two waves per SIMD (221 VGPRs, no spill): 4.16M rows 1.37 ms; bounded to 168 registers for three, 1.46 ms.
__global__ __launch_bounds__(EL_NW * 64, 2) void el_tail_kernel(ElParams p) {
  typedef bf16 T;
  constexpr int NWO = EL_W / El<T>::OUTS, NFF = EL_FF / El<T>::FFC, NS = NWO + 2 * NFF, NB = El<T>::NB;
  constexpr int ES = (int)sizeof(T);
  __shared__ __attribute__((aligned(512))) char ring[EL_RING * EL_STEP];
  __shared__ __attribute__((aligned(16))) float prm[4 * EL_W + EL_FF];
  const float *bo = prm, *lw = prm + EL_W, *lb = prm + 2 * EL_W, *b2 = prm + 3 * EL_W, *b1 = prm + 4 * EL_W;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, m = lane & 31, hh = lane >> 5;
  const int64_t row0 = (int64_t)blockIdx.x * EL_ROWS;
  const int nrow = (int)(p.rows - row0 < EL_ROWS ? p.rows - row0 : EL_ROWS);
  const __amdgpu_buffer_rsrc_t ors =
      __builtin_amdgcn_make_buffer_rsrc((T*)p.out + row0 * EL_W, 0, nrow * El<T>::RB, TA_BUF_WORD3);
  const int xoff = (w * 32 + m) * El<T>::RB + hh * 8 * ES;
  bool keep;
  if (el_skip_tile<T>(p, row0, nrow, w * 32 + m, ors, xoff, keep)) return;
  const uint32_t ring0 = lds_addr(ring);
  // step s: Wo's output features, then W1's features f and W2's columns f in turn
  auto copy_step = [&](int s, int slot) {
    const uint32_t dst = ring0 + slot * EL_STEP;
    if (s < NWO) {
      el_copy_wide<T>((const char*)p.wo + s * EL_STEP, dst, w, lane);
    } else if (((s - NWO) & 1) == 0) {
      el_copy_wide<T>((const char*)p.w1 + ((s - NWO) >> 1) * EL_STEP, dst, w, lane);
    } else {
      el_copy_w2((const char*)p.w2 + ((s - NWO) >> 1) * 128, dst, w, lane);
    }
  };
  copy_step(0, 0);
  copy_step(1, 1);
  const __amdgpu_buffer_rsrc_t ars =
      __builtin_amdgcn_make_buffer_rsrc((T*)p.a + row0 * EL_W, 0, nrow * El<T>::RB, TA_BUF_WORD3);
  const __amdgpu_buffer_rsrc_t xrs =
      __builtin_amdgcn_make_buffer_rsrc((T*)p.x + row0 * EL_W, 0, nrow * El<T>::RB, TA_BUF_WORD3);
  ElOp<T> op;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    op.v[i] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(ars, xoff + i * 16 * ES, 0, 0));
  float sv[64];  // x, then s: feature of register i as in a product's result
#pragma unroll
  for (int i = 0; i < 8; ++i) el_load8<T>(xrs, xoff + i * 16 * ES, sv + 8 * i);
  el_tail_params<T>(p, prm);
  const int prow = el_perm(m);
  const uint32_t rbw = el_wide_base<T>(prow, hh), rb2 = el_w2_base(prow, hh);

  // s = x + a Wo^T + bo
#pragma unroll
  for (int s = 0; s < NWO; ++s) {
    TA_WAIT_JOIN(4);
    copy_step(s + 2, (s + 2) % EL_RING);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      f32x16 y = {}, bias;
      el_mm_wide(y, ring + (s % EL_RING) * EL_STEP, rbw + nb * 32 * El<T>::RB, op);
      el_bias(bias, bo + (s * NB + nb) * 32, hh);
#pragma unroll
      for (int i = 0; i < 16; ++i) sv[(s * NB + nb) * 16 + i] += y[i] + bias[i];
    }
  }
  const auto val = [&](int i) { return sv[i]; };
  const ElNorm norm = el_stats(val, p.eps);
  el_operand([&](int i) { return el_normed(val, i, norm, lw, lb, hh); }, op);
  // out = s + b2 + W2 gelu(W1 LN2(s) + b1), one step of feed-forward features at a time, summed onto s
  f32x16 z[4];
#pragma unroll
  for (int i = 0; i < 64; ++i) z[i >> 4][i & 15] = sv[i];
  int slot = NWO % EL_RING;
  for (int f = 0; f < NFF; ++f) {
    const int s = NWO + 2 * f;
    int next = slot == 0 ? 2 : slot - 1;
    TA_WAIT_JOIN(4);
    if (s + 2 < NS) copy_step(s + 2, next);
    ElOp<T> g;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      f32x16 h = {}, bias;
      el_mm_wide(h, ring + slot * EL_STEP, rbw + nb * 32 * El<T>::RB, op);
      el_bias(bias, b1 + (f * NB + nb) * 32, hh);
      h += bias;
      float t[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) t[i] = el_gelu<T>(h[i]);
#pragma unroll
      for (int k = 0; k < 2; ++k)
        g.v[2 * nb + k] = el_pack8(f32x4{t[8 * k], t[8 * k + 1], t[8 * k + 2], t[8 * k + 3]},
                                   f32x4{t[8 * k + 4], t[8 * k + 5], t[8 * k + 6], t[8 * k + 7]});
    }
    slot = slot == 2 ? 0 : slot + 1;
    next = slot == 0 ? 2 : slot - 1;
    if (s + 2 < NS) {
      TA_WAIT_JOIN(4);
      if (s + 3 < NS) copy_step(s + 3, next);
    } else {
      TA_WAIT_JOIN(0);
    }
#pragma unroll
    for (int ob = 0; ob < 4; ++ob) el_mm_w2(z[ob], ring + slot * EL_STEP, rb2 + ob * 4096, g);
    slot = slot == 2 ? 0 : slot + 1;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = 8 * i + j;
      o[j] = keep ? z[r >> 4][r & 15] + b2[16 * i + 8 * hh + j] : p.skip;
    }
    el_store8<T>(ors, xoff + i * 16 * ES, o);
  }
}

// ---- fp32 through exact bf16 splits -------------------------------------------------------------------
// Products of fp32 matrices as six bf16 products of exact three-way splits (split.h), sums in fp32; a 16-deep
// MFMA rounds once where 16 fp32 steps round 16 times. Error against float64, tail 1.82e-7 (the fp32 MFMA form
// 2.20e-7, separate library GEMMs 2.20e-7), projection 1.74e-7 (2.11e-7). 6 x 32 cycles in place of 512 for a
// 32 x 32 x 16 product.
//
// The weights are split once per call by el_split_kernel into the images that the kernels stream: units of
// 1 KB, lane l's 16 bytes of a plane at 16 l (row el_perm(l % 32) of a 32-feature tile, values 8 (l / 32) ..
// + 7 of a 16-deep slice), in the order of use, 24 units a step. Activations are split in registers,
// 5.5 VALU per value, once per use as an operand.
constexpr int EX_UNITS = 24, EX_STEP = EX_UNITS * 1024, EX_IPW = EX_UNITS / EL_NW;

// The step image's units are numbered kt * 3 + plane, kt = 0..7 the (k slice, tile) pairs in order of use.
struct ElSplit {
  const float *w0, *w1, *w2;  // tail: Wo, W1, W2; projection: the weight, null, null
  char* img;
  int steps;
};
__global__ __launch_bounds__(256) void el_split_kernel(ElSplit p) {
  const int t = blockIdx.x * 256 + threadIdx.x, lane = t & 63, kt = (t >> 6) & 7, step = t >> 9;
  if (step >= p.steps) return;
  const float* w = p.w0;
  int ld = EL_W, o0 = step * 32, k0 = kt * 16;  // a whole 32-feature tile, K = 128
  if (p.w1 && step >= 4) {
    const int f = (step - 4) >> 2, half = step & 1;
    if (((step - 4) & 2) == 0) {  // W1: features 64 f + 32 tile, slices 4 half .. + 3
      w = p.w1;
      o0 = 64 * f + 32 * (kt & 1);
      k0 = 16 * (4 * half + (kt >> 1));
    } else {  // W2: output tile kt % 4, slices 2 half .. + 1 of the 64 features
      w = p.w2;
      ld = EL_FF;
      o0 = 32 * (kt & 3);
      k0 = 64 * f + 16 * (2 * half + (kt >> 2));
    }
  }
  const float* src = w + (int64_t)(o0 + el_perm(lane & 31)) * ld + k0 + 8 * (lane >> 5);
  const Split8 s = split8(*(const f32x4*)src, *(const f32x4*)(src + 4));
  char* dst = p.img + (int64_t)step * EX_STEP + kt * 3072 + lane * 16;
  *(bf16x8*)dst = s.h;
  *(bf16x8*)(dst + 1024) = s.m;
  *(bf16x8*)(dst + 2048) = s.l;
}

__device__ __forceinline__ void ex_copy(const char* img, int step, uint32_t dst, int w, int lane) {
#pragma unroll
  for (int i = 0; i < EX_IPW; ++i)
    lds_dma16_s((uint32_t)((w * EX_IPW + i) * 1024 + lane * 16), img + (int64_t)step * EX_STEP, dst + (w * EX_IPW + i) * 1024);
}
__device__ __forceinline__ Split8 ex_unit(const char* buf, int kt) {
  return {*(const bf16x8*)(buf + kt * 3072), *(const bf16x8*)(buf + kt * 3072 + 1024), *(const bf16x8*)(buf + kt * 3072 + 2048)};
}
// acc += A B in fp32 accuracy, the small terms first.
__device__ __forceinline__ void ex_mm(f32x16& acc, const Split8& a, const Split8& b) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.l, b.h, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.l, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.m, b.m, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.m, b.h, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.m, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.h, acc, 0, 0, 0);
}

// el_proj_kernel<float> through splits: img holds one step per 32 output features.
__global__ __launch_bounds__(EL_NW * 64, 2) void ex_proj_kernel(ElParams p) {
  __shared__ __attribute__((aligned(512))) char ring[EL_RING * EX_STEP];
  __shared__ __attribute__((aligned(16))) float prm[2 * EL_W + 3 * EL_W];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, m = lane & 31, hh = lane >> 5;
  const int64_t row0 = (int64_t)blockIdx.x * EL_ROWS;
  const int nrow = (int)(p.rows - row0 < EL_ROWS ? p.rows - row0 : EL_ROWS);
  const int S = p.n_out / 32;
  const uint32_t ring0 = lds_addr(ring);
  const char* img = (const char*)p.w1;
  ex_copy(img, 0, ring0, w, lane);
  ex_copy(img, 1, ring0 + EX_STEP, w, lane);
  const __amdgpu_buffer_rsrc_t xrs =
      __builtin_amdgcn_make_buffer_rsrc((float*)p.x + row0 * EL_W, 0, nrow * 512, TA_BUF_WORD3);
  const int xoff = (w * 32 + m) * 512 + hh * 32;
  float v[64];
#pragma unroll
  for (int i = 0; i < 8; ++i) el_load8<float>(xrs, xoff + i * 64, v + 8 * i);
  for (int i = threadIdx.x; i < EL_W; i += EL_NW * 64) {
    prm[i] = p.ln_w ? p.ln_w[i] : 1.f;
    prm[EL_W + i] = p.ln_b ? p.ln_b[i] : 0.f;
  }
  for (int i = threadIdx.x; i < p.n_out; i += EL_NW * 64) prm[2 * EL_W + i] = el_param((const float*)p.b1, i);
  if (p.live) {
    bool diff = false;
#pragma unroll
    for (int i = 0; i < 64; ++i) diff |= !(v[i] == p.skip);
    if (diff && w * 32 + m < nrow) p.live[(uint32_t)(row0 + w * 32 + m) / p.group_rows] = 1;
  }
  TA_JOIN_LDS();
  const auto val = [&](int i) { return v[i]; };
  const ElNorm norm = el_stats(val, p.eps);
  Split8 op[8];
#pragma unroll
  for (int k = 0; k < 8; ++k)
    op[k] = split8(el_normed(val, 2 * k, norm, prm, prm + EL_W, hh), el_normed(val, 2 * k + 1, norm, prm, prm + EL_W, hh));
  const __amdgpu_buffer_rsrc_t ors = __builtin_amdgcn_make_buffer_rsrc(
      (float*)p.out + row0 * p.n_out, 0, nrow * p.n_out * 4, TA_BUF_WORD3);
  const int ooff = ((w * 32 + m) * p.n_out + hh * 8) * 4;
  int slot = 0;
  for (int s = 0; s < S; ++s) {
    // younger than step s's copies: the next step's six copies and the last two steps' four stores each
    if (s == 0) TA_WAIT_JOIN(6);
    else if (s == S - 1) TA_WAIT_JOIN(8);
    else if (s == 1) TA_WAIT_JOIN(10);
    else TA_WAIT_JOIN(14);
    if (s + 2 < S) ex_copy(img, s + 2, ring0 + (slot == 0 ? 2 : slot - 1) * EX_STEP, w, lane);
    f32x16 acc = {}, bias;
    const char* buf = ring + slot * EX_STEP + lane * 16;
#pragma unroll
    for (int k = 0; k < 8; ++k) ex_mm(acc, ex_unit(buf, k), op[k]);
    el_bias(bias, prm + 2 * EL_W + s * 32, hh);
    acc += bias;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float o[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = acc[8 * i + j];
      el_store8<float>(ors, ooff + (s * 32 + i * 16) * 4, o);
    }
    slot = slot == 2 ? 0 : slot + 1;
  }
}

// el_tail_kernel<float> through splits: img holds 4 steps of Wo, then per 64 feed-forward features two of W1
// and two of W2 (el_split_kernel).
__global__ __launch_bounds__(EL_NW * 64, 2) void ex_tail_kernel(ElParams p) {
  constexpr int NS = 20;
  __shared__ __attribute__((aligned(512))) char ring[EL_RING * EX_STEP];
  __shared__ __attribute__((aligned(16))) float prm[4 * EL_W + EL_FF];
  const float *bo = prm, *lw = prm + EL_W, *lb = prm + 2 * EL_W, *b2 = prm + 3 * EL_W, *b1 = prm + 4 * EL_W;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, m = lane & 31, hh = lane >> 5;
  const int64_t row0 = (int64_t)blockIdx.x * EL_ROWS;
  const int nrow = (int)(p.rows - row0 < EL_ROWS ? p.rows - row0 : EL_ROWS);
  const __amdgpu_buffer_rsrc_t ors =
      __builtin_amdgcn_make_buffer_rsrc((float*)p.out + row0 * EL_W, 0, nrow * 512, TA_BUF_WORD3);
  const int xoff = (w * 32 + m) * 512 + hh * 32;
  bool keep;
  if (el_skip_tile<float>(p, row0, nrow, w * 32 + m, ors, xoff, keep)) return;
  const uint32_t ring0 = lds_addr(ring);
  const char* img = (const char*)p.w1;
  ex_copy(img, 0, ring0, w, lane);
  ex_copy(img, 1, ring0 + EX_STEP, w, lane);
  const __amdgpu_buffer_rsrc_t ars =
      __builtin_amdgcn_make_buffer_rsrc((float*)p.a + row0 * EL_W, 0, nrow * 512, TA_BUF_WORD3);
  const __amdgpu_buffer_rsrc_t xrs =
      __builtin_amdgcn_make_buffer_rsrc((float*)p.x + row0 * EL_W, 0, nrow * 512, TA_BUF_WORD3);
  float av[64], sv[64];
#pragma unroll
  for (int i = 0; i < 8; ++i) el_load8<float>(ars, xoff + i * 64, av + 8 * i);
#pragma unroll
  for (int i = 0; i < 8; ++i) el_load8<float>(xrs, xoff + i * 64, sv + 8 * i);
  el_tail_params<float>(p, prm);
  {
    Split8 op[8];
#pragma unroll
    for (int k = 0; k < 8; ++k)
      op[k] = split8(f32x4{av[8 * k], av[8 * k + 1], av[8 * k + 2], av[8 * k + 3]},
                        f32x4{av[8 * k + 4], av[8 * k + 5], av[8 * k + 6], av[8 * k + 7]});
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      TA_WAIT_JOIN(6);
      ex_copy(img, s + 2, ring0 + (s + 2) % EL_RING * EX_STEP, w, lane);
      f32x16 y = {}, bias;
      const char* buf = ring + s % EL_RING * EX_STEP + lane * 16;
#pragma unroll
      for (int k = 0; k < 8; ++k) ex_mm(y, ex_unit(buf, k), op[k]);
      el_bias(bias, bo + s * 32, hh);
#pragma unroll
      for (int i = 0; i < 16; ++i) sv[s * 16 + i] += y[i] + bias[i];
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  const auto val = [&](int i) { return sv[i]; };
  ElNorm norm = el_stats(val, p.eps);
  f32x16 z[4];
#pragma unroll
  for (int ob = 0; ob < 4; ++ob) z[ob] = f32x16{};
  int slot = 4 % EL_RING;
  for (int f = 0; f < 4; ++f) {
    const int s = 4 + 4 * f;
    asm volatile("" : "+v"(norm.mean), "+v"(norm.rstd));  // LN(s) and its splits again at each use: kept, they would take 96 registers
    f32x16 h[2] = {};
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      TA_WAIT_JOIN(6);
      ex_copy(img, s + half + 2, ring0 + (slot == 0 ? 2 : slot - 1) * EX_STEP, w, lane);
      const char* buf = ring + slot * EX_STEP + lane * 16;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = 2 * (4 * half + k);
        const Split8 b = split8(el_normed(val, i, norm, lw, lb, hh), el_normed(val, i + 1, norm, lw, lb, hh));
        ex_mm(h[0], ex_unit(buf, 2 * k), b);
        ex_mm(h[1], ex_unit(buf, 2 * k + 1), b);
        __builtin_amdgcn_sched_barrier(0);
      }
      slot = slot == 2 ? 0 : slot + 1;
    }
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      f32x16 bias;
      el_bias(bias, b1 + f * 64 + nb * 32, hh);
#pragma unroll
      for (int i = 0; i < 16; ++i) h[nb][i] = el_gelu<float>(h[nb][i] + bias[i]);
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      if (s + half + 2 < NS - 1) TA_WAIT_JOIN(6);
      else TA_WAIT_JOIN(0);
      if (s + half + 4 < NS) ex_copy(img, s + half + 4, ring0 + (slot == 0 ? 2 : slot - 1) * EX_STEP, w, lane);
      const char* buf = ring + slot * EX_STEP + lane * 16;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const f32x16& g = h[half];
        const Split8 b = split8(f32x4{g[8 * k], g[8 * k + 1], g[8 * k + 2], g[8 * k + 3]},
                                  f32x4{g[8 * k + 4], g[8 * k + 5], g[8 * k + 6], g[8 * k + 7]});
#pragma unroll
        for (int ob = 0; ob < 4; ++ob) ex_mm(z[ob], ex_unit(buf, 4 * k + ob), b);
        __builtin_amdgcn_sched_barrier(0);
      }
      slot = slot == 2 ? 0 : slot + 1;
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = 8 * i + j;
      o[j] = keep ? sv[r] + (z[r >> 4][r & 15] + b2[16 * i + 8 * hh + j]) : p.skip;
    }
    el_store8<float>(ors, xoff + i * 64, o);
  }
}

// The column stage's input: circular feature grouping (slot j holds features (j mod rf + 2^i) mod rf, i < 3, rf = the
// table's real feature count), the group's linear 3 -> 128 and the skip rule, written as [b, columns, t, 128] with
// `reserve` leading columns of the skip value.
// One launch for 21 (gathers, stack, pad, conversion, GEMM, compares, select) and one write of the result: 4.16M rows
// (8 x 5000 x 104) fp32 2.13 -> 0.57 ms, bf16 1.61 -> 0.32 ms; 1 x 50000 x 24 fp32 0.70 -> 0.11; 8 x 60 x 28 146 ->
// 12 us (launches). Bound by the write (3.8 TB/s). Workgroup = one column and 256 rows, 16 threads a row, so that the
// 24 weights of a thread stay in registers; the rows of x it reads are shared through L2 by the columns.
struct EmbedParams {
  const float* x;          // [B, T, H]
  const int64_t* real;     // [B] or null (H)
  const void *w, *b;       // [128, 3], [128] or null
  void* out;
  int T, H, reserve;
  float skip;
};
template <typename T> __global__ __launch_bounds__(256) void el_embed_kernel(EmbedParams p) {
  const int HC = p.H + p.reserve, col = blockIdx.y % HC, b = blockIdx.y / HC;
  const int f = (threadIdx.x & 15) * 8, sub = threadIdx.x >> 4;
  const float skip = to_f32<T>(from_f32<T>(p.skip));
  float w[8][3], bias[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
#pragma unroll
    for (int j = 0; j < 3; ++j) w[i][j] = to_f32<T>(((const T*)p.w)[(f + i) * 3 + j]);
    bias[i] = p.b ? to_f32<T>(((const T*)p.b)[f + i]) : 0.f;
  }
  int idx[3] = {0, 0, 0};
  bool bad = false;
  if (col >= p.reserve) {
    int64_t rf = p.real ? p.real[b] : p.H;
    bad = rf < 1 || rf > p.H;  // no such features: the table's slots become NaN, nothing is read out of range
    rf = bad ? 1 : rf;
    const int base = (int)((col - p.reserve) % rf);
#pragma unroll
    for (int i = 0; i < 3; ++i) idx[i] = (int)((base + (1 << i)) % rf);
  }
  const float* xb = p.x + (int64_t)b * p.T * p.H;
  T* ob = (T*)p.out + ((int64_t)blockIdx.y * p.T) * EL_W + f;
#pragma unroll 4
  for (int i = 0; i < 16; ++i) {
    const int t = blockIdx.x * 256 + i * 16 + sub;
    if (t >= p.T) break;
    float y[8];
    bool dead = true;
    float v[3];
    if (col >= p.reserve) {
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        v[j] = to_f32<T>(from_f32<T>(xb[(int64_t)t * p.H + idx[j]]));
        dead = dead && v[j] == skip;
      }
#pragma unroll
      for (int k = 0; k < 8; ++k)
        y[k] = __builtin_fmaf(v[2], w[k][2], __builtin_fmaf(v[1], w[k][1], v[0] * w[k][0])) + bias[k];
    }
    if (dead || bad) {
#pragma unroll
      for (int k = 0; k < 8; ++k) y[k] = bad ? __builtin_nanf("") : skip;
    }
    T* o = ob + (int64_t)t * EL_W;
    if constexpr (sizeof(T) == 4) {
      *(f32x4*)o = f32x4{y[0], y[1], y[2], y[3]};
      *(f32x4*)(o + 4) = f32x4{y[4], y[5], y[6], y[7]};
    } else {
      *(bf16x8*)o = el_pack8(f32x4{y[0], y[1], y[2], y[3]}, f32x4{y[4], y[5], y[6], y[7]});
    }
  }
}

int el_cus() {
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    return 256;
  return cus;
}

void split_weights(const float* w0, const float* w1, const float* w2, void* img, int steps, hipStream_t stream) {
  const ElSplit e = {w0, w1, w2, (char*)img, steps};
  hipLaunchKernelGGL(el_split_kernel, dim3((unsigned)steps * 2), dim3(256), 0, stream, e);
}

// Rows from which a fp32 projection runs on splits (the tail always does: 39 against 61 us for one tile of
// rows). Below, the launch that splits the weights (3-4 us) costs more than the fp32 MFMA kernel's products:
// 128 features, 480 / 13440 / 16384 rows, 14.5 / 16.8 / 17.0 us against 19.7 / 20.4 / 19.1 us; 4.16M rows
// 1316 against 1172 us.
constexpr int64_t EX_MIN_ROWS = 32768;

}  // namespace

// Bytes of the split weight image of a projection to n_out features (0: of a tail); 0 where none is used.
int64_t tabicl_launch_layer_ws_bytes(int64_t n_out, int64_t rows, int dtype) {
  if (dtype != 1 || (n_out && rows < EX_MIN_ROWS)) return 0;
  return (n_out ? n_out / 32 : 20) * EX_STEP;
}

int tabicl_launch_layer_proj(const void* x, const float* ln_w, const float* ln_b, float eps, const void* w,
                             const void* b, void* out, int64_t rows, int64_t n_out, int dtype, int* live,
                             int64_t group_rows, float skip, void* ws, int64_t ws_bytes, hipStream_t stream) {
  if (rows <= 0) return 0;
  ElParams p = {};
  p.x = x;
  p.ln_w = ln_w;
  p.ln_b = ln_b;
  p.eps = eps;
  p.w1 = w;
  p.b1 = b;
  p.out = out;
  p.rows = rows;
  p.n_out = (int)n_out;
  p.live = live;
  p.group_rows = (uint32_t)group_rows;
  p.skip = skip;
  const int64_t tiles = (rows + EL_ROWS - 1) / EL_ROWS;
  const int64_t need = tabicl_launch_layer_ws_bytes(n_out, rows, dtype);
  if (need && ws && ws_bytes >= need) {
    split_weights((const float*)w, nullptr, nullptr, ws, (int)n_out / 32, stream);
    p.w1 = ws;
    hipLaunchKernelGGL(ex_proj_kernel, dim3((unsigned)tiles), dim3(EL_NW * 64), 0, stream, p);
    return (int)hipGetLastError();
  }
  const int nsteps = (int)n_out / (dtype == 0 ? El<bf16>::OUTS : El<float>::OUTS);
  // few rows: split the output features over workgroups too (each repeats the LayerNorm of its rows), until
  // every CU has two
  int split = (int)((2 * el_cus() + tiles - 1) / tiles);
  if (split > nsteps) split = nsteps;
  p.steps_per_wg = (nsteps + split - 1) / split;
  const dim3 grid((unsigned)tiles, (unsigned)((nsteps + p.steps_per_wg - 1) / p.steps_per_wg));
  if (dtype == 0)
    hipLaunchKernelGGL((el_proj_kernel<bf16>), grid, dim3(EL_NW * 64), 0, stream, p);
  else
    hipLaunchKernelGGL((el_proj_kernel<float>), grid, dim3(EL_NW * 64), 0, stream, p);
  return (int)hipGetLastError();
}

int tabicl_launch_layer_tail(const void* a, const void* x, const void* wo, const void* bo, const float* ln_w,
                             const float* ln_b, float eps, const void* w1, const void* b1, const void* w2,
                             const void* b2, void* out, int64_t rows, int dtype, const int* live, int64_t group_rows,
                             float skip, void* ws, int64_t ws_bytes, hipStream_t stream) {
  if (rows <= 0) return 0;
  ElParams p = {};
  p.a = a;
  p.x = x;
  p.ln_w = ln_w;
  p.ln_b = ln_b;
  p.eps = eps;
  p.wo = wo;
  p.bo = bo;
  p.w1 = w1;
  p.b1 = b1;
  p.w2 = w2;
  p.b2 = b2;
  p.out = out;
  p.rows = rows;
  p.live = (int*)live;
  p.group_rows = (uint32_t)group_rows;
  p.skip = skip;
  const dim3 grid((unsigned)((rows + EL_ROWS - 1) / EL_ROWS));
  if (dtype == 1) {
    split_weights((const float*)wo, (const float*)w1, (const float*)w2, ws, 20, stream);
    p.w1 = ws;
    hipLaunchKernelGGL(ex_tail_kernel, grid, dim3(EL_NW * 64), 0, stream, p);
    return (int)hipGetLastError();
  }
  hipLaunchKernelGGL(el_tail_kernel, grid, dim3(EL_NW * 64), 0, stream, p);
  return (int)hipGetLastError();
}

int tabicl_launch_column_embed(const float* x, const int64_t* real, const void* w, const void* b, void* out, int64_t B,
                               int64_t T, int64_t H, int64_t reserve, float skip, int dtype, hipStream_t stream) {
  const EmbedParams p = {x, real, w, b, out, (int)T, (int)H, (int)reserve, skip};
  const dim3 grid((unsigned)((T + 255) / 256), (unsigned)(B * (H + reserve)));
  if (dtype == 0) hipLaunchKernelGGL((el_embed_kernel<bf16>), grid, dim3(256), 0, stream, p);
  else hipLaunchKernelGGL((el_embed_kernel<float>), grid, dim3(256), 0, stream, p);
  return (int)hipGetLastError();
}
