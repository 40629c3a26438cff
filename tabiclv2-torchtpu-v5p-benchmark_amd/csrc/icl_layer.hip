// The linear layers of an ICL block (width 512, feed-forward 1024, bf16 weights, fp32 residual stream) for a query of
// few rows, each fused with what surrounds it:
//
//   ic_linear_kernel<512, LN>    out = [gelu](LN(x) W^T + b), bf16      (q projection; first feed-forward layer; decoder)
//   ic_linear_kernel<K, residual> out = res + (x W^T + b), fp32          (out projection; second feed-forward layer)
//
// As library GEMMs these are 14 launches a block with norms, activation, casts and adds; at a few hundred rows
// each launch is a few us of GPU time and 10-25 us of host time (the library's heuristics), so the blocks were
// bound by the host.
//
// Workgroup = 32 rows and, per wave, one 32x32 tile (Y^T = W X^T). The rows (normalised to bf16 by the four waves,
// or copied) stay in LDS, chunks XOR-swizzled by row; a wave copies its own weights, steps of 32 rows x 64 values,
// so the sweep has no barrier. Two splits:
//   KS = false  the waves take 32 features each of 128; three steps in flight in a private ring
//   KS = true   the waves take a quarter of K each of the same 32 features, every weight in flight at once, and add
//               their tiles through LDS: four times the workgroups, for launches that leave CUs idle
// Bound by latency: the loads, then K / 64 (K / 256) steps of 128 matrix cycles.
// Measured: a block (everything but the attention kernel) of 480 rows 163 -> 66 us, host time included.
#include "common.h"
#include "launch.h"
#include "layer.h"

namespace {

constexpr int IL_W = 512, IL_ROWS = 32, IL_NW = 4, IL_RING = 3, IL_STEP = 4096;
// Below this many workgroups of the first split, the second. us at 480 rows (60 workgroups per 512 features):
// q projection 7.3 (KS) / 9.3, first feed-forward layer (120) 10.5 / 9.8, out projection 3.7 / 5.6, second
// feed-forward layer 4.7 / 7.1; 1000 rows (128): 9.9 / 9.3, 18.1 / 10.2, 4.4 / 5.6, 7.1 / 7.2; 1600 rows (200):
// 17 / 9.4, 29 / 14, 6.8 / 5.8, 11.4 / 7.4.
constexpr int IL_KS_WGS_LN = 112, IL_KS_WGS_RES = 160;

struct IlParams {
  const void* x;                // LN: fp32 [rows, 512]; residual: bf16 [rows, K]
  const float *ln_w, *ln_b;
  const bf16 *w, *b;            // [n, K], [n] or null
  const float* res;             // [rows, 512]
  void* out;                    // LN: bf16 [rows, n]; residual: fp32 [rows, 512]
  int64_t rows;
  int n, gelu;
  float eps;
};

template <int CTRL> __device__ __forceinline__ float il_dpp_add(float x) {
  return x + __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(x), CTRL, 0xf, 0xf, true));
}
// Sum over the wave: within 16 lanes by quad permutes and mirrors, then the lane quads.
__device__ __forceinline__ float il_wave_sum(float x) {
  x = il_dpp_add<0xb1>(x);   // quad_perm 1,0,3,2
  x = il_dpp_add<0x4e>(x);   // quad_perm 2,3,0,1
  x = il_dpp_add<0x141>(x);  // half mirror
  x = il_dpp_add<0x140>(x);  // mirror
  return quad_sum(x);
}

template <int K, bool LN, bool KS> __global__ __launch_bounds__(IL_NW * 64) void ic_linear_kernel(IlParams p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  constexpr int S = KS ? K / 256 : K / 64, RING = KS ? S : IL_RING;  // steps of a wave, in flight
  constexpr int RB = K * 2, CPR = RB / 16;                            // bytes and 16-byte chunks of a row
  constexpr int NE = KS ? 4 : 16;                                     // output values of a lane
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, m = lane & 31, hh = lane >> 5;
  const int64_t row0 = (int64_t)blockIdx.x * IL_ROWS;
  const int nrow = (int)(p.rows - row0 < IL_ROWS ? p.rows - row0 : IL_ROWS);
  const int f0 = KS ? blockIdx.y * 32 : blockIdx.y * 128 + w * 32;
  const int s0 = KS ? w * S : 0, e0 = KS ? 4 * w : 0;  // first step; first result register this wave finishes
  const int64_t row = row0 + (m < nrow ? m : nrow - 1);
  auto feature = [&](int i) { return f0 + 16 * ((e0 + i) >> 3) + 8 * hh + ((e0 + i) & 7); };
  // the epilogue's operands first: no load waits for the copies below
  float bias[NE], res[NE];
#pragma unroll
  for (int i = 0; i < NE; ++i) bias[i] = p.b ? (float)p.b[feature(i)] : 0.f;
  if constexpr (!LN) {
#pragma unroll
    for (int i = 0; i < NE; i += 4) {
      const f32x4 r = *(const f32x4*)(p.res + row * IL_W + feature(i));
#pragma unroll
      for (int j = 0; j < 4; ++j) res[i + j] = r[j];
    }
  }
  const uint32_t act0 = lds_addr(lds), ring0 = act0 + IL_ROWS * RB + w * (RING * IL_STEP);
  if constexpr (!LN) {  // rows into LDS, eight per wave (rows past the end repeat the last)
#pragma unroll
    for (int i = 0; i < 8 * CPR / 64; ++i) {
      const int c0 = (w * 8 * CPR / 64 + i) * 64, q = c0 + lane, r = q / CPR, pos = q % CPR;
      lds_dma16_s((uint32_t)((r < nrow ? r : nrow - 1) * RB + ((pos ^ (r & 15)) << 4)), (const bf16*)p.x + row0 * K,
                  act0 + c0 * 16);
    }
  }
  // this wave's weight rows, step s: values [64 (s0 + s), + 64) of rows f0 .. f0 + 31
  auto copy_step = [&](int s) {
    const char* src = (const char*)(p.w + (int64_t)f0 * K) + (s0 + s) * 128;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int q = i * 64 + lane, r = q >> 3, pos = q & 7;
      lds_dma16_s((uint32_t)(r * RB + ((pos ^ ((r >> 1) & 7)) << 4)), src, ring0 + (s % RING) * IL_STEP + i * 1024);
    }
  };
#pragma unroll
  for (int s = 0; s < RING; ++s) copy_step(s);
  if constexpr (LN) {
    float lw[8], lb[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      lw[i] = p.ln_w ? p.ln_w[lane * 8 + i] : 1.f;
      lb[i] = p.ln_b ? p.ln_b[lane * 8 + i] : 0.f;
    }
    f32x4 v[8][2];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int lr = w * 8 + r;
      const float* src = (const float*)p.x + (row0 + (lr < nrow ? lr : nrow - 1)) * IL_W + lane * 8;
      v[r][0] = *(const f32x4*)src;
      v[r][1] = *(const f32x4*)(src + 4);
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      float q = 0.f;
      const float mean = il_wave_sum(el_sum<8>([&](int i) { return v[r][i >> 2][i & 3]; }, 0)) * (1.0f / IL_W);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float d = v[r][i >> 2][i & 3] - mean;
        q = __builtin_fmaf(d, d, q);
      }
      const float rstd = __builtin_amdgcn_rsqf(il_wave_sum(q) * (1.0f / IL_W) + p.eps);
      f32x4 y[2];
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i >> 2][i & 3] = __builtin_fmaf((v[r][i >> 2][i & 3] - mean) * rstd, lw[i], lb[i]);
      const int lr = w * 8 + r;
      *(bf16x8*)(lds + lr * RB + ((lane ^ (lr & 15)) << 4)) = el_pack8(y[0], y[1]);
    }
    TA_JOIN_LDS();
  } else {
    // the rows: older than the RING steps of weights
    if constexpr (RING == 4) TA_WAIT_JOIN(16);
    else if constexpr (RING == 3) TA_WAIT_JOIN(12);
    else TA_WAIT_JOIN(8);
  }
  const char* act = lds + m * RB;
  char* ring = lds + IL_ROWS * RB + w * (RING * IL_STEP);
  const int prow = el_perm(m);
  const uint32_t wb = (uint32_t)(prow * 128 + ((hh ^ ((prow >> 1) & 7)) << 4)), ab = (uint32_t)((hh ^ (m & 15)) << 4);
  f32x16 acc = {};
#pragma unroll
  for (int s = 0; s < S; ++s) {
    constexpr int LAST = S - 1;
    const int younger = LAST - s < RING - 1 ? LAST - s : RING - 1;  // steps copied after this one
    if (younger >= 3) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
    else if (younger == 2) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    else if (younger == 1) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int k = s0 + s;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const bf16x8 a = *(const bf16x8*)(ring + (s % RING) * IL_STEP + (wb ^ (kk << 5)));
      const bf16x8 b = *(const bf16x8*)(act + (k >> 1) * 256 + (ab ^ (((k & 1) * 4 + kk) << 5)));
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
    }
    if (s + RING < S) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this step's reads have left the slot
      copy_step(s + RING);
    }
  }
  float y[NE];
  if constexpr (KS) {
    // the four partial tiles through the waves' own (read out) weight slots: [register][lane]
#pragma unroll
    for (int i = 0; i < 16; ++i) *(float*)(ring + i * 256 + lane * 4) = acc[i];
    TA_JOIN_LDS();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      y[i] = 0.f;
#pragma unroll
      for (int q = 0; q < IL_NW; ++q)
        y[i] += *(const float*)(lds + IL_ROWS * RB + q * (RING * IL_STEP) + (e0 + i) * 256 + lane * 4);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) y[i % NE] = acc[i];
  }
  if (m >= nrow) return;
#pragma unroll
  for (int i = 0; i < NE; i += 4) {
    f32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      o[j] = y[i + j] + bias[i + j];
      if constexpr (LN) {
        if (p.gelu) o[j] = el_gelu<bf16>(o[j]);
      } else {
        o[j] += res[i + j];
      }
    }
    if constexpr (LN) *(bf16x4*)((bf16*)p.out + row * p.n + feature(i)) = cvt_bf16x4(o);
    else *(f32x4*)((float*)p.out + row * IL_W + feature(i)) = o;
  }
}

template <int K, bool LN, bool KS> int launch_ic_linear_inst(const IlParams& p, int64_t tiles, hipStream_t stream) {
  constexpr int LDS = IL_ROWS * K * 2 + IL_NW * (KS ? K / 256 : IL_RING) * IL_STEP;
  const hipError_t e = hipFuncSetAttribute((const void*)ic_linear_kernel<K, LN, KS>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL((ic_linear_kernel<K, LN, KS>), dim3((unsigned)tiles, (unsigned)(p.n / (KS ? 32 : 128))),
                     dim3(IL_NW * 64), LDS, stream, p);
  return (int)hipGetLastError();
}
template <int K, bool LN> int launch_ic_linear(const IlParams& p, hipStream_t stream) {
  const int64_t tiles = (p.rows + IL_ROWS - 1) / IL_ROWS;
  return tiles * (p.n / 128) < (LN ? IL_KS_WGS_LN : IL_KS_WGS_RES) ? launch_ic_linear_inst<K, LN, true>(p, tiles, stream)
                                         : launch_ic_linear_inst<K, LN, false>(p, tiles, stream);
}

}  // namespace

int tabicl_launch_ln_linear(const float* x, const float* ln_w, const float* ln_b, float eps, const void* w, const void* b,
                            void* out, int64_t rows, int64_t n, int gelu, hipStream_t stream) {
  if (rows <= 0) return 0;
  IlParams p = {};
  p.x = x;
  p.ln_w = ln_w;
  p.ln_b = ln_b;
  p.eps = eps;
  p.w = (const bf16*)w;
  p.b = (const bf16*)b;
  p.out = out;
  p.rows = rows;
  p.n = (int)n;
  p.gelu = gelu;
  return launch_ic_linear<512, true>(p, stream);
}

int tabicl_launch_linear_residual(const void* x, const void* w, const void* b, const float* res, float* out, int64_t rows,
                                  int64_t k, hipStream_t stream) {
  if (rows <= 0) return 0;
  IlParams p = {};
  p.x = x;
  p.w = (const bf16*)w;
  p.b = (const bf16*)b;
  p.res = res;
  p.out = out;
  p.rows = rows;
  p.n = IL_W;
  return k == 512 ? launch_ic_linear<512, false>(p, stream) : launch_ic_linear<1024, false>(p, stream);
}
