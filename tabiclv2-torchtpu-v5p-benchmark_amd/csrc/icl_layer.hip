// The linear layers of an ICL block (width 512, feed-forward 1024, bf16 weights, fp32 residual stream) for a query of
// few rows, each fused with what surrounds it:
//
//   ic_linear_kernel<512, LN>    out = [gelu](LN(x) W^T + b), bf16      (q projection; first feed-forward layer)
//   ic_linear_kernel<K, residual> out = res + (x W^T + b), fp32          (out projection; second feed-forward layer)
//
// As library GEMMs these are 14 launches a block with norms, activation, casts and adds; at a few hundred rows
// each launch is a few us of GPU time and 10-25 us of host time (the library's heuristics), so the blocks were
// bound by the host.
//
// Workgroup = 32 rows x 128 features, wave = 32 features (one 32x32 tile, Y^T = W X^T). The rows (normalised to
// bf16 by the four waves, or copied) stay in LDS, chunks XOR-swizzled by row; a wave streams its own 32 weight
// rows, 64 values deep, three steps ahead into a private ring, so the sweep has no barrier. Bound by latency:
// the first loads, then K / 64 steps of 128 matrix cycles.
// Measured (480 rows): see the dispatch rule in tabicl_mi355_icl.py.
#include "common.h"
#include "launch.h"
#include "layer.h"

namespace {

constexpr int IL_W = 512, IL_ROWS = 32, IL_NW = 4, IL_RING = 3, IL_STEP = 4096;

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

__device__ __forceinline__ float il_wave_sum(float x) {
#pragma unroll
  for (int m = 1; m < 16; m <<= 1) x += __shfl_xor(x, m, 64);
  return quad_sum(x);
}

template <int K, bool LN> __global__ __launch_bounds__(IL_NW * 64) void ic_linear_kernel(IlParams p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  constexpr int S = K / 64, RB = K * 2, CPR = RB / 16;  // steps; bytes and 16-byte chunks of a row
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, m = lane & 31, hh = lane >> 5;
  const int64_t row0 = (int64_t)blockIdx.x * IL_ROWS;
  const int nrow = (int)(p.rows - row0 < IL_ROWS ? p.rows - row0 : IL_ROWS);
  const int f0 = blockIdx.y * 128 + w * 32;
  const int64_t row = row0 + (m < nrow ? m : nrow - 1);
  // the epilogue's operands first: no load waits for the copies below
  float bias[16], res[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int f = f0 + 16 * (i >> 3) + 8 * hh + (i & 7);
    bias[i] = p.b ? (float)p.b[f] : 0.f;
  }
  if constexpr (!LN) {
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      const f32x4 r = *(const f32x4*)(p.res + row * IL_W + f0 + 16 * (i >> 3) + 8 * hh + (i & 7));
#pragma unroll
      for (int j = 0; j < 4; ++j) res[i + j] = r[j];
    }
  }
  const uint32_t act0 = lds_addr(lds), ring0 = act0 + IL_ROWS * RB + w * (IL_RING * IL_STEP);
  if constexpr (!LN) {  // rows into LDS, eight per wave (rows past the end repeat the last)
#pragma unroll
    for (int i = 0; i < 8 * CPR / 64; ++i) {
      const int c0 = (w * 8 * CPR / 64 + i) * 64, q = c0 + lane, r = q / CPR, pos = q % CPR;
      lds_dma16_s((uint32_t)((r < nrow ? r : nrow - 1) * RB + ((pos ^ (r & 15)) << 4)), (const bf16*)p.x + row0 * K,
                  act0 + c0 * 16);
    }
  }
  // this wave's weight rows, step s: values [64 s, 64 s + 64) of rows f0 .. f0 + 31
  auto copy_step = [&](int s) {
    const char* src = (const char*)(p.w + (int64_t)f0 * K) + s * 128;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int q = i * 64 + lane, r = q >> 3, pos = q & 7;
      lds_dma16_s((uint32_t)(r * RB + ((pos ^ ((r >> 1) & 7)) << 4)), src, ring0 + (s % IL_RING) * IL_STEP + i * 1024);
    }
  };
#pragma unroll
  for (int s = 0; s < IL_RING; ++s) copy_step(s);
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
      float s = 0.f, q = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) s += v[r][i >> 2][i & 3];
      const float mean = il_wave_sum(s) * (1.0f / IL_W);
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
    TA_WAIT_JOIN(12);  // the rows: older than the three steps of weights
  }
  const char* act = lds + m * RB;
  const char* ring = lds + IL_ROWS * RB + w * (IL_RING * IL_STEP);
  const int prow = el_perm(m);
  const uint32_t wb = (uint32_t)(prow * 128 + ((hh ^ ((prow >> 1) & 7)) << 4)), ab = (uint32_t)((hh ^ (m & 15)) << 4);
  f32x16 acc = {};
#pragma unroll
  for (int s = 0; s < S; ++s) {
    if (S - 1 - s >= 2) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    else if (S - 1 - s == 1) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const bf16x8 a = *(const bf16x8*)(ring + (s % IL_RING) * IL_STEP + (wb ^ (kk << 5)));
      const bf16x8 b = *(const bf16x8*)(act + (s >> 1) * 256 + (ab ^ (((s & 1) * 4 + kk) << 5)));
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
    }
    if (s + IL_RING < S) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this step's reads have left the slot
      copy_step(s + IL_RING);
    }
  }
  if (m >= nrow) return;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    f32x4 o[2];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float y = acc[8 * i + j] + bias[8 * i + j];
      if constexpr (LN) {
        if (p.gelu) y = el_gelu<bf16>(y);
      } else {
        y += res[8 * i + j];
      }
      o[j >> 2][j & 3] = y;
    }
    const int64_t f = f0 + 16 * i + 8 * hh;
    if constexpr (LN) {
      *(bf16x8*)((bf16*)p.out + row * p.n + f) = el_pack8(o[0], o[1]);
    } else {
      *(f32x4*)((float*)p.out + row * IL_W + f) = o[0];
      *(f32x4*)((float*)p.out + row * IL_W + f + 4) = o[1];
    }
  }
}

template <int K, bool LN> int launch_ic_linear(const IlParams& p, hipStream_t stream) {
  constexpr int LDS = IL_ROWS * K * 2 + IL_NW * IL_RING * IL_STEP;
  const hipError_t e = hipFuncSetAttribute((const void*)ic_linear_kernel<K, LN>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL((ic_linear_kernel<K, LN>), dim3((unsigned)((p.rows + IL_ROWS - 1) / IL_ROWS), (unsigned)(p.n / 128)),
                     dim3(IL_NW * 64), LDS, stream, p);
  return (int)hipGetLastError();
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
