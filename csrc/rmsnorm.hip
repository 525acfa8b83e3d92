// RMSNorm + fused residual-add RMSNorm, bf16 I/O, fp32 accumulation.
// Memory-bound: vectorized u16x8 loads (G13: scalar bf16 loads cost ~2x).
// Two shapes:
//  - wide rows (hidden_size 1k..16k): one or four waves per row, row kept in
//    registers between the sum-of-squares pass and the normalize pass.
//  - small rows (head_dim 64/128, q/k norm): one wave per row.
#include "common.h"

// ---------------- wide rows ----------------

// WAVES waves hold a row in registers, NV pieces of 8 a lane. Bound by memory.
// Where rows are many, one wave a row: no barrier, no LDS, and a row's loads
// all in flight at once. With a workgroup a row half of it had nothing to do at
// 1024 columns: 24,000 such rows with the residual 59 -> 32 us (6.2 TB/s, some of
// it from the caches). Few rows take four waves each, for the latency.
template <bool FUSED_ADD, int NV, int WAVES>
__global__ void __launch_bounds__(256)
rmsnorm_wide_kernel(u16* __restrict__ out,       // [rows, C]
                    u16* __restrict__ residual,  // [rows, C] or null
                    const u16* __restrict__ in,  // [rows, C]
                    const u16* __restrict__ w,   // [C]
                    float eps, long rows, int C) {
  constexpr int LANES = WAVES * (int)WAVE;
  const int l = threadIdx.x % LANES;
  const long row = (long)blockIdx.x * (256 / LANES) + threadIdx.x / LANES;
  if (WAVES == 1 && row >= rows) return;
  const int pieces = C / 8;
  const long base = row * C;
  u16x8 x[NV], r[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = l + i * LANES;
    if (v < pieces) {
      x[i] = *(const u16x8*)(in + base + v * 8);
      if (FUSED_ADD) r[i] = *(const u16x8*)(residual + base + v * 8);
    }
  }
  float xf[NV][8], ssq = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = l + i * LANES;
    if (v < pieces) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        xf[i][j] = bf2f(x[i][j]) + (FUSED_ADD ? bf2f(r[i][j]) : 0.f);
        ssq += xf[i][j] * xf[i][j];
      }
      if (FUSED_ADD) {   // residual += x
        u16x8 nr;
#pragma unroll
        for (int j = 0; j < 8; ++j) nr[j] = f2bf(xf[i][j]);
        *(u16x8*)(residual + base + v * 8) = nr;
      }
    }
  }
  ssq = wave_sum_f32(ssq);
  if (WAVES > 1) {
    __shared__ float red[WAVES];
    if ((l & (WAVE - 1)) == 0) red[l / WAVE] = ssq;
    __syncthreads();
    ssq = red[0];
#pragma unroll
    for (int i = 1; i < WAVES; ++i) ssq += red[i];
  }
  const float inv = rsqrtf(ssq / (float)C + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = l + i * LANES;
    if (v < pieces) {
      const u16x8 wv = *(const u16x8*)(w + v * 8);
      u16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = f2bf(xf[i][j] * inv * bf2f(wv[j]));
      *(u16x8*)(out + base + v * 8) = o;
    }
  }
}

// ---------------- small rows (head-dim q/k norm) ----------------

__global__ void rmsnorm_small_kernel(u16* __restrict__ out,
                                     const u16* __restrict__ in,
                                     const u16* __restrict__ w,
                                     float eps, long rows, int C) {
  const int lane = threadIdx.x & (WAVE - 1);
  const long wave_id = ((long)blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  if (wave_id >= rows) return;
  const u16* rin = in + wave_id * C;
  u16* rout = out + wave_id * C;
  const int per_lane = C / (int)WAVE;  // C=128 -> 2, C=64 -> 1
  float x[4];
  float ssq = 0.f;
  for (int j = 0; j < per_lane; ++j) {
    x[j] = bf2f(rin[lane * per_lane + j]);
    ssq += x[j] * x[j];
  }
  ssq = wave_sum_f32(ssq);
  float inv = rsqrtf(ssq / (float)C + eps);
  for (int j = 0; j < per_lane; ++j)
    rout[lane * per_lane + j] = f2bf(x[j] * inv * bf2f(w[lane * per_lane + j]));
}

// ---------------- launchers ----------------

template <bool FUSED_ADD>
static void wide_launch(u16* out, u16* residual, const u16* in, const u16* w,
                        float eps, long rows, int C, hipStream_t s) {
  if (rows == 0) return;
#define LAUNCH_WIDE(NV, WAVES)                                              \
  hipLaunchKernelGGL((rmsnorm_wide_kernel<FUSED_ADD, NV, WAVES>),           \
                     dim3((unsigned)((rows * WAVES + 3) / 4)), dim3(256), 0, \
                     s, out, residual, in, w, eps, rows, C)
  if (rows >= 2048 && C <= 4096) {   // eight waves on every CU
    if (C <= 1024) LAUNCH_WIDE(2, 1);
    else if (C <= 2048) LAUNCH_WIDE(4, 1);
    else LAUNCH_WIDE(8, 1);
  } else if (C <= 2048) LAUNCH_WIDE(1, 4);
  else if (C <= 4096) LAUNCH_WIDE(2, 4);
  else if (C <= 8192) LAUNCH_WIDE(4, 4);
  else LAUNCH_WIDE(8, 4);
#undef LAUNCH_WIDE
}

extern "C" void sutro_rmsnorm(void* out, const void* in, const void* w,
                              float eps, long rows, int C, hipStream_t s) {
  if (C % (int)WAVE == 0 && C <= 256 && C / (int)WAVE <= 4) {
    int waves_per_block = 4;
    long blocks = (rows + waves_per_block - 1) / waves_per_block;
    hipLaunchKernelGGL(rmsnorm_small_kernel, dim3((unsigned)blocks),
                       dim3(waves_per_block * WAVE), 0, s, (u16*)out,
                       (const u16*)in, (const u16*)w, eps, rows, C);
    return;
  }
  wide_launch<false>((u16*)out, nullptr, (const u16*)in, (const u16*)w, eps,
                     rows, C, s);
}

extern "C" void sutro_fused_add_rmsnorm(void* x, void* residual, const void* w,
                                        float eps, long rows, int C,
                                        hipStream_t s) {
  wide_launch<true>((u16*)x, (u16*)residual, (const u16*)x, (const u16*)w, eps,
                    rows, C, s);
}
