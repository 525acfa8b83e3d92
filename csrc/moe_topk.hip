// Softmax top-k router of the Qwen3 experts: one wave a token, experts on the
// lanes (NP each), k rounds of a wave-wide arg-max (equal logits: the lower
// index first), weights softmax(logit) / sum of the chosen ones in fp32.
//
// Bound by launches: with the dispatch of moe_dispatch.hip this takes two of them
// a layer (four for long prompts) where softmax, top-k, sort, searchsorted,
// index_add, cumsum, scatters, index puts and wheres of the library took 47: 11
// us instead of about 220 at 128 rows over 32 experts.
//
// Ranks that hold the experts [base, base + n_local) get local numbers; other
// choices come back as n_local with weight 0 (a segment that no GEMM visits).
#include <cfloat>

#include "common.h"

template <int NP>
__global__ void __launch_bounds__(256) moe_topk_kernel(
    int* __restrict__ idx,            // [T, k]
    float* __restrict__ wts,          // [T, k]
    const u16* __restrict__ logits,   // [T, E] bf16
    long T, int E, int k, int base, int n_local) {
  const int lane = threadIdx.x & 63;
  const long t = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  // cmp orders the choice: NaN and -inf logits below every finite one (the
  // lowest float lies below the lowest bf16), chosen and missing experts below
  // those
  float x[NP], cmp[NP];
  float m = -INFINITY;
#pragma unroll
  for (int n = 0; n < NP; ++n) {
    const int e = n * 64 + lane;
    x[n] = e < E ? bf2f(logits[t * E + e]) : -INFINITY;
    cmp[n] = e < E ? (x[n] > -INFINITY ? x[n] : -FLT_MAX) : -INFINITY;
    m = fmaxf(m, x[n]);
  }
  m = wave_max_f32(m);
  float sum = 0.f;
#pragma unroll
  for (int n = 0; n < NP; ++n) sum += expf(x[n] - m);
  sum = wave_sum_f32(sum);
  float total = 0.f, my_p = 0.f;
  int my_e = 0;
  for (int j = 0; j < k; ++j) {
    float bv = -INFINITY;
    int bi = 0;
#pragma unroll
    for (int n = 0; n < NP; ++n)
      if (cmp[n] > bv) {
        bv = cmp[n];
        bi = n * 64 + lane;
      }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ov > bv || (ov == bv && oi < bi)) {
        bv = ov;
        bi = oi;
      }
    }
    const float p = expf(bv - m) / sum;
    total += p;
    if (lane == j) {
      my_e = bi;
      my_p = p;
    }
#pragma unroll
    for (int n = 0; n < NP; ++n)
      if (bi == n * 64 + lane) cmp[n] = -INFINITY;
  }
  if (lane < k) {
    const int e = my_e - base;
    const bool mine = e >= 0 && e < n_local;
    idx[t * k + lane] = mine ? e : n_local;
    wts[t * k + lane] = mine ? my_p / total : 0.f;
  }
}

// k <= 64 and k <= E <= 1024
extern "C" void sutro_moe_topk(int* idx, float* wts, const void* logits, long T,
                               int E, int k, int base, int n_local,
                               hipStream_t s) {
  if (T == 0) return;
#define LAUNCH_TK(NN)                                                       \
  hipLaunchKernelGGL(moe_topk_kernel<NN>, dim3((unsigned)((T + 3) / 4)),    \
                     dim3(256), 0, s, idx, wts, (const u16*)logits, T, E, k, \
                     base, n_local)
  if (E <= 64) LAUNCH_TK(1);
  else if (E <= 128) LAUNCH_TK(2);
  else if (E <= 256) LAUNCH_TK(4);
  else LAUNCH_TK(16);
#undef LAUNCH_TK
}
