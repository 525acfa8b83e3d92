// Layout of routed experts: (token, choice) pairs into per-expert segments that
// are padded to the tile of the expert GEMMs, on the device (no host round
// trip, no sort; launches depend on sizes alone, so decode steps can be
// captured). Both extensions compile this file.
#include "common.h"

// ---- moe_dispatch ----------------------------------------------------------
// The place of a pair inside its expert's segment comes from an LDS counter, so
// it depends on timing; a row's result does not depend on its place, and every
// pair finds its row through padpos. With `ids`, idx is a table [vocab, k] and
// pair i uses its row ids[i / k]. With `row_w`, row r of pair i also gets
// row_w[r] = wts[i] (0 for padding rows).
__device__ __forceinline__ int pair_expert(const int* __restrict__ idx,
                                           const long* __restrict__ ids, int i,
                                           int t, int k) {
  return ids ? idx[ids[t] * k + (i - t * k)] : idx[i];
}

// Small batches: everything in one 1024-thread workgroup.
__global__ void __launch_bounds__(1024) moe_dispatch_kernel(
    int* __restrict__ row_tok, int* __restrict__ tile_off,
    int* __restrict__ counts, int* __restrict__ padpos,
    const int* __restrict__ idx, const long* __restrict__ ids, int n_pairs,
    int k, int E, int bm, long n_rows, const float* __restrict__ wts,
    float* __restrict__ row_w) {
  extern __shared__ int smi[];
  int* cnt = smi;          // [E] pairs per expert, then a running cursor
  int* start = smi + E;    // [E + 1] first padded row of each segment
  const int tid = threadIdx.x;
  for (int e = tid; e < E; e += 1024) cnt[e] = 0;
  __syncthreads();
  for (int i = tid; i < n_pairs; i += 1024)
    atomicAdd(&cnt[pair_expert(idx, ids, i, i / k, k)], 1);
  for (long i = tid; i < n_rows; i += 1024) {
    row_tok[i] = -1;
    if (row_w) row_w[i] = 0.f;
  }
  __syncthreads();
  if (tid == 0) {
    int off = 0;
    for (int e = 0; e < E; ++e) {
      start[e] = off;
      off += (cnt[e] + bm - 1) / bm * bm;
    }
    start[E] = off;
  }
  __syncthreads();
  for (int e = tid; e <= E; e += 1024) {
    tile_off[e] = start[e] / bm;
    if (e < E) counts[e] = cnt[e];
  }
  __syncthreads();
  for (int e = tid; e < E; e += 1024) cnt[e] = 0;
  __syncthreads();
  for (int i = tid; i < n_pairs; i += 1024) {
    const int t = i / k, e = pair_expert(idx, ids, i, t, k);
    const int r = start[e] + atomicAdd(&cnt[e], 1);
    row_tok[r] = t;
    padpos[i] = r;
    if (row_w) row_w[r] = wts[i];
  }
}

// Large batches, in three launches over runs of DCH pairs: every run counts
// its experts; one workgroup turns the counts into segment starts and into
// every run's first place inside each segment; every run places its pairs.
#define DCH 2048

__global__ void __launch_bounds__(256) moe_count_kernel(
    int* __restrict__ hist, int* __restrict__ row_tok,
    const int* __restrict__ idx, const long* __restrict__ ids, int n_pairs,
    int k, int E, long n_rows, float* __restrict__ row_w) {
  extern __shared__ int smi[];
  for (int e = threadIdx.x; e < E; e += 256) smi[e] = 0;
  __syncthreads();
  int ex[DCH / 256];
#pragma unroll
  for (int n = 0; n < DCH / 256; ++n) {
    const int i = blockIdx.x * DCH + n * 256 + threadIdx.x;
    ex[n] = i < n_pairs ? pair_expert(idx, ids, i, i / k, k) : -1;
  }
#pragma unroll
  for (int n = 0; n < DCH / 256; ++n)
    if (ex[n] >= 0) atomicAdd(&smi[ex[n]], 1);
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n_rows;
       i += (long)gridDim.x * 256) {
    row_tok[i] = -1;
    if (row_w) row_w[i] = 0.f;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += 256)
    hist[(long)blockIdx.x * E + e] = smi[e];
}

__global__ void __launch_bounds__(1024) moe_offsets_kernel(
    int* __restrict__ hist, int* __restrict__ tile_off,
    int* __restrict__ counts, int runs, int E, int bm) {
  extern __shared__ int smi[];  // [E] totals
  for (int e = threadIdx.x; e < E; e += 1024) {
    int sum = 0;
#pragma unroll 8
    for (int b = 0; b < runs; ++b) {
      const int c = hist[(long)b * E + e];
      hist[(long)b * E + e] = sum;
      sum += c;
    }
    smi[e] = sum;
    counts[e] = sum;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int off = 0;
    for (int e = 0; e < E; ++e) {
      tile_off[e] = off;
      off += (smi[e] + bm - 1) / bm;
    }
    tile_off[E] = off;
  }
}

__global__ void __launch_bounds__(256) moe_place_kernel(
    int* __restrict__ row_tok, int* __restrict__ padpos,
    const int* __restrict__ hist, const int* __restrict__ tile_off,
    const int* __restrict__ idx, const long* __restrict__ ids, int n_pairs,
    int k, int E, int bm, const float* __restrict__ wts,
    float* __restrict__ row_w) {
  extern __shared__ int smi[];  // [E] next row of each segment
  for (int e = threadIdx.x; e < E; e += 256)
    smi[e] = tile_off[e] * bm + hist[(long)blockIdx.x * E + e];
  __syncthreads();
  int ex[DCH / 256];
#pragma unroll
  for (int n = 0; n < DCH / 256; ++n) {
    const int i = blockIdx.x * DCH + n * 256 + threadIdx.x;
    ex[n] = i < n_pairs ? pair_expert(idx, ids, i, i / k, k) : -1;
  }
#pragma unroll
  for (int n = 0; n < DCH / 256; ++n) {
    const int i = blockIdx.x * DCH + n * 256 + threadIdx.x;
    if (ex[n] < 0) continue;
    const int r = atomicAdd(&smi[ex[n]], 1);
    row_tok[r] = i / k;
    padpos[i] = r;
    if (row_w) row_w[r] = wts[i];
  }
}

// ints of scratch the launch needs (0: none)
extern "C" long mix_moe_dispatch_scratch(long n_pairs, int E) {
  return n_pairs < 4 * DCH ? 0 : (n_pairs + DCH - 1) / DCH * E;
}

extern "C" void mix_moe_dispatch(int* row_tok, int* tile_off, int* counts,
                                 int* padpos, const int* idx, const long* ids,
                                 long n_pairs, int k, int E, int bm,
                                 long n_rows, int* scratch, const float* wts,
                                 float* row_w, hipStream_t s) {
  if (!scratch) {
    const size_t smem = (size_t)(2 * E + 1) * sizeof(int);
    hipLaunchKernelGGL(moe_dispatch_kernel, dim3(1), dim3(1024), smem, s,
                       row_tok, tile_off, counts, padpos, idx, ids,
                       (int)n_pairs, k, E, bm, n_rows, wts, row_w);
    return;
  }
  const int runs = (int)((n_pairs + DCH - 1) / DCH);
  const size_t smem = (size_t)E * sizeof(int);
  hipLaunchKernelGGL(moe_count_kernel, dim3(runs), dim3(256), smem, s, scratch,
                     row_tok, idx, ids, (int)n_pairs, k, E, n_rows, row_w);
  hipLaunchKernelGGL(moe_offsets_kernel, dim3(1), dim3(1024), smem, s, scratch,
                     tile_off, counts, runs, E, bm);
  hipLaunchKernelGGL(moe_place_kernel, dim3(runs), dim3(256), smem, s, row_tok,
                     padpos, scratch, tile_off, idx, ids, (int)n_pairs, k, E,
                     bm, wts, row_w);
}
