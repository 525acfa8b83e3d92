// Causal prefill attention of the dense decoders over the paged KV cache
// (head size 64 or 128, bf16 or e4m3 pages): see attn_paged.h for the kernel.
#include "common.h"
#include "attn_paged.h"

extern "C" void sutro_attn_prefill(void* out, const void* q,
                                   const void* k_cache, const void* v_cache,
                                   const int* block_tables,
                                   const int* seq_lens, const int* qlocs,
                                   const int* tile_seq, const int* tile_q0,
                                   int n_tiles, int n_seqs, int bt_stride, int Hq,
                                   int Hk, int head_dim, int kv_fp8,
                                   float scale, hipStream_t s) {
  if (n_tiles == 0) return;
  PagedArgs A = {};
  A.out = (u16*)out;
  A.ldo = (long)Hq * head_dim;
  A.q = (const u16*)q;
  A.kc = (const u8*)k_cache;
  A.vc = (const u8*)v_cache;
  A.bt = block_tables;
  A.bt_stride = bt_stride;
  A.seq_lens = seq_lens;
  A.qlocs = qlocs;
  A.Hq = Hq;
  A.Hk = Hk;
  A.scale = scale * PA_LOG2E;
  A.tile_seq = tile_seq;
  A.tile_q0 = tile_q0;
  A.n_tiles = n_tiles;
  if (head_dim == 128) {
    if (kv_fp8) pa_launch_prefill<128, true, false>(A, n_seqs, s);
    else pa_launch_prefill<128, false, false>(A, n_seqs, s);
  } else {
    if (kv_fp8) pa_launch_prefill<64, true, false>(A, n_seqs, s);
    else pa_launch_prefill<64, false, false>(A, n_seqs, s);
  }
}

// ---------------------------------------------------------------------------
// MFMA layout probe: C[32,32] = A[32,16] @ B[16,32] using exactly the fragment
// loaders above. Run on hardware against torch.matmul to pin the layout.
// ---------------------------------------------------------------------------

typedef s16x8 bf16frag;

__device__ __forceinline__ f32x16 mfma32(bf16frag a, bf16frag b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ int d_row(int r, int hi) {
  return (r & 3) + 8 * (r >> 2) + 4 * hi;
}

__global__ void mfma32_probe_kernel(float* __restrict__ c,
                                    const u16* __restrict__ a,   // [32,16]
                                    const u16* __restrict__ b) { // [16,32]
  const int lane = threadIdx.x & (WAVE - 1);
  const int hi = lane >> 5;
  bf16frag af, bf;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    af[j] = (short)a[(lane & 31) * 16 + hi * 8 + j];
    bf[j] = (short)b[(hi * 8 + j) * 32 + (lane & 31)];
  }
  f32x16 d = (f32x16)(0.f);
  d = mfma32(af, bf, d);
#pragma unroll
  for (int r = 0; r < 16; ++r)
    c[d_row(r, hi) * 32 + (lane & 31)] = d[r];
}

extern "C" void sutro_mfma32_probe(float* c, const void* a, const void* b,
                                   hipStream_t s) {
  hipLaunchKernelGGL(mfma32_probe_kernel, dim3(1), dim3(64), 0, s, c,
                     (const u16*)a, (const u16*)b);
}
