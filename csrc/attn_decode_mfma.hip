// Decode attention of the dense decoders (head size 64 or 128, bf16 or e4m3
// pages): see attn_paged.h for the kernel. Below, a probe of the fragment
// layouts it relies on.
#include "common.h"
#include "attn_paged.h"

typedef s16x8 bf16frag;

__device__ __forceinline__ f32x4 mfma16(bf16frag a, bf16frag b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// runs the decode kernel cuts a row's pages into (workspace: n_dec * Hq * runs
// * (head_dim + 2) floats when there is more than one)
extern "C" int sutro_attn_decode_splits(int n_dec, int Hk, int bt_stride) {
  return pa_splits(n_dec, Hk, bt_stride);
}

extern "C" void sutro_attn_decode_mfma(void* out, const void* q,
                                       const void* k_cache,
                                       const void* v_cache,
                                       const int* block_tables,
                                       const int* seq_lens, int bt_stride,
                                       int n_dec, int Hq, int Hk,
                                       int seq_offset, float scale, int kv_fp8,
                                       int head_dim, int nsplit, float* part_o,
                                       float* part_ml, hipStream_t s) {
  PagedArgs A = {};
  A.out = (u16*)out;
  A.ldo = (long)Hq * head_dim;
  A.q = (const u16*)q;
  A.kc = (const u8*)k_cache;
  A.vc = (const u8*)v_cache;
  A.bt = block_tables;
  A.bt_stride = bt_stride;
  A.seq_lens = seq_lens;
  A.Hq = Hq;
  A.Hk = Hk;
  A.scale = scale * PA_LOG2E;
  A.seq_offset = seq_offset;
  A.n_rows = n_dec;
  A.nsplit = nsplit;
  A.part_o = part_o;
  A.part_ml = part_ml;
  if (head_dim == 128) {
    if (kv_fp8) pa_launch_decode<128, true, false>(A, bt_stride, s);
    else pa_launch_decode<128, false, false>(A, bt_stride, s);
  } else {
    if (kv_fp8) pa_launch_decode<64, true, false>(A, bt_stride, s);
    else pa_launch_decode<64, false, false>(A, bt_stride, s);
  }
}

// ---- probe: C[16,16] = A[16,32] @ B[32,16] with the exact frag loaders ----
__global__ void mfma16_probe_kernel(float* __restrict__ c,
                                    const u16* __restrict__ a,   // [16,32]
                                    const u16* __restrict__ b) { // [32,16]
  const int lane = threadIdx.x & (WAVE - 1);
  const int lo16 = lane & 15, hi4 = lane >> 4;
  bf16frag af, bf;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    af[j] = (short)a[lo16 * 32 + hi4 * 8 + j];
    bf[j] = (short)b[(hi4 * 8 + j) * 16 + lo16];
  }
  f32x4 d = (f32x4)(0.f);
  d = mfma16(af, bf, d);
#pragma unroll
  for (int r = 0; r < 4; ++r) c[(hi4 * 4 + r) * 16 + lo16] = d[r];
}

extern "C" void sutro_mfma16_probe(float* c, const void* a, const void* b,
                                   hipStream_t s) {
  hipLaunchKernelGGL(mfma16_probe_kernel, dim3(1), dim3(64), 0, s, c,
                     (const u16*)a, (const u16*)b);
}
