// Decode attention of the dense decoders (head size 64 or 128, bf16 or e4m3
// pages): see attn_paged.h for the kernel. Below, probes of the fragment
// layouts and of the stages of a one-wave form of it.
#include "common.h"
#include "attn_paged.h"

#define BS 32
#define PV_PAD 40    // padded row length (elems) for P and Vt tiles

typedef s16x8 bf16frag;

__device__ __forceinline__ f32x4 mfma16(bf16frag a, bf16frag b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// 8 consecutive KV elements at byte pointer p -> bf16 fragment.
// bf16 cache: one 16B load. e4m3 cache: 8B load + native pk converts.
template <bool KV8>
__device__ __forceinline__ bf16frag load_kv_frag(const u8* p) {
  if constexpr (!KV8) return *(const s16x8*)p;
  const u32x2 raw = *(const u32x2*)p;
  float f[8];
  fp8x4_to_f32(raw[0], f);
  fp8x4_to_f32(raw[1], f + 4);
  bf16frag r;
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = (short)f2bf(f[j]);
  return r;
}

template <int D>
struct MfmaSmem {
  u16 qt[16 * D];           // Q^T as [head16][kD], row-swizzled
  u16 vt[D * PV_PAD];       // V^T [dD][pos32+pad]
  u16 p[16 * PV_PAD];       // P [head16][pos32+pad] (1.25 KB)
  float alpha[16];
  float linv[16];
};

// row-local XOR swizzle; mask keeps the offset inside the 2*D-byte row
template <int D>
__device__ __forceinline__ int qt_swz(int head, int byte_in_row) {
  constexpr int mask = (D == 128) ? 15 : 7;
  return head * (2 * D) + (byte_in_row ^ ((head & mask) << 4));
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

// ---- debug probe: run the D=64 decode stages for one (seq, kv_head) and
// dump the vt and p LDS images plus the output, to localize a stage that
// breaks on hardware but not in the CPU simulation (tools/sim_mfma_decode.py)
__global__ void hd64_stage_probe_kernel(
    float* __restrict__ vt_dump,     // [64 * PV_PAD]
    float* __restrict__ p_dump,      // [16 * PV_PAD]
    u16* __restrict__ out,           // [Hq=1, 64]
    const u16* __restrict__ q,       // [1, 64]
    const u16* __restrict__ k_cache, // one page [32, 64]
    const u16* __restrict__ v_cache,
    int L, float scale) {
  constexpr int D = 64;
  const int lane = threadIdx.x & (WAVE - 1);
  __shared__ MfmaSmem<D> smw;
  MfmaSmem<D>* sm = &smw;
  const int lo16 = lane & 15;
  const int hi4 = lane >> 4;
  const int G = 1;
  {
    const int head = lo16;
#pragma unroll
    for (int t = 0; t < D / 32; ++t) {
      const int k0 = hi4 * 8 + t * 32;
      u16x8 val = {};
      if (head < G) {
        const u16* qrow = q + head * D;
#pragma unroll
        for (int j = 0; j < 8; ++j) val[j] = f2bf(bf2f(qrow[k0 + j]) * scale);
      }
      *(u16x8*)((char*)sm->qt + qt_swz<D>(head, k0 * 2)) = val;
    }
  }
  float m_run = -1e30f, l_run = 0.f;
  constexpr int DB = D / 16;
  f32x4 acc[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b) acc[b] = (f32x4)(0.f);
  const int valid = L;
  {
    const u8* vsrc = (const u8*)v_cache;
#pragma unroll
    for (int it = 0; it < (BS * D) / ((int)WAVE * 8); ++it) {
      const int flat = it * (int)WAVE + lane;
      const int pos = flat & 31;
      const int d0 = (flat >> 5) * 8;
      const bf16frag vx = load_kv_frag<false>(vsrc + (pos * D + d0) * 2);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        sm->vt[(d0 + j) * PV_PAD + pos] = (u16)vx[j];
    }
  }
  // dump vt
  for (int i = lane; i < D * PV_PAD; i += WAVE)
    vt_dump[i] = bf2f(sm->vt[i]);
  f32x4 s01[2];
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    f32x4 d = (f32x4)(0.f);
#pragma unroll
    for (int kk = 0; kk < D / 32; ++kk) {
      const u8* krow = (const u8*)k_cache +
                       ((long)(half * 16 + lo16) * D + kk * 32 + hi4 * 8) * 2;
      bf16frag ka = load_kv_frag<false>(krow);
      bf16frag qb = *(const s16x8*)((char*)sm->qt +
                                    qt_swz<D>(lo16, (kk * 32 + hi4 * 8) * 2));
      d = mfma16(ka, qb, d);
    }
    s01[half] = d;
  }
  float sv[8];
#pragma unroll
  for (int half = 0; half < 2; ++half)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int pos = half * 16 + hi4 * 4 + r;
      float x = s01[half][r];
      if (pos >= valid) x = -1e30f;
      sv[half * 4 + r] = x;
    }
  float tmax = sv[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) tmax = fmaxf(tmax, sv[i]);
  tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
  tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
  const float m_new = fmaxf(m_run, tmax);
  const float al = __expf(m_run - m_new);
  m_run = m_new;
  float psum = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    sv[i] = __expf(sv[i] - m_new);
    psum += sv[i];
  }
  psum += __shfl_xor(psum, 16, 64);
  psum += __shfl_xor(psum, 32, 64);
  l_run = l_run * al + psum;
  if (hi4 == 0) sm->alpha[lo16] = al;
#pragma unroll
  for (int half = 0; half < 2; ++half)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      sm->p[lo16 * PV_PAD + half * 16 + hi4 * 4 + r] = f2bf(sv[half * 4 + r]);
  // dump p
  for (int i = lane; i < 16 * PV_PAD; i += WAVE)
    p_dump[i] = bf2f(sm->p[i]);
  float alr[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) alr[r] = sm->alpha[hi4 * 4 + r];
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[b][r] *= alr[r];
  bf16frag pa = *(const s16x8*)(sm->p + lo16 * PV_PAD + hi4 * 8);
#pragma unroll
  for (int b = 0; b < DB; ++b) {
    bf16frag vb = *(const s16x8*)(sm->vt + (b * 16 + lo16) * PV_PAD + hi4 * 8);
    acc[b] = mfma16(pa, vb, acc[b]);
  }
  if (hi4 == 0) sm->linv[lo16] = 1.0f / l_run;
  float li[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) li[r] = sm->linv[hi4 * 4 + r];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int head = hi4 * 4 + r;
    if (head >= G) continue;
    u16* orow = out + head * D;
#pragma unroll
    for (int b = 0; b < DB; ++b) orow[b * 16 + lo16] = f2bf(acc[b][r] * li[r]);
  }
}

extern "C" void sutro_hd64_stage_probe(float* vt_dump, float* p_dump, void* out,
                                       const void* q, const void* k,
                                       const void* v, int L, float scale,
                                       hipStream_t s) {
  hipLaunchKernelGGL(hd64_stage_probe_kernel, dim3(1), dim3(64), 0, s, vt_dump,
                     p_dump, (u16*)out, (const u16*)q, (const u16*)k,
                     (const u16*)v, L, scale);
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
