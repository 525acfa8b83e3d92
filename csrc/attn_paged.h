// Softmax attention over paged keys and values on the matrix cores: prompt
// pieces (paged_prefill_kernel) and single decoded tokens
// (paged_decode_kernel + paged_join_kernel), bf16 or e4m3 pages of 32 tokens
// [blocks, kv heads, 32, D], head size D = 64 or 128 for keys and values.
// LOCAL adds what layer-list decoders ask for: chunk and window masks with
// kept first keys, a logarithmic distance bias, sinks, output gates and an
// output section.
//
// Both kernels make S^T = K Q^T, so a lane holds the scores of ONE query row:
// softmax is lane-local, the weights are already in the B layout of
// O^T += V^T P^T (with the contraction index permuted alike on both sides) and
// never pass through LDS, and rescaling O is one multiplication by a lane's own
// factor. V^T fragments come out of row-major LDS tiles through the transposed
// read. The running maximum moves only when a score exceeds it by more than
// 2^PA_SLACK: weights then stay below 2^PA_SLACK, which fp32 sums and bf16
// weights hold without loss of relative precision.
//
// Fragment layouts (gfx950), lane l:
//   mfma_f32_32x32x16_bf16: A[l%32][(l/32)*8 + j], B[(l/32)*8 + j][l%32],
//     D[(r&3) + 8*(r>>2) + 4*(l/32)][l%32], r = 0..15
//   mfma_f32_16x16x32_bf16: A[l%16][(l/16)*8 + j], B[(l/16)*8 + j][l%16],
//     D[(l/16)*4 + r][l%16], r = 0..3
//   ds_read_tr16_b64: in a group of 16 lanes lane i addresses the 4 columns
//     (i%4)*4.. of row i/4 and receives column i of those 4 rows.
#pragma once

#define PA_PG 32       // page size
#define PA_KEYS 64     // keys per prefill step (two pages)
#define PA_SLACK 8.f   // log2 of the largest weight against a stale maximum
#define PA_NONE -1e30f // no key seen yet
#define PA_LOG2E 1.4426950408889634f

typedef s16x8 pa_frag;
typedef short pa_s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 pa_bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 pa_bf16x8 __attribute__((ext_vector_type(8)));
typedef float pa_f32x8 __attribute__((ext_vector_type(8)));

struct PagedArgs {
  u16* out;             // row t: out + t * ldo + out_off + head * D
  long ldo;
  int out_off;
  const u16* q;         // [T, Hq, D]
  const u8* kc;         // pages
  const u8* vc;
  const int* bt;        // [S, bt_stride]
  int bt_stride;
  const int* seq_lens;  // [S]
  const int* qlocs;     // [S + 1]
  int Hq, Hk;
  float scale;          // times log2(e)
  // prefill: one entry per 32 rows of new tokens
  const int* tile_seq;
  const int* tile_q0;
  int n_tiles, hpb, rpb;  // heads and 32-row blocks of a workgroup
  // decode: rows t0 .. t0 + n_rows, row t of sequence token_seq[t] or
  // seq_offset + t - t0
  const int* token_seq;
  int seq_offset, n_rows, nsplit;
  long t0;
  float* part_o;        // [n_rows * Hq][nsplit][D]
  float* part_ml;       // [n_rows * Hq][nsplit][2]
  // LOCAL
  int chunk, window, keep_first;
  const float* r1;      // [Hq] distance bias r1 * ln(1 + r2 * distance)
  const float* r2;
  int sink;
  const float* sink_w;  // [Hq] or null (0)
  const u16* proj;      // gate logits at column gate_off
  long ld;
  int gate_off, gate_n;
  float out_scale;
};

__device__ __forceinline__ f32x16 pa_mfma32(pa_frag a, pa_frag b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 pa_mfma16(pa_frag a, pa_frag b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ pa_frag pa_pack8(pa_f32x8 v) {
  return __builtin_bit_cast(pa_frag, __builtin_convertvector(v, pa_bf16x8));
}
__device__ __forceinline__ u32x2 pa_pack4(f32x4 v) {
  return __builtin_bit_cast(u32x2, __builtin_convertvector(v, pa_bf16x4));
}
__device__ __forceinline__ void pa_glds16(const void* g, void* lds) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) u32*)g,
      (__attribute__((address_space(3))) u32*)lds, 16, 0, 0);
}
// transposed reads of rows base..base+3 and base+8.. (or +16..) of a V tile
__device__ __forceinline__ pa_frag pa_tr(const char* a, const char* b) {
  const pa_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) pa_s16x4*)a);
  const pa_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) pa_s16x4*)b);
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
// 8 cached elements as bf16
template <bool KV8>
__device__ __forceinline__ u16x8 pa_cached8(const u8* p) {
  if constexpr (!KV8) {
    return *(const u16x8*)p;
  } else {
    const u32x2 raw = *(const u32x2*)p;
    float f[8];
    fp8x4_to_f32(raw[0], f);
    fp8x4_to_f32(raw[1], f + 4);
    return __builtin_bit_cast(
        u16x8, pa_pack8(pa_f32x8{f[0], f[1], f[2], f[3], f[4], f[5], f[6],
                                 f[7]}));
  }
}
// Tiles in LDS are row-major; 16-byte chunks are XOR-swizzled by the row so
// that 8 rows of one chunk (keys, read in 16-byte fragments) and 4 rows of two
// neighbouring chunks (values, read transposed) lie on different banks.
__device__ __forceinline__ int pa_kchunk(int row, int c) { return c ^ (row & 7); }
__device__ __forceinline__ int pa_vchunk(int row, int c) {
  return c ^ ((row & 3) << 1);
}

__device__ __forceinline__ int pa_lower(const PagedArgs& A, int p, int& kept) {
  int lo = 0;
  if (A.chunk > 0) lo = (p / A.chunk) * A.chunk;
  kept = lo;              // kept first keys: [kept, keep_first)
  if (A.window > 0) lo = max(lo, p - A.window + 1);
  return lo;
}

// ---------------------------------------------------------------------------
// Single tokens. One workgroup of 4 waves per (row, kv head, run of pages); the
// G <= 16 query heads of the kv head are the 16 columns of the products. The
// waves take the run's pages in turn, each with the next page's K and V on the
// way in registers while this one is computed (V passes through the wave's own
// LDS tile to be read transposed), and their partial results meet in LDS. Few
// rows over long contexts would leave most of the chip idle: their pages are
// cut into up to nsplit runs of at least PA_RUN pages, whose partial results
// paged_join_kernel joins. A context of one run is finished here.
//
// Bound by memory: K and V of a row are read once. One wave a row, each page
// loaded and then computed, took 1.9 us a page; a call now takes (with the
// join) 28 us instead of 2390 for one row of 40 k keys and 4 kv heads (82 MB,
// 3 TB/s), 24 instead of 314 for 7 rows of 3 k e4m3 keys and 8 heads, 24
// instead of 128 for 16 rows of 2 k keys and 4 heads, and 37 instead of 41 for
// 256 rows of 130 keys and 8 heads (138 MB, 3.7 TB/s, one run each). Runs of 8
// pages give every wave two pages, the fewest that hide one load behind
// another's work.
// ---------------------------------------------------------------------------
#define PA_RUN 8

// runs of a context of n pages: (pages per run, number of runs)
__device__ __forceinline__ int pa_run_pages(int n, int nsplit) {
  return max(PA_RUN, (n + nsplit - 1) / nsplit);
}

struct PagedSpan {  // the pages of a row: kept ones first, then the window's
  int s, p, lo, c_lo, pg0, kf0, n_kept, total;
};
template <bool LOCAL>
__device__ __forceinline__ PagedSpan pa_span(const PagedArgs& A, int i) {
  PagedSpan v;
  const long t = A.t0 + i;
  v.s = A.token_seq ? A.token_seq[t] : A.seq_offset + i;
  v.p = A.token_seq ? A.seq_lens[v.s] - (int)(A.qlocs[v.s + 1] - t)
                    : A.seq_lens[v.s] - 1;
  v.lo = v.c_lo = v.pg0 = v.kf0 = v.n_kept = 0;
  if (LOCAL) {
    v.lo = pa_lower(A, v.p, v.c_lo);
    v.pg0 = v.lo / PA_PG;
    v.kf0 = v.c_lo / PA_PG;
    v.n_kept = max(min(v.pg0, (A.keep_first + PA_PG - 1) / PA_PG) - v.kf0, 0);
  }
  v.total = v.n_kept + v.p / PA_PG + 1 - v.pg0;
  return v;
}

// final factor and store of column c of (row, head)
template <bool LOCAL>
__device__ __forceinline__ void pa_store(const PagedArgs& A, long t, int hq,
                                         int D, int c, float o, float l) {
  float f = l > 0.f ? 1.0f / l : 0.f;
  if (LOCAL) {
    f *= A.out_scale;
    if (A.gate_off >= 0) {
      const u16* gp = A.proj + t * A.ld + A.gate_off + (long)hq * A.gate_n;
      f *= 1.f / (1.f + expf(-bf2f(gp[A.gate_n > 1 ? c : 0])));
    }
  }
  A.out[t * A.ldo + A.out_off + (long)hq * D + c] = f2bf(o * f);
}

template <int D, bool KV8, bool LOCAL>
__global__ void __launch_bounds__(256) paged_decode_kernel(PagedArgs A) {
  constexpr int ES = KV8 ? 1 : 2;
  constexpr int KK = D / 32;                 // k-steps of the scores
  constexpr int DB = D / 16;                 // 16-column blocks of O
  constexpr int VL = PA_PG * D / (64 * 8);   // 8-element pieces a lane stages
  constexpr int VT = PA_PG * D * 2;          // bytes of a V page in LDS
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lo16 = lane & 15, g4 = lane >> 4;
  const int G = A.Hq / A.Hk;
  const int kh = blockIdx.x % A.Hk;
  const int i = blockIdx.x / A.Hk;
  const PagedSpan v = pa_span<LOCAL>(A, i);
  const int run = pa_run_pages(v.total, A.nsplit);
  const int begin = blockIdx.y * run;
  if (begin >= v.total) return;
  const int end = min(v.total, begin + run);
  const bool alone = run >= v.total;
  const long t = A.t0 + i;

  // V tiles of the waves, then (behind a barrier) their results [4][16][D]
  __shared__ __attribute__((aligned(16))) char smem[4 * 16 * D * 4];
  __shared__ float ml[4][16][2];
  char* vt = smem + w * VT;

  pa_frag qb[KK];   // B: query head lo16, dims kk*32 + g4*8; zero past G
  {
    const u16* qp = A.q + (t * A.Hq + kh * G + min(lo16, G - 1)) * D + g4 * 8;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
      qb[kk] = lo16 < G ? *(const s16x8*)(qp + kk * 32) : (s16x8)(0);
  }
  const int hq = kh * G + min(lo16, G - 1);
  const float r1 = LOCAL && A.r1 ? A.r1[hq] : 0.f;
  const float r2 = LOCAL && A.r1 ? A.r2[hq] : 0.f;
  f32x4 acc[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b) acc[b] = (f32x4)(0.f);
  float m_run = PA_NONE, l_run = 0.f;

  const int* table = A.bt + (long)v.s * A.bt_stride;
  auto page_of = [&](int x) {
    return x < v.n_kept ? v.kf0 + x : v.pg0 + (x - v.n_kept);
  };
  u16x8 kx[2 * KK], vx[VL];
  auto load = [&](int x) {
    const long base =
        (((long)table[page_of(x)] * A.Hk + kh) * PA_PG) * D;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
        kx[h * KK + kk] = pa_cached8<KV8>(
            A.kc + (base + (h * 16 + lo16) * D + kk * 32 + g4 * 8) * ES);
#pragma unroll
    for (int j = 0; j < VL; ++j)
      vx[j] = pa_cached8<KV8>(A.vc + (base + (j * 64 + lane) * 8) * ES);
  };
  // V fragment addresses: rows 4*g4 + ti/4 (+16), columns of 16-block b
  int vad[4];
#pragma unroll
  for (int o = 0; o < 4; ++o)
    vad[o] = (4 * g4 + (lo16 >> 2)) * (2 * D) +
             pa_vchunk(lo16 >> 2, o * 2 + ((lo16 & 3) >> 1)) * 16 +
             (lo16 & 1) * 8;

  int x = begin + w;
  if (x < end) load(x);
  for (; x < end; x += 4) {
    // this page's V into the wave's tile, then the next page's loads
#pragma unroll
    for (int j = 0; j < VL; ++j) {
      const int row = (j * 64 + lane) / (D / 8), c = (j * 64 + lane) % (D / 8);
      *(u16x8*)(vt + row * (2 * D) + pa_vchunk(row, c) * 16) = vx[j];
    }
    f32x4 sc[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      sc[h] = (f32x4)(0.f);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
        sc[h] = pa_mfma16(__builtin_bit_cast(pa_frag, kx[h * KK + kk]), qb[kk],
                          sc[h]);
    }
    const int kv0 = page_of(x) * PA_PG;
    if (x + 4 < end) load(x + 4);
    // ---- this lane: head lo16, keys kv0 + h*16 + g4*4 + r
    float tmax = PA_NONE;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kp = kv0 + h * 16 + g4 * 4 + r;
        float z = sc[h][r] * A.scale;
        bool vis = kp <= v.p;
        if (LOCAL) {
          if (A.r1)
            z -= r1 * __builtin_amdgcn_logf(1.f +
                                            r2 * (float)max(v.p - kp, 0));
          vis = vis && (kp >= v.lo || (kp < A.keep_first && kp >= v.c_lo));
        }
        sc[h][r] = vis ? z : PA_NONE;
        tmax = fmaxf(tmax, sc[h][r]);
      }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float m_new = fmaxf(m_run, tmax);
    const float al = __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    // kept pages need not hold a visible key: weights are exp2(-1e30) = 0 then
    const float m_sub = LOCAL && m_new < 0.1f * PA_NONE ? 0.f : m_new;
    pa_f32x8 p;
    l_run *= al;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      p[j] = __builtin_amdgcn_exp2f(sc[j >> 2][j & 3] - m_sub);
      l_run += p[j];
    }
    const pa_frag pb = pa_pack8(p);
#pragma unroll
    for (int b = 0; b < DB; ++b) {
      const char* at = vt + vad[b & 3] + (b >> 2) * 128;
      f32x4 a = acc[b] * al;
      acc[b] = pa_mfma16(pa_tr(at, at + 16 * 2 * D), pb, a);
    }
  }
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);

  __syncthreads();   // the V tiles are done with
  float* res = (float*)smem;
  if (g4 == 0) {
    ml[w][lo16][0] = m_run;
    ml[w][lo16][1] = l_run;
  }
  if (lo16 < G) {
#pragma unroll
    for (int b = 0; b < DB; ++b)
      *(f32x4*)(res + (w * 16 + lo16) * D + b * 16 + g4 * 4) = acc[b];
  }
  __syncthreads();
  for (int z = threadIdx.x; z < G * D; z += 256) {
    const int h = z / D, c = z % D;
    float m = fmaxf(fmaxf(ml[0][h][0], ml[1][h][0]),
                    fmaxf(ml[2][h][0], ml[3][h][0]));
    float l = 0.f, o = 0.f, sk = 0.f;
    const bool snk = LOCAL && A.sink && alone;
    if (snk) {
      sk = A.sink_w ? A.sink_w[kh * G + h] * PA_LOG2E : 0.f;
      m = fmaxf(m, sk);
      l = __builtin_amdgcn_exp2f(sk - m);
    }
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      const float f = __builtin_amdgcn_exp2f(ml[y][h][0] - m);
      l += f * ml[y][h][1];
      o += f * res[(y * 16 + h) * D + c];
    }
    if (alone) {
      pa_store<LOCAL>(A, t, kh * G + h, D, c, o, l);
    } else {
      const long at = ((long)i * A.Hq + kh * G + h) * A.nsplit + blockIdx.y;
      A.part_o[at * D + c] = o;
      if (c == 0) {
        A.part_ml[at * 2] = m;
        A.part_ml[at * 2 + 1] = l;
      }
    }
  }
}

// Joins the runs of one (row, head). The threads of a column share its runs:
// one thread a column walked up to 157 of them one after the other, 48 us at
// 40 k keys against 20 us for the kernel above.
#define PA_JOIN 512
#define PA_MOST_RUNS 256
template <int D, bool LOCAL>
__global__ void __launch_bounds__(PA_JOIN) paged_join_kernel(PagedArgs A) {
  constexpr int SH = PA_JOIN / D;   // threads a column
  const int i = blockIdx.x / A.Hq, hq = blockIdx.x % A.Hq;
  const PagedSpan v = pa_span<LOCAL>(A, i);
  const int run = pa_run_pages(v.total, A.nsplit);
  const int n = (v.total + run - 1) / run;
  if (n <= 1) return;               // finished by the kernel above
  __shared__ float wgt[PA_MOST_RUNS], red[PA_JOIN], lw[PA_JOIN / 64];
  const long at = ((long)i * A.Hq + hq) * A.nsplit;
  const float* ml = A.part_ml + at * 2;
  const int c = threadIdx.x % D, sh = threadIdx.x / D;
  float m = PA_NONE;
  for (int y = threadIdx.x & 63; y < n; y += 64) m = fmaxf(m, ml[2 * y]);
  m = wave_max_f32(m);              // every wave on its own
  float sk = 0.f;
  if (LOCAL && A.sink) {
    sk = A.sink_w ? A.sink_w[hq] * PA_LOG2E : 0.f;
    m = fmaxf(m, sk);
  }
  float l = 0.f;
  for (int y = threadIdx.x; y < n; y += PA_JOIN) {
    wgt[y] = __builtin_amdgcn_exp2f(ml[2 * y] - m);
    l += wgt[y] * ml[2 * y + 1];
  }
  l = wave_sum_f32(l);
  if ((threadIdx.x & 63) == 0) lw[threadIdx.x >> 6] = l;
  __syncthreads();
  float o = 0.f;
#pragma unroll 4
  for (int y = sh; y < n; y += SH)
    o += wgt[y] * A.part_o[(at + y) * D + c];
  red[threadIdx.x] = o;
  __syncthreads();
  if (sh > 0) return;
  l = LOCAL && A.sink ? __builtin_amdgcn_exp2f(sk - m) : 0.f;
#pragma unroll
  for (int y = 0; y < PA_JOIN / 64; ++y) l += lw[y];
  o = 0.f;
#pragma unroll
  for (int y = 0; y < SH; ++y) o += red[y * D + c];
  pa_store<LOCAL>(A, A.t0 + i, hq, D, c, o, l);
}

// runs to cut contexts of up to max_pages pages into: as many as give every CU
// four workgroups, none shorter than PA_RUN pages
static inline int pa_splits(long rows, int Hk, int max_pages) {
  const long items = rows * Hk;
  const long want = (1024 + items - 1) / (items > 0 ? items : 1);
  const long most = (max_pages + PA_RUN - 1) / PA_RUN;
  long n = want < most ? want : most;
  if (n > PA_MOST_RUNS) n = PA_MOST_RUNS;
  return n < 1 ? 1 : (int)n;
}

template <int D, bool KV8, bool LOCAL>
static inline void pa_launch_decode(const PagedArgs& A, hipStream_t s) {
  hipLaunchKernelGGL((paged_decode_kernel<D, KV8, LOCAL>),
                     dim3((unsigned)(A.n_rows * A.Hk), (unsigned)A.nsplit),
                     dim3(256), 0, s, A);
  if (A.nsplit > 1)
    hipLaunchKernelGGL((paged_join_kernel<D, LOCAL>),
                       dim3((unsigned)(A.n_rows * A.Hq)), dim3(PA_JOIN), 0, s,
                       A);
}
