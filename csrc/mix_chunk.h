// Linear recurrences with one decay per head, S <- a S + b k v^T, o = S^T q, over
// chunks of 32 tokens on the matrix cores (decay_scan of mix_decay.hip, mLSTM of
// mix_mlstm.hip). With P_t the product of a chunk's decays up to token t,
// L_ti that of the tokens behind i up to t and R_i that of all behind i:
//   o_t = P_t (S0^T q_t) + sum_{i<=t} (q_t . k_i) L_ti (b_i v_i)
//   S   = P_32 S0 + sum_i k_i (R_i b_i v_i)^T
// Decays are multiplied up (no logarithms, no quotients), so a decay of zero and
// one above 1 are ordinary numbers.
//
// fp32 operands are split into three bf16 terms (8 + 8 + 8 bits: exact) and a
// product is the sum of the six terms above 2^-24 of it, added from the smallest
// up in fp32; bf16 operands (mLSTM's q, k and v) are one term. S is rounded once a
// chunk and term, not once a token. Errors against 64 bits, scan and chunks, 4096 tokens
// of 128 x 64: decays near 1 (0.9987654, 0.99 to 1, 0.9999 to 1) read-out 7.5e-8 to 1.3e-6
// and 8.3e-8 to 2.0e-7, state 3.6e-7 to 1.6e-6 and 7.2e-8 to 2.2e-7; decays anywhere
// from 0 to 1, where both are single roundings, 5.2e-8 (keys that resemble each other),
// 7.2e-8 (behind silu) and 9.8e-8 (independent), and 8.3e-8 to 8.9e-8, state 4.4e-8 to
// 4.7e-8 and 4.4e-8 to 5.2e-8.
// Infinities and NaN do not survive a split: a sequence in which any read-out or state is
// not finite is done once more, token by token (chunk_serial), from the state that is
// still in memory, by each wave with such a column and without LDS: 16 rows of 1024 tokens
// of 32 heads 441 us, with a NaN in one of them 1824, in all 4517; 1 row of 4000 of 16
// heads 526, 6464 and 7397.
//
// A wave owns 16 columns of S in registers, laid out as the products leave them (row
// dk = 16 m + 4 (lane / 16) + r of tile m, column lane % 16).
// The contraction over dk is permuted alike in q, k (in LDS, 32 at a time:
// place 8 g + 4 hi + r holds 16 hi + 4 g + r) and S, and the one over tokens in v,
// so neither S nor v passes through LDS; k^T comes from the rows of k through the
// transposed read.
//
// The scan does four fp32 operations an element of S and token, at 70 % of the VALU's
// rate, one token behind the other; here they are 80,000 operations a token of a head
// of 128 x 128 on the matrix cores, six times over. Times, scan and chunks: 13 rows of
// 30,001 tokens in all, 16 heads of 128 x 128, 1280 and 495 us; 16 rows of 1024, 32
// heads, 990 and 375; 1 row of 4000, 16 heads, 1240 and 532; MLSTM with its gates, 61 rows
// of 30,000 in all, 8 heads, 891 and 237. What bounds it: a chunk takes 9950 cycles of a CU, its
// SIMDs issue VALU instructions in 5900 of them (the splits above all) and are at
// products in 3750, and the two overlap little. Slower: waves of 32 columns (half the
// reads of LDS, but half the waves: 620 instead of 350 us), workgroups without
// producers (652 instead of 455), one barrier a chunk with three buffers (the same).
#pragma once

#include <type_traits>

#include "mix_common.h"
#include "lds_limit.h"

#define CH_T 32

typedef short ch_s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 ch_bf16x2 __attribute__((ext_vector_type(2)));

struct ChunkArgs {
  float* o;             // [T, H, ov]
  const void* q;        // rows ldq apart, heads dense: fp32, or bf16 (MLSTM)
  const void* k;
  const void* v;
  long ldq, ldk, ldv;
  const float* a;       // [T, H], or [H] with lda = 0
  long lda;
  const float* b;       // [T, H] or null (1)
  const float* skip;    // [H] or null: o += skip v
  float* state;         // [slots, H, dk, ov]
  const int* state_slots;
  const int* qlocs;
  const int* seq_lens;
  int S, H, G, dk, dv;
  int ov;               // dv; MLSTM dv + 1: the last column's value is 1
  int cgs;              // column groups of a head
  int n_wg, run;        // see ch_wg
  float qscale;         // of the read-out
  int least;            // new tokens from which a sequence is done here
};

__device__ __forceinline__ f32x4 ch_mfma(s16x8 a, s16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// two fp32 numbers -> their bf16 terms of rank n, leaving the rest in x, y
__device__ __forceinline__ u32 ch_term(float& x, float& y) {
  const f32x2 v = {x, y};
  const u32 t = __builtin_bit_cast(u32, __builtin_convertvector(v, ch_bf16x2));
  x -= __uint_as_float(t << 16);
  y -= __uint_as_float(t & 0xffff0000u);
  return t;
}

// N / 2 words of each term (N = 4 or 8)
template <int NT, int N>
__device__ __forceinline__ void ch_split(u32 (&w)[NT][N / 2],
                                         const float (&x)[N]) {
#pragma unroll
  for (int j = 0; j < N; j += 2) {
    float a = x[j], b = x[j + 1];
#pragma unroll
    for (int n = 0; n < NT; ++n) w[n][j / 2] = ch_term(a, b);
  }
}
template <int NT>
__device__ __forceinline__ void ch_frag(s16x8 (&f)[NT], const float (&x)[8]) {
  u32 w[NT][4];
  ch_split<NT, 8>(w, x);
#pragma unroll
  for (int n = 0; n < NT; ++n)
    f[n] = __builtin_bit_cast(s16x8, (u32x4){w[n][0], w[n][1], w[n][2], w[n][3]});
}

// sums of products by the order of their terms: the large ones are added to few
// times, and three short chains follow one another faster than a long one
struct ChSum {
  f32x4 c[3];
  __device__ __forceinline__ ChSum() { c[0] = c[1] = c[2] = (f32x4)(0.f); }
  template <int NA, int NB>
  __device__ __forceinline__ void mul(const s16x8 (&a)[NA],
                                      const s16x8 (&b)[NB]) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int o = 2; o >= i; --o)
        if (i < NA && o - i < NB) c[o] = ch_mfma(a[i], b[o - i], c[o]);
  }
  __device__ __forceinline__ f32x4 total() const { return c[0] + (c[1] + c[2]); }
};

// the same with the two small orders in one sum
struct ChSum2 {
  f32x4 c[2];
  __device__ __forceinline__ ChSum2() { c[0] = c[1] = (f32x4)(0.f); }
  template <int NA, int NB>
  __device__ __forceinline__ void mul(const s16x8 (&a)[NA],
                                      const s16x8 (&b)[NB]) {
#pragma unroll
    for (int o = 2; o >= 0; --o)
#pragma unroll
      for (int i = 0; i <= o; ++i)
        if (i < NA && o - i < NB)
          c[o > 0] = ch_mfma(a[i], b[o - i], c[o > 0]);
  }
  __device__ __forceinline__ f32x4 total() const { return c[0] + c[1]; }
};

// lane n of a row of 16 <- lane n - N (shr) or n + N (shl), 1 from outside
template <int CTRL>
__device__ __forceinline__ float ch_dpp1(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(
      __float_as_int(1.f), __float_as_int(v), CTRL, 0xF, 0xF, false));
}
// product of a row's lanes up to this one, or from this one on
__device__ __forceinline__ float ch_prefix(float v) {
  v *= ch_dpp1<0x111>(v);
  v *= ch_dpp1<0x112>(v);
  v *= ch_dpp1<0x114>(v);
  return v * ch_dpp1<0x118>(v);
}
__device__ __forceinline__ float ch_suffix(float v) {
  v *= ch_dpp1<0x101>(v);
  v *= ch_dpp1<0x102>(v);
  v *= ch_dpp1<0x104>(v);
  return v * ch_dpp1<0x108>(v);
}
// lane N of the row of 16
template <int N>
__device__ __forceinline__ float ch_lane(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(
      0, __float_as_int(v), 0x150 + N, 0xF, 0xF, true));
}

// byte of place (row t, 16-byte piece c) in a plane of rows of DK bf16. Pieces are
// mixed with the row: equal pieces of eight rows (row reads) fill 128 bytes of banks,
// and so do four neighbouring pieces of two rows (transposed reads, writes).
template <int DK>
__device__ __forceinline__ int ch_place(int t, int c) {
  return t * (DK * 2) + ((c ^ ((DK == 128 ? t & 8 : 0) | ((t & 1) << 2) |
                               ((t >> 1) & 3))) << 4);
}

// Rows of a chunk through buffer accesses: what lies past the chunk's last row (or at
// CH_OUT) reads as zero and is not written, without branches
#define CH_OUT 0x80000000u
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ch_rows(const void* p,
                                                          u32 bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, bytes, 0x00027000);
}
template <typename T>
__device__ __forceinline__ T ch_load(__amdgpu_buffer_rsrc_t r, u32 at) {
  if constexpr (sizeof(T) == 16)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0));
  else if constexpr (sizeof(T) == 8)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, at, 0, 0));
  else if constexpr (sizeof(T) == 4)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, at, 0, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b16(r, at, 0, 0));
}

// a uniform number the compiler knows nothing of: row pointers are made anew in every
// chunk instead of being carried along, in two registers a lane, for each load
__device__ __forceinline__ int ch_plain(int v) {
  asm("" : "+s"(v));
  return v;
}

// Token by token, without LDS, for sequences with numbers that are not finite:
// eight lanes a column, DK / 8 rows each
template <int DK, bool MLSTM>
__device__ __forceinline__ void chunk_serial(const ChunkArgs& A, int s, int h,
                                          int col0, int ncols, int lane) {
  const int q0 = A.qlocs[s], n = A.qlocs[s + 1] - q0;
  const bool old = A.seq_lens[s] > n;
  const int g = h / (A.H / A.G), r = lane & 7;
  float* Sg = A.state + ((long)A.state_slots[s] * A.H + h) * A.dk * A.ov;
  for (int c = col0 + (lane >> 3); c < col0 + ncols; c += 8) {
    if (c >= A.ov) continue;
    float S[DK / 8];
#pragma unroll
    for (int m = 0; m < DK / 8; ++m) {
      const int d = m * 8 + r;
      S[m] = old && d < A.dk ? Sg[(long)d * A.ov + c] : 0.f;
    }
    for (int t = q0; t < q0 + n; ++t) {
      const float at = A.a[(long)t * A.lda + h];
      const float bt = A.b ? A.b[(long)t * A.H + h] : 1.f;
      float vt;
      if (MLSTM)
        vt = c < A.dv ? bf2f(((const u16*)A.v)[t * A.ldv + (long)h * A.dv + c])
                      : 1.f;
      else
        vt = ((const float*)A.v)[t * A.ldv + (long)h * A.dv + c];
      float sum = 0.f;
#pragma unroll
      for (int m = 0; m < DK / 8; ++m) {
        const int d = m * 8 + r;
        float kt = 0.f, qt = 0.f;
        if (d < A.dk) {
          if (MLSTM) {
            kt = bf2f(((const u16*)A.k)[t * A.ldk + (long)g * A.dk + d]) * bt;
            qt = bf2f(((const u16*)A.q)[t * A.ldq + (long)g * A.dk + d]) *
                 A.qscale;
          } else {
            kt = ((const float*)A.k)[t * A.ldk + (long)g * A.dk + d];
            qt = ((const float*)A.q)[t * A.ldq + (long)g * A.dk + d];
          }
        }
        S[m] = at * S[m] + kt * (MLSTM ? vt : bt * vt);
        sum += S[m] * qt;
      }
      sum = group_sum<8>(sum);
      if (r == 0)
        A.o[((long)t * A.H + h) * A.ov + c] =
            MLSTM ? sum : sum + (A.skip ? A.skip[h] : 0.f) * vt;
    }
#pragma unroll
    for (int m = 0; m < DK / 8; ++m) {
      const int d = m * 8 + r;
      if (d < A.dk) Sg[(long)d * A.ov + c] = S[m];
    }
  }
}

// product of the lanes of a row of 16 up to this one, or from this one on, in 64
// bits: with a constant decay the same error would return in every chunk
template <bool UP>
__device__ __forceinline__ double ch_scan64(double v) {
#define CH_STEP(N)                                                             \
  {                                                                            \
    const u64 b = __builtin_bit_cast(u64, v);                                  \
    const int c1 = (UP ? 0x110 : 0x100) + N;                                   \
    const u32 lo = __builtin_amdgcn_update_dpp(0, (int)(u32)b, c1, 0xF, 0xF,   \
                                               false);                         \
    const u32 hi = __builtin_amdgcn_update_dpp(0x3ff00000, (int)(u32)(b >> 32),\
                                               c1, 0xF, 0xF, false);           \
    v *= __builtin_bit_cast(double, (u64)hi << 32 | lo);                       \
  }
  CH_STEP(1) CH_STEP(2) CH_STEP(4) CH_STEP(8)
#undef CH_STEP
  return v;
}

// Workgroups are numbered by the rank of their sequence among those of `least` or more
// new tokens, of which there are no more than T / least: single tokens beside a few
// prompts need none that way. Runs of up to four go to one XCD (k and q are shared where
// heads share them), the next run to the next XCD. All sequences, an eighth of them for
// each XCD, left the prompts of a batch to few XCDs: 3 of 1200 tokens beside 48 single
// ones, 32 heads of 128 x 128, 617 us (the scan 418) and 236 now, the delta rule 636
// (730) and 275; 16 rows of 2048, 16 heads, 385 and 347.
__device__ __forceinline__ int ch_wg(int run) {
  const int x = blockIdx.x % 8, j = blockIdx.x / 8;
  return (j / run * 8 + x) * run + j % run;
}
static inline int ch_run(int n_wg) { return n_wg < 32 ? (n_wg + 7) / 8 : 4; }
static inline unsigned ch_grid(int n_wg, int run) {
  return (unsigned)((n_wg + 8 * run - 1) / (8 * run) * (8 * run));
}
// the sequence of rank k, or -1
__device__ __forceinline__ int ch_sequence(const int* qlocs, int S, int least, int k) {
  const int lane = threadIdx.x & 63;
  for (int b = 0; b < S; b += 64) {
    const int i = b + lane < S ? b + lane : S - 1;
    const bool is = b + lane < S && qlocs[i + 1] - qlocs[i] >= least;
    const u64 all = __ballot(is);
    if (k < __popcll(all))
      return b + __builtin_ctzll(
                     __ballot(is && __popcll(all & ((1ull << lane) - 1)) == k));
    k -= __popcll(all);
  }
  return -1;
}

// One workgroup: a sequence, a head and NC tiles of 16 columns. NC consumer waves
// hold a tile each; four (MLSTM: three) producer waves bring k, q and the weights of
// the next chunk into the other half of LDS meanwhile. Two barriers a chunk:
//   producers  terms of k and q       | weights, products of decays
//   consumers  S0^T q of the chunk    | its own tokens, the state behind it
template <bool MLSTM> struct ChunkWaves {
  static constexpr int NC = MLSTM ? 9 : 8, NPW = MLSTM ? 3 : 4;
};

template <int DK, bool MLSTM>
__global__ void __launch_bounds__(768, 3) chunk_scan_kernel(const ChunkArgs A) {
  constexpr int NC = ChunkWaves<MLSTM>::NC, NPW = ChunkWaves<MLSTM>::NPW;
  constexpr int NP = MLSTM ? 1 : 3;        // terms of q and k
  constexpr int PLANE = CH_T * DK * 2;     // bytes
  constexpr int WPLANE = CH_T * CH_T * 2;
  constexpr int NT = DK / 16;              // tiles of 16 rows of S
  constexpr int UNITS = 2 * (DK / 32);     // pieces of 32 rows x 32 to stage
  constexpr int UN = (UNITS + NPW - 1) / NPW;
  constexpr int HALF = 16 * DK * 2;        // 16 rows further
  typedef typename std::conditional<MLSTM, u16, float>::type E;
  typedef E e4 __attribute__((ext_vector_type(4)));
  constexpr u32 ES = sizeof(E);
  struct Buf {
    char q[NP * PLANE], k[NP * PLANE], w[3 * WPLANE];
    float P[CH_T], R[CH_T], B[CH_T], tot[4];
  };
  extern __shared__ __attribute__((aligned(16))) char ch_lds[];
  Buf* const buf = (Buf*)ch_lds;

  int wg = ch_wg(A.run);
  if (wg >= A.n_wg) return;
  const int cg = wg % A.cgs;
  wg /= A.cgs;
  const int h = wg % A.H, s = ch_sequence(A.qlocs, A.S, A.least, wg / A.H);
  if (s < 0) return;
  const int q0 = A.qlocs[s], n = A.qlocs[s + 1] - q0;
  const bool old = A.seq_lens[s] > n;
  const int tid = threadIdx.x;
  const int lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int dk = A.dk, ov = A.ov;
  const int steps = (n + CH_T - 1) / CH_T;
  float odd = 0.f;      // NaN once a result was not finite

  // places in LDS: rows of 16 q or k at piece 4 ks + lg; the transposed read's rows
  // 4 lg + lr / 4 (and 16 behind) at piece 4 ks + lr % 4
  int at_row[DK / 32], at_tr[DK / 32];
#pragma unroll
  for (int ks = 0; ks < DK / 32; ++ks) {
    at_row[ks] = ch_place<DK>(lr, ks * 4 + lg);
    at_tr[ks] = ch_place<DK>(lg * 4 + (lr >> 2), ks * 4 + (lr & 3));
  }
  // tokens 0..15 see nothing of tokens 16..31
  if (tid < 2 * 3 * 16 * 4)
    *(u32x2*)(buf[tid / 192].w + tid % 192 / 64 * WPLANE + tid % 64 / 4 * 64 +
              tid % 4 * 16 + 8) = (u32x2){0u, 0u};

  if (w >= NC) {
    // ---------------------------------------------------------- producers
    // a lane stages 4 rows (8 apart) of 4 neighbours. Row pointers are uniform, lanes add 32
    // bits; rows past the last token and dk are zeros.
    const int pw = w - NC;
    const int g = h / (A.H / A.G);
    const int st = lane >> 3, sd = (lane & 7) * 4;
    const u32 ldq = (u32)A.ldq * ES, ldk = (u32)A.ldk * ES;   // bytes
    const u32 lda = (u32)A.lda, ldb = (u32)A.H * 4u;
    e4 pkq[UN][4];
    float pa0, pa1, pb = 1.f;
    auto fetch = [&](int base) {
      const long row = ch_plain(q0 + base);
      const int left = n - base < CH_T ? n - base : CH_T;
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const int unit = pw + u * NPW;
        if (UNITS % NPW && unit >= UNITS) break;
        const int arr = unit / (DK / 32), d = unit % (DK / 32) * 32 + sd;
        const u32 ld = arr ? ldq : ldk;
        const E* src = arr ? (const E*)A.q + row * A.ldq + (long)g * dk
                           : (const E*)A.k + row * A.ldk + (long)g * dk;
        const auto rows = ch_rows(src, (u32)left * ld);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          pkq[u][i] =
              ch_load<e4>(rows, d < dk ? (u32)(st + i * 8) * ld + d * ES : CH_OUT);
      }
      const float* arow = A.a + row * A.lda + h;
      pa0 = lr < left ? arow[lr * lda] : 1.f;
      pa1 = 16 + lr < left ? arow[(16 + lr) * lda] : 1.f;
      if (A.b && pw == NPW - 1)
        pb = ch_load<float>(ch_rows(A.b + row * A.H + h, (u32)left * ldb),
                            (lane & 31) * ldb);
    };
    fetch(0);
    for (int c = -1; c + 1 < steps; ++c) {
      Buf& L = buf[(c + 1) & 1];
      const int left = n - (c + 1) * CH_T;
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const int unit = pw + u * NPW;
        if (UNITS % NPW && unit >= UNITS) break;
        const int d32 = unit % (DK / 32);
        char* dst = unit / (DK / 32) ? L.q : L.k;
        const int piece = d32 * 4 + (sd & 15) / 4, half = (sd >> 4) * 8;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          char* p = dst + ch_place<DK>(st + i * 8, piece) + half;
          const e4 y = pkq[u][i];
          if constexpr (MLSTM) {
            *(e4*)p = y;
          } else {
            const float x[4] = {y[0], y[1], y[2], y[3]};
            u32 t[3][2];
            ch_split<3, 4>(t, x);
#pragma unroll
            for (int r = 0; r < 3; ++r)
              *(u32x2*)(p + r * PLANE) = (u32x2){t[r][0], t[r][1]};
          }
        }
      }
      const float a0 = pa0, a1 = pa1, b0 = pb;
      if (left > CH_T) fetch((c + 2) * CH_T);
      __syncthreads();
      // weights (q_t . k_i) L_ti, a tile of 16 x 16 a wave
      if (pw < 3) {
        const int it = pw == 2, tt = pw > 0;   // keys' and queries' half
        ChSum sum;
#pragma unroll
        for (int ks = 0; ks < DK / 32; ++ks) {
          s16x8 fk[NP], fq[NP];
#pragma unroll
          for (int p = 0; p < NP; ++p) {
            fk[p] = *(const s16x8*)(L.k + p * PLANE + it * HALF + at_row[ks]);
            fq[p] = *(const s16x8*)(L.q + p * PLANE + tt * HALF + at_row[ks]);
          }
          sum.mul(fk, fq);
        }
        const f32x4 acc = sum.total();
        const float at = it ? a1 : a0;
        const float pre1 = ch_prefix(a1);
        float x[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = lg * 4 + r;
          const float sc = ch_prefix(lr > i ? at : 1.f);
          if (pw == 1) x[r] = acc[r] * (pre1 * ch_lane<15>(sc));
          else x[r] = lr >= i ? acc[r] * sc : 0.f;
        }
        u32 t[3][2];
        ch_split<3, 4>(t, x);
#pragma unroll
        for (int p = 0; p < 3; ++p)
          *(u32x2*)(L.w + p * WPLANE + (tt * 16 + lr) * 64 + lg * 16 + it * 8) =
              (u32x2){t[p][0], t[p][1]};
      }
      if (pw == NPW - 1) {
        // lanes 0..15: tokens 0..15, then 16..31; the others repeat them
        const double up0 = ch_scan64<true>(a0), up1 = ch_scan64<true>(a1);
        const double dn0 = ch_scan64<false>(a0), dn1 = ch_scan64<false>(a1);
        const double t0 = __shfl(up0, 15, 64), t1 = __shfl(up1, 15, 64);
        const double x0 = __shfl_down(dn0, 1, 64), x1 = __shfl_down(dn1, 1, 64);
        if (lane < 32) {
          const bool lo = lane < 16;
          L.P[lane] = (float)(lo ? up0 : t0 * up1);
          L.R[lane] = (float)(lo ? (lr < 15 ? x0 * t1 : t1) : lr < 15 ? x1 : 1.0);
          L.B[lane] = b0;
        }
        const double tot = t0 * t1;
        const float hi = (float)tot;
        if (lane == 0) {
          L.tot[0] = hi;
          L.tot[1] = fabsf(hi) <= 3.4e38f ? (float)(tot - (double)hi) : 0.f;
        }
      }
      __syncthreads();
    }
    __syncthreads();    // the consumers' last chunk
    __syncthreads();
  } else {
    // ---------------------------------------------------------- consumers
    const int colb = (cg * NC + w) * 16, col = colb + lr;
    const bool live = colb < ov, own = col < ov;  // a tile, and a column, to work on
    float* Sg = A.state + ((long)A.state_slots[s] * A.H + h) * dk * ov;
    const float sk = A.skip ? A.skip[h] : 0.f;
    if (!live) {
      for (int c = -1; c < steps; ++c) {
        __syncthreads();
        __syncthreads();
      }
      return;
    }
    const u32 ldv = (u32)A.ldv * ES, ldo = (u32)ov * (u32)A.H * 4u;
    const u32 vcol = col < A.dv ? col * ES : CH_OUT;
    const u32 ocol = own ? col * 4u : CH_OUT;
    E pv[8];
    auto fetch = [&](int base) {
      const int left = n - base < CH_T ? n - base : CH_T;
      const auto rows = ch_rows(
          (const E*)A.v + ch_plain(q0 + base) * A.ldv + (long)h * A.dv,
          (u32)left * ldv);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        pv[e] = ch_load<E>(
            rows, (u32)((e >> 2) * 16 + (e & 3) + lg * 4) * ldv + vcol);
    };
    f32x4 S[NT];
    fetch(0);
#pragma unroll
    for (int m = 0; m < NT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = m * 16 + lg * 4 + r;
        S[m][r] = old && own && d < dk ? Sg[(long)d * ov + col] : 0.f;
      }
    __syncthreads();
    __syncthreads();
    for (int c = 0; c < steps; ++c) {
      const Buf& L = buf[c & 1];
      const int left = n - c * CH_T;
      float v[8];
      ChSum O[2];
      {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          v[e] = ldf<E>(&pv[e]);
          // the column of ones; its input gates are 0 past the last token
          if (MLSTM && col == A.dv) v[e] = 1.f;
        }
        if (left > CH_T) fetch((c + 1) * CH_T);
        // ---- S0^T q
#pragma unroll
        for (int ks = 0; ks < DK / 32; ++ks) {
          s16x8 fq[2][NP];
#pragma unroll
          for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int p = 0; p < NP; ++p)
              fq[rt][p] =
                  *(const s16x8*)(L.q + p * PLANE + rt * HALF + at_row[ks]);
          const f32x4 lo = S[2 * ks], hi = S[2 * ks + 1];
          const float x[8] = {lo[0], lo[1], lo[2], lo[3],
                              hi[0], hi[1], hi[2], hi[3]};
          s16x8 fs[3];
          ch_frag<3>(fs, x);
          O[0].mul(fq[0], fs);
          O[1].mul(fq[1], fs);
        }
      }
      __syncthreads();
      // ---- the chunk's own tokens, and the state behind it
      {
        s16x8 fv[3], fr[3];
        {
          float x[8], y[8];
#pragma unroll
          for (int rt = 0; rt < 2; ++rt) {
            const f32x4 R = *(const f32x4*)(L.R + rt * 16 + lg * 4);
            const f32x4 B = *(const f32x4*)(L.B + rt * 16 + lg * 4);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              x[rt * 4 + r] = A.b ? B[r] * v[rt * 4 + r] : v[rt * 4 + r];
              y[rt * 4 + r] = R[r] * x[rt * 4 + r];
            }
          }
          ch_frag<3>(fv, x);
          ch_frag<3>(fr, y);
        }
        const auto orows = ch_rows(
            A.o + ((long)ch_plain(q0 + c * CH_T) * A.H + h) * ov,
            (u32)(left < CH_T ? left : CH_T) * ldo);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
          s16x8 fw[3];
#pragma unroll
          for (int p = 0; p < 3; ++p)
            fw[p] = *(const s16x8*)(L.w + p * WPLANE + (rt * 16 + lr) * 64 +
                                    lg * 16);
          ChSum near;
          near.mul(fw, fv);
          const f32x4 P = *(const f32x4*)(L.P + rt * 16 + lg * 4);
          const f32x4 y = O[rt].total() * P + near.total();
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float res =
                MLSTM ? y[r] * A.qscale : y[r] + sk * v[rt * 4 + r];
            odd += res * 0.f;
            __builtin_amdgcn_raw_buffer_store_b32(
                __float_as_uint(res), orows,
                (u32)(rt * 16 + r + lg * 4) * ldo + ocol, 0, 0);
          }
        }
        const float ph = L.tot[0], pl = L.tot[1];
        // four tiles side by side: a chain's products wait for one another
#pragma unroll
        for (int m0 = 0; m0 < NT; m0 += 4) {
          s16x8 fk[4][NP];
          f32x4 u[4];
#pragma unroll
          for (int m = m0; m < m0 + 4; ++m) {
            u[m - m0] = (f32x4)(0.f);
#pragma unroll
            for (int p = 0; p < NP; ++p) {
              const char* at = L.k + p * PLANE + (m & 1) * 8 + at_tr[m >> 1];
              const ch_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                  (__attribute__((address_space(3))) ch_s16x4*)at);
              const ch_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                  (__attribute__((address_space(3))) ch_s16x4*)(at + HALF));
              fk[m - m0][p] =
                  __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            }
          }
#pragma unroll
          for (int o = 2; o >= 0; --o)
#pragma unroll
            for (int i = 0; i <= o; ++i)
              if (i < NP)
#pragma unroll
                for (int m = 0; m < 4; ++m)
                  u[m] = ch_mfma(fk[m][i], fr[o - i], u[m]);
#pragma unroll
          for (int m = 0; m < 4; ++m)
            S[m0 + m] = S[m0 + m] * ph + (S[m0 + m] * pl + u[m]);
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < NT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) odd += S[m][r] * 0.f;
    // a wave whose columns are not finite does them again by itself
    if (__any(odd != 0.f)) {
      chunk_serial<DK, MLSTM>(A, s, h, colb, 16, lane);
      return;
    }
#pragma unroll
      for (int m = 0; m < NT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = m * 16 + lg * 4 + r;
          if (own && d < dk) Sg[(long)d * ov + col] = S[m][r];
        }
  }
}

// New tokens from which a sequence goes through chunks (0: none of the batch does); the
// scans keep the shorter ones (single tokens among them: state in, state out). A chunk
// takes a CU as long whatever its columns, and one workgroup is on a CU; the scan takes
// what its rows and columns cost, several workgroups a CU. So where more than a round of
// workgroups is at work, small heads stay with the scan for long, or always: `few`, `mid`
// and `many` for up to 256 workgroups, up to 512, and more. But only T / n sequences can
// have n tokens: longer ones may be few where shorter ones were many.
// One kernel runs behind the other, so that sequences on both sides of the line take
// the time of both: not where the longest (`longest` new tokens; 0: not known) has less than
// twice the line and the mean is below 5/4 of it.
struct ChunkNeed { int few, mid, many; };
#define CH_NEVER (1 << 30)
static inline int chunk_least(ChunkNeed need, long T, long longest, int S, long wgs) {
  long least = need.many;
  const long caps[2] = {256, 512}, needs[2] = {need.few, need.mid};
  for (int i = 0; i < 2; ++i) {
    const long seqs = caps[i] / wgs;          // sequences within `caps`
    if (!seqs) continue;
    long n = S > seqs ? T / (seqs + 1) + 1 : 0;
    if (n < needs[i]) n = needs[i];
    if (n < least) least = n;
  }
  if (longest <= 0) longest = T - S + 1;     // (a token for each of the others)
  if (S < 1 || least > T || least > longest || (longest < 2 * least && 4 * T < 5 * S * least))
    return 0;
  return (int)least;
}

// Measured, tokens from which chunks are ahead in batches of equal sequences, 32 to 256
// workgroups, 512, and 1024 to 4096 (keys x values of a head):
//   decay  16 x 64    24        96   never     MLSTM  16 x 64     8    16   24 to 32
//          16 x 128   32        96   192, 256         64 x 64    16    16    4 to 8
//          32 x 64    24        64   192, 256         64 x 128   16    16    8
//          64 x 16    24        48   96 to 192       128 x 16    24    32   32
//          64 x 64    24        24   48              128 x 64    24    48   32 to 48
//          64 x 128   24        16   24              128 x 128   32    16   16 to 24
//         128 x 16    48       192   never
//         128 x 64    64       128   128 to 256
//         128 x 128   64        64   48 to 96
// (128 x 32, 256 sequences of 64 tokens, 16 heads: 170 and 440 us; 128 x 128, 1024 workgroups
// of 40 111 and 127, of 64 157 and 132; 1 row of 40 18.5 and 26, of 96 36 and 31.)
static inline ChunkNeed chunk_need(bool mlstm, int dk, int columns) {
  if (mlstm) {
    if (dk > 64) return columns > 80 ? ChunkNeed{28, 24, 24} : ChunkNeed{28, 48, 48};
    return dk > 32 ? ChunkNeed{12, 12, 12} : ChunkNeed{12, 32, 32};
  }
  if (dk > 64) {
    if (columns > 80) return {64, 64, columns > 112 ? 80 : 96};
    return columns > 48 ? ChunkNeed{64, 128, 256} : ChunkNeed{64, 192, CH_NEVER};
  }
  if (dk > 32) {
    if (columns > 96) return {24, 24, 24};
    return {24, 48, columns > 48 ? 48 : columns > 24 ? 128 : 192};
  }
  if (columns > 96) return {24, 96, dk > 16 ? 96 : 256};
  return {24, 96, dk > 16 ? 256 : CH_NEVER};
}

// 0 also where rows are not in whole 16-byte (8-byte) pieces, or less than a head apart
// (one row for all tokens): what a chunk may read ends a row's distance behind its last.
static inline int chunk_scan_least(int dk, long ldq, long ldk, long ldv, long ldo,
                                   const void* q, const void* k, int dv,
                                   int align, bool mlstm, long T, long longest,
                                   int S, int H) {
  const long most = 1 << 23;               // 32 rows within 2^31 bytes
  if (dk > 128 || dk % 4 || ldq % 4 || ldk % 4 || (size_t)q % align ||
      (size_t)k % align || ldq >= most || ldk >= most || ldv >= most ||
      ldo >= most || ldq < dk || ldk < dk || ldv < dv)
    return 0;
  const int ov = mlstm ? dv + 1 : dv, per = mlstm ? 144 : 128;
  const int cgs = (ov + per - 1) / per;
  return chunk_least(chunk_need(mlstm, dk, dv / cgs), T, longest, S, (long)H * cgs);
}

template <int DK, bool MLSTM>
static void chunk_scan_go(const ChunkArgs& A, hipStream_t s) {
  constexpr int NP = MLSTM ? 1 : 3;
  constexpr int bytes =
      2 * (NP * 2 * CH_T * DK * 2 + 3 * CH_T * CH_T * 2 + (3 * CH_T + 4) * 4);
  static std::atomic<unsigned long long> asked{0};
  const auto fn = chunk_scan_kernel<DK, MLSTM>;
  lds_limit((const void*)fn, bytes, asked);
  hipLaunchKernelGGL(fn, dim3(ch_grid(A.n_wg, A.run)), dim3(768), bytes, s, A);
}
template <bool MLSTM>
static void chunk_scan_launch(ChunkArgs A, long T, int S, int least, hipStream_t s) {
  const int per = ChunkWaves<MLSTM>::NC * 16;
  A.cgs = (A.ov + per - 1) / per;
  A.S = S;
  A.n_wg = (int)(T / least < S ? T / least : S) * A.H * A.cgs;
  A.run = ch_run(A.n_wg);
  A.least = least;
  if (A.dk <= 64) chunk_scan_go<64, MLSTM>(A, s);
  else chunk_scan_go<128, MLSTM>(A, s);
}
