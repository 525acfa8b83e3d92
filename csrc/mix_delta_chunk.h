// The gated delta rule over chunks of 32 tokens on the matrix cores (delta_scan of
// mix_delta.hip does the same token by token). In a chunk that starts from S0, with
// g_t the product of the decays up to token t and g_ti that of those behind i up to t
// (a number a key channel each):
//   u_t = beta_t (v_t - S0^T (g_t k_t) - sum_{i<t} (k_t . g_ti k_i) u_i)
//   o_t = S0^T (g_t q_t) + sum_{i<=t} (q_t . g_ti k_i) u_i
//   S   = g_32 S0 + sum_i (g_32,i k_i) u_i^T
// The first line is a triangular system of the chunk's tokens alone: with A the
// matrix of its sums, U = M (V - S0^T K+), M = (1 + diag(beta) A)^-1 diag(beta). The
// diagonal of M, beta, is applied in fp32: most of u_t is that.
//
//   delta_pairs   M off its diagonal and the sums of the second line, for all chunks side by side
//   delta_chunks  the recurrence from chunk to chunk
//
// Decays are only multiplied up, never divided: g_ti is split where the binary
// digits of t and i part. For a half size h = 1, 2, 4, 8, 16, t in an upper and i in
// the lower half of the same 2h tokens, it is the product from the middle to t times
// that from i to the middle, and both are shared by all pairs of the 2h tokens; one
// tile of 16 x 16 holds the pairs of a level. fp32 operands are split into three bf16
// terms as in mix_chunk.h, whose layouts are used here as well; sequences with
// numbers that are not finite are done once more token by token (as there; 16 rows of
// 1024 tokens of 32 heads 727 us, with a NaN in one of them 3640, in all 8629; 1 row of
// 4000 of 16 heads 399 and 12,300).
//
// Times for 16 rows of 2048 tokens with a decay a channel, heads of 128 x 128, scan and
// both kernels: 16 heads 1530 and 619 us (pairs 235), 8 heads 1000 and 354 (pairs 133);
// 1 row of 4000, 16 heads, 1641 and 397; 16 rows of 1024, 32 heads with a decay a head,
// 1300 and 600. The scan was bound by VALU issue, one token behind the other. Here a
// chunk takes 10,300 cycles of a CU in delta_chunks (VALU 6300, products 5400: the
// splits of S, U and the producers' rows) and 7700 in delta_pairs (VALU 5200). Slower
// in delta_pairs: adding the halves of a product with LDS atomics (328 instead of 235
// us), two channels of eight tokens a lane; in delta_chunks: loading the next chunk's
// rows at once (443 us instead of 380 for 16 heads), K- through the transposed read.
// Errors against 64 bits, scan and chunks: at those sizes read-out 1.3e-7 and 9.8e-8,
// state 6.8e-8 both; 4096 tokens of the same decay, 0.9987654 or 0.99987, beta 0.02 to
// 0.98, independent keys, keys behind silu, keys that resemble each other, keys that
// leave half of the channels alone: read-out 2.7e-7 to 1.4e-6 and 1.2e-7 to 3.2e-7,
// state 2.1e-7 to 2.2e-6 and 9.7e-8 to 2.9e-7. Larger than the scan's are those of keys
// that resemble each other (cosine 0.9) with beta 0.98 and decays that change, 1.4e-7
// and 2.1e-7: there u_t is the small difference of large numbers of S0.
#pragma once

#include "mix_chunk.h"

struct DeltaChunkArgs {
  float* o;             // [T, H, dv]
  const float* q;       // [T, G, dk]
  const float* k;
  const float* v;       // [T, H, dv]
  const float* d;       // [T, H, dk], or [T, H] (HEAD)
  const float* beta;    // [T, H]
  float* state;         // [slots, H, dk, dv]
  const int* state_slots;
  const int* qlocs;
  const int* seq_lens;
  float* pairs;         // [T / 32 + T / least, H, DC_PAIRS]
  int S, H, G, dk, dv;
  int cgs, n_wg, run;   // as in ChunkArgs
  int least;
};

// tiles (0, 0), (1, 0), (1, 1) of 16 x 16: M, then the read-out's sums
#define DC_PAIRS (2 * 3 * 256)

// chunks of the sequence of rank k (see ch_wg) are numbered from this on: no two have
// the same number, and all are below T / 32 + T / least
__device__ __forceinline__ int dc_slot(int q0, int k) { return (q0 >> 5) + k; }

// two channels of a row -> three terms at `p`, PLANE bytes apart
template <int PLANE>
__device__ __forceinline__ void dc_put(char* p, float x, float y) {
#pragma unroll
  for (int n = 0; n < 3; ++n) *(u32*)(p + n * PLANE) = ch_term(x, y);
}

// A product of decays times one more, and what its roundings left out (of first
// order). The state is multiplied by a product in every chunk, and where the decays
// stay the same, so does its rounding: over 4096 tokens of 0.9987654 errors were 2 to 9
// times the scan's (beta 0.02, keys that resemble each other: state 8.2e-6 and 9.4e-7).
// So what the product of a chunk lacks is handed on to that of the next (2.3e-7). It
// costs nothing where the chip is full and 1 % for one row of 4000 tokens; a second
// factor in the consumers took 5 % there.
__device__ __forceinline__ void dc_times(f32x2& p, f32x2& lost, f32x2 d) {
#pragma clang fp contract(off)    // (the product is the rounded one also behind this)
  const f32x2 x = p * d;
#pragma unroll
  for (int e = 0; e < 2; ++e)
    lost[e] = fmaf(lost[e], d[e], fmaf(p[e], d[e], -x[e]));
  p = x;
}

// ---- pairs of tokens -----------------------------------------------------------
// rows of 16 lanes (rows of 32 lanes): the even one's value in both, the odd one's
__device__ __forceinline__ void dc_rows16(float x, float& even, float& odd) {
  const u32 v = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  even = __uint_as_float(r[0]);
  odd = __uint_as_float(r[1]);
}
__device__ __forceinline__ void dc_rows32(float x, float& even, float& odd) {
  const u32 v = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  even = __uint_as_float(r[0]);
  odd = __uint_as_float(r[1]);
}

// One workgroup: a chunk of a head. A lane has eight channels of the tokens
// 8 w + 2 lg and the next, so that a term goes to LDS in 16 bytes. Pairs within four
// tokens are summed over the 16 lanes, the levels of h = 4, 8, 16 are products of
// 16 x 16 x dk, half of dk a wave.
template <int DK, bool HEAD>
__global__ void __launch_bounds__(256, 3)
delta_pairs_kernel(const DeltaChunkArgs A) {
  constexpr int PLANE = 16 * DK * 2;
  // upper halves: k and q; lower halves: k. Later the inverse, and a product
  __shared__ __attribute__((aligned(16))) char Lk[3 * PLANE], Lq[3 * PLANE],
      Rk[3 * PLANE];
  __shared__ __attribute__((aligned(16))) float Ma[32][36], Mb[32][36];
  __shared__ __attribute__((aligned(16))) float tot8[4][DK], bt[32];
  float (*const Mi)[36] = (float (*)[36])Lk;
  float (*const Y)[17] = (float (*)[17])Lq;

  const int tid = threadIdx.x, lane = tid & 63;
  const int lr = lane & 15, lg = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = blockIdx.x % A.H, slot = blockIdx.x / A.H;
  int s = -1, rank = 0;    // the last sequence that begins at or in front of the slot
  for (int b = 0, before = 0; b < A.S; b += 64) {
    const int i = b + lane < A.S ? b + lane : A.S - 1, q = A.qlocs[i];
    const bool is = b + lane < A.S && A.qlocs[i + 1] - q >= A.least;
    const u64 all = __ballot(is);
    const int k = before + __popcll(all & ((1ull << lane) - 1));
    const u64 hit = __ballot(is && dc_slot(q, k) <= slot);
    if (hit) {
      const int last = 63 - __builtin_clzll(hit);
      s = b + last;
      rank = before + __popcll(all & ((1ull << last) - 1));
    }
    before += __popcll(all);
  }
  if (s < 0) return;       // none
  const int q0 = A.qlocs[s], n = A.qlocs[s + 1] - q0;
  const int base = (slot - dc_slot(q0, rank)) * CH_T;
  if (base >= n) return;
  const int left = n - base < CH_T ? n - base : CH_T;
  const int dk = A.dk, g = h / (A.H / A.G);
  const int ch = lr * 8, r0 = w * 8 + lg * 2;   // channels and tokens of this lane

  float k[2][8], q[2][8], d[2][8];
  {
    const long row = q0 + base;
    const u32 ldk = (u32)(A.G * dk) * 4u, ldd = (u32)(HEAD ? A.H : A.H * dk) * 4u;
    const auto kr = ch_rows(A.k + (row * A.G + g) * dk, left * ldk);
    const auto qr = ch_rows(A.q + (row * A.G + g) * dk, left * ldk);
    const auto dr = HEAD ? ch_rows(A.d + row * A.H + h, left * ldd)
                         : ch_rows(A.d + (row * A.H + h) * dk, left * ldd);
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int x = 0; x < 8; x += 4) {
        const u32 t = r0 + r, off = ch + x < dk ? (ch + x) * 4u : CH_OUT;
        const f32x4 a = ch_load<f32x4>(kr, t * ldk + off);
        const f32x4 b = ch_load<f32x4>(qr, t * ldk + off);
        f32x4 c;
        if (HEAD) c = (f32x4)(ch_load<float>(dr, t * ldd));
        else c = ch_load<f32x4>(dr, t * ldd + off);
        if ((int)t >= left) c = (f32x4)(1.f);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          k[r][x + e] = a[e];
          q[r][x + e] = b[e];
          d[r][x + e] = c[e];
        }
      }
  }
  for (int i = tid; i < 32 * 36; i += 256) (&Ma[0][0])[i] = (&Mb[0][0])[i] = 0.f;
  if (tid < 32)
    bt[tid] = tid < left ? A.beta[(long)(q0 + base + tid) * A.H + h] : 0.f;
  __syncthreads();
  float pre[2][8], suf[2][8], tot[8];
  {
    // a lane's own two tokens, then (in the odd rows of lanes) with the two before
    float a10 = 0.f, b10 = 0.f, b00 = 0.f, b11 = 0.f;
    float a[2][2] = {{0.f, 0.f}, {0.f, 0.f}}, b[2][2] = {{0.f, 0.f}, {0.f, 0.f}};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float z = k[0][e] * d[1][e], t2 = d[0][e] * d[1][e];
      a10 += k[1][e] * z;
      b10 += q[1][e] * z;
      b00 += q[0][e] * k[0][e];
      b11 += q[1][e] * k[1][e];
      float lo0, lo1, t_lo, t_hi, no;
      dc_rows16(z, lo0, no);
      dc_rows16(k[1][e], lo1, no);
      dc_rows16(t2, t_lo, t_hi);
      const float k0 = k[0][e] * d[0][e], k1 = k[1][e] * t2;
      const float q0e = q[0][e] * d[0][e], q1e = q[1][e] * t2;
      a[0][0] += k0 * lo0; a[0][1] += k0 * lo1;
      a[1][0] += k1 * lo0; a[1][1] += k1 * lo1;
      b[0][0] += q0e * lo0; b[0][1] += q0e * lo1;
      b[1][0] += q1e * lo0; b[1][1] += q1e * lo1;
      // products over four tokens
      pre[0][e] = lg & 1 ? t_lo * d[0][e] : d[0][e];
      pre[1][e] = lg & 1 ? t_lo * t2 : t2;
      suf[0][e] = lg & 1 ? d[1][e] : d[1][e] * t_hi;
      suf[1][e] = lg & 1 ? 1.f : t_hi;
      tot[e] = t_lo * t_hi;
    }
    a10 = group_sum<16>(a10); b10 = group_sum<16>(b10);
    b00 = group_sum<16>(b00); b11 = group_sum<16>(b11);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[t][i] = group_sum<16>(a[t][i]);
        b[t][i] = group_sum<16>(b[t][i]);
      }
    if (lr == 0) {
      Ma[r0 + 1][r0] = a10;
      *(f32x2*)&Mb[r0 + 1][r0] = (f32x2){b10, b11};
      Mb[r0][r0] = b00;
      if (lg & 1)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          *(f32x2*)&Ma[r0 + t][r0 - 2] = (f32x2){a[t][0], a[t][1]};
          *(f32x2*)&Mb[r0 + t][r0 - 2] = (f32x2){b[t][0], b[t][1]};
        }
    }
  }

  // two rows of terms (x times f), `row` and the next
  auto put = [&](char* dst, int row, const float (&x)[2][8], const float (&f)[2][8]) {
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = x[r][e] * f[r][e];
      s16x8 t[3];
      ch_frag<3>(t, y);
      if (DK == 128 || lr < 8)
#pragma unroll
        for (int p = 0; p < 3; ++p)
          *(s16x8*)(dst + p * PLANE + ch_place<DK>(row + r, lr)) = t[p];
    }
  };
  // a level: the operands in LDS -> this wave's half of the sums over dk
  f32x4 part[3];
  auto level = [&](f32x4& x) {
    __syncthreads();
    const char* L = w & 1 ? Lq : Lk;
    ChSum sum;
#pragma unroll
    for (int y = 0; y < DK / 64; ++y) {
      const int ks = (w >> 1) * (DK / 64) + y;
      s16x8 a[3], b[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const int at = p * PLANE + ch_place<DK>(lr, ks * 4 + lg);
        a[p] = *(const s16x8*)(L + at);
        b[p] = *(const s16x8*)(Rk + at);
      }
      sum.mul(a, b);
    }
    x = sum.total();
    __syncthreads();
  };
  {
    float f[2][8];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int e = 0; e < 8; ++e) f[r][e] = lg & 2 ? pre[r][e] : suf[r][e];
    put(lg & 2 ? Lk : Rk, w * 4 + (lg & 1) * 2, k, f);
    if (lg & 2) put(Lq, w * 4 + (lg & 1) * 2, q, f);
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float lo, hi;
    dc_rows32(tot[e], lo, hi);
    if (lg & 2) { pre[0][e] *= lo; pre[1][e] *= lo; }
    else { suf[0][e] *= hi; suf[1][e] *= hi; }
    tot[e] = lo * hi;
  }
  if (lg == 0 && (DK == 128 || lr < 8)) {
    *(f32x4*)&tot8[w][ch] = (f32x4){tot[0], tot[1], tot[2], tot[3]};
    *(f32x4*)&tot8[w][ch + 4] = (f32x4){tot[4], tot[5], tot[6], tot[7]};
  }
  level(part[0]);
  if (w & 1) {
    put(Lk, (w >> 1) * 8 + lg * 2, k, pre);
    put(Lq, (w >> 1) * 8 + lg * 2, q, pre);
  } else {
    put(Rk, (w >> 1) * 8 + lg * 2, k, suf);
  }
  level(part[1]);
  if (DK == 128 || lr < 8) {
#pragma unroll
    for (int x = 0; x < 8; x += 4) {
      const f32x4 t = *(const f32x4*)&tot8[w ^ 1][ch + x];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (w & 1) { pre[0][x + e] *= t[e]; pre[1][x + e] *= t[e]; }
        else { suf[0][x + e] *= t[e]; suf[1][x + e] *= t[e]; }
      }
    }
  }
  if (w >= 2) {
    put(Lk, (w & 1) * 8 + lg * 2, k, pre);
    put(Lq, (w & 1) * 8 + lg * 2, q, pre);
  } else {
    put(Rk, (w & 1) * 8 + lg * 2, k, suf);
  }
  level(part[2]);
  // both halves; then to their places
  if (w >= 2) {
#pragma unroll
    for (int x = 0; x < 3; ++x)
      *(f32x4*)(Rk + ((x * 2 + (w & 1)) * 64 + lane) * 16) = part[x];
  }
  __syncthreads();
  if (w < 2) {
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      const int hs = 4 << x;
      const f32x4 y =
          part[x] + *(const f32x4*)(Rk + ((x * 2 + w) * 64 + lane) * 16);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int li = lg * 4 + r, blk = li / hs;
        if (lr / hs == blk)
          (w ? Mb : Ma)[blk * 2 * hs + hs + li % hs][blk * 2 * hs + lr % hs] = y[r];
      }
    }
  }
  __syncthreads();
  // (1 + diag(beta) A)^-1: both blocks of 16 on the diagonal, a lane a column
  if (tid < 32) {
    const int b0 = tid & 16, j = tid & 15;
    float m[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      float x = 0.f;
#pragma unroll
      for (int i = 0; i < t; ++i) x += Ma[b0 + t][b0 + i] * m[i];
      m[t] = (t == j ? 1.f : 0.f) - bt[b0 + t] * x;
    }
#pragma unroll
    for (int t = 0; t < 16; ++t) Mi[b0 + t][b0 + j] = m[t];
  }
  __syncthreads();
  const int t = tid >> 4, j = tid & 15;
  {
    float x = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) x += Ma[16 + t][i] * Mi[i][j];
    Y[t][j] = bt[16 + t] * x;
  }
  __syncthreads();
  float x = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) x += Mi[16 + t][16 + i] * Y[i][j];
  float* out = A.pairs + ((long)slot * A.H + h) * DC_PAIRS + tid;
  out[0] = t == j ? 0.f : Mi[t][j] * bt[j];   // (the diagonal is beta)
  out[256] = -x * bt[j];
  out[512] = t == j ? 0.f : Mi[16 + t][16 + j] * bt[16 + j];
  out[768] = Mb[t][j];
  out[1024] = Mb[16 + t][j];
  out[1280] = Mb[16 + t][16 + j];
}

// ---- token by token, for numbers that are not finite ---------------------------
template <int DK, bool HEAD>
__device__ __forceinline__ void delta_serial(const DeltaChunkArgs& A, int s, int h,
                                             int col0, int lane) {
  const int q0 = A.qlocs[s], n = A.qlocs[s + 1] - q0;
  const bool old = A.seq_lens[s] > n;
  const int g = h / (A.H / A.G), r = lane & 7, dk = A.dk, dv = A.dv;
  float* Sg = A.state + ((long)A.state_slots[s] * A.H + h) * dk * dv;
  for (int c = col0 + (lane >> 3); c < col0 + 16; c += 8) {
    if (c >= dv) continue;
    float S[DK / 8];
#pragma unroll
    for (int m = 0; m < DK / 8; ++m) {
      const int i = m * 8 + r;
      S[m] = old && i < dk ? Sg[(long)i * dv + c] : 0.f;
    }
    for (long t = q0; t < q0 + n; ++t) {
      float kk[DK / 8], dot = 0.f, out = 0.f;
#pragma unroll
      for (int m = 0; m < DK / 8; ++m) {
        const int i = m * 8 + r;
        kk[m] = i < dk ? A.k[(t * A.G + g) * dk + i] : 0.f;
        S[m] *= HEAD ? A.d[t * A.H + h]
                     : i < dk ? A.d[(t * A.H + h) * dk + i] : 1.f;
        dot += S[m] * kk[m];
      }
      const float u = A.beta[t * A.H + h] *
                      (A.v[(t * A.H + h) * dv + c] - group_sum<8>(dot));
#pragma unroll
      for (int m = 0; m < DK / 8; ++m) {
        const int i = m * 8 + r;
        S[m] += kk[m] * u;
        out += S[m] * (i < dk ? A.q[(t * A.G + g) * dk + i] : 0.f);
      }
      out = group_sum<8>(out);
      if (r == 0) A.o[(t * A.H + h) * dv + c] = out;
    }
#pragma unroll
    for (int m = 0; m < DK / 8; ++m) {
      const int i = m * 8 + r;
      if (i < dk) Sg[(long)i * dv + c] = S[m];
    }
  }
}

// ---- from chunk to chunk -------------------------------------------------------
// One workgroup: a sequence, a head and 16 NC columns, as in chunk_scan_kernel: NC
// consumer waves with a tile of 16 columns of S each, four producers (wave pw tokens
// 8 pw .. 8 pw + 7, a lane two channels). Two barriers a chunk, what is read in one
// half is written in the other:
//   consumers  S0^T K+, S0^T Q+            | U, the read-out, S
//   producers  K- and the pairs of c,      | K+ and Q+ of c + 1
//              products over 8 of c + 1    |
template <int DK, bool HEAD, int NC>
__global__ void __launch_bounds__((NC + 4) * 64, (NC + 4) / 4)
delta_chunks_kernel(const DeltaChunkArgs A) {
  constexpr int PLANE = CH_T * DK * 2, WPLANE = CH_T * CH_T * 2;
  constexpr int NT = DK / 16, HALF = 16 * DK * 2;
  struct Lds {
    char kp[3 * PLANE], qp[3 * PLANE], km[3 * PLANE];
    char m[3 * WPLANE], b[3 * WPLANE];
    float tot8[2][2][4][DK], all[DK], beta[CH_T];   // (products over 8: hi, lo)
  };
  extern __shared__ __attribute__((aligned(16))) char dc_lds[];
  Lds& L = *(Lds*)dc_lds;

  int wg = ch_wg(A.run);
  if (wg >= A.n_wg) return;
  const int cg = wg % A.cgs;
  wg /= A.cgs;
  const int h = wg % A.H, rank = wg / A.H;
  const int s = ch_sequence(A.qlocs, A.S, A.least, rank);
  if (s < 0) return;
  const int q0 = A.qlocs[s], n = A.qlocs[s + 1] - q0;
  const bool old = A.seq_lens[s] > n;
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int dk = A.dk, dv = A.dv;
  const int steps = (n + CH_T - 1) / CH_T;

  // pairs of tokens 0..15 with 16..31 are zero
  if (tid < 3 * 64) {
    const int at = tid / 64 * WPLANE + tid % 64 / 4 * 64 + tid % 4 * 16 + 8;
    *(u32x2*)(L.m + at) = (u32x2){0u, 0u};
    *(u32x2*)(L.b + at) = (u32x2){0u, 0u};
  }
  if (w >= NC) {
    // ---------------------------------------------------------- producers
    const int pw = w - NC, g = h / (A.H / A.G);
    const int ch = lane * 2;
    const bool in = ch < dk;
    const u32 ldk = (u32)(A.G * dk) * 4u;                     // bytes
    const u32 ldd = (u32)(HEAD ? A.H : A.H * dk) * 4u;
    const u32 off = in ? ch * 4u : CH_OUT;
    f32x2 rk[8], rq[8], rd[8], rm[8];    // loaded rows; K- on its way
    f32x4 rp[2];                         // pairs on their way
    f32x2 owed = (f32x2)(0.f);           // by the last chunk's product, as a part of it
    float rb = 0.f;                      // and beta (wave 2)
    auto fetch_d = [&](int c) {
      const long row = ch_plain(q0 + c * CH_T);
      const int left = n - c * CH_T < CH_T ? n - c * CH_T : CH_T;
      const auto dr = HEAD ? ch_rows(A.d + row * A.H + h, left * ldd)
                           : ch_rows(A.d + (row * A.H + h) * dk, left * ldd);
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const u32 t = pw * 8 + r;
        if (HEAD) rd[r] = (f32x2)(ch_load<float>(dr, t * ldd));
        else rd[r] = ch_load<f32x2>(dr, t * ldd + off);
      }
    };
    auto kq_rows = [&](const float* p, int c) {
      const int left = n - c * CH_T < CH_T ? n - c * CH_T : CH_T;
      return ch_rows(p + ((long)ch_plain(q0 + c * CH_T) * A.G + g) * dk,
                     left > 0 ? left * ldk : 0u);
    };
    // tiles pw and (waves 0, 1) 4 + pw of the chunk's six
    const int slot0 = dc_slot(q0, rank);
    auto fetch_pairs = [&](int c) {
      const float* p = A.pairs + ((long)(slot0 + c) * A.H + h) * DC_PAIRS + lane * 4;
      rp[0] = *(const f32x4*)(p + pw * 256);
      if (pw < 2) rp[1] = *(const f32x4*)(p + (pw + 4) * 256);
      if (pw == 2) {
        const int t = c * CH_T + (lane & 31);
        rb = t < n ? A.beta[(long)(q0 + t) * A.H + h] : 0.f;
      }
    };
    auto put_pairs = [&](int tile, const f32x4 v) {
      char* dst = tile < 3 ? L.m : L.b;
      const int k3 = tile % 3, tt = k3 > 0, it = k3 == 2;
      const float x[4] = {v[0], v[1], v[2], v[3]};
      u32 t[3][2];
      ch_split<3, 4>(t, x);
#pragma unroll
      for (int p = 0; p < 3; ++p)
        *(u32x2*)(dst + p * WPLANE + (tt * 16 + (lane >> 2)) * 64 +
                  (lane & 3) * 16 + it * 8) = (u32x2){t[p][0], t[p][1]};
    };
    // place of the lane's channels in a row: piece, half and word (see mix_chunk.h)
    const int piece = (ch >> 5) * 4 + ((ch & 15) >> 2);
    const int sub = ((ch >> 4) & 1) * 8 + (ch & 2) * 2;
    auto put = [&](char* dst, int r, f32x2 x) {
      if (DK == 128 || lane < 32)
        dc_put<PLANE>(dst + ch_place<DK>(pw * 8 + r, piece) + sub, x[0], x[1]);
    };
    f32x2 pre[8], suf[8];
    auto local = [&](int c) {            // products over the wave's 8 tokens
      // rows past the last token were read as zero: no decay behind it
      const int left = n - c * CH_T - pw * 8;
#pragma unroll
      for (int r = 0; r < 8; ++r)
        if (r >= left) rd[r] = (f32x2)(1.f);
      // what the products behind the first lose (see dc_times)
      f32x2 lost = (f32x2)(0.f);
      pre[0] = rd[0];
#pragma unroll
      for (int r = 1; r < 8; ++r) {
        pre[r] = pre[r - 1];
        dc_times(pre[r], lost, rd[r]);
      }
      suf[7] = (f32x2)(1.f);
#pragma unroll
      for (int r = 6; r >= 0; --r) suf[r] = suf[r + 1] * rd[r + 1];
      if (DK == 128 || lane < 32) {
        *(f32x2*)&L.tot8[c & 1][0][pw][ch] = pre[7];
        *(f32x2*)&L.tot8[c & 1][1][pw][ch] = lost;
      }
    };
    // K+ and Q+ into LDS, K- into registers; rows of the next chunk take the place of
    // those that are done (loads all at once would wait for the memory)
    auto plus = [&](int c) {
      const auto kr = kq_rows(A.k, c + 1), qr = kq_rows(A.q, c + 1);
      f32x2 before = (f32x2)(1.f), behind = (f32x2)(1.f);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x2 t = DK == 128 || lane < 32
                            ? *(const f32x2*)&L.tot8[c & 1][0][i][ch] : (f32x2)(1.f);
        if (i < pw) before *= t;
        if (i > pw) behind *= t;
      }
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const f32x2 p = before * pre[r];
        put(L.kp, r, rk[r] * p);
        put(L.qp, r, rq[r] * p);
        rm[r] = rk[r] * (suf[r] * behind);
        rk[r] = ch_load<f32x2>(kr, (u32)(pw * 8 + r) * ldk + off);
        rq[r] = ch_load<f32x2>(qr, (u32)(pw * 8 + r) * ldk + off);
      }
    };
    // K- by channel: rows of 32 tokens, in the places of the contraction over tokens;
    // pieces are mixed with the channel, so that lanes write to all of a row's banks
    auto put_minus = [&]() {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const float y[4] = {rm[i * 4][x], rm[i * 4 + 1][x], rm[i * 4 + 2][x],
                              rm[i * 4 + 3][x]};
          u32 t[3][2];
          ch_split<3, 4>(t, y);
          const int at = (ch + x) * 64 + ((((pw & 1) * 2 + i) ^ (lane & 3)) << 4) +
                         (pw >> 1) * 8;
          if (DK == 128 || lane < 32)
#pragma unroll
            for (int p = 0; p < 3; ++p)
              *(u32x2*)(L.km + p * PLANE + at) = (u32x2){t[p][0], t[p][1]};
        }
    };
    fetch_d(0);
    {
      const auto kr = kq_rows(A.k, 0), qr = kq_rows(A.q, 0);
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        rk[r] = ch_load<f32x2>(kr, (u32)(pw * 8 + r) * ldk + off);
        rq[r] = ch_load<f32x2>(qr, (u32)(pw * 8 + r) * ldk + off);
      }
    }
    local(0);
    if (steps > 1) fetch_d(1);
    fetch_pairs(0);
    __syncthreads();
    plus(0);
    __syncthreads();
    for (int c = 0; c < steps; ++c) {
      put_minus();
      put_pairs(pw, rp[0]);
      if (pw < 2) put_pairs(pw + 4, rp[1]);
      if (pw == 2 && lane < 32) L.beta[lane] = rb;
      if (pw == 3 && (DK == 128 || lane < 32)) {
        f32x2 t = *(const f32x2*)&L.tot8[c & 1][0][0][ch];
        f32x2 lost = *(const f32x2*)&L.tot8[c & 1][1][0][ch];
#pragma unroll
        for (int i = 1; i < 4; ++i) {
          const f32x2 y = t * *(const f32x2*)&L.tot8[c & 1][1][i][ch];
          dc_times(t, lost, *(const f32x2*)&L.tot8[c & 1][0][i][ch]);
          lost += y;
        }
        // what this product lacks goes into the next chunk's
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float more = fmaf(t[e], owed[e], lost[e]), all = t[e] + more;
          owed[e] = fabsf(all) > 1e-30f
                        ? (t[e] - all + more) * __builtin_amdgcn_rcpf(all) : 0.f;
          t[e] = all;
        }
        *(f32x2*)&L.all[ch] = t;
      }
      if (c + 1 < steps) {
        fetch_pairs(c + 1);
        local(c + 1);
        if (c + 2 < steps) fetch_d(c + 2);
      }
      __syncthreads();
      if (c + 1 < steps) plus(c + 1);
      __syncthreads();
    }
    return;
  }
  // ------------------------------------------------------------ consumers
  const int colb = (cg * NC + w) * 16, col = colb + lr;
  if (colb >= dv) {
    for (int c = -1; c < steps; ++c) {
      __syncthreads();
      __syncthreads();
    }
    return;
  }
  int at_row[DK / 32];
#pragma unroll
  for (int ks = 0; ks < DK / 32; ++ks) at_row[ks] = ch_place<DK>(lr, ks * 4 + lg);
  const int at_km = lr * 64 + ((lg ^ ((lr >> 1) & 3)) << 4);
  float* Sg = A.state + ((long)A.state_slots[s] * A.H + h) * dk * dv;
  const u32 ldv = (u32)(A.H * dv) * 4u;
  const u32 vcol = col < dv ? col * 4u : CH_OUT;
  float pv[8];
  auto fetch = [&](int c) {
    const int left = n - c * CH_T < CH_T ? n - c * CH_T : CH_T;
    const auto rows = ch_rows(
        A.v + ((long)ch_plain(q0 + c * CH_T) * A.H + h) * dv, left * ldv);
#pragma unroll
    for (int e = 0; e < 8; ++e)
      pv[e] = ch_load<float>(
          rows, (u32)((e >> 2) * 16 + (e & 3) + lg * 4) * ldv + vcol);
  };
  f32x4 S[NT];
  fetch(0);
#pragma unroll
  for (int m = 0; m < NT; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = m * 16 + lg * 4 + r;
      S[m][r] = old && col < dv && i < dk ? Sg[(long)i * dv + col] : 0.f;
    }
  float odd = 0.f;      // NaN once a result was not finite
  __syncthreads();
  __syncthreads();
  for (int c = 0; c < steps; ++c) {
    const int left = n - c * CH_T < CH_T ? n - c * CH_T : CH_T;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = pv[e];
    if (c + 1 < steps) fetch(c + 1);
    ChSum2 K[2], O[2];
#pragma unroll
    for (int ks = 0; ks < DK / 32; ++ks) {
      const f32x4 lo = S[2 * ks], hi = S[2 * ks + 1];
      const float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      s16x8 fs[3];
      ch_frag<3>(fs, x);
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        s16x8 fk[3], fq[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          fk[p] = *(const s16x8*)(L.kp + p * PLANE + rt * HALF + at_row[ks]);
          fq[p] = *(const s16x8*)(L.qp + p * PLANE + rt * HALF + at_row[ks]);
        }
        K[rt].mul(fk, fs);
        O[rt].mul(fq, fs);
      }
    }
    __syncthreads();
    s16x8 fu[3];
    {
      float x[8], u[8];
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        const f32x4 y = K[rt].total();
#pragma unroll
        for (int r = 0; r < 4; ++r) x[rt * 4 + r] = v[rt * 4 + r] - y[r];
      }
      s16x8 fx[3];
      ch_frag<3>(fx, x);
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        s16x8 fm[3];
#pragma unroll
        for (int p = 0; p < 3; ++p)
          fm[p] = *(const s16x8*)(L.m + p * WPLANE + (rt * 16 + lr) * 64 + lg * 16);
        ChSum sum;
        sum.mul(fm, fx);
        const f32x4 y = sum.total();
        const f32x4 b = *(const f32x4*)(L.beta + rt * 16 + lg * 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) u[rt * 4 + r] = b[r] * x[rt * 4 + r] + y[r];
      }
      ch_frag<3>(fu, u);
    }
    const auto orows = ch_rows(
        A.o + ((long)ch_plain(q0 + c * CH_T) * A.H + h) * dv, left * ldv);
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      s16x8 fb[3];
#pragma unroll
      for (int p = 0; p < 3; ++p)
        fb[p] = *(const s16x8*)(L.b + p * WPLANE + (rt * 16 + lr) * 64 + lg * 16);
      ChSum near;
      near.mul(fb, fu);
      const f32x4 y = O[rt].total() + near.total();
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        odd += y[r] * 0.f;
        __builtin_amdgcn_raw_buffer_store_b32(
            __float_as_uint(y[r]), orows, (u32)(rt * 16 + r + lg * 4) * ldv + vcol,
            0, 0);
      }
    }
    // four tiles side by side: a chain's products wait for one another
#pragma unroll
    for (int m0 = 0; m0 < NT; m0 += 4) {
      s16x8 fk[4][3];
      f32x4 y[4];
#pragma unroll
      for (int m = m0; m < m0 + 4; ++m) {
        y[m - m0] = (f32x4)(0.f);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          fk[m - m0][p] =
              *(const s16x8*)(L.km + p * PLANE + m * 16 * 64 + at_km);
        }
      }
#pragma unroll
      for (int o = 2; o >= 0; --o)
#pragma unroll
        for (int i = 0; i <= o; ++i)
#pragma unroll
          for (int m = 0; m < 4; ++m) y[m] = ch_mfma(fk[m][i], fu[o - i], y[m]);
#pragma unroll
      for (int m = 0; m < 4; ++m)
        S[m0 + m] = S[m0 + m] * *(const f32x4*)(L.all + (m0 + m) * 16 + lg * 4) + y[m];
    }
    __syncthreads();
  }
#pragma unroll
  for (int m = 0; m < NT; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) odd += S[m][r] * 0.f;
  // a wave whose columns are not finite does them again by itself
  if (__any(odd != 0.f)) {
    delta_serial<DK, HEAD>(A, s, h, colb, lane);
    return;
  }
#pragma unroll
  for (int m = 0; m < NT; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = m * 16 + lg * 4 + r;
      if (col < dv && i < dk) Sg[(long)i * dv + col] = S[m][r];
    }
}

template <int DK, bool HEAD, int NC>
static void delta_chunks_go(DeltaChunkArgs A, int seqs, hipStream_t s) {
  constexpr int bytes =
      9 * CH_T * DK * 2 + 6 * CH_T * CH_T * 2 + (2 * 2 * 4 + 1) * DK * 4 + CH_T * 4;
  static std::atomic<unsigned long long> asked{0};
  const auto fn = delta_chunks_kernel<DK, HEAD, NC>;
  lds_limit((const void*)fn, bytes, asked);
  A.cgs = (A.dv + 16 * NC - 1) / (16 * NC);
  A.n_wg = seqs * A.H * A.cgs;
  A.run = ch_run(A.n_wg);
  hipLaunchKernelGGL(fn, dim3(ch_grid(A.n_wg, A.run)), dim3((NC + 4) * 64), bytes, s, A);
}
static inline long dc_slots(long T, int least) { return T / CH_T + T / least; }

template <int DK, bool HEAD>
static void delta_chunks_launch(const DeltaChunkArgs& A, long T, hipStream_t s) {
  hipLaunchKernelGGL((delta_pairs_kernel<DK, HEAD>),
                     dim3((unsigned)(dc_slots(T, A.least) * A.H)), dim3(256), 0, s, A);
  const int seqs = (int)(T / A.least < A.S ? T / A.least : A.S);
  const long wgs = (long)seqs * A.H * ((A.dv + 127) / 128);
  if (A.dv > 64 && wgs > 128) delta_chunks_go<DK, HEAD, 8>(A, seqs, s);
  else delta_chunks_go<DK, HEAD, 4>(A, seqs, s);
}

// New tokens from which a sequence goes through chunks (0: none of the batch does), as in
// chunk_scan_least. Measured, 32 to 256 workgroups, 512, and 1024 to 4096:
//            a decay a channel                 a decay a head
//   16 x 64    24, 32   64   128 to never       32        64   never
//   32 x 128   48, 64   64   never              48, 64   128   never
//   64 x 16    48, 64   64    48                48, 64    64    64 to 192
//   64 x 64    48, 64   64    64                48, 64    96    64 to 128
//   64 x 128   48, 64   96    64                48, 64    96    96 to never
//  128 x 16    48, 96   96    64 to 128         64, 128  128   128
//  128 x 64    48, 64  128    96 to 128         64, 96   128   128 to 192
//  128 x 128   48, 64   48    48                64        64    48 to 64
// (16 heads of 32 x 64 with a decay a head, 256 sequences of 128 tokens: 370 and 481 us; of
// 64 x 128, 32 heads, 128 of 64: 306 and 389; of 128 x 128, 256 of 64: 663 and 560.)
static inline int delta_chunks_least(const float* q, const float* k,
                                     const float* d, bool head, long T,
                                     long longest, int S, int H, int dk, int dv) {
  const long most = 1 << 23;               // 32 rows within 2^31 bytes
  if (dk > 128 || dk % 4 || (size_t)q % 16 || (size_t)k % 16 ||
      (!head && (size_t)d % 16) || (long)H * dk >= most || (long)H * dv >= most)
    return 0;
  const int cgs = (dv + 127) / 128, columns = dv / cgs;
  ChunkNeed need;
  if (dk > 64)
    need = columns > 80 ? ChunkNeed{64, 64, 64} : ChunkNeed{96, 128, head ? 192 : 128};
  else if (dk > 32)
    need = head ? ChunkNeed{64, 96, 192} : ChunkNeed{64, 96, 64};
  else
    need = ChunkNeed{64, 192, CH_NEVER};   // (ragged, 480 workgroups, from 128: 148 -> 166)
  return chunk_least(need, T, longest, S, (long)H * cgs);
}
