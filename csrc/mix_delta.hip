// Gated delta rule with one decay per head and key channel, or per head.
//
//   delta_prep         short causal depthwise filter + silu on the q|k|v
//                      channels, unit-norm q (times dk^-1/2) and k; with one
//                      decay per head also beta = sigmoid and decay =
//                      exp(-exp(A_log) softplus(a + dt_bias)); a sequence with
//                      one new token gets its filter history brought up to
//                      date here
//   delta_gates        beta = sigmoid, decay = exp(-exp(A_log) *
//                      softplus(a2 a1 + dt_bias)) per head and key channel
//   conv_state_update  keeps the last taps-1 raw filter inputs of sequences
//                      with several new tokens
//   delta_scan         S <- decay * S; u = beta (v - S^T k); S <- S + k u^T;
//                      o = S^T q, token by token, S [dk, dv] fp32 per head
//   delta_out          o / rms(o) * w * sigmoid(g2 g1), cast, into the
//                      output-projection input
//
// Everything the recurrence consumes is fp32. A sequence whose first token
// (position 0) is in the batch starts from zero filter history and zero S,
// whatever its state slot held before.
//
// delta_scan maps the state onto lanes by COLUMN: the dv columns of S never
// interact, so a column is owned by R adjacent lanes holding dk/R rows each
// in registers; one token costs two R-lane sums (DPP moves) and broadcast
// reads of the staged k, q and decay rows. Blocks cover (sequence, head,
// group of columns). Longer pieces of prompts go through chunks instead
// (mix_delta_chunk.h).
#include <climits>

#include "mix_delta_chunk.h"

#define WPB 4
#define PT 8   // tokens per wave in delta_prep

// merged channel c (q | k | v order) -> column of the projection buffer
__device__ __forceinline__ int chan_col(int c, int Cq, int q_off, int k_off,
                                        int v_off) {
  return c < Cq ? q_off + c : (c < 2 * Cq ? k_off + c - Cq : v_off + c - 2 * Cq);
}

// The per-head gates of one token, spread over lanes l, l + n, ...: beta from
// column b_off, decay from column a_off (both H wide).
struct HeadGates {
  float* decay;           // [T, H]; null: the gates are made elsewhere
  float* beta;            // [T, H]
  int b_off, a_off;
  const float* dt_bias;   // [H]
  const float* a_log;     // [H]
};

template <typename A>
__device__ __forceinline__ void head_gates(const HeadGates& hg, const A* row,
                                           long t, int H, int l, int n) {
  for (int h = l; h < H; h += n) {
    const float a = ldf<A>(row + hg.a_off + h) + hg.dt_bias[h];
    hg.decay[t * H + h] = expf(-expf(hg.a_log[h]) * softplus_f(a));
    hg.beta[t * H + h] = sigmoid_f(ldf<A>(row + hg.b_off + h));
  }
}

// A filter pass walks back from the current token: history row taps-1-back is
// read, and in a sequence with one new token the input `back` tokens ago moves
// to history row taps-2-back. The move is made one step late, when the row it
// overwrites has been read; nobody else touches these channels.
template <typename A>
__global__ void delta_prep_kernel(
    float* __restrict__ qn, float* __restrict__ kn, float* __restrict__ vv,
    HeadGates hg, const A* __restrict__ proj, long ld, int q_off, int k_off,
    int v_off, const float* __restrict__ conv_w, int taps, float* conv_state,
    const int* __restrict__ state_slots, const int* __restrict__ qlocs,
    const int* __restrict__ seq_lens, const int* __restrict__ token_seq,
    long T, int H, int G, int dk, int dv) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = threadIdx.x / WAVE;
  const int heads = 2 * G + H;
  const int units = heads + (hg.decay ? 1 : 0);
  // a wave owns one head unit and PT consecutive tokens
  const long wv = (long)blockIdx.x * WPB + wid;
  const long tg = wv / units;
  const int j = (int)(wv - tg * units);
  const int Cq = G * dk, C = 2 * Cq + H * dv;
  for (long t = tg * PT; t < T && t < (tg + 1) * PT; ++t) {
  if (j == heads) {  // wave-uniform
    head_gates<A>(hg, proj + t * ld, t, H, lane, WAVE);
    continue;
  }
  // filter + silu of one q, k or v head
  const int kind = j < G ? 0 : (j < 2 * G ? 1 : 2);
  const int head = kind == 0 ? j : (kind == 1 ? j - G : j - 2 * G);
  const int d = kind == 2 ? dv : dk;
  const int c0 = (kind == 0 ? 0 : (kind == 1 ? Cq : 2 * Cq)) + head * d;
  const int s = token_seq[t];
  const int q0 = qlocs[s], n = qlocs[s + 1] - q0;
  const int start = seq_lens[s] - n;      // position of the chunk's first token
  const int jl = (int)t - q0;             // local index in the chunk
  float* hist = conv_state + (long)state_slots[s] * (taps - 1) * C;

  float y[4];  // d <= 256
  float ssq = 0.f;
  int k = 0;
  for (int i = lane; i < d; i += WAVE, ++k) {
    const int c = c0 + i;
    const int col = chan_col(c, Cq, q_off, k_off, v_off);
    float acc = 0.f, newer = 0.f;
    for (int back = 0; back < taps; ++back) {
      float x = 0.f;
      if (jl - back >= 0)
        x = ldf<A>(proj + (t - back) * ld + col);
      else if (start > 0)  // start + jl - back >= 0 is implied: the history
        x = hist[(long)(taps - 1 - back + jl) * C + c];  // holds zeros there
      if (n == 1 && back > 0) hist[(long)(taps - 1 - back) * C + c] = newer;
      newer = x;
      acc += conv_w[(long)c * taps + (taps - 1 - back)] * x;
    }
    const float a = acc * sigmoid_f(acc);
    y[k] = a;
    ssq += a * a;
  }
  ssq = wave_sum_f32(ssq);
  float f = 1.f;
  if (kind != 2) {
    f = 1.f / sqrtf(ssq + 1e-6f);
    if (kind == 0) f *= 1.f / sqrtf((float)dk);
  }
  float* dst = kind == 0 ? qn + (t * G + head) * (long)dk
                         : (kind == 1 ? kn + (t * G + head) * (long)dk
                                      : vv + (t * H + head) * (long)dv);
  k = 0;
  for (int i = lane; i < d; i += WAVE, ++k) dst[i] = y[k] * f;
  }  // tokens of this wave
}

// bf16 fast path of delta_prep: a group of GS lanes owns one (token, head)
// unit, lane gl its 8-channel chunk (16-byte loads of the raw rows, float4
// loads of the transposed filter [taps, C] and of the history, float4
// stores). Needs dk, dv and all offsets to be multiples of 8.
template <int GS>
__global__ void delta_prep_vec_kernel(
    float* __restrict__ qn, float* __restrict__ kn, float* __restrict__ vv,
    HeadGates hg, const u16* __restrict__ proj, long ld, int q_off, int k_off,
    int v_off, const float* __restrict__ conv_wt, int taps, float* conv_state,
    const int* __restrict__ state_slots, const int* __restrict__ qlocs,
    const int* __restrict__ seq_lens, const int* __restrict__ token_seq,
    long T, int H, int G, int dk, int dv) {
  constexpr int UPWV = 64 / GS;
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = threadIdx.x / WAVE;
  const int gi = lane / GS, gl = lane % GS;
  const int heads = 2 * G + H;
  const int units = heads + (hg.decay ? 1 : 0);
  const long total = T * units;
  const long u = ((long)blockIdx.x * WPB + wid) * UPWV + gi;
  const bool valid = u < total;
  const long t = valid ? u / units : 0;
  const int j = valid ? (int)(u - t * units) : 0;
  const int Cq = G * dk, C = 2 * Cq + H * dv;
  const int kind = j < G ? 0 : (j < 2 * G ? 1 : 2);
  const int head = kind == 0 ? j : (kind == 1 ? j - G : j - 2 * G);
  const int d = kind == 2 ? dv : dk;
  const int c0 = gl * 8;
  const bool act = valid && j < heads && c0 < d;
  const int c = (kind == 0 ? 0 : (kind == 1 ? Cq : 2 * Cq)) + head * d + c0;
  if (valid && j == heads) head_gates<u16>(hg, proj + t * ld, t, H, gl, GS);
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  if (act) {
    const int col = chan_col(c, Cq, q_off, k_off, v_off);
    const int s = token_seq[t];
    const int q0 = qlocs[s], n = qlocs[s + 1] - q0;
    const int start = seq_lens[s] - n;
    const int jl = (int)t - q0;
    float* hist = conv_state + (long)state_slots[s] * (taps - 1) * C;
    float newer[8];
    for (int back = 0; back < taps; ++back) {
      float x[8];
      if (jl - back >= 0) {
        bf8_to_f32(*(const u16x8*)(proj + (t - back) * ld + col), x);
      } else if (start > 0) {
        const float* hp = hist + (long)(taps - 1 - back + jl) * C + c;
        const f32x4 a = *(const f32x4*)hp, b = *(const f32x4*)(hp + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) { x[e] = a[e]; x[e + 4] = b[e]; }
      } else {  // before the start of the sequence: zeros
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = 0.f;
      }
      if (n == 1) {
        if (back > 0) {
          float* hp = hist + (long)(taps - 1 - back) * C + c;
          f32x4 a, b;
#pragma unroll
          for (int e = 0; e < 4; ++e) { a[e] = newer[e]; b[e] = newer[e + 4]; }
          *(f32x4*)hp = a;
          *(f32x4*)(hp + 4) = b;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) newer[e] = x[e];
      }
      const float* wp = conv_wt + (long)(taps - 1 - back) * C + c;
      const f32x4 w0 = *(const f32x4*)wp, w1 = *(const f32x4*)(wp + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc[e] += w0[e] * x[e];
        acc[e + 4] += w1[e] * x[e + 4];
      }
    }
  }
  float ssq = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    acc[e] = acc[e] * sigmoid_f(acc[e]);
    ssq += acc[e] * acc[e];
  }
#pragma unroll
  for (int off = GS / 2; off > 0; off >>= 1) ssq += __shfl_xor(ssq, off, WAVE);
  if (!act) return;
  float f = 1.f;
  if (kind != 2) {
    f = 1.f / sqrtf(ssq + 1e-6f);
    if (kind == 0) f *= 1.f / sqrtf((float)dk);
  }
  float* dst = (kind == 0 ? qn + (t * G + head) * (long)dk
                          : (kind == 1 ? kn + (t * G + head) * (long)dk
                                       : vv + (t * H + head) * (long)dv)) + c0;
  f32x4 o0, o1;
#pragma unroll
  for (int e = 0; e < 4; ++e) { o0[e] = acc[e] * f; o1[e] = acc[e + 4] * f; }
  *(f32x4*)dst = o0;
  *(f32x4*)(dst + 4) = o1;
}

// The same with four taps for many tokens: a group of lanes takes its unit over
// RUN consecutive tokens, with the filter and the last three inputs in registers
// and the run's inputs loaded together. Token by token the filter alone was
// eight times the bytes of the input, and every input was read four times, which
// took 555 us for 32,768 tokens of 48 heads of 128: now 303 (4 TB/s).
template <int GS, int RUN>
__global__ void __launch_bounds__(WPB * WAVE) delta_prep_run_kernel(
    float* __restrict__ qn, float* __restrict__ kn, float* __restrict__ vv,
    HeadGates hg, const u16* __restrict__ proj, long ld, int q_off, int k_off,
    int v_off, const float* __restrict__ conv_wt, float* conv_state,
    const int* __restrict__ state_slots, const int* __restrict__ qlocs,
    const int* __restrict__ seq_lens, const int* __restrict__ token_seq,
    long T, int H, int G, int dk, int dv) {
  const int gl = threadIdx.x % GS;
  const int heads = 2 * G + H;
  const u32 units = heads + (hg.decay ? 1 : 0);
  const u32 u = blockIdx.x * (u32)(WPB * WAVE / GS) + threadIdx.x / GS;
  const long t0 = (long)(u / units) * RUN;
  const int j = (int)(u % units);
  if (t0 >= T) return;                    // whole groups
  const int len = (int)(T - t0 < RUN ? T - t0 : RUN);
  if (j == heads) {
    for (int i = 0; i < len; ++i)
      head_gates<u16>(hg, proj + (t0 + i) * ld, t0 + i, H, gl, GS);
    return;
  }
  const int Cq = G * dk, C = 2 * Cq + H * dv;
  const int kind = j < G ? 0 : (j < 2 * G ? 1 : 2);
  const int head = kind == 0 ? j : (kind == 1 ? j - G : j - 2 * G);
  const int d = kind == 2 ? dv : dk;
  const bool act = gl * 8 < d;
  const int c0 = act ? gl * 8 : 0;        // idle lanes follow the first
  const int c = (kind == 0 ? 0 : (kind == 1 ? Cq : 2 * Cq)) + head * d + c0;
  const int col = chan_col(c, Cq, q_off, k_off, v_off);

  u16x8 raw[RUN];
#pragma unroll
  for (int i = 0; i < RUN; ++i)
    raw[i] = *(const u16x8*)(proj + (t0 + (i < len ? i : 0)) * ld + col);
  float wt[4][8], x[4][8];                // x[back]: the input `back` ago
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const f32x4 w0 = *(const f32x4*)(conv_wt + (long)(3 - b) * C + c);
    const f32x4 w1 = *(const f32x4*)(conv_wt + (long)(3 - b) * C + c + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) { wt[b][e] = w0[e]; wt[b][e + 4] = w1[e]; }
  }
  float* dst = (kind == 0 ? qn + (t0 * G + head) * (long)dk
                          : (kind == 1 ? kn + (t0 * G + head) * (long)dk
                                       : vv + (t0 * H + head) * (long)dv)) + c0;
  const long step = kind == 2 ? (long)H * dv : (long)G * dk;
  int s = -1;
#pragma unroll
  for (int i = 0; i < RUN; ++i) {
    if (i >= len) break;
    const long t = t0 + i;
#pragma unroll
    for (int b = 3; b > 0; --b)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[b][e] = x[b - 1][e];
    bf8_to_f32(raw[i], x[0]);
    const int st = token_seq[t];
    if (st != s) {                        // the inputs before a new sequence
      s = st;
      const int q0 = qlocs[s], n = qlocs[s + 1] - q0;
      const int start = seq_lens[s] - n;
      const int jl = (int)t - q0;
      float* hist = conv_state + (long)state_slots[s] * 3 * C + c;
#pragma unroll
      for (int b = 1; b < 4; ++b) {
        if (jl - b >= 0) {
          bf8_to_f32(*(const u16x8*)(proj + (t - b) * ld + col), x[b]);
        } else if (start > 0) {
          const f32x4 h0 = *(const f32x4*)(hist + (long)(3 - b + jl) * C);
          const f32x4 h1 = *(const f32x4*)(hist + (long)(3 - b + jl) * C + 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) { x[b][e] = h0[e]; x[b][e + 4] = h1[e]; }
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) x[b][e] = 0.f;
        }
      }
      if (n == 1 && act)                  // one new token: its history moves on
#pragma unroll
        for (int b = 1; b < 4; ++b) {
          f32x4 h0, h1;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            h0[e] = x[b - 1][e];
            h1[e] = x[b - 1][e + 4];
          }
          *(f32x4*)(hist + (long)(3 - b) * C) = h0;
          *(f32x4*)(hist + (long)(3 - b) * C + 4) = h1;
        }
    }
    float acc[8], ssq = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float a = 0.f;
#pragma unroll
      for (int b = 0; b < 4; ++b) a += wt[b][e] * x[b][e];
      acc[e] = a * sigmoid_f(a);
      ssq += act ? acc[e] * acc[e] : 0.f;
    }
#pragma unroll
    for (int off = GS / 2; off > 0; off >>= 1)
      ssq += __shfl_xor(ssq, off, WAVE);
    float f = 1.f;
    if (kind != 2) {
      f = 1.f / sqrtf(ssq + 1e-6f);
      if (kind == 0) f *= 1.f / sqrtf((float)dk);
    }
    if (act) {
      f32x4 o0, o1;
#pragma unroll
      for (int e = 0; e < 4; ++e) { o0[e] = acc[e] * f; o1[e] = acc[e + 4] * f; }
      *(f32x4*)(dst + i * step) = o0;
      *(f32x4*)(dst + i * step + 4) = o1;
    }
  }
}

// ---- low-rank gates ---------------------------------------------------------
// Both gate kernels evaluate act(W2 (W1 h) + bias) where W1 h (`rank` numbers
// a token) is a section of the merged projection and W2 arrives transposed
// [rank, rows]. A wave owns GT consecutive tokens and one head: a lane keeps
// the W2 column of its output channel in registers across those tokens, the
// token's `rank` inputs sit one per lane and reach the FMAs through readlane
// (scalar operands), so the inner loop issues no loads at all.
#define GT 8     // tokens per wave
#define RMAX 32  // W2 rows held per pass

__device__ __forceinline__ float lane_bcast(float v, int src) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}

// acc[tt] += sum_r w2t[(r0 + r) * stride + col] * in[t_base + tt][r0 + r]
template <typename A>
__device__ __forceinline__ void low_rank_acc(
    float (&acc)[GT], const float* __restrict__ w2t, long stride, long col,
    bool col_ok, int rank, const A* __restrict__ in, long ld, long t_base,
    long T, int lane) {
  for (int r0 = 0; r0 < rank; r0 += RMAX) {
    float w[RMAX];
#pragma unroll
    for (int r = 0; r < RMAX; ++r)
      w[r] = (col_ok && r0 + r < rank) ? w2t[(long)(r0 + r) * stride + col] : 0.f;
    float x[GT];  // lane r holds input r of token tt
#pragma unroll
    for (int tt = 0; tt < GT; ++tt)
      x[tt] = (t_base + tt < T && lane < RMAX && r0 + lane < rank)
                  ? ldf<A>(in + (t_base + tt) * ld + r0 + lane) : 0.f;
    // r outer, tokens inner: GT independent readlane + FMA chains
#pragma unroll
    for (int r = 0; r < RMAX; ++r)
#pragma unroll
      for (int tt = 0; tt < GT; ++tt) acc[tt] += w[r] * lane_bcast(x[tt], r);
  }
}

// decay[t,h,i] = exp(-exp(a_log[h]) * softplus(a2 a1 + dt_bias)), beta[t,h] =
// sigmoid(b section). grid (token groups, H).
template <typename A>
__global__ void delta_gates_kernel(
    float* __restrict__ decay, float* __restrict__ beta,
    const A* __restrict__ proj, long ld, int b_off, int a1_off,
    const float* __restrict__ a2t, int rank, const float* __restrict__ dt_bias,
    const float* __restrict__ a_log, long T, int H, int dk) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int h = blockIdx.y;
  const long t_base = ((long)blockIdx.x * WPB + wid) * GT;
  if (t_base >= T) return;
  const float rate = expf(a_log[h]);
  const long HD = (long)H * dk;
  for (int k0 = 0; k0 < dk; k0 += WAVE) {
    const int i = k0 + lane;
    const bool in = i < dk;
    float acc[GT];
    const float bias = in ? dt_bias[h * dk + i] : 0.f;
#pragma unroll
    for (int tt = 0; tt < GT; ++tt) acc[tt] = bias;
    low_rank_acc<A>(acc, a2t, HD, (long)h * dk + i, in, rank, proj + a1_off, ld,
                    t_base, T, lane);
#pragma unroll
    for (int tt = 0; tt < GT; ++tt)
      if (in && t_base + tt < T)
        decay[((t_base + tt) * H + h) * (long)dk + i] =
            expf(-rate * softplus_f(acc[tt]));
  }
  if (lane < GT && t_base + lane < T)
    beta[(t_base + lane) * H + h] =
        sigmoid_f(ldf<A>(proj + (t_base + lane) * ld + b_off + h));
}

// one thread per (sequence, channel): new history = last taps-1 raw inputs
// (delta_prep has done it for sequences with one new token)
template <typename A>
__global__ void conv_state_update_kernel(
    float* __restrict__ conv_state, const A* __restrict__ proj, long ld,
    int q_off, int k_off, int v_off, int taps,
    const int* __restrict__ state_slots, const int* __restrict__ qlocs,
    const int* __restrict__ seq_lens, int S, int Cq, int C) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)S * C) return;
  const int s = (int)(idx / C), c = (int)(idx - (long)s * C);
  const int q0 = qlocs[s], n = qlocs[s + 1] - q0;
  if (n <= 1) return;
  const int start = seq_lens[s] - n;
  const int col = chan_col(c, Cq, q_off, k_off, v_off);
  float* hist = conv_state + (long)state_slots[s] * (taps - 1) * C + c;
  for (int i = 0; i < taps - 1; ++i) {
    const int tau = n - (taps - 1) + i;  // chunk-local time of history row i
    float x = 0.f;
    if (tau >= 0)
      x = ldf<A>(proj + (long)(q0 + tau) * ld + col);
    else if (start > 0 && i + n <= taps - 2)
      x = hist[(long)(i + n) * C];       // read before row i+n is rewritten
    hist[(long)i * C] = x;
  }
}

#define TB 8    // tokens staged per step

// Token-by-token scan. Block = (sequence, head, group of 256/R columns);
// lane (col, r) keeps rows {((n/4)*R + r)*4 + n%4 : n < RPT} of its column of
// S in registers (RPT = 32, or 16 to double the number of waves when a
// launch would leave SIMDs idle) (rows past dk stay zero: their k and q are staged as 0 and
// their decay as 1). k, q, decay, v and beta of TB tokens at a time are
// staged through a double-buffered LDS tile: the global loads of tile s+1
// are issued before the arithmetic of tile s and parked in registers. With
// this row mapping the R lanes of a column read consecutive float4s of a
// staged row, and all columns read the same addresses (LDS broadcast).
// HEAD: decay [T, H], one number a token and head (staged beside beta).
// Sequences of `below` or more new tokens are left to the chunks.
template <int R, int RPT, bool HEAD>
__global__ void __launch_bounds__(256) delta_scan_kernel(
    float* __restrict__ o, const float* __restrict__ qn,
    const float* __restrict__ kn, const float* __restrict__ vv,
    const float* __restrict__ decay, const float* __restrict__ beta,
    float* __restrict__ ssm, const int* __restrict__ state_slots,
    const int* __restrict__ qlocs, const int* __restrict__ seq_lens, int H,
    int G, int dk, int dv, int col_groups, int below) {
  constexpr int DKP = R * RPT;
  constexpr int CPB = 256 / R;            // columns per block
  constexpr int KQD = HEAD ? 2 : 3;       // rows of DKP floats a token
  constexpr int NK = KQD * TB * DKP / 256;  // staged k|q(|decay) per lane
  constexpr int NV = TB * CPB / 256 > 0 ? TB * CPB / 256 : 1;
  constexpr int VOFF = KQD * TB * DKP;    // v, then beta, then head decays
  constexpr int TILE = VOFF + TB * CPB + (HEAD ? 2 : 1) * TB;
  __shared__ __attribute__((aligned(16))) float lds[2][TILE];

  int b = blockIdx.x;
  const int cg = b % col_groups; b /= col_groups;
  const int h = b % H;
  const int s = b / H;
  const int tid = threadIdx.x;
  const int r = tid % R;
  const int cl = tid / R;                 // column within the block
  const int col = cg * CPB + cl;
  const bool cv = col < dv;
  const int g = h / (H / G);
  const int q0 = qlocs[s], q1 = qlocs[s + 1];
  if (q1 <= q0 || q1 - q0 >= below) return;
  const int start = seq_lens[s] - (q1 - q0);
  float* Sg = ssm + (((long)state_slots[s] * H + h) * dk) * dv;

  float S[RPT];
#pragma unroll
  for (int n = 0; n < RPT; ++n) {
    const int i = ((n >> 2) * R + r) * 4 + (n & 3);
    S[n] = (start > 0 && cv && i < dk) ? Sg[(long)i * dv + col] : 0.f;
  }

  float pk[NK], pv[NV], pb = 0.f, pd = 1.f;
  auto prefetch = [&](int t0) {
#pragma unroll
    for (int n = 0; n < NK; ++n) {
      const int e = tid + n * 256;
      const int arr = e / (TB * DKP), rem = e % (TB * DKP);
      const int tok = rem / DKP, i = rem % DKP;
      const int t = t0 + tok;
      float x = arr == 2 ? 1.f : 0.f;
      if (t < q1 && i < dk) {
        if (arr == 0) x = kn[((long)t * G + g) * dk + i];
        else if (arr == 1) x = qn[((long)t * G + g) * dk + i];
        else x = decay[((long)t * H + h) * dk + i];
      }
      pk[n] = x;
    }
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int e = tid + n * 256;
      const int tok = e / CPB, c = cg * CPB + e % CPB;
      const int t = t0 + tok;
      pv[n] = (e < TB * CPB && t < q1 && c < dv)
                  ? vv[((long)t * H + h) * dv + c] : 0.f;
    }
    if (tid < TB) {
      const bool in = t0 + tid < q1;
      pb = in ? beta[(long)(t0 + tid) * H + h] : 0.f;
      if (HEAD) pd = in ? decay[(long)(t0 + tid) * H + h] : 1.f;
    }
  };

  prefetch(q0);
  int buf = 0;
  for (int t0 = q0; t0 < q1; t0 += TB, buf ^= 1) {
    float* L = lds[buf];
#pragma unroll
    for (int n = 0; n < NK; ++n) L[tid + n * 256] = pk[n];
#pragma unroll
    for (int n = 0; n < NV; ++n)
      if (tid + n * 256 < TB * CPB) L[VOFF + tid + n * 256] = pv[n];
    if (tid < TB) {
      L[VOFF + TB * CPB + tid] = pb;
      if (HEAD) L[VOFF + TB * CPB + TB + tid] = pd;
    }
    __syncthreads();
    if (t0 + TB < q1) prefetch(t0 + TB);
    const int nt = min(TB, q1 - t0);
    for (int tok = 0; tok < nt; ++tok) {
      const f32x4* K4 = (const f32x4*)(L + tok * DKP);
      const f32x4* Q4 = (const f32x4*)(L + (TB + tok) * DKP);
      const f32x4* D4 = (const f32x4*)(L + (HEAD ? 0 : 2 * TB + tok) * DKP);
      const float vt = L[VOFF + tok * CPB + cl];
      const float bt = L[VOFF + TB * CPB + tok];
      const float gt = HEAD ? L[VOFF + TB * CPB + TB + tok] : 1.f;
      float kk[RPT];
      float dot = 0.f;
#pragma unroll
      for (int m = 0; m < RPT / 4; ++m) {
        const f32x4 k4 = K4[m * R + r];
        f32x4 d4;
        if (!HEAD) d4 = D4[m * R + r];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          kk[m * 4 + j] = k4[j];
          S[m * 4 + j] *= HEAD ? gt : d4[j];
          dot += S[m * 4 + j] * k4[j];
        }
      }
      dot = group_sum<R>(dot);
      const float uu = bt * (vt - dot);
      float out = 0.f;
#pragma unroll
      for (int m = 0; m < RPT / 4; ++m) {
        const f32x4 q4 = Q4[m * R + r];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          S[m * 4 + j] += kk[m * 4 + j] * uu;
          out += S[m * 4 + j] * q4[j];
        }
      }
      out = group_sum<R>(out);
      if (r == 0 && cv) o[((long)(t0 + tok) * H + h) * dv + col] = out;
    }
  }
  if (cv) {
#pragma unroll
    for (int n = 0; n < RPT; ++n) {
      const int i = ((n >> 2) * R + r) * 4 + (n & 3);
      if (i < dk) Sg[(long)i * dv + col] = S[n];
    }
  }
}

// out[t, out_off + h*dv + c] = out_scale * o[t,h,c] / rms(o[t,h,:]) * w[c] *
// sigmoid(g2 g1)[h*dv + c]. grid (token groups, H); a wave owns GT tokens.
template <typename A>
__global__ void delta_out_kernel(A* __restrict__ out, long ldo, int out_off,
                                 const float* __restrict__ o,
                                 const float* __restrict__ norm_w,
                                 const A* __restrict__ proj, long ld,
                                 int g1_off, const float* __restrict__ g2t,
                                 int rank, float eps, float out_scale, long T,
                                 int H, int dv) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int h = blockIdx.y;
  const long t_base = ((long)blockIdx.x * WPB + wid) * GT;
  if (t_base >= T) return;
  float inv[GT];
#pragma unroll
  for (int tt = 0; tt < GT; ++tt) {
    inv[tt] = 0.f;
    const long t = t_base + tt;
    if (t >= T) break;
    const float* orow = o + (t * H + h) * (long)dv;
    float ssq = 0.f;
    for (int c = lane; c < dv; c += WAVE) ssq += orow[c] * orow[c];
    ssq = wave_sum_f32(ssq);
    inv[tt] = out_scale / sqrtf(ssq / (float)dv + eps);
  }
  const long HV = (long)H * dv;
  for (int k0 = 0; k0 < dv; k0 += WAVE) {
    const int c = k0 + lane;
    const bool in = c < dv;
    float acc[GT];
#pragma unroll
    for (int tt = 0; tt < GT; ++tt) acc[tt] = 0.f;
    low_rank_acc<A>(acc, g2t, HV, (long)h * dv + c, in, rank, proj + g1_off, ld,
                    t_base, T, lane);
    const float wn = in ? norm_w[c] : 0.f;
#pragma unroll
    for (int tt = 0; tt < GT; ++tt) {
      const long t = t_base + tt;
      if (in && t < T)
        stf<A>(out + t * ldo + out_off + (long)h * dv + c,
               o[(t * H + h) * (long)dv + c] * inv[tt] * wn *
                   sigmoid_f(acc[tt]));
    }
  }
}

// ---- low-rank gates on the matrix cores ----
// bf16 projections of rank up to 32 and heads of whole tiles: W2 x is a product
// of [16 channels x 32] by [32 x 16 tokens] tiles. W2 is fp32: it is split into
// three bf16 terms (24 bits: exact), held as fragments in registers across the
// wave's tokens, and the three products are summed in fp32 from the smallest
// term up, so that nothing is rounded that the FMA chain did not round. A lane
// ends with four neighbouring channels of one token (16-byte loads and stores).
// The chain spent 64 instructions an output on readlane and FMA; 32,768 tokens
// of 16 heads x 128 channels, rank 32: gates 516 -> 227 us
// (what is left is exp and log1p), read-out 442 -> 140 us (2.9 TB/s).
#define LR_TOK 128   // tokens per wave, at most

__device__ __forceinline__ f32x4 lr_mfma(s16x8 a, s16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// the fragments of 16 channels: this lane's is channel `col`, k = k0 .. k0 + 7
__device__ __forceinline__ void lr_split(s16x8 (&w)[3],
                                         const float* __restrict__ w2t,
                                         long stride, long col, int k0,
                                         int rank) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    float v = k0 + j < rank ? w2t[(long)(k0 + j) * stride + col] : 0.f;
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      const u16 b = f2bf(v);
      w[n][j] = (short)b;
      const float f = bf2f(b);
      v = fabsf(f) <= 3.4e38f ? v - f : 0.f;   // nothing below an infinity
    }
  }
}

// eight inputs of a token; infinities become the largest numbers, because a
// term of W2 that is zero must not make them NaN
__device__ __forceinline__ s16x8 lr_input(const u16* p, bool in) {
  s16x8 x = (s16x8)(short)0;
  if (in) x = *(const s16x8*)p;
#pragma unroll
  for (int j = 0; j < 8; ++j)
    if ((x[j] & 0x7fff) == 0x7f80) x[j] = x[j] - 1;
  return x;
}

__device__ __forceinline__ f32x4 lr_dot(const s16x8 (&w)[3], s16x8 x,
                                        f32x4 acc) {
#pragma unroll
  for (int n = 2; n >= 0; --n) acc = lr_mfma(w[n], x, acc);
  return acc;
}

// grid (token groups, H, channel groups of 64); block of four waves, each with
// its own `per` tokens
__global__ void __launch_bounds__(WPB * WAVE) delta_gates_mfma_kernel(
    float* __restrict__ decay, float* __restrict__ beta,
    const u16* __restrict__ proj, long ld, int b_off, int a1_off,
    const float* __restrict__ a2t, int rank, const float* __restrict__ dt_bias,
    const float* __restrict__ a_log, long T, int H, int dk, int per) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int h = blockIdx.y, c0 = blockIdx.z * 64;
  const int lr = lane & 15, g = lane >> 4;
  const long t_end0 = ((long)blockIdx.x * WPB + wid) * per;
  if (t_end0 >= T) return;
  const long t_end = t_end0 + per < T ? t_end0 + per : T;
  const float rate = expf(a_log[h]);
  s16x8 w[4][3];
  f32x4 bias[4];
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    lr_split(w[n], a2t, (long)H * dk, (long)h * dk + c0 + n * 16 + lr, g * 8,
             rank);
    bias[n] = *(const f32x4*)(dt_bias + (long)h * dk + c0 + n * 16 + g * 4);
  }
  for (long t0 = t_end0; t0 < t_end; t0 += 16) {
    const long t = t0 + lr < t_end ? t0 + lr : t_end - 1;
    const s16x8 x = lr_input(proj + t * ld + a1_off + g * 8, g * 8 < rank);
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const f32x4 a = lr_dot(w[n], x, bias[n]);
      f32x4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = expf(-rate * softplus_f(a[e]));
      if (t0 + lr < t_end)
        *(f32x4*)(decay + (t * H + h) * (long)dk + c0 + n * 16 + g * 4) = y;
    }
    if (blockIdx.z == 0 && g == 0 && t0 + lr < t_end)
      beta[t * H + h] = sigmoid_f(bf2f(proj[t * ld + b_off + h]));
  }
}

// grid (token groups, H); a wave owns all dv = 16 NT channels of a head
template <int NT>
__global__ void __launch_bounds__(WPB * WAVE) delta_out_mfma_kernel(
    u16* __restrict__ out, long ldo, int out_off, const float* __restrict__ o,
    const float* __restrict__ norm_w, const u16* __restrict__ proj, long ld,
    int g1_off, const float* __restrict__ g2t, int rank, float eps,
    float out_scale, long T, int H, int per) {
  constexpr int dv = NT * 16;
  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int h = blockIdx.y;
  const int lr = lane & 15, g = lane >> 4;
  const long t_end0 = ((long)blockIdx.x * WPB + wid) * per;
  if (t_end0 >= T) return;
  const long t_end = t_end0 + per < T ? t_end0 + per : T;
  s16x8 w[NT][3];
#pragma unroll
  for (int n = 0; n < NT; ++n)
    lr_split(w[n], g2t, (long)H * dv, (long)h * dv + n * 16 + lr, g * 8, rank);
  for (long t0 = t_end0; t0 < t_end; t0 += 16) {
    const long t = t0 + lr < t_end ? t0 + lr : t_end - 1;
    const float* orow = o + (t * H + h) * (long)dv + g * 4;
    f32x4 v[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) v[n] = *(const f32x4*)(orow + n * 16);
    const s16x8 x = lr_input(proj + t * ld + g1_off + g * 8, g * 8 < rank);
    float ssq = 0.f;
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int e = 0; e < 4; ++e) ssq += v[n][e] * v[n][e];
    ssq += __shfl_xor(ssq, 16, 64);
    ssq += __shfl_xor(ssq, 32, 64);
    const float inv = out_scale / sqrtf(ssq / (float)dv + eps);
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const f32x4 a = lr_dot(w[n], x, (f32x4)(0.f));
      const f32x4 wn = *(const f32x4*)(norm_w + n * 16 + g * 4);
      u16x4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        y[e] = f2bf(v[n][e] * inv * wn[e] * sigmoid_f(a[e]));
      if (t0 + lr < t_end)
        *(u16x4*)(out + t * ldo + out_off + (long)h * dv + n * 16 + g * 4) = y;
    }
  }
}

// 16-byte pieces of the rank inputs, whole tiles of channels
static bool lr_fits(const void* proj, long ld, int off, int rank,
                    const void* w2, const void* vec) {
  return rank > 0 && rank <= 32 && rank % 8 == 0 && ld % 8 == 0 &&
         off % 8 == 0 && (size_t)proj % 16 == 0 && (size_t)vec % 16 == 0 &&
         (size_t)w2 % 4 == 0;
}

// Tokens a wave: 128 to read W2 seldom, fewer (whole tiles of 16) where that
// leaves less than 4096 waves. With 128 always, 200 tokens of 16 heads x 128 took
// 53 us for the inputs with their gates and 30 for the read-out (the readlane
// chain 26 and 19), now 18 and 10; 8192 tokens of 8 heads 84 and 40, now 68 and 24.
static int lr_tokens(long T, long groups) {
  const long per = (T * groups + 4096 * 16 - 1) / (4096 * 16) * 16;
  return per < 16 ? 16 : (per > LR_TOK ? LR_TOK : (int)per);
}

extern "C" void mix_delta_prep(
    float* qn, float* kn, float* vv, float* decay, float* beta,
    const void* proj, long ld, int q_off, int k_off, int v_off, int b_off,
    int a1_off, const float* conv_w, const float* conv_wt, int taps,
    const float* a2, int rank,  // a2 null: one decay per head, a1_off = a
    const float* dt_bias, const float* a_log, float* conv_state,
    const int* state_slots, const int* qlocs, const int* seq_lens,
    const int* token_seq, long T, int S, int H, int G, int dk, int dv, int f32,
    hipStream_t s) {
  // a2 null: the gates are one more unit of the filter kernel
  const HeadGates hg = {a2 ? nullptr : decay, beta, b_off, a1_off, dt_bias,
                        a_log};
  const int n_units = 2 * G + H + (a2 ? 0 : 1);
  const bool hist = taps > 1 && T != (long)S;  // some sequence has more tokens
  const long units = ((T + PT - 1) / PT) * n_units;
  const int grid = (int)((units + WPB - 1) / WPB);
  if (grid == 0) return;
  const dim3 ggrid((unsigned)((T + WPB * GT - 1) / (WPB * GT)), (unsigned)H);
  const bool lr = !f32 && a2 && dk % 64 == 0 && (size_t)decay % 16 == 0 &&
                  lr_fits(proj, ld, a1_off, rank, a2, dt_bias);
  if (lr) {
    const int per = lr_tokens(T, H * (dk / 64));
    hipLaunchKernelGGL(delta_gates_mfma_kernel,
                       dim3((unsigned)((T + WPB * per - 1) / (WPB * per)),
                            (unsigned)H, (unsigned)(dk / 64)),
                       dim3(WPB * WAVE), 0, s, decay, beta, (const u16*)proj,
                       ld, b_off, a1_off, a2, rank, dt_bias, a_log, T, H, dk,
                       per);
  }
  const int Cq = G * dk, C = 2 * Cq + H * dv;
  const long su = (long)S * C;
  const int sgrid = (int)((su + 255) / 256);
  const int dmax = dk > dv ? dk : dv;
  const int dm8 = (dmax + 7) / 8;
  const bool vec = !f32 && conv_wt && dk % 8 == 0 && dv % 8 == 0 &&
                   ld % 8 == 0 && q_off % 8 == 0 && k_off % 8 == 0 &&
                   v_off % 8 == 0 && dm8 <= 32;
  if (vec) {
    const int GS = dm8 <= 4 ? 4 : (dm8 <= 8 ? 8 : (dm8 <= 16 ? 16 : 32));
    const long tot = T * n_units;
    const long waves = (tot + 64 / GS - 1) / (64 / GS);
    const int vgrid = (int)((waves + WPB - 1) / WPB);
#define LAUNCH_DV(GG)                                                          \
  hipLaunchKernelGGL(delta_prep_vec_kernel<GG>, dim3(vgrid), dim3(WPB * WAVE), \
                     0, s, qn, kn, vv, hg, (const u16*)proj, ld, q_off, k_off, \
                     v_off, conv_wt, taps, conv_state, state_slots, qlocs,     \
                     seq_lens, token_seq, T, H, G, dk, dv)
    const long run_units = (T + 7) / 8 * n_units;
#define LAUNCH_DR(GG)                                                          \
  hipLaunchKernelGGL((delta_prep_run_kernel<GG, 8>),                           \
                     dim3((unsigned)((run_units * GG + WPB * WAVE - 1) /       \
                                     (WPB * WAVE))),                           \
                     dim3(WPB * WAVE), 0, s, qn, kn, vv, hg,                   \
                     (const u16*)proj, ld, q_off, k_off, v_off, conv_wt,       \
                     conv_state, state_slots, qlocs, seq_lens, token_seq, T,   \
                     H, G, dk, dv)
    // runs of eight tokens where they leave two workgroups for every CU (24 heads:
    // 276 -> 170 us); a decode step keeps a group for every token
    if (taps == 4 && run_units * GS >= 512 * WPB * WAVE &&
        run_units < (1L << 31) && (GS == 8 || GS == 16)) {
      if (GS == 8) LAUNCH_DR(8);
      else LAUNCH_DR(16);
    }
#undef LAUNCH_DR
    else if (GS == 4) LAUNCH_DV(4);
    else if (GS == 8) LAUNCH_DV(8);
    else if (GS == 16) LAUNCH_DV(16);
    else LAUNCH_DV(32);
#undef LAUNCH_DV
    if (a2 && !lr)
    hipLaunchKernelGGL(delta_gates_kernel<u16>, ggrid, dim3(WPB * WAVE), 0, s,
                       decay, beta, (const u16*)proj, ld, b_off, a1_off, a2,
                       rank, dt_bias, a_log, T, H, dk);
    if (hist)
      hipLaunchKernelGGL(conv_state_update_kernel<u16>, dim3(sgrid), dim3(256),
                         0, s, conv_state, (const u16*)proj, ld, q_off, k_off,
                         v_off, taps, state_slots, qlocs, seq_lens, S, Cq, C);
    return;
  }
  if (f32) {
    hipLaunchKernelGGL(delta_prep_kernel<float>, dim3(grid), dim3(WPB * WAVE),
                       0, s, qn, kn, vv, hg, (const float*)proj, ld, q_off, k_off,
                       v_off, conv_w, taps, conv_state, state_slots, qlocs,
                       seq_lens, token_seq, T, H, G, dk, dv);
    if (a2 && !lr)
    hipLaunchKernelGGL(delta_gates_kernel<float>, ggrid, dim3(WPB * WAVE), 0, s,
                       decay, beta, (const float*)proj, ld, b_off, a1_off, a2,
                       rank, dt_bias, a_log, T, H, dk);
    if (hist)
      hipLaunchKernelGGL(conv_state_update_kernel<float>, dim3(sgrid),
                         dim3(256), 0, s, conv_state, (const float*)proj, ld,
                         q_off, k_off, v_off, taps, state_slots, qlocs,
                         seq_lens, S, Cq, C);
  } else {
    hipLaunchKernelGGL(delta_prep_kernel<u16>, dim3(grid), dim3(WPB * WAVE), 0,
                       s, qn, kn, vv, hg, (const u16*)proj, ld, q_off, k_off, v_off,
                       conv_w, taps, conv_state, state_slots, qlocs, seq_lens,
                       token_seq, T, H, G, dk, dv);
    if (a2 && !lr)
    hipLaunchKernelGGL(delta_gates_kernel<u16>, ggrid, dim3(WPB * WAVE), 0, s,
                       decay, beta, (const u16*)proj, ld, b_off, a1_off, a2,
                       rank, dt_bias, a_log, T, H, dk);
    if (hist)
      hipLaunchKernelGGL(conv_state_update_kernel<u16>, dim3(sgrid), dim3(256),
                         0, s, conv_state, (const u16*)proj, ld, q_off, k_off,
                         v_off, taps, state_slots, qlocs, seq_lens, S, Cq, C);
  }
}

// New tokens from which a sequence goes through chunks (mix_delta_chunk.h), 0 if none
// of the batch can be that long or rows are not in whole 16-byte pieces
extern "C" int mix_delta_least(const float* qn, const float* kn,
                               const float* decay, int head_decay, long T,
                               long longest, int S, int H, int dk, int dv) {
  return delta_chunks_least(qn, kn, decay, head_decay, T, longest, S, H, dk, dv);
}
extern "C" long mix_delta_pairs_floats(long T, int least, int H) {
  return dc_slots(T, least) * H * (long)DC_PAIRS;
}

// pairs: mix_delta_pairs_floats(T, least, H) floats of scratch if least is not 0
extern "C" void mix_delta_scan(float* o, const float* qn, const float* kn,
                               const float* vv, const float* decay,
                               int head_decay, const float* beta, float* ssm,
                               const int* state_slots, const int* qlocs,
                               const int* seq_lens, float* pairs, int least,
                               long T, int S, int H, int G, int dk, int dv,
                               hipStream_t s) {
  if (least) {
    DeltaChunkArgs a = {};
    a.o = o; a.q = qn; a.k = kn; a.v = vv; a.d = decay; a.beta = beta;
    a.state = ssm; a.state_slots = state_slots;
    a.qlocs = qlocs; a.seq_lens = seq_lens; a.pairs = pairs;
    a.S = S; a.H = H; a.G = G; a.dk = dk; a.dv = dv; a.least = least;
    if (head_decay) {
      if (dk <= 64) delta_chunks_launch<64, true>(a, T, s);
      else delta_chunks_launch<128, true>(a, T, s);
    } else {
      if (dk <= 64) delta_chunks_launch<64, false>(a, T, s);
      else delta_chunks_launch<128, false>(a, T, s);
    }
  }
  const int below = least ? least : INT_MAX;
  int R = 1;
  while (R * 32 < dk) R <<= 1;  // dk <= 256 -> R <= 8 at 32 rows a lane
  int rpt = 32;
  {
    // few sequences x heads: 16 rows a lane doubles the waves in flight
    const long blocks32 = (long)S * H * ((dv + 256 / R - 1) / (256 / R));
    if (blocks32 < 512 && dk > 16) {
      rpt = 16;
      R = 2;
      while (R * 16 < dk) R <<= 1;  // R <= 16
    }
  }
  const int cols_pb = 256 / R;
  const int col_groups = (dv + cols_pb - 1) / cols_pb;
  const long grid = (long)S * H * col_groups;
  if (grid == 0) return;
#define LAUNCH_SCAN_D(RR, PP, HD)                                            \
  hipLaunchKernelGGL((delta_scan_kernel<RR, PP, HD>), dim3((unsigned)grid),  \
                     dim3(256), 0, s, o, qn, kn, vv, decay, beta, ssm,       \
                     state_slots, qlocs, seq_lens, H, G, dk, dv, col_groups, \
                     below)
#define LAUNCH_SCAN(RR, PP)                                                  \
  do {                                                                       \
    if (head_decay) LAUNCH_SCAN_D(RR, PP, true);                             \
    else LAUNCH_SCAN_D(RR, PP, false);                                       \
  } while (0)
  if (rpt == 32) {
    if (R == 1) LAUNCH_SCAN(1, 32);
    else if (R == 2) LAUNCH_SCAN(2, 32);
    else if (R == 4) LAUNCH_SCAN(4, 32);
    else LAUNCH_SCAN(8, 32);
  } else {
    if (R == 2) LAUNCH_SCAN(2, 16);
    else if (R == 4) LAUNCH_SCAN(4, 16);
    else if (R == 8) LAUNCH_SCAN(8, 16);
    else LAUNCH_SCAN(16, 16);
  }
#undef LAUNCH_SCAN
#undef LAUNCH_SCAN_D
}

extern "C" void mix_delta_out(void* out, long ldo, int out_off, const float* o,
                              const float* norm_w, const void* proj, long ld,
                              int g1_off, const float* g2, int rank, float eps,
                              float out_scale, long T, int H, int dv, int f32,
                              hipStream_t s) {
  if (T == 0) return;
  const dim3 grid((unsigned)((T + WPB * GT - 1) / (WPB * GT)), (unsigned)H);
  if (!f32 && (dv == 64 || dv == 128) && ldo % 4 == 0 && out_off % 4 == 0 &&
      (size_t)out % 8 == 0 && (size_t)o % 16 == 0 &&
      lr_fits(proj, ld, g1_off, rank, g2, norm_w)) {
    const auto fn = dv == 128 ? delta_out_mfma_kernel<8>
                              : delta_out_mfma_kernel<4>;
    const int per = lr_tokens(T, H);
    hipLaunchKernelGGL(fn,
                       dim3((unsigned)((T + WPB * per - 1) / (WPB * per)),
                            (unsigned)H),
                       dim3(WPB * WAVE), 0, s, (u16*)out, ldo, out_off, o,
                       norm_w, (const u16*)proj, ld, g1_off, g2, rank, eps,
                       out_scale, T, H, per);
  } else if (f32)
    hipLaunchKernelGGL(delta_out_kernel<float>, grid, dim3(WPB * WAVE),
                       0, s, (float*)out, ldo, out_off, o, norm_w,
                       (const float*)proj, ld, g1_off, g2, rank, eps,
                       out_scale, T, H, dv);
  else
    hipLaunchKernelGGL(delta_out_kernel<u16>, grid, dim3(WPB * WAVE), 0,
                       s, (u16*)out, ldo, out_off, o, norm_w,
                       (const u16*)proj, ld, g1_off, g2, rank, eps, out_scale,
                       T, H, dv);
}
