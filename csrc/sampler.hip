// Fused sampling kernel (CDNA4 / gfx950): FSM bitmask + temperature +
// top-k/top-p + inverse-CDF sample + logprob, one workgroup per row, NO sort.
//
// Semantics (shared with sutro_amd/engine/sampler.py::sample_torch_reference):
//   alive_i = (i < vl) && mask bit i
//   s_i = (logit_i - max_alive) / T   (f32; greedy rows use T = 1)
//   p_i = expf(s_i); Z = sum p_i
//   keep_i = alive_i && count{s_j > s_i} < k && mass{s_j > s_i} < top_p * Z
//            (value thresholds; ALL ties at a boundary are kept)
//   c = prefix-sum of p_i * keep_i in INDEX order; token = first c > u * M
//   logprob = s_token - log(Z)
//
// Mass bookkeeping runs in 32.32 fixed point (q_i = floor(p_i * 2^32), exact
// for f32 p since *2^32 is an exponent shift): integer sums are order-
// independent, so LDS atomics and wave reductions are bit-deterministic
// across replays — preemption restarts and async/sync A-B runs regenerate
// identical tokens. The value thresholds (top-k count, top-p mass) resolve
// by a 4-level radix descent over the monotonic u32 transform of s_i
// (256-bucket count+mass histograms per level; boundary bucket recursed).
//
// Throughput notes (a first version ran 2.33 ms per 2048x151,936 bf16 call,
// about 5x the pass-count HBM bound; bf16 rows count values instead, see
// sampler_count_kernel):
//  - all full-vocab passes consume u16x8 (16 B) per lane per step — the
//    scalar-u16 version dispatched 8x the instructions for the same bytes;
//  - the level-0 histogram is 8-way lane-replicated (hist[lane&7][bucket]):
//    scaled logits cluster in a handful of exponent buckets, so per-element
//    atomics serialized on a few LDS addresses; replication cuts that 8x
//    and the replicas are reduced once at scan time (integer = order-free);
//  - the final index-order selection streams the crossing chunk with a
//    whole-wave u64 scan (ballot early-exit) instead of a single-lane walk.
//   Passes: A max/argmax | B Z + level-0 hist | R1-R3 refine | F select.

#include <hip/hip_runtime.h>

#include "common.h"

#define SMP_THREADS 256
#define HREP 8  // level-0 histogram replicas
#define SMP_LEFT -2  // token of a row that another kernel has to sample

struct SmpArgs {
  const void* logits;
  const float* temps;
  const float* topps;
  const int* topks;
  const float* us;
  const u32* mask;
  long v_row;
  int n, vl, w_words;
  int* out_tok;
  float* out_lp;
  bool left;            // only rows whose token is SMP_LEFT
};

// monotonic u32 key: key(a) < key(b)  <=>  a < b (floats, no NaN)
__device__ __forceinline__ u32 f32key(float s) {
  u32 b = __float_as_uint(s);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
// and back
__device__ __forceinline__ float f32val(u32 k) {
  return __uint_as_float((k & 0x80000000u) ? k & 0x7fffffffu : ~k);
}

struct Boundary {
  u32 pref;        // resolved key prefix (eventually the exact 32-bit key)
  u64 above_mass;  // total q of keys strictly above the prefix region
  u32 above_cnt;
  u64 eq_mass;     // totals of the chosen bucket (after last level: exact key)
  u32 eq_cnt;
  int active;
};

template <int SMP_WAVES>
struct SmpShared {
  float wmax[SMP_WAVES];
  int warg[SMP_WAVES];
  float wsum[SMP_WAVES];
  u64 wfix[SMP_WAVES];
  float m;        // row max
  int argmax;
  float zf;       // float Z (logprob)
  u64 zfix;       // fixed-point Z (thresholds)
  // level 0 uses all HREP replicas (reduced into replica 0 at scan time);
  // refinement levels use replicas 0 (count descent) and 1 (mass descent)
  u32 hist_cnt[HREP][256];
  u64 hist_mass[HREP][256];
  Boundary bk, bp;
  u32 tau;        // combined threshold key
  u64 kept_mass;  // M
  u64 target;
  u64 chunk_sum[SMP_WAVES];
  int last_kept[SMP_WAVES];
  int token;
  int done;
  int chunk;   // of the crossing
  u64 base;
  int lastk;
};

template <bool BF16>
__device__ __forceinline__ float load_logit(const void* row, int i) {
  if (BF16) return bf2f(((const u16*)row)[i]);
  return ((const float*)row)[i];
}

// 8 consecutive logits starting at i0 (16B/32B aligned vector loads)
template <bool BF16>
__device__ __forceinline__ void load_logit8(const void* row, int i0,
                                            float* out) {
  if (BF16) {
    const u16x8 v = *(const u16x8*)((const u16*)row + i0);
#pragma unroll
    for (int j = 0; j < 8; ++j) out[j] = bf2f(v[j]);
  } else {
    const f32x4 a = *(const f32x4*)((const float*)row + i0);
    const f32x4 b = *(const f32x4*)((const float*)row + i0 + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      out[j] = a[j];
      out[4 + j] = b[j];
    }
  }
}

__device__ __forceinline__ bool alive_bit(const u32* mrow, int i) {
  return mrow == nullptr || ((mrow[i >> 5] >> (i & 31)) & 1u);
}

// mask bits for 8 consecutive tokens at i0 (i0 % 8 == 0: never crosses a word)
__device__ __forceinline__ u32 alive_bits8(const u32* mrow, int i0) {
  if (mrow == nullptr) return 0xFFu;
  return (mrow[i0 >> 5] >> (i0 & 31)) & 0xFFu;
}

// deterministic block max+argmax (lowest index wins ties)
template <int SMP_WAVES>
__device__ __forceinline__ void block_argmax(SmpShared<SMP_WAVES>* sm, float v,
                                             int idx, int tid) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    float ov = __shfl_xor(v, off, 64);
    int oi = __shfl_xor(idx, off, 64);
    if (ov > v || (ov == v && oi >= 0 && (idx < 0 || oi < idx))) {
      v = ov;
      idx = oi;
    }
  }
  if ((tid & 63) == 0) {
    sm->wmax[tid >> 6] = v;
    sm->warg[tid >> 6] = idx;
  }
  __syncthreads();
  if (tid == 0) {
    float bv = sm->wmax[0];
    int bi = sm->warg[0];
    for (int w = 1; w < SMP_WAVES; ++w) {
      float ov = sm->wmax[w];
      int oi = sm->warg[w];
      if (ov > bv || (ov == bv && oi >= 0 && (bi < 0 || oi < bi))) {
        bv = ov;
        bi = oi;
      }
    }
    sm->m = bv;
    sm->argmax = bi;
  }
  __syncthreads();
}

// scan one histogram level from the top bucket down; absolute thresholds
__device__ __forceinline__ void scan_level(const u32* cnt, const u64* mass,
                                           Boundary* b, u64 thr_mass,
                                           u32 thr_cnt, bool by_mass) {
  u64 macc = b->above_mass;
  u32 cacc = b->above_cnt;
  for (int bu = 255; bu >= 0; --bu) {
    u64 nm = macc + mass[bu];
    u32 nc = cacc + cnt[bu];
    bool crossed = by_mass ? (nm >= thr_mass) : (nc >= thr_cnt);
    if (crossed) {
      b->pref = (b->pref << 8) | (u32)bu;
      b->above_mass = macc;
      b->above_cnt = cacc;
      b->eq_mass = mass[bu];
      b->eq_cnt = cnt[bu];
      return;
    }
    macc = nm;
    cacc = nc;
  }
  b->active = 0;  // never crossed: threshold keeps everything
}

// any logits, any row: one workgroup of THREADS
template <bool BF16, int THREADS>
__device__ __forceinline__ void sample_row(const SmpArgs& A, int row, int tid,
                                           SmpShared<THREADS / 64>& sm) {
  constexpr int SMP_WAVES = THREADS / 64;
  const void* lrow =
      BF16 ? (const void*)((const u16*)A.logits + (long)row * A.v_row)
           : (const void*)((const float*)A.logits + (long)row * A.v_row);
  const u32* mrow = A.mask ? A.mask + (long)row * A.w_words : nullptr;
  const int vl = A.vl;
  const float T = A.temps[row];
  const bool greedy = T < 1e-5f;
  const float inv_t = greedy ? 1.0f : 1.0f / T;
  const int vl8 = vl & ~7;

  // ---- pass A: max + argmax over alive (vectorized) ----
  float lmax = -INFINITY;
  int larg = -1;
  for (int i0 = tid * 8; i0 < vl8; i0 += THREADS * 8) {
    const u32 ab = alive_bits8(mrow, i0);
    if (ab == 0) continue;
    float v[8];
    load_logit8<BF16>(lrow, i0, v);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (((ab >> j) & 1u) && v[j] > lmax) {
        lmax = v[j];
        larg = i0 + j;
      }
  }
  for (int i = vl8 + tid; i < vl; i += THREADS)
    if (alive_bit(mrow, i)) {
      float v = load_logit<BF16>(lrow, i);
      if (v > lmax) {
        lmax = v;
        larg = i;
      }
    }
  block_argmax(&sm, lmax, larg, tid);
  const float m = (sm.argmax >= 0) ? sm.m : 0.0f;
  if (sm.argmax < 0) {  // no alive token (should not happen): emit 0
    if (tid == 0) {
      A.out_tok[row] = 0;
      A.out_lp[row] = -INFINITY;
    }
    return;
  }

  // ---- pass B: Z (float + fixed) and 8-way replicated level-0 hist ----
  for (int i = tid; i < HREP * 256; i += THREADS) {
    ((u32*)sm.hist_cnt)[i] = 0;
    ((u64*)sm.hist_mass)[i] = 0;
  }
  __syncthreads();
  const int rep = tid & (HREP - 1);
  float zf_part = 0.0f;
  u64 zx_part = 0;
  for (int i0 = tid * 8; i0 < vl8; i0 += THREADS * 8) {
    const u32 ab = alive_bits8(mrow, i0);
    if (ab == 0) continue;
    float v[8];
    load_logit8<BF16>(lrow, i0, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (!((ab >> j) & 1u)) continue;
      const float s = (v[j] - m) * inv_t;
      const float p = __expf(s);
      zf_part += p;
      if (!greedy) {
        const u64 q = (u64)(p * 4294967296.0f);  // exact exponent shift
        zx_part += q;
        const u32 bu = f32key(s) >> 24;
        atomicAdd(&sm.hist_cnt[rep][bu], 1u);
        atomicAdd((unsigned long long*)&sm.hist_mass[rep][bu],
                  (unsigned long long)q);
      }
    }
  }
  for (int i = vl8 + tid; i < vl; i += THREADS) {
    if (!alive_bit(mrow, i)) continue;
    const float s = (load_logit<BF16>(lrow, i) - m) * inv_t;
    const float p = __expf(s);
    zf_part += p;
    if (!greedy) {
      const u64 q = (u64)(p * 4294967296.0f);
      zx_part += q;
      const u32 bu = f32key(s) >> 24;
      atomicAdd(&sm.hist_cnt[rep][bu], 1u);
      atomicAdd((unsigned long long*)&sm.hist_mass[rep][bu],
                (unsigned long long)q);
    }
  }
  // deterministic float Z: fixed per-thread partials + fixed tree
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) zf_part += __shfl_xor(zf_part, off, 64);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    zx_part += __shfl_xor(zx_part, off, 64);
  if ((tid & 63) == 0) {
    sm.wsum[tid >> 6] = zf_part;
    sm.wfix[tid >> 6] = zx_part;
  }
  __syncthreads();
  // reduce histogram replicas into replica 0 (integers: order-free)
  if (!greedy) {
    for (int b = tid; b < 256; b += THREADS) {
      u32 c = 0;
      u64 q = 0;
#pragma unroll
      for (int r = 0; r < HREP; ++r) {
        c += sm.hist_cnt[r][b];
        q += sm.hist_mass[r][b];
      }
      sm.hist_cnt[0][b] = c;
      sm.hist_mass[0][b] = q;
    }
  }
  if (tid == 0) {
    float z = 0.0f;
    u64 zx = 0;
    for (int w = 0; w < SMP_WAVES; ++w) {
      z += sm.wsum[w];
      zx += sm.wfix[w];
    }
    sm.zf = z;
    sm.zfix = zx;
  }
  __syncthreads();

  if (greedy) {
    if (tid == 0) {
      A.out_tok[row] = sm.argmax;
      A.out_lp[row] = -logf(sm.zf);  // s_argmax == 0 at T=1
    }
    return;
  }

  // ---- radix descent: resolve tau_k (count) and tau_p (mass) ----
  const u32 k_thr = (u32)max(1, A.topks[row]);
  if (tid == 0) {
    double pd = (double)A.topps[row] * (double)sm.zfix;
    u64 p_thr = (pd >= (double)sm.zfix) ? sm.zfix : (u64)pd;
    if (p_thr == 0) p_thr = 1;  // top_p ~ 0: keep at least the max token
    sm.bk = Boundary{0u, 0, 0, 0, 0, 1};
    sm.bp = Boundary{0u, 0, 0, 0, 0, 1};
    scan_level(sm.hist_cnt[0], sm.hist_mass[0], &sm.bk, 0, k_thr, false);
    scan_level(sm.hist_cnt[0], sm.hist_mass[0], &sm.bp, p_thr, 0, true);
    sm.done = (!sm.bk.active && !sm.bp.active);
  }
  __syncthreads();

  for (int level = 1; level < 4 && !sm.done; ++level) {
    const int shift_prev = 32 - 8 * level;
    const int shift_cur = shift_prev - 8;
    for (int i = tid; i < 256; i += THREADS) {
      sm.hist_cnt[0][i] = 0;
      sm.hist_mass[0][i] = 0;
      sm.hist_cnt[1][i] = 0;
      sm.hist_mass[1][i] = 0;
    }
    __syncthreads();
    const int ka = sm.bk.active, pa = sm.bp.active;
    const u32 kpref = sm.bk.pref, ppref = sm.bp.pref;
    for (int i0 = tid * 8; i0 < vl8; i0 += THREADS * 8) {
      const u32 ab = alive_bits8(mrow, i0);
      if (ab == 0) continue;
      float v[8];
      load_logit8<BF16>(lrow, i0, v);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (!((ab >> j) & 1u)) continue;
        const float s = (v[j] - m) * inv_t;
        const u32 key = f32key(s);
        const u32 hp = key >> shift_prev;
        if (hp != kpref && hp != ppref) continue;
        const u64 q = (u64)(__expf(s) * 4294967296.0f);
        const u32 bu = (key >> shift_cur) & 0xFFu;
        if (ka && hp == kpref) {
          atomicAdd(&sm.hist_cnt[0][bu], 1u);
          atomicAdd((unsigned long long*)&sm.hist_mass[0][bu],
                    (unsigned long long)q);
        }
        if (pa && hp == ppref) {
          atomicAdd(&sm.hist_cnt[1][bu], 1u);
          atomicAdd((unsigned long long*)&sm.hist_mass[1][bu],
                    (unsigned long long)q);
        }
      }
    }
    for (int i = vl8 + tid; i < vl; i += THREADS) {
      if (!alive_bit(mrow, i)) continue;
      const float s = (load_logit<BF16>(lrow, i) - m) * inv_t;
      const u32 key = f32key(s);
      const u32 hp = key >> shift_prev;
      if (hp != kpref && hp != ppref) continue;
      const u64 q = (u64)(__expf(s) * 4294967296.0f);
      const u32 bu = (key >> shift_cur) & 0xFFu;
      if (ka && hp == kpref) {
        atomicAdd(&sm.hist_cnt[0][bu], 1u);
        atomicAdd((unsigned long long*)&sm.hist_mass[0][bu],
                  (unsigned long long)q);
      }
      if (pa && hp == ppref) {
        atomicAdd(&sm.hist_cnt[1][bu], 1u);
        atomicAdd((unsigned long long*)&sm.hist_mass[1][bu],
                  (unsigned long long)q);
      }
    }
    __syncthreads();
    if (tid == 0) {
      double pd = (double)A.topps[row] * (double)sm.zfix;
      u64 p_thr = (pd >= (double)sm.zfix) ? sm.zfix : (u64)pd;
      if (p_thr == 0) p_thr = 1;
      if (sm.bk.active)
        scan_level(sm.hist_cnt[0], sm.hist_mass[0], &sm.bk, 0, k_thr, false);
      if (sm.bp.active)
        scan_level(sm.hist_cnt[1], sm.hist_mass[1], &sm.bp, p_thr, 0, true);
    }
    __syncthreads();
  }

  if (tid == 0) {
    u32 tk = sm.bk.active ? sm.bk.pref : 0u;
    u32 tp = sm.bp.active ? sm.bp.pref : 0u;
    if (!sm.bk.active && !sm.bp.active) {
      sm.tau = 0u;
      sm.kept_mass = sm.zfix;
    } else if (tk >= tp) {
      sm.tau = tk;
      sm.kept_mass = sm.bk.above_mass + sm.bk.eq_mass;
    } else {
      sm.tau = tp;
      sm.kept_mass = sm.bp.above_mass + sm.bp.eq_mass;
    }
    sm.target = (u64)((double)A.us[row] * (double)sm.kept_mass);
    sm.token = -1;
  }
  __syncthreads();
  const u32 tau = sm.tau;
  const u64 target = sm.target;

  // ---- pass F: index-order inverse CDF, hierarchical first-crossing ----
  // phase 1: per-wave contiguous chunks, lane-strided vectorized sums
  const int chunk = ((vl + SMP_WAVES * 8 - 1) / (SMP_WAVES * 8)) * 8;
  const int wv = tid >> 6, lane = tid & 63;
  const int c0 = min(vl, wv * chunk), c1 = min(vl, c0 + chunk);
  u64 wsum = 0;
  int wlast = -1;
  for (int i0 = c0 + lane * 8; i0 + 8 <= c1; i0 += 64 * 8) {
    const u32 ab = alive_bits8(mrow, i0);
    if (ab == 0) continue;
    float v[8];
    load_logit8<BF16>(lrow, i0, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (!((ab >> j) & 1u)) continue;
      const float s = (v[j] - m) * inv_t;
      if (f32key(s) < tau) continue;
      wsum += (u64)(__expf(s) * 4294967296.0f);
      wlast = i0 + j;
    }
  }
  // scalar remainder: the vectorized loop covers every FULL 8-block of
  // [c0, c1) (block b -> lane b%64, iteration b/64); at most 7 elements of
  // the last (vl-tail) chunk remain
  {
    const int rem0 = c0 + ((c1 - c0) & ~7);
    const int i = rem0 + lane;
    if (i < c1 && alive_bit(mrow, i)) {
      const float s = (load_logit<BF16>(lrow, i) - m) * inv_t;
      if (f32key(s) >= tau) {
        wsum += (u64)(__expf(s) * 4294967296.0f);
        wlast = max(wlast, i);
      }
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    wsum += __shfl_xor(wsum, off, 64);
    wlast = max(wlast, __shfl_xor(wlast, off, 64));
  }
  if (lane == 0) {
    sm.chunk_sum[wv] = wsum;
    sm.last_kept[wv] = wlast;
  }
  __syncthreads();
  // phase 1b: pick the crossing chunk (thread 0)
  if (tid == 0) {
    u64 acc = 0;
    int pick = -1, lastk = -1;
    for (int w2 = 0; w2 < SMP_WAVES; ++w2) {
      if (sm.last_kept[w2] >= 0) lastk = sm.last_kept[w2];
      if (pick < 0 && acc + sm.chunk_sum[w2] > target) {
        pick = w2;
        sm.base = acc;
      }
      acc += sm.chunk_sum[w2];
    }
    sm.chunk = pick;
    sm.lastk = lastk;
    if (pick < 0) sm.token = lastk;  // float-edge fallback: last kept
  }
  __syncthreads();

  if (sm.token < 0 && wv == 0 && sm.chunk >= 0) {
    // phase 2: wave 0 streams the chosen chunk with a whole-wave u64 scan
    // (cache-hot after phase 1); ballot early-exit at the crossing
    const int p0 = min(vl, sm.chunk * chunk), p1 = min(vl, p0 + chunk);
    const u64 rem = target - sm.base;
    u64 running = 0;
    for (int j = p0; j < p1; j += 64) {
      const int i = j + lane;
      u64 q = 0;
      if (i < p1 && alive_bit(mrow, i)) {
        const float s = (load_logit<BF16>(lrow, i) - m) * inv_t;
        if (f32key(s) >= tau) q = (u64)(__expf(s) * 4294967296.0f);
      }
      u64 inc = q;
      for (int off = 1; off < 64; off <<= 1) {
        const u64 t = __shfl_up(inc, off, 64);
        if (lane >= off) inc += t;
      }
      const bool mine = q > 0 && (running + inc - q) <= rem
                        && rem < (running + inc);
      const u64 total = __shfl(inc, 63, 64);
      const u64 found = __ballot(mine);
      if (found) {  // wave-uniform: broadcast the winner's index and stop
        const int src = __ffsll((unsigned long long)found) - 1;
        const int tok = __shfl(mine ? i : -1, src, 64);
        if (lane == 0) sm.token = tok;
        break;
      }
      running += total;
    }
    if (lane == 0 && sm.token < 0) sm.token = sm.lastk;
  }
  __syncthreads();
  if (tid == 0) {
    int tok = sm.token >= 0 ? sm.token : sm.argmax;
    float s = (load_logit<BF16>(lrow, tok) - m) * inv_t;
    A.out_tok[row] = tok;
    A.out_lp[row] = s - logf(sm.zf);
  }
}

template <bool BF16>
__global__ void __launch_bounds__(SMP_THREADS) sampler_kernel(SmpArgs A) {
  __shared__ SmpShared<SMP_THREADS / 64> sm;
  sample_row<BF16, SMP_THREADS>(A, blockIdx.x, threadIdx.x, sm);
}

// ---- bf16 rows: count the values ----
//
// A bf16 logit has one of 65,536 values, and everything above (p, q, the
// sampling key) is a function of the value alone. So one pass over the row
// counts the values in LDS, and masses, thresholds and Z come from the counts:
// the exponential is taken once per value present (about 2,500 of 151,936
// logits) instead of five times per logit, the sums are the same integers, and
// the thresholds are found by one scan in order of value. The row stays in
// registers (1,024 threads, up to 155,648 logits), so that the selection in
// order of index reads no memory; longer rows are read twice.
//
// Counters are 16 bits wide, those of v and -v share a word (128 KB). A row
// with a value that occurs 65,536 times overflows one; every overflow lowers
// the sum of the counters, so comparing it with the number of alive tokens
// finds all of them, and such a row is sampled by the general code. So is a row
// with a NaN or +inf.
//
// Bound by instruction issue: four to count and sixteen to select per logit.
// 1024 x 151,936 by the general kernel and here: 1382 -> 197 us (top_p 0.95 at
// temperature 0.8), 1393 -> 151 with top_k 20, 1338 -> 250
// with a mask; one row 636 -> 41 us. Of the 50 us that a row takes its
// workgroup 16 are fixed, clearing and scanning 128 KB of counters. Greedy batches, rows
// of more than 155,648 logits and what sampler_fast_kernel leaves come here.
#define CNT_MIN 2048
#define CNT_THREADS 1024
#define CNT_WAVES (CNT_THREADS / 64)
#define CNT_CHUNKS 19                          // of 8 logits a thread
#define CNT_CHUNK (CNT_THREADS * 8)
#define CNT_TILE (CNT_CHUNKS * CNT_CHUNK)
#define CNT_SEGS 512                           // of 64 magnitudes

typedef short s16x2 __attribute__((ext_vector_type(2)));

struct CountShared {
  u32 words[CNT_SEGS * 64];     // [magnitude]: low half of v, high half of -v
  u64 seg_mass[2 * CNT_SEGS];   // in descending order of value
  u32 seg_cnt[2 * CNT_SEGS];
  u64 blk[CNT_CHUNKS];          // of the wave's part that u falls into
  u64 wave_mass[CNT_WAVES];
  u32 wave_cnt[CNT_WAVES];
  u32 wave_alive[CNT_WAVES];
  float wave_z[CNT_WAVES];
  int max_pos, min_neg;         // magnitudes of the extremes
  int seg[2];                   // where the count / the mass crosses
  u64 above[2];
  u32 tau[2];
  int tcode;                    // lowest kept value, as an ordered code
  int one;                      // and lowest value with p = 1
  u64 kept;
  int last, token;
  u64 base;
};

// order of the values: as signed 16-bit numbers
__device__ __forceinline__ s16x2 ordered2(u32 w) {
  const s16x2 v = __builtin_bit_cast(s16x2, w);
  const s16x2 m = {0x7fff, 0x7fff};
  return v ^ ((v >> (short)15) & m);
}

// whole part, 2**32 - 1 for 2**32 (which a C++ conversion leaves undefined)
__device__ __forceinline__ u32 to_u32(float v) {
  u32 r;
  asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}

template <class T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

template <class T>
__device__ __forceinline__ T wave_scan(T v, int lane) {  // inclusive
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const T t = __shfl_up(v, off, 64);
    if (lane >= off) v += t;
  }
  return v;
}

template <bool MASKED>
__global__ void __launch_bounds__(CNT_THREADS)
sampler_count_kernel(SmpArgs A) {
  extern __shared__ __attribute__((aligned(16))) char cnt_lds[];
  CountShared& sm = *(CountShared*)cnt_lds;
  const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  if (A.left && A.out_tok[row] != SMP_LEFT) return;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const u16* lrow = (const u16*)A.logits + (long)row * A.v_row;
  const u8* mrow = MASKED ? (const u8*)(A.mask + (long)row * A.w_words)
                          : nullptr;
  const int vl = A.vl;
  const int tiles = (vl + CNT_TILE - 1) / CNT_TILE;
  const int last8 = (vl - 1) & ~7;   // rows are whole eights: readable
  const float T = A.temps[row];
  const bool greedy = T < 1e-5f;
  const float inv_t = greedy ? 1.0f : 1.0f / T;

  // a wave's part of a tile is contiguous: `part` chunks of 512 logits
  auto part_of = [&](int tile) {
    return (min(vl - tile * CNT_TILE, CNT_TILE) + CNT_CHUNK - 1) / CNT_CHUNK;
  };
  auto eight = [&](int i0) {
    return *(const u32x4*)((const char*)lrow + 2 * (u32)min(i0, last8));
  };
  auto bits8 = [&](int i0) -> u32 {
    return MASKED ? mrow[min(i0, last8) >> 3] : 0xffu;
  };
  // logits that are not alive become 0xffff, the lowest of all values (and, as
  // a NaN, nobody's logit)
  auto patch = [&](u32x4& w, u32 bits, int i0) {
    const int left = vl - i0;
    if (!MASKED && left >= 8) return;
    u32 dead = ~bits;
    if (left < 8) dead |= left > 0 ? 0xffu << left : 0xffu;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      w[j] |= ((dead >> (2 * j)) & 1u) * 0xffffu |
              ((dead >> (2 * j + 1)) & 1u) * 0xffff0000u;
  };
  u32x4 r[CNT_CHUNKS];
  auto load = [&](int tile) {
    const int part = part_of(tile);
    const int t0 = tile * CNT_TILE + wave * part * 512 + lane * 8;
    u32 bits[CNT_CHUNKS];
#pragma unroll
    for (int c = 0; c < CNT_CHUNKS; ++c)
      if (c < part) bits[c] = bits8(t0 + c * 512);
#pragma unroll
    for (int c = 0; c < CNT_CHUNKS; ++c)
      if (c < part) r[c] = eight(t0 + c * 512);
#pragma unroll
    for (int c = 0; c < CNT_CHUNKS; ++c)
      if (c < part) patch(r[c], bits[c], t0 + c * 512);
  };

  // ---- greedy rows: the first of the largest, and Z, from the registers ----
  // Nothing is counted. 1024 rows of 151,936 / 65,536 / 32,000 / 2048 logits: with
  // counts 139 / 91 / 75 / 60 us, now 111 / 51 / 34 / 20 (the general kernel, of which
  // more rows fit a CU, 153 / 53 / 30 / 8; one row 73 / 34 / 20 / 8 and here 24 / 13
  // / 10 / 8).
  if (greedy && tiles == 1) {
    const int part = part_of(0), t0 = wave * part * 512 + lane * 8;
    load(0);
    float best = -INFINITY;
    int ones = 0;      // logits that look like one that is not alive
#pragma unroll
    for (int c = 0; c < CNT_CHUNKS; ++c)
      if (c < part) {
        int dead = 0;
        if (MASKED || t0 + c * 512 + 8 > vl) {
          u32 bits = bits8(t0 + c * 512);
          const int left = vl - (t0 + c * 512);
          if (left < 8) bits &= left > 0 ? (1u << left) - 1 : 0u;
          dead = 8 - __popc(bits);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const u32 w = r[c][j];
          ones += ((w & 0xffffu) == 0xffffu) + (w >= 0xffff0000u);
          best = fmaxf(best, fmaxf(__uint_as_float(w << 16),
                                   __uint_as_float(w & 0xffff0000u)));
        }
        ones -= dead;
      }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
      best = fmaxf(best, __shfl_xor(best, off, 64));
    if (lane == 0) sm.wave_z[wave] = best;
    const bool odd = __ballot(ones != 0) != 0;
    if (lane == 0) sm.wave_cnt[wave] = odd;
    __syncthreads();
    const int l16 = lane & (CNT_WAVES - 1);
    best = sm.wave_z[l16];
    u32 any = sm.wave_cnt[l16];
#pragma unroll
    for (int off = 1; off < CNT_WAVES; off <<= 1) {
      best = fmaxf(best, __shfl_xor(best, off, CNT_WAVES));
      any |= __shfl_xor(any, off, CNT_WAVES);
    }
    if (!any) {
      float z = 0.f;
      int first = 0x7fffffff;
#pragma unroll
      for (int c = 0; c < CNT_CHUNKS; ++c)
        if (c < part)
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const u32 w = r[c][j >> 1];
            const u32 h = j & 1 ? w & 0xffff0000u : w << 16;
            const float v = __uint_as_float(h);
            z += h == 0xffff0000u ? 0.f : __expf(v - best);
            if (v == best) first = min(first, t0 + c * 512 + j);
          }
      z = wave_sum(z);
#pragma unroll
      for (int off = 32; off > 0; off >>= 1)
        first = min(first, __shfl_xor(first, off, 64));
      if (lane == 0) {
        sm.seg_cnt[wave] = (u32)first;
        sm.seg_cnt[CNT_WAVES + wave] = __float_as_uint(z);
      }
      __syncthreads();
      if (tid == 0) {
        z = 0.f;
        for (int w = 0; w < CNT_WAVES; ++w) {
          first = min(first, (int)sm.seg_cnt[w]);
          z += __uint_as_float(sm.seg_cnt[CNT_WAVES + w]);
        }
        const bool none = best == -INFINITY;
        A.out_tok[row] = none ? 0 : first;
        A.out_lp[row] = none ? -INFINITY : -logf(z);
      }
      return;
    }
    __syncthreads();
  }

  {
    u32x4* z = (u32x4*)sm.words;
#pragma unroll
    for (int i = 0; i < CNT_SEGS * 16 / CNT_THREADS; ++i)
      z[i * CNT_THREADS + tid] = (u32x4)(0u);
    sm.seg_mass[tid] = 0;
    sm.seg_cnt[tid] = 0;
    if (tid == 0) {
      sm.max_pos = -1;
      sm.min_neg = 0x8000;
      sm.seg[0] = sm.seg[1] = -1;
      sm.tau[0] = sm.tau[1] = 0;
      sm.tcode = sm.one = 0x7fff;
      sm.kept = 0;
      sm.last = sm.token = -1;
      sm.base = 0;
    }
  }
  __syncthreads();

  // ---- count the values ----
  for (int tile = 0; tile < tiles; ++tile) {
    load(tile);
    const int part = part_of(tile);
#pragma unroll
    for (int c = 0; c < CNT_CHUNKS; ++c) {
      // lanes without a live logit would all add to one counter
      if (c < part && (MASKED || r[c][0] != ~0u))
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const u32 w = r[c][j];
        const u32 lo = w & 0x7fffu, hi = (w >> 16) & 0x7fffu;
        if (!MASKED || (w & 0xffffu) != 0xffffu)
          atomicAdd(&sm.words[lo], (w & 0x8000u) ? 0x10000u : 1u);
        if (!MASKED || w < 0xffff0000u)
          atomicAdd(&sm.words[hi], (int)w < 0 ? 0x10000u : 1u);
      }
    }
  }
  // alive tokens, for the check of the counters
  u32 n_alive = 0;
  if (MASKED)
    for (int i = tid; i * 32 < vl; i += CNT_THREADS) {
      u32 w = ((const u32*)mrow)[i];
      if (vl - i * 32 < 32) w &= (1u << (vl - i * 32)) - 1;
      n_alive += __popc(w);
    }
  else if (tid == 0)
    n_alive = vl;
  __syncthreads();
  if (tid == 0) sm.words[0x7fff] &= 0xffffu;   // 0xffff: not alive
  __syncthreads();

  // ---- segments that hold a value, and the largest value ----
  // segment j * CNT_WAVES + wave is this wave's, so that neighbours spread
  u32 present = 0;
  int max_pos = -1, min_neg = 0x8000;
#pragma unroll 4
  for (int j = 0; j < CNT_SEGS / CNT_WAVES; ++j) {
    const int mag0 = (j * CNT_WAVES + wave) * 64;
    const u32 w = sm.words[mag0 + lane];
    if (__ballot(w != 0) == 0) continue;
    present |= 1u << j;
    const bool number = mag0 + lane <= 0x7f80;   // not a NaN
    const u64 p = __ballot(number && (w & 0xffffu) != 0);
    const u64 n = __ballot(number && (w >> 16) != 0);
    if (p) max_pos = mag0 + 63 - __clzll(p);
    if (n) min_neg = min(min_neg, mag0 + __ffsll((unsigned long long)n) - 1);
  }
  if (lane == 0) {
    atomicMax(&sm.max_pos, max_pos);
    atomicMin(&sm.min_neg, min_neg);
  }
  __syncthreads();
  const bool pos = sm.max_pos >= 0;
  // nothing above -inf counted: none alive, or a counter overflowed
  const bool none = !pos && sm.min_neg >= 0x7f80;
  float m = bf2f((u16)(pos ? sm.max_pos : 0x8000 | sm.min_neg));

  // ---- Z, and counts and masses by segment ----
  float z = 0.f;
  int one = 0x7fff;
  for (u32 left = present; left; left &= left - 1) {
    const int seg = (__ffs(left) - 1) * CNT_WAVES + wave;
    const int mag = seg * 64 + lane;
    const u32 w = sm.words[mag];
    const u32 cp = w & 0xffffu, cn = w >> 16;
    const float v = bf2f((u16)mag);
    if (__ballot(cp != 0)) {
      const float p = __expf((v - m) * inv_t);
      if (cp) z += (float)cp * p;
      if (cp && p >= 1.f) one = min(one, mag);
      const u64 q = (u64)(p * 4294967296.0f);
      const u64 ms = wave_sum(cp ? q * cp : (u64)0);
      const u32 cs = wave_sum(cp);
      if (lane == 0) {
        sm.seg_mass[CNT_SEGS - 1 - seg] = ms;
        sm.seg_cnt[CNT_SEGS - 1 - seg] = cs;
      }
    }
    if (__ballot(cn != 0)) {
      const float p = __expf((-v - m) * inv_t);
      if (cn) z += (float)cn * p;
      if (cn && p >= 1.f) one = min(one, -1 - mag);
      const u64 q = (u64)(p * 4294967296.0f);
      const u64 ms = wave_sum(cn ? q * cn : (u64)0);
      const u32 cs = wave_sum(cn);
      if (lane == 0) {
        sm.seg_mass[CNT_SEGS + seg] = ms;
        sm.seg_cnt[CNT_SEGS + seg] = cs;
      }
    }
  }
  if (one != 0x7fff) atomicMin(&sm.one, one);
  z = wave_sum(z);
  n_alive = wave_sum(n_alive);
  if (lane == 0) {
    sm.wave_z[wave] = z;
    sm.wave_alive[wave] = n_alive;
  }
  __syncthreads();

  // ---- running count and mass, from the largest value down ----
  const u64 my_mass = sm.seg_mass[tid];
  const u32 my_cnt = sm.seg_cnt[tid];
  u64 mass = wave_scan(my_mass, lane);
  u32 cnt = wave_scan(my_cnt, lane);
  if (lane == 63) {
    sm.wave_mass[wave] = mass;
    sm.wave_cnt[wave] = cnt;
  }
  __syncthreads();
  // every wave scans the sixteen sums
  const int l16 = lane & (CNT_WAVES - 1);
  u64 wm = sm.wave_mass[l16];
  u32 wc = sm.wave_cnt[l16], want = sm.wave_alive[l16];
  float zf = sm.wave_z[l16];
#pragma unroll
  for (int off = 1; off < CNT_WAVES; off <<= 1) {
    const u64 tm = __shfl_up(wm, off, CNT_WAVES);
    const u32 tc = __shfl_up(wc, off, CNT_WAVES);
    wm += l16 >= off ? tm : 0;
    wc += l16 >= off ? tc : 0;
    want += __shfl_xor(want, off, CNT_WAVES);
    zf += __shfl_xor(zf, off, CNT_WAVES);
  }
  const u64 zfix = __shfl(wm, CNT_WAVES - 1, 64);
  const u32 counted = __shfl(wc, CNT_WAVES - 1, 64);
  const u64 mass0 = wave ? __shfl(wm, wave - 1, 64) : 0;
  const u32 cnt0 = wave ? __shfl(wc, wave - 1, 64) : 0;
  // ... or zeros of both signs on top, of which the first is the maximum and
  // decides whether the other sign ranks below
  const bool zeros = pos && sm.max_pos == 0 && sm.min_neg == 0;
  // ... or NaN or +inf (then Z is NaN), whose differences have no order
  if (none || counted != want || (zeros && !greedy) || zf != zf) {
    __syncthreads();
    sample_row<true, CNT_THREADS>(A, row, tid,
                                  *(SmpShared<CNT_WAVES>*)cnt_lds);
    return;
  }
  // a greedy row: the first of the tokens of the largest value
  u64 target = 0;
  int tcode = m > 0.f ? sm.max_pos : (m < 0.f ? -1 - sm.min_neg : -1);
  if (!greedy) {
    mass += mass0;
    cnt += cnt0;
    const u32 k_thr = (u32)max(1, A.topks[row]);
    const double pd = (double)A.topps[row] * (double)zfix;
    u64 p_thr = (pd >= (double)zfix) ? zfix : (u64)pd;
    if (p_thr == 0) p_thr = 1;   // top_p ~ 0: keep at least the max token
    if (cnt >= k_thr && cnt - my_cnt < k_thr) {
      sm.seg[0] = tid;
      sm.above[0] = cnt - my_cnt;
    }
    if (mass >= p_thr && mass - my_mass < p_thr) {
      sm.seg[1] = tid;
      sm.above[1] = mass - my_mass;
    }
    __syncthreads();
    // the crossing value within its segment: wave 0 the count's, wave 1 the
    // mass's
    if (wave < 2 && sm.seg[wave] >= 0) {
      const int e = sm.seg[wave];
      const bool up = e < CNT_SEGS;
      const int mag = up ? (CNT_SEGS - 1 - e) * 64 + 63 - lane
                         : (e - CNT_SEGS) * 64 + lane;
      const u32 w = sm.words[mag];
      const u32 cv = up ? w & 0xffffu : w >> 16;
      const float v = bf2f((u16)(up ? mag : 0x8000 | mag));
      const float s = (v - m) * inv_t;
      u64 own = cv;
      if (wave == 1) own = cv ? (u64)(__expf(s) * 4294967296.0f) * cv : 0;
      const u64 sum = wave_scan(own, lane) + sm.above[wave];
      const u64 thr = wave == 0 ? (u64)k_thr : p_thr;
      if (sum >= thr && sum - own < thr) sm.tau[wave] = f32key(s);
    }
    __syncthreads();

    // ---- kept mass, and the lowest kept value ----
    // different values can have one key (v - m rounds): all of them are kept
    const u32 tau = max(sm.tau[0], sm.tau[1]);
    u64 kept = 0;
    tcode = 0x7fff;
    for (u32 left = present; left; left &= left - 1) {
      const int mag = ((__ffs(left) - 1) * CNT_WAVES + wave) * 64 + lane;
      const u32 w = sm.words[mag];
      const u32 cp = w & 0xffffu, cn = w >> 16;
      const float v = bf2f((u16)mag);
      const float sp = (v - m) * inv_t, sn = (-v - m) * inv_t;
      if (cp && f32key(sp) >= tau) {
        kept += (u64)(__expf(sp) * 4294967296.0f) * cp;
        tcode = min(tcode, mag);
      }
      if (cn && f32key(sn) >= tau) {
        kept += (u64)(__expf(sn) * 4294967296.0f) * cn;
        tcode = min(tcode, -1 - mag);
      }
    }
    kept = wave_sum(kept);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
      tcode = min(tcode, __shfl_xor(tcode, off, 64));
    if (lane == 0 && tcode != 0x7fff) {
      atomicAdd((unsigned long long*)&sm.kept, (unsigned long long)kept);
      atomicMin(&sm.tcode, tcode);
    }
    __syncthreads();
    target = (u64)((double)A.us[row] * (double)sm.kept);
    tcode = sm.tcode;
  }

  // ---- selection in order of index ----
  // by float order: apart from the zeros (see above) that of the codes
  const float low = bf2f((u16)(tcode >= 0 ? tcode : 0x7fff ^ tcode));
  // floor(p 2**32) of one logit; the conversion stops at 2**32 - 1, so that
  // values of p = 1 lack one
  auto q32 = [&](float v) -> u32 {
    return v >= low ? to_u32(__expf((v - m) * inv_t) * 4294967296.0f) : 0u;
  };
  auto mass8 = [&](const u32x4& w) {
    u64 sum = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      sum += q32(__uint_as_float(w[j] << 16));
      sum += q32(__uint_as_float(w[j] & 0xffff0000u));
    }
    return sum;
  };
  // kept values of p = 1 (a value just below the maximum may round to it and
  // still be cut off)
  const int top_code = max(sm.one, tcode);
  const float top = bf2f((u16)(top_code >= 0 ? top_code : 0x7fff ^ top_code));
  auto ones8 = [&](const u32x4& w) {
    u32 n = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      n += (__uint_as_float(w[j] << 16) >= top) +
           (__uint_as_float(w[j] & 0xffff0000u) >= top);
    return n;
  };
  auto best8 = [&](const u32x4& w) {
    s16x2 t = ordered2(w[0]);
#pragma unroll
    for (int j = 1; j < 4; ++j) t = __builtin_elementwise_max(t, ordered2(w[j]));
    return max((int)t[0], (int)t[1]);
  };
  auto mass_of = [&](const u32x4& w) -> u64 {   // a wave together
    const int best = best8(w);
    if (!__ballot(best >= tcode)) return 0;
    u64 sum = mass8(w);
    if (__ballot(best >= top_code)) sum += ones8(w);
    return sum;
  };
  for (int tile = 0; tile < tiles; ++tile) {
    if (tiles > 1) load(tile);
    const int part = part_of(tile), t0 = tile * CNT_TILE;
#pragma unroll
    for (int c = 0; c < CNT_CHUNKS; ++c) asm volatile("" : "+v"(r[c]));
    u64 sum = 0;
#pragma unroll
    for (int c = 0; c < CNT_CHUNKS; ++c) {
      if (c < part) sum += mass_of(r[c]);
    }
    sum = wave_sum(sum);
    if (lane == 0) sm.wave_mass[wave] = sum;
    __syncthreads();
    // the wave's part that holds u (every wave finds it), its chunks again
    u64 at = sm.base, next = at;
    int own = -1;
    for (int w2 = 0; w2 < CNT_WAVES; ++w2) {
      next = at + sm.wave_mass[w2];
      if (next > target) {
        own = w2;
        break;
      }
      at = next;
    }
    if (own >= 0) {
      const int p0 = t0 + own * part * 512 + lane * 8;
      for (int c = wave; c < part; c += CNT_WAVES) {
        u32x4 w = eight(p0 + c * 512);
        patch(w, bits8(p0 + c * 512), p0 + c * 512);
        const u64 s8 = wave_sum(mass_of(w));
        if (lane == 0) sm.blk[c] = s8;
      }
      __syncthreads();
      if (wave == 0) {
        int c = 0;
        while (c < part - 1 && at + sm.blk[c] <= target) at += sm.blk[c++];
        const int i0 = p0 + c * 512;
        u32x4 w = eight(i0);
        patch(w, bits8(i0), i0);
        u64 q[8], mine = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float v = __uint_as_float(j & 1 ? w[j >> 1] & 0xffff0000u
                                                : w[j >> 1] << 16);
          q[j] = (u64)q32(v) + (v >= top);
          mine += q[j];
        }
        const u64 to = wave_scan(mine, lane) + at;
        u64 from = to - mine;
        if (to > target && from <= target) {
          int tok = i0;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            if (from <= target) tok = i0 + j;
            from += q[j];
          }
          sm.token = tok;
        }
      }
      __syncthreads();
      break;
    }
    __syncthreads();   // all have read base
    if (tid == 0) sm.base = next;
  }
  if (sm.token < 0) {   // u at the upper edge: the last kept token
    for (int i = tid; i < vl; i += CNT_THREADS)
      if ((!MASKED || ((mrow[i >> 3] >> (i & 7)) & 1u)) &&
          ordered2((u32)lrow[i])[0] >= tcode)
        atomicMax(&sm.last, i);
    __syncthreads();
    if (tid == 0) sm.token = sm.last;
    __syncthreads();
  }
  if (tid == 0) {
    const int tok = sm.token;
    A.out_tok[row] = tok;
    A.out_lp[row] = (bf2f(lrow[tok]) - m) * inv_t - logf(zf);
  }
}

// ---- bf16 rows, most of them: counts of fewer values, by quarters of the row ----
//
// The counts above are of 65,536 values, so that a CU has room for one row's, and what
// selects has to go through the whole row again, a dozen instructions a logit. Here a
// logit is counted under its sign and its magnitude between 2^-24 and 255, 8192 values
// in 32 bits, in four tables, one for each quarter of the row. They tell the kept mass of
// every quarter, and only the one that u falls into is read again. What lies outside is
// counted at the ends. That is exact where the largest logit is above 1 (a magnitude of
// 2^-24 or less then vanishes in the difference to it) or no magnitude is as small, and
// where none is above 254, or those are negative and 0 as weights; other rows, with NaN
// or +inf among them, are left to the kernel above, which runs behind this one.
//
// One workgroup a CU stays for all of its rows: where a piece of the row has been counted,
// the same piece of the next row is asked for, so that the copies run on beside the
// counting, the thresholds and the selection.
// Bound by instruction issue and LDS additions while it counts (four instructions and an
// addition a logit, 9 of 20 us a row), the chain of eight barriers behind it (7 us), and
// the quarter (4). 1024 / 256 / 1 rows of 151,936, top_p 0.95 at temperature 0.8: 193 /
// 49 / 41 us by the kernel above, 109 / 29 / 24 here; top_k 20 150 -> 105, with a mask
// 248 -> 136, at temperature 3 194 -> 113; 1024 of 32,000 92 -> 53, of 2048 69 -> 39. Of
// these 4.7 us are the launch that finds nothing left to do. Flat rows (normal, 0.3) 198 ->
// 115, log-probabilities 185 -> 117, all at -20 and less 185 -> 119.
// That a row is left is known when it has been counted, which is then lost: 1024 / 64 /
// 1 rows of 151,936 with logits above 254 152 / 33 / 31 us by the kernel above alone and
// 219 / 46 / 44 with this one in front, with NaN 1693 / 418 / 411 and 1885 / 467 / 458,
// with a largest logit of 0 1716 / 415 / 363 and 1999 / 485 / 433.
#define FAST_PARTS 4
#define FAST_BASE 0x3380        // bits of 2^-24
#define FAST_TOP 4095           // 255, and what is larger
#define FAST_SIGN 4096
#define FAST_CODES 8192
#define FAST_DEAD 0xc37fc37fu   // -255 twice
#define FAST_BLK (FAST_PARTS * CNT_CHUNKS)
#define FAST_RING 8             // pieces of a wave that are asked for ahead

struct FastShared {
  u32 cnt[FAST_PARTS][FAST_CODES];
  u64 part[FAST_PARTS];         // kept mass
  u64 blk[128];                 // of 512 logits of the quarter that u falls into
  u64 wave_mass[CNT_WAVES];
  u32 wave_cnt[CNT_WAVES];
  float wave_z[CNT_WAVES];
  int first, code;              // of the largest value: its thread and what it is,
  int low;                      // and the lowest kept one: magnitude, or -1 - magnitude
  u32 one;                      // lowest value with p = 1, by its key
  u32 odd, tau[2];
  int token, last;
};

// v of the lane that CTRL names, `none` where there is none or ROWS leaves it out
template <int CTRL, int ROWS = 15>
__device__ __forceinline__ u32 dpp(u32 none, u32 v) {
  return __builtin_amdgcn_update_dpp(none, v, CTRL, ROWS, 15, false);
}
template <int CTRL, int ROWS = 15>
__device__ __forceinline__ u64 dpp(u64 none, u64 v) {
  return (u64)dpp<CTRL, ROWS>((u32)(none >> 32), (u32)(v >> 32)) << 32 |
         dpp<CTRL, ROWS>((u32)none, (u32)v);
}
template <int CTRL, int ROWS = 15>
__device__ __forceinline__ float dpp(float none, float v) {
  return __uint_as_float(
      dpp<CTRL, ROWS>(__float_as_uint(none), __float_as_uint(v)));
}
// Inclusive scans over rows of 16 lanes and over the wave, without the LDS: of 16 waves
// one may be alone with this.
template <class T, class Op>
__device__ __forceinline__ T row_scan(T v, T none, Op op) {
  v = op(v, dpp<0x111>(none, v));    // from 1, 2, 4, 8 lanes below
  v = op(v, dpp<0x112>(none, v));
  v = op(v, dpp<0x114>(none, v));
  return op(v, dpp<0x118>(none, v));
}
template <class T, class Op>
__device__ __forceinline__ T lane_scan(T v, T none, Op op) {
  v = row_scan(v, none, op);
  v = op(v, dpp<0x142, 0xa>(none, v));   // lane 15 to the next row's, then 31
  return op(v, dpp<0x143, 0xc>(none, v));
}
__device__ __forceinline__ u32 from_lane(u32 v, int l) {
  return __builtin_amdgcn_readlane(v, l);
}
__device__ __forceinline__ u64 from_lane(u64 v, int l) {
  return (u64)from_lane((u32)(v >> 32), l) << 32 | from_lane((u32)v, l);
}
struct AddOp {
  template <class T>
  __device__ T operator()(T a, T b) const { return a + b; }
};
struct MinOp {
  __device__ u32 operator()(u32 a, u32 b) const { return min(a, b); }
};

// The first pieces of 512 logits of each wave's part of a row, and their masks.
template <bool MASKED>
struct FastRing {
  u32x4 w[FAST_RING];
  u32 bits[MASKED ? FAST_RING : 1];
  __device__ __forceinline__ void load(const SmpArgs& A, int row, int slot, int i0) {
    const int i = min(i0, (A.vl - 1) & ~7);
    w[slot] = *(const u32x4*)((const u16*)A.logits + (long)row * A.v_row + i);
    if (MASKED)
      bits[MASKED ? slot : 0] =
          ((const u8*)(A.mask + (long)row * A.w_words))[i >> 3];
  }
};

// Samples the row that begins in r, and leaves the beginning of row `ahead` there, if that
// is not negative. False: nothing was done.
template <bool MASKED>
__device__ __forceinline__ bool fast_row(const SmpArgs& A, int row, int ahead,
                                         char* lds, FastRing<MASKED>& r) {
  FastShared& sm = *(FastShared*)lds;
  // (what follows from these is made for each row: kept for all of them it took more
  // registers than there are)
  int tid = threadIdx.x, vl = A.vl;
  asm volatile("" : "+v"(tid), "+s"(vl));
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const u16* lrow = (const u16*)A.logits + (long)row * A.v_row;
  const u8* mrow = MASKED ? (const u8*)(A.mask + (long)row * A.w_words)
                          : nullptr;
  const int last8 = (vl - 1) & ~7;
  const int part = (vl + CNT_CHUNK - 1) / CNT_CHUNK;   // pieces of a wave
  // weight of a difference to the largest logit, and its whole part of 2^32 (of which
  // those of 1 lack one: the conversion stops at 2^32 - 1)
  const float inv_t = 1.0f / A.temps[row];
  auto weight = [&](float d) { return __expf(d * inv_t); };
  auto q32 = [&](float p) { return to_u32(p * 4294967296.0f); };

  // logits that are not alive become `dead` (twice 16 bits)
  auto patch = [&](u32x4& w, u32 bits, int i0, u32 dead) {
    const int left = vl - i0;
    if (left < 8) bits &= left > 0 ? (1u << left) - 1 : 0u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u32 keep = ((bits >> (2 * j)) & 1u) * 0xffffu |
                       ((bits >> (2 * j + 1)) & 1u) * 0xffff0000u;
      w[j] = (w[j] & keep) | (dead & ~keep);
    }
  };

  {
    u32x4* z = (u32x4*)sm.cnt;
#pragma unroll
    for (int i = 0; i < FAST_PARTS * FAST_CODES / 4 / CNT_THREADS; ++i)
      z[i * CNT_THREADS + tid] = (u32x4)(0u);
    if (tid < FAST_PARTS) sm.part[tid] = 0;
    if (tid == 0) {
      sm.first = CNT_THREADS;
      sm.code = -FAST_CODES;
      sm.one = f32key(INFINITY);
      sm.low = FAST_CODES;
      sm.odd = sm.tau[0] = sm.tau[1] = 0;
      sm.token = sm.last = -1;
    }
  }
  __syncthreads();

  // ---- count ----
  u16x2 most = (u16x2)(0);
  {
    typedef __attribute__((address_space(3))) u32 lds_u32;
    lds_u32* const table = (lds_u32*)sm.cnt[wave * FAST_PARTS / CNT_WAVES];
    const u32 base = (u32)(size_t)table;
#pragma unroll
    for (int c = 0; c < CNT_CHUNKS; ++c) {
      const int i0 = (wave * part + c) * 512;
      if (c < part) {
        if (i0 < vl) {
          u32x4 w = r.w[c % FAST_RING];
          if (MASKED || i0 + 512 > vl) {
            patch(w, MASKED ? r.bits[MASKED ? c % FAST_RING : 0] : 0xffu, i0 + lane * 8,
                  FAST_DEAD);
            if (!MASKED && lane == 0)      // they are not to be counted
              atomicSub(&sm.cnt[wave * FAST_PARTS / CNT_WAVES][FAST_SIGN | FAST_TOP],
                        (u32)(i0 + 512 - vl));
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const u16x2 mag = __builtin_bit_cast(u16x2, w[j] & 0x7fff7fffu);
            most = __builtin_elementwise_max(most, mag);
            u16x2 d = __builtin_elementwise_sub_sat(mag, (u16x2)(FAST_BASE));
            d = __builtin_elementwise_min(d, (u16x2)(FAST_TOP));
            const u32 a = ((w[j] >> 3) & (FAST_SIGN * 0x10001u)) |
                          __builtin_bit_cast(u32, d);
            u32 lo, hi;
            asm("v_mad_u32_u16 %0, %1, 4, %2" : "=v"(lo) : "v"(a), "v"(base));
            asm("v_mad_u32_u16 %0, %1, 4, %2 op_sel:[1,0,0,0]"
                : "=v"(hi) : "v"(a), "v"(base));
            // (under a mask -255 is not counted: all that are not alive would add there)
            if (!MASKED || (a & 0xffffu) != (FAST_SIGN | FAST_TOP))
              __hip_atomic_fetch_add((lds_u32*)(size_t)lo, 1u, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_WORKGROUP);
            if (!MASKED || a >> 16 != (FAST_SIGN | FAST_TOP))
              __hip_atomic_fetch_add((lds_u32*)(size_t)hi, 1u, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_WORKGROUP);
          }
        }
        if (c + FAST_RING < part)
          r.load(A, row, c % FAST_RING, i0 + FAST_RING * 512 + lane * 8);
        else if (ahead >= 0)
          r.load(A, ahead, c % FAST_RING,
                 (wave * part + c % FAST_RING) * 512 + lane * 8);
      }
    }
  }
  {
    const u32 mag = max((u32)most[0], (u32)most[1]);
    const u32 nan = __any(mag > 0x7f80u) ? 1u : 0u;
    const u32 far = __any(mag > FAST_BASE + FAST_TOP) ? 2u : 0u;
    if (lane == 0 && (nan | far)) atomicOr(&sm.odd, nan | far);
  }
  __syncthreads();

  // ---- a thread has eight values, from the largest (thread 0) down ----
  const bool up = wave < CNT_WAVES / 2;
  const int mag0 = up ? (CNT_THREADS / 2 - 1 - tid) * 8 : (tid - CNT_THREADS / 2) * 8;
  const int at0 = up ? mag0 : FAST_SIGN + mag0;
  auto mag_of = [&](int j) { return up ? mag0 + 7 - j : mag0 + j; };
  auto value = [&](int j) {
    const int mag = mag_of(j);
    const float v = mag ? bf2f((u16)(FAST_BASE + mag)) : 0.f;
    return up ? v : -v;
  };
  auto counts = [&](int p, u32 (&c)[8]) {
    const u32x4 a = *(const u32x4*)&sm.cnt[p][at0];
    const u32x4 b = *(const u32x4*)&sm.cnt[p][at0 + 4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      c[j] = up ? b[3 - j] : a[j];
      c[4 + j] = up ? a[3 - j] : b[j];
    }
  };
  u32 tot[8], my_cnt = 0;
  counts(0, tot);
#pragma unroll
  for (int p = 1; p < FAST_PARTS; ++p) {
    u32 c[8];
    counts(p, c);
#pragma unroll
    for (int j = 0; j < 8; ++j) tot[j] += c[j];
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) my_cnt += tot[j];
  {
    const u64 any = __ballot(my_cnt != 0);
    if (lane == 0 && any)
      atomicMin(&sm.first, wave * 64 + __ffsll((unsigned long long)any) - 1);
    if (mag0 == 0 && (up ? tot[7] : tot[0])) atomicOr(&sm.odd, 4u);
  }
  __syncthreads();
  if (tid == sm.first) {
    int code = 0;
#pragma unroll
    for (int j = 7; j >= 0; --j)
      if (tot[j]) code = up ? mag_of(j) : -1 - mag_of(j);
    sm.code = code;
  }
  __syncthreads();
  const int code = sm.code;
  const int mag = code >= 0 ? code : -1 - code;
  const float size = bf2f((u16)(FAST_BASE + mag)), m = code >= 0 ? size : -size;
  const u32 odd = sm.odd;
  const float range = (255.f + m) * inv_t;
  if (mag >= FAST_TOP || (size <= 1.f && (odd & 4)) || (odd & 1) ||
      ((odd & 2) && !(range > 104.f)) || (MASKED && !(range > 40.f)))
    return false;

  // ---- Z, and running count and mass ----
  const AddOp add;
  u64 mass = 0, my_mass = 0;
  u32 cnt = 0, q[8];
  float z = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) q[j] = 0;
  u32 ones = 0;            // which values have a weight of 1
  if (__any(my_cnt != 0)) {
    u32 one = f32key(INFINITY);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float v = value(j);
      // (no value above m has a count, but its exponential may be infinite)
      const float p = weight(fminf(v, m) - m);
      z += (float)tot[j] * p;
      q[j] = q32(p);
      my_mass += (u64)q[j] * tot[j];
      if (p >= 1.f) {
        ones |= 1u << j;
        my_mass += tot[j];
        // (what is counted as 0 is kept together)
        if (tot[j]) one = min(one, f32key(mag_of(j) ? v : -bf2f(FAST_BASE)));
      }
    }
    if (__any(one != f32key(INFINITY))) {
      one = lane_scan(one, f32key(INFINITY), MinOp());
      if (lane == 63) atomicMin(&sm.one, one);
    }
    mass = lane_scan(my_mass, (u64)0, add);
    cnt = lane_scan(my_cnt, 0u, add);
    z = lane_scan(z, 0.f, add);
  }
  if (lane == 63) {
    sm.wave_mass[wave] = mass;
    sm.wave_cnt[wave] = cnt;
    sm.wave_z[wave] = z;
  }
  __syncthreads();
  const int l16 = lane & (CNT_WAVES - 1);
  const u64 wm = row_scan(sm.wave_mass[l16], (u64)0, add);
  const u32 wc = row_scan(sm.wave_cnt[l16], 0u, add);
  float zf = row_scan(sm.wave_z[l16], 0.f, add);
  zf = __uint_as_float(from_lane(__float_as_uint(zf), CNT_WAVES - 1));
  const u64 zfix = from_lane(wm, CNT_WAVES - 1);
  if (wave) {
    mass += from_lane(wm, wave - 1);
    cnt += from_lane(wc, wave - 1);
  }
  const u32 k_thr = (u32)max(1, A.topks[row]);
  const double pd = (double)A.topps[row] * (double)zfix;
  u64 p_thr = (pd >= (double)zfix) ? zfix : (u64)pd;
  if (p_thr == 0) p_thr = 1;   // top_p ~ 0: keep at least the max token
  if (cnt >= k_thr && cnt - my_cnt < k_thr) {
    u32 run = cnt - my_cnt;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (run < k_thr && run + tot[j] >= k_thr)
        sm.tau[0] = f32key((value(j) - m) * inv_t);
      run += tot[j];
    }
  }
  if (mass >= p_thr && mass - my_mass < p_thr) {
    u64 run = mass - my_mass;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const u64 own = ((u64)q[j] + ((ones >> j) & 1u)) * tot[j];
      if (run < p_thr && run + own >= p_thr)
        sm.tau[1] = f32key((value(j) - m) * inv_t);
      run += own;
    }
  }
  __syncthreads();

  // ---- kept mass of the quarters, and the lowest kept value ----
  const u32 tau = max(sm.tau[0], sm.tau[1]);
  {
    u32 kept = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      kept |= (tot[j] && f32key((value(j) - m) * inv_t) >= tau) ? 1u << j : 0u;
    if (__any(kept)) {
      u32 low = 2 * FAST_CODES;          // FAST_CODES for the magnitude 0
      u64 sum[FAST_PARTS] = {};
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if ((kept >> j) & 1u)
          low = up ? FAST_CODES + mag_of(j) : FAST_CODES - 1 - mag_of(j);
#pragma unroll
      for (int p = 0; p < FAST_PARTS; ++p) {
        u32 c[8];
        counts(p, c);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if ((kept >> j) & 1u) {
            sum[p] += (u64)q[j] * c[j];
            if ((ones >> j) & 1u) sum[p] += c[j];
          }
      }
#pragma unroll
      for (int p = 0; p < FAST_PARTS; ++p) sum[p] = lane_scan(sum[p], (u64)0, add);
      low = lane_scan(low, (u32)2 * FAST_CODES, MinOp());
      if (lane == 63) {
#pragma unroll
        for (int p = 0; p < FAST_PARTS; ++p)
          atomicAdd((unsigned long long*)&sm.part[p], (unsigned long long)sum[p]);
        atomicMin(&sm.low, (int)low - FAST_CODES);
      }
    }
  }
  __syncthreads();

  // ---- selection, in order of index ----
  u64 total = 0;
#pragma unroll
  for (int p = 0; p < FAST_PARTS; ++p) total += sm.part[p];
  const u64 target = (u64)((double)A.us[row] * (double)total);
  u64 at = 0;
  int own = 0;
#pragma unroll
  for (int p = 0; p < FAST_PARTS - 1; ++p)
    if (own == p && at + sm.part[p] <= target) {
      at += sm.part[p];
      own = p + 1;
    }
  const int lc = sm.low;
  const int lm = lc >= 0 ? lc : -1 - lc;
  const float low = lm == 0 ? -bf2f(FAST_BASE)
                            : bf2f((u16)((lc < 0 ? 0x8000 : 0) | (FAST_BASE + lm)));
  const float top = fmaxf(f32val(sm.one), low);
  auto mass_of = [&](float v) { return v >= low ? q32(weight(v - m)) : 0u; };
  auto half = [](u32 w, int j) {
    return __uint_as_float(j & 1 ? w & 0xffff0000u : w << 16);
  };
  const int first = own * (CNT_WAVES / FAST_PARTS) * part;   // piece of 512
  const int pieces = CNT_WAVES / FAST_PARTS * part;
  constexpr int TURNS = (FAST_BLK + CNT_WAVES - 1) / CNT_WAVES;
  {
    u32x4 w[TURNS];
    u32 alive[TURNS];
#pragma unroll
    for (int k = 0; k < TURNS; ++k) {
      const int i = min((first + wave + k * CNT_WAVES) * 512 + lane * 8, last8);
      w[k] = *(const u32x4*)(lrow + i);
      alive[k] = MASKED ? mrow[i >> 3] : 0xffu;
    }
#pragma unroll
    for (int k = 0; k < TURNS; ++k) {
      const int c = wave + k * CNT_WAVES;
      if (c >= pieces) break;
      const int i0 = (first + c) * 512;
      if (MASKED || i0 + 512 > vl) patch(w[k], alive[k], i0 + lane * 8, 0xffffffffu);
      u64 sum = 0;
      float best = half(w[k][0], 0);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float v = half(w[k][j >> 1], j);
        sum += mass_of(v);
        best = fmaxf(best, v);
      }
      if (__any(best >= top))
#pragma unroll
        for (int j = 0; j < 8; ++j) sum += half(w[k][j >> 1], j) >= top;
      sum = lane_scan(sum, (u64)0, add);
      if (lane == 63) sm.blk[c] = sum;
    }
  }
  __syncthreads();
  if (wave == 0) {
    const u64 a = 2 * lane < pieces ? sm.blk[2 * lane] : 0;
    const u64 b = 2 * lane + 1 < pieces ? sm.blk[2 * lane + 1] : 0;
    const u64 to = lane_scan(a + b, (u64)0, add) + at, from = to - a - b;
    const u64 mine = __ballot(to > target && from <= target);
    if (mine) {
      const int src = __ffsll((unsigned long long)mine) - 1;
      const bool second = from + a <= target;
      const int c = (int)from_lane((u32)(2 * lane + second), src);
      const u64 begin = from_lane(second ? from + a : from, src);
      const int i0 = (first + c) * 512 + lane * 8;
      u32x4 w = *(const u32x4*)(lrow + min(i0, last8));
      if (MASKED || i0 + 8 > vl)
        patch(w, MASKED ? mrow[min(i0, last8) >> 3] : 0xffu, i0, 0xffffffffu);
      u64 q[8], sum = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float v = half(w[j >> 1], j);
        q[j] = (u64)mass_of(v) + (v >= top);
        sum += q[j];
      }
      const u64 end = lane_scan(sum, (u64)0, add) + begin;
      u64 run = end - sum;
      if (end > target && run <= target) {
        int tok = i0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (run <= target) tok = i0 + j;
          run += q[j];
        }
        sm.token = tok;
      }
    }
  }
  __syncthreads();
  if (sm.token < 0) {   // u at the upper edge: the last kept token
    for (int i = tid; i < vl; i += CNT_THREADS)
      if ((!MASKED || ((mrow[i >> 3] >> (i & 7)) & 1u)) && bf2f(lrow[i]) >= low)
        atomicMax(&sm.last, i);
    __syncthreads();
    if (tid == 0) sm.token = sm.last;
    __syncthreads();
  }
  if (tid == 0) {
    const int tok = sm.token;
    A.out_tok[row] = tok;
    A.out_lp[row] = (bf2f(lrow[tok]) - m) * inv_t - logf(zf);
  }
  return true;
}

// A greedy row among others: the same sums as the kernel above makes of it, in the same
// order, but the row is read twice, eight pieces a wave and turn, for want of registers.
// Left to the kernel above, which runs behind, one greedy row in three made a batch wait
// for it: 3 / 116 / 378 rows of 151,936 43 / 45 / 93 us, now 30 / 30 / 76 (by the kernel
// above alone 32 / 35 / 90). False: nothing was done (the NaN that stands for logits that are not alive is one).
template <bool MASKED>
__device__ __forceinline__ bool fast_greedy(const SmpArgs& A, int row, char* lds) {
  u32* red = (u32*)lds;
  int tid = threadIdx.x, vl = A.vl;
  asm volatile("" : "+v"(tid), "+s"(vl));
  const int lane = tid & 63, l16 = lane & (CNT_WAVES - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const u16* lrow = (const u16*)A.logits + (long)row * A.v_row;
  const u8* mrow = MASKED ? (const u8*)(A.mask + (long)row * A.w_words)
                          : nullptr;
  const int last8 = (vl - 1) & ~7;
  const int part = (vl + CNT_CHUNK - 1) / CNT_CHUNK, t0 = wave * part * 512 + lane * 8;
  // f(logits, how many of them are not alive, index); those are 0xffff
  auto pieces = [&](auto f) {
#pragma unroll 1
    for (int c = 0; c < part; c += FAST_RING) {
      u32x4 w[FAST_RING];
      u32 bits[FAST_RING];
#pragma unroll
      for (int k = 0; k < FAST_RING; ++k) {
        const int i = min(t0 + (c + k) * 512, last8);
        w[k] = *(const u32x4*)(lrow + i);
        bits[k] = MASKED ? mrow[i >> 3] : 0xffu;
      }
#pragma unroll
      for (int k = 0; k < FAST_RING; ++k) {
        const int i = t0 + (c + k) * 512, left = c + k < part ? vl - i : 0;
        if (left < 8) bits[k] &= left > 0 ? (1u << left) - 1 : 0u;
        if (MASKED || left < 8)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            w[k][j] |= ((~bits[k] >> (2 * j)) & 1u) * 0xffffu |
                       ((~bits[k] >> (2 * j + 1)) & 1u) * 0xffff0000u;
        f(w[k], 8 - __popc(bits[k]), i);
      }
    }
  };
  float best = -INFINITY;
  int ones = 0;
  pieces([&](const u32x4& w, int dead, int) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ones += ((w[j] & 0xffffu) == 0xffffu) + (w[j] >= 0xffff0000u);
      best = fmaxf(best, fmaxf(__uint_as_float(w[j] << 16),
                               __uint_as_float(w[j] & 0xffff0000u)));
    }
    ones -= dead;
  });
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    best = fmaxf(best, __shfl_xor(best, off, 64));
  const bool odd = __any(ones != 0);
  if (lane == 0) {
    red[wave] = __float_as_uint(best);
    red[CNT_WAVES + wave] = odd;
  }
  __syncthreads();
  best = __uint_as_float(red[l16]);
  u32 any = red[CNT_WAVES + l16];
#pragma unroll
  for (int off = 1; off < CNT_WAVES; off <<= 1) {
    best = fmaxf(best, __shfl_xor(best, off, CNT_WAVES));
    any |= __shfl_xor(any, off, CNT_WAVES);
  }
  if (any) return false;
  float z = 0.f;
  int first = 0x7fffffff;
  pieces([&](const u32x4& w, int, int i) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const u32 h = j & 1 ? w[j >> 1] & 0xffff0000u : w[j >> 1] << 16;
      const float v = __uint_as_float(h);
      z += h == 0xffff0000u ? 0.f : __expf(v - best);
      if (v == best) first = min(first, i + j);
    }
  });
  z = wave_sum(z);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    first = min(first, __shfl_xor(first, off, 64));
  red += 2 * CNT_WAVES;
  if (lane == 0) {
    red[wave] = (u32)first;
    red[CNT_WAVES + wave] = __float_as_uint(z);
  }
  __syncthreads();
  if (tid == 0) {
    z = 0.f;
    for (int w = 0; w < CNT_WAVES; ++w) {
      first = min(first, (int)red[w]);
      z += __uint_as_float(red[CNT_WAVES + w]);
    }
    const bool none = best == -INFINITY;
    A.out_tok[row] = none ? 0 : first;
    A.out_lp[row] = none ? -INFINITY : -logf(z);
  }
  return true;
}

template <bool MASKED>
__global__ void __launch_bounds__(CNT_THREADS)
sampler_fast_kernel(SmpArgs A) {
  extern __shared__ __attribute__((aligned(16))) char fast_lds[];
  FastRing<MASKED> r;
  bool have = false;       // r is this row's
  for (int row = blockIdx.x; row < A.n; row += gridDim.x) {
    const int next = row + gridDim.x;
    bool done = false;
    if (!(A.temps[row] < 1e-5f)) {
      if (!have) {
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int part = (A.vl + CNT_CHUNK - 1) / CNT_CHUNK;
#pragma unroll
        for (int c = 0; c < FAST_RING; ++c)
          if (c < part)
            r.load(A, row, c, ((tid >> 6) * part + c) * 512 + (tid & 63) * 8);
      }
      have = next < A.n;
      done = fast_row<MASKED>(A, row, have ? next : -1, fast_lds, r);
    } else {
      have = false;
      done = fast_greedy<MASKED>(A, row, fast_lds);
      r = {};                // (not kept meanwhile)
    }
    __syncthreads();
    if (!done && threadIdx.x == 0) A.out_tok[row] = SMP_LEFT;
  }
}

extern "C" void sutro_sampler_fused(const void* logits, int logits_f32,
                                    const float* temps, const float* topps,
                                    const int* topks, const float* us,
                                    const unsigned int* mask, int n,
                                    long v_row, int vl, int w_words,
                                    int* out_tok, float* out_lp, int greedy,
                                    hipStream_t stream) {
  if (n == 0) return;
  SmpArgs A = {logits, temps, topps, topks, us, mask, v_row, n, vl, w_words,
               out_tok, out_lp, false};
  dim3 grid((unsigned)n), block(SMP_THREADS);
  // counting: rows of whole, aligned 16-byte pieces, from 2048 logits on (there
  // 124 -> 67 us for 1024 rows and 91 -> 17 us for one; below that no
  // vocabulary in use, and the general kernel has no 128 KB to clear)
  if (!logits_f32 && vl >= CNT_MIN && v_row % 8 == 0 &&
      (size_t)logits % 16 == 0) {
    auto run = [&](void (*fn)(SmpArgs), unsigned groups, int lds) {
      (void)hipFuncSetAttribute((const void*)fn,
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      hipLaunchKernelGGL(fn, dim3(groups), dim3(CNT_THREADS), lds, stream, A);
    };
    if (vl <= CNT_TILE && !greedy) {
      run(mask ? sampler_fast_kernel<true> : sampler_fast_kernel<false>,
          n < 256 ? n : 256, sizeof(FastShared));
      A.left = true;
    }
    // (a workgroup a row: in a loop over four rows each, the kernel needs more registers
    // than there are, 109 -> 113 us for 1024 rows of which none is left)
    run(mask ? sampler_count_kernel<true> : sampler_count_kernel<false>, n,
        sizeof(CountShared) > sizeof(SmpShared<CNT_WAVES>)
            ? sizeof(CountShared)
            : sizeof(SmpShared<CNT_WAVES>));
  } else if (logits_f32) {
    hipLaunchKernelGGL((sampler_kernel<false>), grid, block, 0,
                       stream, A);
  } else {
    hipLaunchKernelGGL((sampler_kernel<true>), grid, block, 0, stream, A);
  }
  HIP_CHECK_LAUNCH();
}
