// Softmax attention over paged keys and values on the matrix cores: prompt
// pieces (paged_prefill_kernel) and single decoded tokens
// (paged_decode_kernel + paged_join_kernel), bf16 or e4m3 pages of 32 tokens
// [blocks, kv heads, 32, D], head size D = 64 or 128 for keys and values.
// LOCAL adds what layer-list decoders ask for: chunk and window masks with
// kept first keys, a logarithmic distance bias, sinks, output gates and an
// output section.
//
// Both kernels make S^T = K Q^T, so a lane holds scores of ONE query row (a prompt's
// waves of 32 rows: of two, each in registers of its own):
// softmax is lane-local, the weights are already in the B layout of
// O^T += V^T P^T (with the contraction index permuted alike on both sides) and
// never pass through LDS, and rescaling O is one multiplication by a lane's own
// factor. V^T fragments come out of row-major LDS tiles through the transposed
// read. The running maximum moves only when a score exceeds it by more than
// 2^PA_SLACK: weights then stay below 2^PA_SLACK, which fp32 sums and bf16
// weights hold without loss of relative precision.
//
// Fragment layouts (gfx950), lane l:
//   mfma_f32_16x16x32_bf16: A[l%16][(l/16)*8 + j], B[(l/16)*8 + j][l%16],
//     D[(l/16)*4 + r][l%16], r = 0..3
//   ds_read_tr16_b64: in a group of 16 lanes lane i addresses the 4 columns
//     (i%4)*4.. of row i/4 and receives column i of those 4 rows.
#pragma once

#include "lds_limit.h"

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
  int G, per, groups;     // heads a kv head; workgroups a kv head and in all,
  int leads;              // each for entries rpb apart
  // decode: rows t0 .. t0 + n_rows, row t of sequence token_seq[t] or
  // seq_offset + t - t0
  const int* token_seq;
  int seq_offset, n_rows, nsplit;
  int quad;             // pages up to which a wave takes an item (0: none)
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

__device__ __forceinline__ f32x4 pa_mfma16(pa_frag a, pa_frag b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ pa_frag pa_pack8(pa_f32x8 v) {
  return __builtin_bit_cast(pa_frag, __builtin_convertvector(v, pa_bf16x8));
}
__device__ __forceinline__ u32x2 pa_pack4(f32x4 v) {
  return __builtin_bit_cast(u32x2, __builtin_convertvector(v, pa_bf16x4));
}
__device__ __forceinline__ int pa_same(int v) {
  return __builtin_amdgcn_readfirstlane(v);
}
// an entry of the block table, through the scalar cache (no kernel writes it)
__device__ __forceinline__ int pa_entry(const int* p, int i) {
  return ((const __attribute__((address_space(4))) int*)p)[i];
}
// transposed reads of rows base..base+3 and base+8.. (or +16..) of a V tile
__device__ __forceinline__ pa_frag pa_tr(const char* a, const char* b) {
  const pa_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) pa_s16x4*)a);
  const pa_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) pa_s16x4*)b);
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
// Issue order of a run of LDS reads feeding matrix products: AHEAD reads first,
// then EACH reads behind every PER products of MFMAS times PER (left alone, the
// compiler waits for every fragment in front of its product).
template <int READS, int MFMAS, int AHEAD, int EACH, int PER = 1>
__device__ __forceinline__ void pa_order() {
  constexpr int STEPS = (READS - AHEAD) / EACH;
  __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x8, PER, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, EACH, 0);
  }
  __builtin_amdgcn_sched_group_barrier(0x8, (MFMAS - STEPS) * PER, 0);
}
// maximum over the four lanes of equal lane % 16
__device__ __forceinline__ float pa_max4(float v) {
  const u32 x = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  const u32 y = __float_as_uint(
      fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
  const auto b = __builtin_amdgcn_permlane16_swap(y, y, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
// 8 cached elements as they are stored, and as bf16
template <bool KV8> struct PaRaw { typedef u16x8 type; };
template <> struct PaRaw<true> { typedef u32x2 type; };
template <bool KV8>
__device__ __forceinline__ u16x8 pa_widen(typename PaRaw<KV8>::type raw) {
  if constexpr (!KV8) {
    return raw;
  } else {
    float f[8];
    fp8x4_to_f32(raw[0], f);
    fp8x4_to_f32(raw[1], f + 4);
    return __builtin_bit_cast(
        u16x8, pa_pack8(pa_f32x8{f[0], f[1], f[2], f[3], f[4], f[5], f[6],
                                 f[7]}));
  }
}
// Tiles in LDS are row-major; 16-byte chunks are XOR-swizzled by the row. Of a
// prompt's tiles 256 bytes are read in a cycle: 16 rows of one chunk (keys) or 8 rows
// of two neighbouring ones (values, read transposed), which cover all 64 banks. That
// takes twice the addresses, which tiles that come through registers (REGS) have no
// registers for: with e4m3 pages and heads of 128 it was 2 % slower in the median of 55
// sizes and up to 5 (34 prompts of 120 behind 1500 keys, 20 and 4 heads, 101 -> 106 us), as
// was one new operand a product. They cover half of the banks.
template <int D, bool REGS>
__device__ __forceinline__ int pa_kswz(int row, int c) {
  return c ^ (REGS ? row & 7 : D == 128 ? row & 15 : row >> 1 & 7);
}
template <int D, bool REGS>
__device__ __forceinline__ int pa_vswz(int row, int c) {
  return c ^ (REGS ? row & 3 : D == 128 ? row & 7 : row >> 1 & 3) << 1;
}
// single tokens: 4 rows of two chunks
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
// Prompt pieces. A workgroup owns (up to) hpb query heads of one kv head times
// rpb blocks of 32 rows, one wave each (hpb * rpb = 4), and walks the visible keys
// 64 at a time: K and V of the next step go to the other half of a double-buffered
// LDS tile while this step is computed, straight from memory (REGS: through
// registers), one barrier a step. Through registers that way
// took a fifth of the time: without any copies at all, on one tile over and over, the
// 40 k prompt below was at 0.79 of it. Now, in turn on one card: 40 k 6549 -> 6079 us
// (1.01 -> 1.09 PFLOP/s), 16 of 2 k 356 -> 334, one of 3000 with 16 heads and 8 kv heads
// 76.7 -> 71.9, of 3850 with one head 88.8 -> 82.8, 256 of 200 with 8 heads of 64 49.0 ->
// 46.7, 160 of 150 with 16 and 8 heads 82 and 82.
//
// Bound by the products (0.47 of the matrix cores' cycles), the exponentials and the
// other operations of the softmax (0.5 of the vector unit's): the two waves of a SIMD
// cover each other's by little. Mixing them within a wave as well, a run of 32 keys'
// weights among the next one's scores and its values among the next one's maximum, is
// slower (40 k without copies 4.86 and 6.11 ms: more branches, one wave's order fixed).
// LDS reads are 0.35 of its cycles; with two rows on the same banks, as it was, 0.58, at
// the same time. The
// form before, 32 keys a step, two barriers, V scattered into a transposed tile
// two bytes at a time and weights passed through LDS, ran at 337 TFLOP/s on a
// 32 k prompt (16 heads, 4 kv heads, 128; useful flops) and 250 on prompts of
// 2 k; this one at 860 and 640 (13.1 -> 5.1 ms, 1.10 -> 0.43 ms), 0.78 instead
// of 1.61 ms on 7 prompts of 3 k with 32 heads over e4m3 pages, 0.11 instead of
// 0.22 ms on 160 short ones (24 k tokens). Two workgroups a CU (64 KB of LDS,
// up to 256 registers a lane) are what both limits allow.
//
// Products are of 16 x 16 x 32: those of 32 x 32 x 16 do as much a cycle but read
// and write every sum twice as often, which the power limit takes off the clock.
// In turn on one card: 32 k prompt (16 heads, 4 kv heads, 128) 4.42 -> 4.18 ms (996 ->
// 1052 TFLOP/s, the clock 1.99 -> 2.08 GHz, the matrix cores as busy as before), 40 k
// 6.63 -> 6.19, 16 of 2 k 361 -> 339 us, 7 of 3 k with 32 heads over e4m3 603 -> 552, 2
// of 20 k with 16 heads of 64 2.18 -> 2.04 ms, 16 of 2 k in chunks of 1024 235 -> 225 us.
// Between a decoder's other kernels: the 40 k prompt 31.6 -> 29.6 ms for four layers
// (0.83 -> 0.89 PFLOP/s), 16 ragged ones of 2 k 443 and 446 us.
// Where the power limit is out of reach a step takes as long as before or a little
// longer: one prompt of 3000 tokens with 16 heads and 8 kv heads 76.2 and 76.5 us, of
// 3850 with one head 86.2 and 88.8. Four keys' fragments are read ahead for it (six,
// which the larger products wanted: 78.6 and 91.4; two 79.0 and 92.1; all 84.3 and 99.5).
//
// BLOCKS: more than one block of rows in a workgroup. REGS: keys and values through
// registers, where they are widened or begin elsewhere than at 16 bytes.
//
// Entries of the tile map that continue each other (same sequence, 32 rows on)
// share a workgroup; the entry at a multiple of rpb, or one that continues
// nothing, leads.
// ---------------------------------------------------------------------------
template <int D, bool KV8, bool LOCAL, bool BLOCKS, int WAVES_PER_SIMD, bool REGS>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(WAVES_PER_SIMD, WAVES_PER_SIMD)))
paged_prefill_kernel(PagedArgs A) {
  constexpr int CPR = D / 8;                // 16-byte chunks per row
  constexpr int TILE = PA_KEYS * D * 2;     // bytes of a K or V tile
  constexpr int PER = TILE / 1024;          // 1 KB pieces per tile
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 15, g = lane >> 4;
  // heads vary fastest: workgroup id i runs on XCD i % 8, so an XCD works on
  // few kv heads and the tiles that share their pages meet in its L2; long
  // contexts first. Entries rpb apart follow each other, the rest comes after
  // them (z): in the order of the map the leaders of prompts of rpb blocks would
  // all be dispatched to the same quarter of the chip (128 prompts of 100 tokens,
  // 8 heads and kv heads of 64: 39 us, now 18; 16 and 8 heads of 128: 72, now 45)
  const int turn = blockIdx.x / A.groups, hg = blockIdx.x - turn * A.groups;
  const int e = (A.leads - 1 - turn) * A.rpb + blockIdx.z;
  if (e >= A.n_tiles) return;
  // (the same for all lanes: kept in scalar registers)
  const int s = pa_same(A.tile_seq[e]), q0 = pa_same(A.tile_q0[e]);
  const int k0 = (q0 >> 5) & (A.rpb - 1);
  if (k0 > 0 && e > 0 && A.tile_seq[e - 1] == s && A.tile_q0[e - 1] == q0 - 32)
    return;
  int cnt = 1;
  while (k0 + cnt < A.rpb && e + cnt < A.n_tiles && A.tile_seq[e + cnt] == s &&
         A.tile_q0[e + cnt] == q0 + 32 * cnt)
    ++cnt;
  const int kh = hg / A.per, rb = w >> (A.hpb >> 1);
  const int head = (hg - kh * A.per) * A.hpb + (w & (A.hpb - 1));  // of kh's
  const int hq = kh * A.G + min(head, A.G - 1);

  const int q_first = pa_same(A.qlocs[s]);
  const int nq_total = pa_same(A.qlocs[s + 1]) - q_first;
  const int rows = min(cnt * 32, nq_total - q0);   // of the workgroup
  if (rows <= 0) return;                    // a padding entry
  const int row_base = q_first + q0;
  const int L = pa_same(A.seq_lens[s]);
  const int p0 = L - nq_total + q0;         // position of the first row
  const int kv_end = p0 + rows;             // causal bound (exclusive)
  // this lane's rows of the workgroup, one of each sixteen, and their positions
  const int my_r[2] = {rb * 32 + ln, rb * 32 + 16 + ln};
  const int my_p[2] = {p0 + my_r[0], p0 + my_r[1]};
  const bool live = rb * 32 < rows && head < A.G;     // this wave has work
  const int w_end = min(kv_end, p0 + rb * 32 + 32);

  extern __shared__ __attribute__((aligned(16))) char pa_smem[];

  pa_frag qb[2][D / 32];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const u16* qp =
        A.q + ((long)(row_base + min(my_r[u], rows - 1)) * A.Hq + hq) * D +
        g * 8;
#pragma unroll
    for (int kk = 0; kk < D / 32; ++kk) {
      qb[u][kk] = *(const s16x8*)(qp + kk * 32);
      // scores are compared before they are scaled: by a positive number
      if (A.scale < 0.f) qb[u][kk] ^= (short)0x8000;
    }
  }
  const float scale = fabsf(A.scale);
  f32x4 acc[D / 16][2];
#pragma unroll
  for (int b = 0; b < D / 16; ++b) acc[b][0] = acc[b][1] = (f32x4)(0.f);
  float m_run[2] = {PA_NONE, PA_NONE}, l_run[2] = {0.f, 0.f};
  if (LOCAL && A.sink) {
    m_run[0] = m_run[1] = A.sink_w ? A.sink_w[hq] * PA_LOG2E : 0.f;
    l_run[0] = l_run[1] = g == 0 ? 1.f : 0.f;   // four lanes' sums are added
  }
  const float r1 = LOCAL && A.r1 ? A.r1[hq] : 0.f;
  const float r2 = LOCAL && A.r1 ? A.r2[hq] : 0.f;
  // lower key bounds: of this lane's row, of the workgroup's first row, and of
  // this wave's last row (above which a step needs no mask)
  int lo_row[2] = {0, 0}, c_row[2] = {0, 0}, kt0 = 0, kf0 = 0, n_kept = 0, lo_last = 0;
  int lo_first = 0, c_first = 0, w_lo = 0, w_c = 0;  // w: this wave's first row
  if (LOCAL) {
    int c_last;
    lo_row[0] = pa_lower(A, my_p[0], c_row[0]);
    lo_row[1] = pa_lower(A, my_p[1], c_row[1]);
    lo_first = pa_lower(A, p0, c_first);
    lo_last = pa_lower(A, w_end - 1, c_last);
    w_lo = pa_lower(A, p0 + rb * 32, w_c);
    kt0 = lo_first / PA_KEYS;
    kf0 = c_first / PA_KEYS;
    n_kept = max(min(kt0, (A.keep_first + PA_KEYS - 1) / PA_KEYS) - kf0, 0);
  }
  const u32 kept_n[2] = {(u32)max(A.keep_first - c_row[0], 0),
                         (u32)max(A.keep_first - c_row[1], 0)};
  const int kt1 = (kv_end + PA_KEYS - 1) / PA_KEYS;
  const int steps = n_kept + kt1 - kt0;
  const int last_page = (kv_end - 1) / PA_PG;
  const int* table = A.bt + (long)s * A.bt_stride;

  auto step_tile = [&](int it) {
    return it < n_kept ? kf0 + it : kt0 + (it - n_kept);
  };
  // A step is 2 * PER pieces of 1 KB of LDS, of K and then of V, piece c on wave
  // c % 4; all of its addresses but the lane's own offset are wave-uniform
  // (made per lane they cost more than the step's products). The second page of
  // the last step may lie past the context and is then fetched from the last
  // one (masked).
  constexpr int ES = KV8 ? 1 : 2;
  constexpr int RPP = 64 / CPR;             // rows per piece
  const int st_row = lane / CPR;
  const int t_row = w * RPP + st_row;       // of the tile, modulo 4 * RPP
  const u32 koff = (st_row * D + pa_kswz<D, REGS>(t_row, lane % CPR) * 8) * ES;
  const u32 voff = (st_row * D + pa_vswz<D, REGS>(t_row, lane % CPR) * 8) * ES;
  // LATE: four workgroups a CU, no registers to hold them while a step is computed
  constexpr bool LATE = REGS && WAVES_PER_SIMD == 4;
  typedef typename PaRaw<KV8>::type raw_t;
  typedef raw_t page_t __attribute__((aligned(KV8 ? 8 : 2)));   // as it lies in a page
  raw_t st[REGS ? PER / 2 : 1];
  int pa = 0, pb = 0;    // pages of the next step to load
  auto pages = [&](int kt) {
    pa = pa_entry(table, min(2 * kt, last_page));
    pb = pa_entry(table, min(2 * kt + 1, last_page));
  };
  // REGS: the pieces in registers, on their way to LDS
  auto load = [&]() {
#pragma unroll
    for (int j = 0; REGS && j < PER / 2; ++j) {
      const bool isv = j >= PER / 4;
      const int piece = (isv ? j - PER / 4 : j) * 4 + w;
      const long blk = j % (PER / 4) >= PER / 8 ? pb : pa;
      const u8* base = (isv ? A.vc : A.kc) +
                       ((blk * A.Hk + kh) * PA_PG + piece % (PER / 2) * RPP) *
                           (D * ES);
      st[j] = *(const page_t*)(base + (isv ? voff : koff));
    }
  };
  // Keys that a row does not see have weight 0, but their values may be infinite
  // or NaN (behind the context lies what an earlier request left there), which
  // 0 does not take away: values of keys that no row of the workgroup sees are
  // stored as zeros, and a wave takes 16 keys that none of its own rows see from
  // a tile of zeros.
  const u32 g_kept = max(A.keep_first - c_first, 0);
  auto edge = [&](int kv) {
    return kv + PA_KEYS > kv_end || (LOCAL && kv < lo_first);
  };
  auto any_sees = [&](int kp) {
    bool any = kp < kv_end;
    if (LOCAL) any &= (kp >= lo_first) | ((u32)(kp - c_first) < g_kept);
    return any;
  };
  auto store = [&](char* buf, int kv) {
    if (edge(kv))
#pragma unroll
      for (int j = PER / 4; REGS && j < PER / 2; ++j)
        if (!any_sees(kv + ((j - PER / 4) * 4 + w) * RPP + st_row))
          st[j] = raw_t(0);
#pragma unroll
    for (int j = 0; REGS && j < PER / 2; ++j)
      *(u16x8*)(buf + (j * 4 + w) * 1024 + lane * 16) = pa_widen<KV8>(st[j]);
  };

  // Otherwise straight to LDS, a page (of one kv head) a buffer, past whose end a lane of an
  // unseen value reads zeros. Written as assembly, since the compiler would wait for all
  // of them in front of every transposed read; without results, so that it has
  // nothing to wait for: the end of the step does.
  auto copy = [&](char* buf, int kv) {
    const bool e = edge(kv);
#pragma unroll
    for (int j = 0; j < PER / 2; ++j) {
      const bool isv = j >= PER / 4;
      const int piece = (isv ? j - PER / 4 : j) * 4 + w;
      const long blk = j % (PER / 4) >= PER / 8 ? pb : pa;
      const u64 base =
          (u64)(isv ? A.vc : A.kc) + (u64)(blk * A.Hk + kh) * (PA_PG * D * 2);
      const u32x4 page = {(u32)base, (u32)(base >> 32) & 0xffffu, PA_PG * D * 2,
                          0x00027000u};
      u32 off = isv ? voff : koff;
      if (isv && e && !any_sees(kv + piece * RPP + st_row)) off = 1u << 30;
      const u32 to = (u32)(size_t)(__attribute__((address_space(3))) char*)(
          buf + (j * 4 + w) * 1024);
      asm volatile(
          "s_mov_b32 m0, %0\n\ts_nop 3\n\t"
          "buffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(to),
          "v"(off), "s"(page), "s"(piece % (PER / 2) * RPP * (D * 2))
          : "m0", "memory");
    }
  };
  auto landed = [&]() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };

  // fragment addresses: keys row ln (+16 a tile), chunk kk*4 + g; values rows
  // 4*g + ti/4 (+16), columns of 16-block b
  constexpr int KA = REGS ? 2 : D / 32, VA = REGS ? 4 : D / 16;
  int kad[KA];
#pragma unroll
  for (int kk = 0; kk < KA; ++kk)
    kad[kk] = ln * (2 * D) + pa_kswz<D, REGS>(ln, kk * 4 + g) * 16;
  const int ti = lane & 15;
  int vad[VA];
#pragma unroll
  for (int b = 0; b < VA; ++b)
    vad[b] = (4 * g + (ti >> 2)) * (2 * D) +
             pa_vswz<D, REGS>(4 * g + (ti >> 2), b * 2 + ((ti & 3) >> 1)) * 16 +
             (ti & 1) * 8;

  pages(step_tile(0));
  if (REGS) load();
  else copy(pa_smem, step_tile(0) * PA_KEYS);
  if (steps > 1) pages(step_tile(1));
  if (REGS) store(pa_smem, step_tile(0) * PA_KEYS);
  else landed();
  if (BLOCKS)
#pragma unroll
    for (int z = 0; z < D / 64; ++z)
      *(u32x2*)(pa_smem + 4 * TILE + threadIdx.x * (D / 8) + z * 8) =
          u32x2{0u, 0u};
  for (int it = 0; it < steps; ++it) {
    __syncthreads();
    const int kv0 = step_tile(it) * PA_KEYS;
    const bool more = it + 1 < steps;
    char* const other = pa_smem + ((it + 1) & 1) * 2 * TILE;
    if (more && !REGS) copy(other, step_tile(it + 1) * PA_KEYS);
    if (more && REGS && !LATE) load();
    if (!LATE && it + 2 < steps) pages(step_tile(it + 2));
    // With several row blocks in the workgroup a step may be for the rows of
    // others: which of its four times 16 keys does a row of this wave see?
    u32 seen = 15;
    if (BLOCKS) {
      auto below = [&](int key) {       // the sixteens that begin before `key`
        return (1u << min(max((key - kv0 + 15) >> 4, 0), 4)) - 1;
      };
      seen = below(w_end);
      if (LOCAL)
        seen &= ~below(w_lo - 15) | (below(A.keep_first) & ~below(w_c - 15));
    }
    const bool mine = live && seen;
    if (mine) {
    const char* kb = pa_smem + (it & 1) * 2 * TILE;
    const char* vb = kb + TILE;

    f32x4 d[2][4];      // scores: row u, keys kv0 + t*16 + 4*g + r
#pragma unroll
    for (int t = 0; t < 4; ++t) d[0][t] = d[1][t] = (f32x4)(0.f);
#pragma unroll
    for (int kk = 0; kk < D / 32; ++kk)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const pa_frag ka = *(const s16x8*)(kb + kad[kk % KA] + kk / KA * 128 +
                                           t * 16 * 2 * D);
        const int f = REGS ? 0 : t & 1;     // (one new operand a product)
        d[f][t] = pa_mfma16(ka, qb[f][kk], d[f][t]);
        d[1 - f][t] = pa_mfma16(ka, qb[1 - f][kk], d[1 - f][t]);
      }
    pa_order<D / 8, D / 8, WAVES_PER_SIMD == 4 ? 2 : 4, 1, 2>();
    // without a distance bias scores stay unscaled until the exponential
    const bool whole = kv0 + PA_KEYS <= p0 + rb * 32 + 1 &&
                       (!LOCAL || kv0 >= lo_last);
    const bool biased = (LOCAL && A.r1) || scale < 1e-20f;
    if (biased) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int kp = kv0 + t * 16 + 4 * g + r;
            d[u][t][r] =
                d[u][t][r] * scale -
                r1 * __builtin_amdgcn_logf(
                         1.f + r2 * (float)max(my_p[u] - kp, 0));
          }
    }
    const float mul = biased ? 1.f : scale;
    if (!whole) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int kp = kv0 + t * 16 + 4 * g + r;
            bool vis = kp <= my_p[u];
            if (LOCAL)  // no short circuits: 32 selects, not 32 branches
              vis &= (kp >= lo_row[u]) | ((u32)(kp - c_row[u]) < kept_n[u]);
            d[u][t][r] = vis ? d[u][t][r] : -INFINITY;
          }
    }
    float tmax[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float m = PA_NONE;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) m = fmaxf(m, d[u][t][r]);
      tmax[u] = pa_max4(m) * mul;
    }
    const bool up0 = tmax[0] > m_run[0] + PA_SLACK,
               up1 = tmax[1] > m_run[1] + PA_SLACK;
    if (__any(up0 | up1)) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const float m_new = (u ? up1 : up0) ? tmax[u] : m_run[u];
        const float al = __builtin_amdgcn_exp2f(m_run[u] - m_new);
        m_run[u] = m_new;
        l_run[u] *= al;
#pragma unroll
        for (int b = 0; b < D / 16; ++b) acc[b][u] *= al;
      }
    }
    // a row that has seen no key yet: every weight is exp2(-inf) = 0
    float m_sub[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
      m_sub[u] = LOCAL && m_run[u] < 0.1f * PA_NONE ? 0.f : m_run[u];
    // a step's weights are summed by themselves: added one by one to the sum of
    // 20,000 they would each lose bits (0.7 at 14,000: 3e-4 of the sum)
    float sum[2] = {0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      pa_frag pb[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        pa_f32x8 p;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          p[j] = __builtin_amdgcn_exp2f(
              __builtin_fmaf(d[u][2 * ks + (j >> 2)][j & 3], mul, -m_sub[u]));
          sum[u] += p[j];
        }
        pb[u] = pa_pack8(p);
      }
      const char* v0 = vb + ks * 32 * 2 * D;
      const char* v1 = v0 + 16 * 2 * D;
      if (BLOCKS) {
        v0 = seen & (1u << 2 * ks) ? v0 : pa_smem + 4 * TILE;
        v1 = seen & (2u << 2 * ks) ? v1 : pa_smem + 4 * TILE;
      }
#pragma unroll
      for (int b = 0; b < D / 16; ++b) {
        const int at = vad[b % VA] + b / VA * 128;
        const pa_frag va = pa_tr(v0 + at, v1 + at);
        const int f = REGS ? 0 : b & 1;
        acc[b][f] = pa_mfma16(va, pb[f], acc[b][f]);
        acc[b][1 - f] = pa_mfma16(va, pb[1 - f], acc[b][1 - f]);
      }
    }
    pa_order<D / 4, D / 8, WAVES_PER_SIMD == 4 ? 4 : 8, 2, 2>();
    l_run[0] += sum[0];
    l_run[1] += sum[1];
    }
    if (more && REGS) {
      if (LATE) load();
      if (LATE && it + 2 < steps) pages(step_tile(it + 2));
      store(other, step_tile(it + 1) * PA_KEYS);
    }
    if (!REGS) landed();
  }

  if (!live) return;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    float l = l_run[u] + __shfl_xor(l_run[u], 32, 64);
    l += __shfl_xor(l, 16, 64);
    float f = l > 0.f ? 1.0f / l : 0.f;
    const long row = row_base + my_r[u];
    if (my_r[u] >= rows) continue;
    const u16* gp = nullptr;
    if (LOCAL) {
      f *= A.out_scale;
      if (A.gate_off >= 0) {
        gp = A.proj + row * A.ld + A.gate_off + (long)hq * A.gate_n;
        if (A.gate_n == 1) f *= 1.f / (1.f + expf(-bf2f(gp[0])));
      }
    }
    u16* op = A.out + row * A.ldo + A.out_off + (long)hq * D;
#pragma unroll
    for (int b = 0; b < D / 16; ++b) {
      const int col = b * 16 + 4 * g;
      f32x4 o = acc[b][u] * f;
      if (LOCAL && gp && A.gate_n > 1) {
#pragma unroll
        for (int e2 = 0; e2 < 4; ++e2)
          o[e2] *= 1.f / (1.f + expf(-bf2f(gp[col + e2])));
      }
      *(u32x2*)(op + col) = pa_pack4(o);
    }
  }
}

// ---------------------------------------------------------------------------
// Single tokens. One workgroup of 4 waves per item (row and kv head) and run of
// pages; the G <= 16 query heads of the kv head are the 16 columns of the
// products. The waves take the run's pages in turn, each with the next page's K
// and V on the way in registers while this one is computed (V passes through the
// wave's own LDS tile to be read transposed), and their partial results meet in
// LDS. Few rows over long contexts would leave most of the chip idle: their pages
// are cut into up to nsplit runs of at least PA_RUN pages, whose partial results
// a second kernel joins. A context of one run is finished here, one of a single
// page by one wave.
//
// Bound by memory: K and V of a row are read once. One wave a row, each page
// loaded and then computed, took 1.9 us a page; a call now takes (with the
// join) 28 us instead of 2390 for one row of 40 k keys and 4 kv heads (82 MB,
// 3 TB/s), 24 instead of 314 for 7 rows of 3 k e4m3 keys and 8 heads, 24
// instead of 128 for 16 rows of 2 k keys and 4 heads, and 33 instead of 41 for
// 256 rows of 130 keys and 8 heads (138 MB, 4.1 TB/s; a wave each, see below).
// Runs of 8 pages give every wave two pages, the fewest that hide one load
// behind another's work.
//
// Many rows over short contexts are bound by the workgroups themselves: two of
// them fit a CU, and one that has a page or two leaves most of its waves idle.
// From PA_QUAD_ITEMS items on a first layer of workgroups takes four neighbouring
// items each, a wave one, where none has more than PA_QUAD_PAGES pages; four more
// layers take the other items one by one as above (no layer where the table or
// the window bounds all of them). 4 kv heads, 1024 rows of 20 / 60 / 130 / 400
// keys: 30 / 35 / 68 / 153 us a workgroup an item, 20 / 28 / 62 / 153 this way; 2048
// rows of 20 keys 55 -> 35. (A wave alone with a long context beside short ones
// would take as long as four together: therefore the layers, not more pages.)
// ---------------------------------------------------------------------------
#define PA_RUN 8
#define PA_QUAD_ITEMS 1024  // items from which a wave takes a short one alone,
#define PA_QUAD_PAGES 6     // short: up to so many pages

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

// the same for columns c .. c + 3
template <bool LOCAL>
__device__ __forceinline__ void pa_store4(const PagedArgs& A, long t, int hq,
                                          int D, int c, f32x4 o, float l) {
  float f = l > 0.f ? 1.0f / l : 0.f;
  if (LOCAL) {
    f *= A.out_scale;
    if (A.gate_off >= 0) {
      const u16* gp = A.proj + t * A.ld + A.gate_off + (long)hq * A.gate_n;
      if (A.gate_n > 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] *= 1.f / (1.f + expf(-bf2f(gp[c + e])));
      } else {
        f *= 1.f / (1.f + expf(-bf2f(gp[0])));
      }
    }
  }
  *(u32x2*)(A.out + t * A.ldo + A.out_off + (long)hq * D + c) = pa_pack4(o * f);
}

template <int D, bool KV8, bool LOCAL>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(D == 64 ? 4 : 2)))
paged_decode_kernel(PagedArgs A) {
  constexpr int ES = KV8 ? 1 : 2;
  constexpr int KK = D / 32;                 // k-steps of the scores
  constexpr int DB = D / 16;                 // 16-column blocks of O
  constexpr int VL = PA_PG * D / (64 * 8);   // 8-element pieces a lane stages
  constexpr int VT = PA_PG * D * 2;          // bytes of a V page in LDS
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lo16 = lane & 15, g4 = lane >> 4;
  const int G = A.Hq / A.Hk;
  const int items = A.n_rows * A.Hk;   // (row, kv head)
  // with A.quad: the first layer of workgroups (y = 0) takes four items each,
  // one a wave, where all four are short; the other four layers take the items
  // of the rest one by one, neighbours side by side
  int item = blockIdx.x;
  bool solo = false;
  if (A.quad) {
    if (blockIdx.y) item += (blockIdx.y - 1) * gridDim.x;
    const int first = blockIdx.y ? item & ~3 : item * 4;
    if (first >= items) return;
    int longest = 0;
    for (int r = first / A.Hk; r <= min(first + 3, items - 1) / A.Hk; ++r)
      longest = max(longest, pa_span<LOCAL>(A, r).total);
    solo = blockIdx.y == 0;
    if (solo != (longest <= A.quad)) return;
    if (solo) item = first + w;
    if (item >= items) return;
  }
  const int kh = item % A.Hk;
  const int i = item / A.Hk;
  const PagedSpan v = pa_span<LOCAL>(A, i);
  const int run = pa_run_pages(v.total, A.nsplit);
  const int begin = A.quad ? 0 : blockIdx.y * run;
  if (begin >= v.total) return;
  const int end = min(v.total, begin + run);
  const bool alone = run >= v.total;
  if (!A.quad && v.total == 1) {
    solo = true;
    if (w) return;
  }
  const int step = solo ? 1 : 4;
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
  const u32 kept_n = max(A.keep_first - v.c_lo, 0);

  const int* table = A.bt + (long)v.s * A.bt_stride;
  auto page_of = [&](int x) {
    return x < v.n_kept ? v.kf0 + x : v.pg0 + (x - v.n_kept);
  };
  typedef typename PaRaw<KV8>::type Raw;
  Raw kx[2 * KK], vx[VL];
  int next = 0;      // page to load next
  auto load = [&]() {
    const long base = (((long)next * A.Hk + kh) * PA_PG) * D;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
        kx[h * KK + kk] = *(const Raw*)(
            A.kc + (base + (h * 16 + lo16) * D + kk * 32 + g4 * 8) * ES);
#pragma unroll
    for (int j = 0; j < VL; ++j)
      vx[j] = *(const Raw*)(A.vc + (base + (j * 64 + lane) * 8) * ES);
  };
  // V fragment addresses: rows 4*g4 + ti/4 (+16), columns of 16-block b
  int vad[4];
#pragma unroll
  for (int o = 0; o < 4; ++o)
    vad[o] = (4 * g4 + (lo16 >> 2)) * (2 * D) +
             pa_vchunk(lo16 >> 2, o * 2 + ((lo16 & 3) >> 1)) * 16 +
             (lo16 & 1) * 8;

  int x = solo ? begin : begin + w;
  if (x < end) {
    next = pa_entry(table, page_of(x));
    load();
    if (x + step < end) next = pa_entry(table, page_of(x + step));
  }
  for (; x < end; x += step) {
    const int kv0 = page_of(x) * PA_PG;
    auto visible = [&](int kp) {
      bool vis = kp <= v.p;
      if (LOCAL) vis &= (kp >= v.lo) | ((u32)(kp - v.c_lo) < kept_n);
      return vis;
    };
    // this page's V into the wave's tile, then the next page's loads; rows of
    // keys that are not visible as zeros (their weight is 0, but what lies there
    // may be infinite or NaN, which 0 does not take away)
    if (kv0 + PA_PG - 1 > v.p || (LOCAL && kv0 < v.lo))
#pragma unroll
      for (int j = 0; j < VL; ++j)
        if (!visible(kv0 + (j * 64 + lane) / (D / 8))) vx[j] = Raw(0);
#pragma unroll
    for (int j = 0; j < VL; ++j) {
      const int row = (j * 64 + lane) / (D / 8), c = (j * 64 + lane) % (D / 8);
      *(u16x8*)(vt + row * (2 * D) + pa_vchunk(row, c) * 16) =
          pa_widen<KV8>(vx[j]);
    }
    f32x4 sc[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      sc[h] = (f32x4)(0.f);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
        sc[h] = pa_mfma16(
            __builtin_bit_cast(pa_frag, pa_widen<KV8>(kx[h * KK + kk])), qb[kk],
            sc[h]);
    }
    if (x + step < end) load();
    if (x + 2 * step < end) next = pa_entry(table, page_of(x + 2 * step));
    // ---- this lane: head lo16, keys kv0 + h*16 + g4*4 + r
    float tmax = PA_NONE;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kp = kv0 + h * 16 + g4 * 4 + r;
        float z = sc[h][r] * A.scale;
        if (LOCAL && A.r1)
          z -= r1 * __builtin_amdgcn_logf(1.f +
                                          r2 * (float)max(v.p - kp, 0));
        sc[h][r] = visible(kp) ? z : PA_NONE;
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
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      p[j] = __builtin_amdgcn_exp2f(sc[j >> 2][j & 3] - m_sub);
      sum += p[j];
    }
    l_run = l_run * al + sum;
    const pa_frag pb = pa_pack8(p);
    // LOCAL keeps the weights' 24 bits: three bf16 terms (the products are
    // idle here), the other form rounds them to one
    pa_frag pb2, pb3;
    if (LOCAL) {
      p -= __builtin_convertvector(__builtin_bit_cast(pa_bf16x8, pb), pa_f32x8);
      pb2 = pa_pack8(p);
      p -= __builtin_convertvector(__builtin_bit_cast(pa_bf16x8, pb2),
                                   pa_f32x8);
      pb3 = pa_pack8(p);
    }
#pragma unroll
    for (int b = 0; b < DB; ++b) {
      const char* at = vt + vad[b & 3] + (b >> 2) * 128;
      const pa_frag va = pa_tr(at, at + 16 * 2 * D);
      f32x4 a = acc[b] * al;
      if (LOCAL) {
        a = pa_mfma16(va, pb3, a);
        a = pa_mfma16(va, pb2, a);
      }
      acc[b] = pa_mfma16(va, pb, a);
    }
  }
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);

  if (solo) {
    if (lo16 >= G) return;
    float m = m_run, l = l_run, f = 1.f;
    if (LOCAL && A.sink) {
      const float sk = A.sink_w ? A.sink_w[hq] * PA_LOG2E : 0.f;
      m = fmaxf(m_run, sk);
      f = __builtin_amdgcn_exp2f(m_run - m);
      l = f * l_run + __builtin_amdgcn_exp2f(sk - m);
    }
#pragma unroll
    for (int b = 0; b < DB; ++b)
      pa_store4<LOCAL>(A, t, hq, D, b * 16 + g4 * 4, acc[b] * f, l);
    return;
  }
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

// Joins the runs of a (row, head). The threads of a column share its runs:
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

// The same for few runs (then rows are many): a thread a column, nothing shared,
// and as few workgroups as that leaves, since rows of one run have nothing to
// join. 32 rows of 64 heads over 20 keys 8.8 -> 6.0 us
// for the call, over 400 keys 20.7 -> 17.1.
#define PA_FEW_RUNS 8
template <int D, bool LOCAL>
__global__ void __launch_bounds__(PA_JOIN) paged_join_few_kernel(PagedArgs A) {
  const int idx = blockIdx.x * (PA_JOIN / D) + threadIdx.x / D;
  if (idx >= A.n_rows * A.Hq) return;
  const int i = idx / A.Hq, hq = idx % A.Hq, c = threadIdx.x % D;
  const PagedSpan v = pa_span<LOCAL>(A, i);
  const int run = pa_run_pages(v.total, A.nsplit);
  const int n = (v.total + run - 1) / run;
  if (n <= 1) return;
  const long at = (long)idx * A.nsplit;
  float po[PA_FEW_RUNS], pm[PA_FEW_RUNS], pl[PA_FEW_RUNS];
#pragma unroll
  for (int y = 0; y < PA_FEW_RUNS; ++y)
    if (y < n) {
      po[y] = A.part_o[(at + y) * D + c];
      pm[y] = A.part_ml[(at + y) * 2];
      pl[y] = A.part_ml[(at + y) * 2 + 1];
    }
  float m = PA_NONE, sk = 0.f;
#pragma unroll
  for (int y = 0; y < PA_FEW_RUNS; ++y)
    if (y < n) m = fmaxf(m, pm[y]);
  if (LOCAL && A.sink) {
    sk = A.sink_w ? A.sink_w[hq] * PA_LOG2E : 0.f;
    m = fmaxf(m, sk);
  }
  float l = LOCAL && A.sink ? __builtin_amdgcn_exp2f(sk - m) : 0.f, o = 0.f;
#pragma unroll
  for (int y = 0; y < PA_FEW_RUNS; ++y)
    if (y < n) {
      const float f = __builtin_amdgcn_exp2f(pm[y] - m);
      l += f * pl[y];
      o += f * po[y];
    }
  pa_store<LOCAL>(A, A.t0 + i, hq, D, c, o, l);
}

// Runs to cut contexts of up to max_pages pages into: as many as give every CU
// four workgroups, none shorter than PA_RUN pages. From 512 items (row, kv head)
// on contexts stay whole: 128 rows of 400 keys, 4 heads, 28 us in two runs and
// 21 in one, 2500 keys 127 and 116.
static inline int pa_splits(long rows, int Hk, int max_pages) {
  const long items = rows * Hk;
  if (items >= 512) return 1;
  const long want = (1024 + items - 1) / (items > 0 ? items : 1);
  const long most = (max_pages + PA_RUN - 1) / PA_RUN;
  long n = want < most ? want : most;
  if (n > PA_MOST_RUNS) n = PA_MOST_RUNS;
  return n < 1 ? 1 : (int)n;
}

template <int D, bool KV8, bool LOCAL, bool BLOCKS, int WAVES_PER_SIMD, bool REGS>
static inline void pa_start_prefill(const PagedArgs& A, hipStream_t s) {
  // K and V twice, and zeros for 16 keys
  const size_t smem =
      2 * 2 * (size_t)PA_KEYS * D * 2 + (BLOCKS ? 16 * D * 2 : 0);
  const auto kernel =
      paged_prefill_kernel<D, KV8, LOCAL, BLOCKS, WAVES_PER_SIMD, REGS>;
  static std::atomic<unsigned long long> asked{0};
  if (smem > 65536) lds_limit((const void*)kernel, (int)smem, asked);
  hipLaunchKernelGGL(kernel, dim3((unsigned)A.leads * A.groups, 1, A.rpb),
                     dim3(256), smem, s, A);
}

// n_seqs: prompts that the tile map is of
template <int D, bool KV8, bool LOCAL, bool REGS = KV8>
static inline void pa_launch_prefill(PagedArgs A, int n_seqs, hipStream_t s) {
  // The copies to LDS take 16 bytes from multiples of 16. Pages that are a part of a
  // larger buffer may begin at any number (of layer lists they go to another kernel):
  // 16 of 2048 tokens, 16 and 4 heads of 128, 400 us from an odd one, as before, and
  // 317 straight from multiples of 16.
  if constexpr (!REGS && !LOCAL)
    if (((size_t)A.kc | (size_t)A.vc) % 16)
      return pa_launch_prefill<D, KV8, LOCAL, true>(A, n_seqs, s);
  // K and V are read once for 128 rows: 4, 2 or 1 query heads (what divides
  // their group) times 1, 2 or 4 row blocks. Prompts of one or two blocks have no
  // more of them: where workgroups are many they take 4 or 2 heads of any group,
  // the last workgroup of a kv head with fewer. Heads of 64, 500 prompts of 30
  // tokens, 14 and 2 heads 38 -> 23 us; 160 of 60 tokens 23 -> 19.
  A.G = A.Hq / A.Hk;
  A.hpb = A.G % 4 == 0 ? 4 : (A.G % 2 == 0 ? 2 : 1);
  if (A.G > 2 && (long)A.n_tiles * A.Hq / A.hpb > 512) {
    if (A.n_tiles <= n_seqs) A.hpb = 4;
    else if (A.n_tiles <= 2 * n_seqs && A.hpb == 1) A.hpb = 2;
  }
  A.rpb = 4 / A.hpb;
  A.per = (A.G + A.hpb - 1) / A.hpb;
  A.groups = A.Hk * A.per;
  A.leads = (A.n_tiles + A.rpb - 1) / A.rpb;
  // Heads of 64 leave room for four workgroups a CU in 128 registers, if a step's
  // keys and values are loaded behind the one before it (LATE). Many short prompts, a
  // few steps each with nothing to overlap them, are faster that way: 128 of 100
  // tokens, 8 heads and kv heads 18.3 -> 15.1 us, 160 of 150, 14 and 2 heads, 60 -> 44,
  // 500 of 30, 16 and 8, 37 -> 25, 256 of 200 117 -> 94 (three workgroups in 168
  // registers 16.0, 47.6, 28.3 and 97.7); long ones and few are not. (Layer lists would
  // spill registers: 32 prompts of 200 tokens, 8 heads and kv heads, 19 -> 24 us.)
  if constexpr (D == 64 && !LOCAL) {
    if ((long)A.n_tiles * A.groups >= 512 && A.n_tiles <= 8 * n_seqs) {
      if (A.rpb == 1) pa_start_prefill<D, KV8, LOCAL, false, 4, REGS>(A, s);
      else pa_start_prefill<D, KV8, LOCAL, true, 4, REGS>(A, s);
      return;
    }
  }
  if (A.rpb == 1) pa_start_prefill<D, KV8, LOCAL, false, 2, REGS>(A, s);
  else pa_start_prefill<D, KV8, LOCAL, true, 2, REGS>(A, s);
}

// max_pages: of a row at most (by the table, the window or the chunk)
template <int D, bool KV8, bool LOCAL>
static inline void pa_launch_decode(PagedArgs A, int max_pages, hipStream_t s) {
  const long items = (long)A.n_rows * A.Hk;
  dim3 grid((unsigned)items, (unsigned)A.nsplit);
  if (A.nsplit == 1 && items >= PA_QUAD_ITEMS) {
    A.quad = PA_QUAD_PAGES;
    grid = dim3((unsigned)((items + 3) / 4), max_pages <= A.quad ? 1u : 5u);
  }
  hipLaunchKernelGGL((paged_decode_kernel<D, KV8, LOCAL>), grid, dim3(256), 0,
                     s, A);
  if (A.nsplit > PA_FEW_RUNS)
    hipLaunchKernelGGL((paged_join_kernel<D, LOCAL>),
                       dim3((unsigned)(A.n_rows * A.Hq)), dim3(PA_JOIN), 0, s,
                       A);
  else if (A.nsplit > 1)
    hipLaunchKernelGGL((paged_join_few_kernel<D, LOCAL>),
                       dim3((unsigned)((A.n_rows * A.Hq + PA_JOIN / D - 1) /
                                       (PA_JOIN / D))),
                       dim3(PA_JOIN), 0, s, A);
}
