// Attention over one shared latent per token (all query heads read the same
// cached row; the row is the key, its leading columns are the value), on the
// MFMA matrix cores: bf16, pages of 32.
//
// The heads of a token are query rows like any other: the new tokens of a
// sequence times its H heads form one block of rows (the folded queries lie
// that way in memory), cut into tiles of 64, so prompt pieces and single
// decoded tokens run the same kernel and every cached row is fetched once for
// 64 query rows. A workgroup of 4 waves owns a tile and walks the visible keys
// 64 at a time (double-buffered in LDS, 16-byte chunks XOR-swizzled by row; the
// next tile's pages are copied straight there meanwhile, their places in the block
// table looked up a step before):
//   scores   wave (a, b) makes the 32 x 32 block of row half a and key half b,
//            S^T = mfma(A = K, B = Q^T), Q in registers; soft-max statistics
//            meet in LDS
//   values   wave w owns DV / 4 columns of all 64 rows, O^T += mfma(A = V^T,
//            B = P^T); V^T fragments come out of the key tile through the
//            transposed LDS read, P through LDS
// The running maximum of a row moves only when a score exceeds it by more than
// 2^LT_SLACK (weights then stay below 2^LT_SLACK, which fp32 sums and bf16
// weights hold without loss), so the accumulators are hardly ever rescaled.
//
// Workgroup id i runs on XCD i % 8: the tiles of 64 rows of one 32-token piece
// stay on one XCD, neighbouring pieces go to the eight XCDs in turn, so all
// XCDs work through the same sequence and its pages stay in their L2.
// When there are too few tiles for the chip the keys are also cut into
// `nsplit` runs whose partial results a second kernel joins.
//
// Times: 16 prompts of 1024 tokens, 32 heads of 576 and 512, 1343 -> 990 us; 61 prompts
// of 490, 16 heads of 256 and 256, window 1024, 441 -> 246 (590 and 480 TFLOP/s). Pages
// through registers waited for two memory latencies (table, page) twice a step; 64 rows
// of queries read and of results written in pieces of 8 to 32 bytes were 17 K cycles a
// tile. A step now takes 5.6 K cycles (products 2.2 K, the softmax between them 1.5 K,
// one wave a SIMD), a tile's begin and end 15 K.
//
// Fragment layouts (gfx950 v_mfma_f32_32x32x16_bf16): lane l holds
//   A[l%32][(l/32)*8 + j], B[(l/32)*8 + j][l%32], j = 0..7;
//   D[(r&3) + 8*(r>>2) + 4*(l/32)][l%32], r = 0..15.
// ds_read_tr16_b64: in a group of 16 lanes lane i addresses 4 consecutive
// columns (i%4)*4.. of row i/4; it receives column i of those 4 rows.
#include "mix_common.h"
#include "lds_limit.h"

#define LT_ROWS 64   // query rows per tile
#define LT_KEYS 64   // keys per step (two pages)
#define LT_PG 32     // page size
#define LT_PP 72     // padded row of the P tile
#define LT_SLACK 8.f // log2 of the largest weight against a stale maximum

typedef s16x8 bfrag;
typedef short s16x4l __attribute__((ext_vector_type(4)));
typedef u16 u16x4l __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4l __attribute__((ext_vector_type(4)));

__device__ __forceinline__ u16x4l pack_bf4(f32x4 v) {
  return __builtin_bit_cast(u16x4l, __builtin_convertvector(v, bf16x4l));
}

__device__ __forceinline__ f32x16 mfma32l(bfrag a, bfrag b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// A [64][DK] tile: row r's logical 16-byte chunk c lies at byte
//   r * 2 * DK + (c & ~7) * 16 + ((c ^ r) & 7) * 16.
// Only the low three bits of c and r decide the swizzle, so a lane keeps a few
// addresses and reaches the rest by constant offsets.

struct LatentArgs {
  u16* out;             // rows [t][out_off + h * dv ..], multiples of 16 bytes
  long ldo;
  int out_off;
  const u16* q;         // [T, H, dk]
  const u16* cache;     // [blocks, 1, 32, dk]
  const int* bt;
  int bt_stride;
  const int* seq_lens;
  const int* qlocs;
  const int* tile_seq;  // prompt pieces: 32 tokens a tile; null: single tokens
  const int* tile_q0;
  const int* token_seq;
  float scale;          // times log2(e)
  int window, H, dk, dv, nsplit;
  int pieces, n_sub;    // 32-token pieces (or tokens) and row tiles of each
  long t0, rows;        // first token and (token, head) rows of this launch
  float* part_o;        // [nsplit][rows][dv]
  float* part_ml;       // [nsplit][rows][2]
};

// keeps the accumulators in the accumulation registers between steps (they
// leave them for the rare rescaling only)
template <int NC>
__device__ __forceinline__ void lt_pin(f32x16 (&acc)[2][NC]) {
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int c = 0; c < NC; ++c) asm volatile("" : "+a"(acc[a][c]));
}

// Issue order of a run of `reads` LDS reads feeding `mfmas` matrix products:
// `ahead` reads first, then two products for every two further reads.
template <int READS, int MFMAS, int AHEAD>
__device__ __forceinline__ void lt_sched() {
  constexpr int A0 = AHEAD < READS ? AHEAD : READS;
  constexpr int P = (READS - A0) / 2 < MFMAS / 2 ? (READS - A0) / 2 : MFMAS / 2;
  __builtin_amdgcn_sched_group_barrier(0x100, A0, 0);
#pragma unroll
  for (int i = 0; i < P; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
  }
  __builtin_amdgcn_sched_group_barrier(0x100, READS - A0 - 2 * P, 0);
  __builtin_amdgcn_sched_group_barrier(0x8, MFMAS - 2 * P, 0);
}

// v[r] *= f inside the accumulation registers
__device__ __forceinline__ void lt_scale(f32x16& v, int r, float f) {
  float x = v[r], t;
  asm("v_accvgpr_read_b32 %1, %0\n\t"
      "s_nop 0\n\t"
      "v_mul_f32 %1, %1, %2\n\t"
      "v_accvgpr_write_b32 %0, %1\n\t"
      "s_nop 1"
      : "+a"(x), "=&v"(t) : "v"(f));
  v[r] = x;
}

template <int DK, int DV>
__device__ __forceinline__ void latent_body(const LatentArgs& A) {
  constexpr int CPR = DK / 8;             // chunks per row
  constexpr int CPT = LT_KEYS * CPR / 256;  // staged chunks per thread
  constexpr int NC = DV / 128;            // 32-column blocks per wave
  constexpr int QF = DK / 16;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int ln = lane & 31, hi = lane >> 5;
  const int wr = w >> 1, wk = w & 1;
  const int H = A.H, dk = A.dk, dv = A.dv;

  // grid.x = (pieces in groups of 8) x sub x 8
  const int x8 = blockIdx.x & 7, j8 = blockIdx.x >> 3;
  const int piece = (j8 / A.n_sub) * 8 + x8, sub = j8 % A.n_sub;
  if (piece >= A.pieces) return;
  int s, tok0, ntok;
  if (A.tile_seq) {
    const int b = A.pieces - 1 - piece;  // long contexts first
    s = A.tile_seq[b];
    const int q0 = A.tile_q0[b];
    tok0 = A.qlocs[s] + q0;
    ntok = min(32, A.qlocs[s + 1] - tok0);
  } else {
    tok0 = (int)A.t0 + piece;
    s = A.token_seq[tok0];
    ntok = 1;
  }
  const int row0 = sub * LT_ROWS;  // among ntok * H rows
  const int nrow = min(LT_ROWS, ntok * H - row0);
  if (nrow <= 0) return;
  // position of token tok0
  const int p0 = A.seq_lens[s] - (A.qlocs[s + 1] - tok0);
  const int pf = p0 + row0 / H;                    // first and last row
  const int kv_end = p0 + (row0 + nrow - 1) / H + 1;
  const int my_row = min(wr * 32 + ln, nrow - 1);
  const int my_p = p0 + (row0 + my_row) / H;
  const int my_lo = A.window > 0 ? max(0, my_p - A.window + 1) : 0;
  int kt0 = (A.window > 0 ? max(0, pf - A.window + 1) : 0) / LT_KEYS;
  int kt1 = (kv_end + LT_KEYS - 1) / LT_KEYS;
  if (A.nsplit > 1) {
    const int per = (kt1 - kt0 + A.nsplit - 1) / A.nsplit;
    kt0 += blockIdx.y * per;
    kt1 = min(kt1, kt0 + per);
  }
  const long prow = (long)(tok0 - A.t0) * H + row0;  // row of this launch
  float* pml = A.part_ml + ((long)blockIdx.y * A.rows + prow) * 2;
  if (kt0 >= kt1) {  // an empty run of keys (uniform over the workgroup)
    if (tid < nrow) {
      pml[tid * 2] = -1e30f;
      pml[tid * 2 + 1] = 0.f;
    }
    return;
  }

  extern __shared__ __attribute__((aligned(16))) char lt_smem[];
  constexpr int TILE = LT_KEYS * DK * 2;
  u16* P = (u16*)(lt_smem + 2 * TILE);               // [64][LT_PP]
  float* mx = (float*)(lt_smem + 2 * TILE + LT_ROWS * LT_PP * 2);  // [2][64]
  float* alpha_lds = mx + 2 * LT_ROWS;               // [64]

  f32x16 acc[2][NC];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int c = 0; c < NC; ++c)  // zeros made where they stay
      acc[a][c] = mfma32l((s16x8)(0), (s16x8)(0), (f32x16)(0.f));
  float m_run = -1e30f, l_run = 0.f;

  const int* table = A.bt + (long)s * A.bt_stride;
  const int last_page = (kv_end - 1) / LT_PG;
  // Pages go straight to LDS, 16 bytes a lane; a thread's chunks of either page sit at
  // the same places of the page. Columns past the row end are fetched from its start:
  // the query is zero there, so any finite value does.
  constexpr int HC = CPT / 2;
  u32 src[HC];
#pragma unroll
  for (int i = 0; i < HC; ++i) {
    const int L = i * 256 + tid, row = L / CPR, pc = L % CPR;
    int c = ((pc & ~7) | ((pc ^ row) & 7)) * 8;
    if (c >= dk) c = 0;
    src[i] = (u32)(row * dk + c) * 2;
  }
  const int wu = __builtin_amdgcn_readfirstlane(w);
  // entries of the block table through the scalar cache (no kernel writes it)
  auto page = [&](int i) {
    return ((const __attribute__((address_space(4))) int*)table)[min(i, last_page)];
  };
  auto copy = [&](int buf, int half, int pg) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(A.cache + (long)pg * LT_PG * dk), 0, 0xffffffffu, 0x00027000);
    char* dst = lt_smem + buf * TILE + half * (TILE / 2) + wu * 1024;
#pragma unroll
    for (int i = 0; i < HC; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          r, (__attribute__((address_space(3))) void*)(dst + i * 4096), 16, src[i],
          0, 0, 0);
  };

  // key fragments: row wk*32 + ln, logical chunks kk*2 + hi
  const int krow = wk * 32 + ln;
  int kad[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    kad[j] = krow * (2 * DK) + (((j * 2 + hi) ^ krow) & 7) * 16;
  // value fragments: rows hi*8 + ti/4 (+ 4), columns of block w*NC + c
  const int ti = lane & 15;
  int vad[2][2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      const int row = hi * 8 + (ti >> 2) + 4 * h;
      const int c = (w * NC + o) * 4 + ((lane >> 4) & 1) * 2 + ((ti & 3) >> 1);
      vad[h][o] = row * (2 * DK) + (c & ~7) * 16 + ((c ^ row) & 7) * 16 +
                  (ti & 1) * 8;
    }
  copy(0, 0, page(2 * kt0));
  copy(0, 1, page(2 * kt0 + 1));
  int pg0 = page(2 * kt0 + 2), pg1 = page(2 * kt0 + 3);
  // The queries come through the second buffer, laid out like 64 keys (read where the
  // products want them, a load touched 32 rows of 32 bytes: 8 K cycles a tile), and
  // through registers: copies straight to LDS do some 28 bytes a cycle.
  {
    const u16* qp = A.q + ((long)tok0 * H + row0) * dk;
    u16x8 v[CPT];
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int L = i * 256 + tid, row = L / CPR, pc = L % CPR;
      int c = ((pc & ~7) | ((pc ^ row) & 7)) * 8;
      if (c >= dk) c = 0;
      v[i] = *(const u16x8*)(qp + min(row, nrow - 1) * dk + c);
    }
#pragma unroll
    for (int i = 0; i < CPT; ++i)
      *(u16x8*)(lt_smem + TILE + i * 4096 + tid * 16) = v[i];
  }
  __syncthreads();
  bfrag qb[QF];
  {
    const int row = wr * 32 + ln;
    int qad[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      qad[j] = TILE + row * (2 * DK) + (((j * 2 + hi) ^ row) & 7) * 16;
#pragma unroll
    for (int kk = 0; kk < QF; ++kk) {
      qb[kk] = *(const s16x8*)(lt_smem + qad[kk & 3] + (kk >> 2) * 128);
      if (kk * 16 + hi * 8 >= dk) qb[kk] = (s16x8)(0);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  // each step's end waits for the next one's pages and sends for those of the step
  // behind it
  if (kt0 + 1 < kt1) {
    copy(1, 0, pg0);
    copy(1, 1, pg1);
    pg0 = page(2 * kt0 + 4);
    pg1 = page(2 * kt0 + 5);
  }
  int buf = 0;
  for (int kt = kt0; kt < kt1; ++kt, buf ^= 1) {
    lt_pin<NC>(acc);
    const char* tile = lt_smem + buf * TILE;
    // ---- scores: keys wk*32.., rows wr*32..
    f32x16 d = (f32x16)(0.f), d2 = (f32x16)(0.f);  // two independent chains
#pragma unroll
    for (int kk = 0; kk < QF; kk += 2) {
      d = mfma32l(*(const s16x8*)(tile + kad[kk & 3] + (kk >> 2) * 128), qb[kk],
                  d);
      d2 = mfma32l(*(const s16x8*)(tile + kad[(kk + 1) & 3] +
                                   ((kk + 1) >> 2) * 128), qb[kk + 1], d2);
    }
    const int kv0 = kt * LT_KEYS + wk * 32;
    float tmax = -1e30f;
    // (uniform) every row of the tile sees all keys of the step
    const bool all = kt * LT_KEYS + LT_KEYS - 1 <= pf &&
                     (A.window <= 0 || kt * LT_KEYS >= kv_end - A.window);
    if (all) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        d[r] = (d[r] + d2[r]) * A.scale;
        tmax = fmaxf(tmax, d[r]);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kp = kv0 + (r & 3) + 8 * (r >> 2) + 4 * hi;
        d[r] = kp <= my_p && kp >= my_lo ? (d[r] + d2[r]) * A.scale : -1e30f;
        tmax = fmaxf(tmax, d[r]);
      }
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    if (hi == 0) mx[wk * LT_ROWS + wr * 32 + ln] = tmax;
    __syncthreads();
    const float m_tile = fmaxf(mx[wr * 32 + ln], mx[LT_ROWS + wr * 32 + ln]);
    const float m_new = m_tile > m_run + LT_SLACK ? m_tile : m_run;
    const float al = exp2f(m_run - m_new);
    m_run = m_new;
    // a row that has seen no key yet: every weight is exp2(-1e30) = 0
    const float m_sub = m_new > -1e29f ? m_new : 0.f;
    float psum = 0.f;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 p;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        p[e] = __builtin_amdgcn_exp2f(d[g * 4 + e] - m_sub);
        psum += p[e];
      }
      *(u16x4l*)(P + (wr * 32 + ln) * LT_PP + wk * 32 + g * 8 + hi * 4) =
          pack_bf4(p);
    }
    l_run = l_run * al + psum;  // this lane's share of this wave's keys
    if (wk == 0 && hi == 0) alpha_lds[wr * 32 + ln] = al;
    __syncthreads();
    // ---- values: columns w * NC * 32.. of all rows
    const float al0 = alpha_lds[ln], al1 = alpha_lds[32 + ln];
    if (kt > kt0 && __any(al0 != 1.f || al1 != 1.f)) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          lt_scale(acc[0][c], r, al0);
          lt_scale(acc[1][c], r, al1);
        }
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const bfrag pb0 =
          *(const s16x8*)(P + ln * LT_PP + ks * 16 + hi * 8);
      const bfrag pb1 =
          *(const s16x8*)(P + (32 + ln) * LT_PP + ks * 16 + hi * 8);
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int at = ks * 16 * 2 * DK + (c >> 1) * 128;
        const char* a0 = tile + vad[0][c & 1] + at;
        const char* a1 = tile + vad[1][c & 1] + at;
        const s16x4l lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4l*)a0);
        const s16x4l hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4l*)a1);
        const bfrag va = __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7);
        acc[0][c] = mfma32l(va, pb0, acc[0][c]);
        acc[1][c] = mfma32l(va, pb1, acc[1][c]);
      }
    }
    lt_sched<4 * (2 + 2 * NC), 8 * NC, 4 + 2 * NC>();
    lt_pin<NC>(acc);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (kt + 2 < kt1) {
      copy(buf, 0, pg0);
      copy(buf, 1, pg1);
      pg0 = page(2 * kt + 6);
      pg1 = page(2 * kt + 7);
    }
  }

  // ---- epilogue: the row sums meet in LDS
  l_run += __shfl_xor(l_run, 32, 64);
  if (hi == 0) mx[wk * LT_ROWS + wr * 32 + ln] = l_run;
  if (wk == 0 && hi == 0) alpha_lds[wr * 32 + ln] = m_run;
  __syncthreads();
  if (A.nsplit > 1 && tid < nrow) {
    pml[tid * 2] = alpha_lds[tid];
    pml[tid * 2 + 1] = mx[tid] + mx[LT_ROWS + tid];
  }
  if (A.nsplit > 1) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const int row = a * 32 + ln;
      if (row >= nrow) continue;
      float* pp = A.part_o + ((long)blockIdx.y * A.rows + prow + row) * dv;
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int col = (w * NC + c) * 32 + g * 8 + hi * 4;
          f32x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = acc[a][c][g * 4 + e];
          if (col < dv) *(f32x4*)(pp + col) = o;
        }
    }
    return;
  }
  // Results go through the key buffers, so that lanes write neighbouring places of a
  // row (8 bytes of 32 rows a store took 9 K cycles a tile).
  constexpr int OS = DV * 2 + 16;
  static_assert(LT_ROWS * OS <= 2 * TILE, "results fit the key buffers");
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int row = a * 32 + ln;
    const float l = mx[row] + mx[LT_ROWS + row];
    const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = acc[a][c][g * 4 + e] * inv;
        *(u16x4l*)(lt_smem + row * OS +
                   ((w * NC + c) * 32 + g * 8 + hi * 4) * 2) = pack_bf4(o);
      }
  }
  __syncthreads();
  constexpr int PER = DV / 8;              // 16-byte pieces of a row
  const int c8 = tid % PER * 8;
  int row = tid / PER, t = (row0 + row) / H, h = row0 + row - t * H;
#pragma unroll 4
  for (; row < nrow; row += 256 / PER) {
    const u16x8 v = *(const u16x8*)(lt_smem + row * OS + c8 * 2);
    u16* op = A.out + (long)(tok0 + t) * A.ldo + A.out_off + (long)h * dv + c8;
    for (h += 256 / PER; h >= H; h -= H) ++t;
    if (c8 < dv) *(u16x8*)op = v;
  }
}

template <int DK, int DV>
__global__ void __launch_bounds__(256, 1)
latent_attention_kernel(const LatentArgs A) {
  latent_body<DK, DV>(A);
}

// one 128-thread block a (token, head) row: joins the partial results
__global__ void __launch_bounds__(128) latent_join_kernel(
    u16* __restrict__ out, long ldo, int out_off, const float* __restrict__ po,
    const float* __restrict__ pml, int nsplit, long t0, long rows, int H,
    int dv) {
  __shared__ float wz[64];
  const long r = blockIdx.x;
  if (threadIdx.x < 64) {  // the first wave: one run of keys a lane
    const int z = threadIdx.x;
    float m = -1e30f, l = 0.f;
    if (z < nsplit) {
      m = pml[(z * rows + r) * 2];
      l = pml[(z * rows + r) * 2 + 1];
    }
    if (!(l > 0.f)) m = -1e30f;
    const float top = wave_max_f32(m);
    const float w = l > 0.f ? exp2f(m - top) : 0.f;  // 0: an empty run
    const float sum = wave_sum_f32(w * l);
    wz[z] = w / sum;
  }
  __syncthreads();
  u16* op = out + (t0 + r / H) * ldo + out_off + (r % H) * (long)dv;
  for (int c = threadIdx.x * 4; c < dv; c += 512) {
    f32x4 a = (f32x4)(0.f);
#pragma unroll 4
    for (int z = 0; z < nsplit; ++z) {
      const float f = wz[z];
      if (f == 0.f) continue;  // an empty run left nothing behind
      a += f * *(const f32x4*)(po + (z * rows + r) * dv + c);
    }
    *(u16x4l*)(op + c) = pack_bf4(a);
  }
}

// Padded (key, value) sizes of a shape, or 0 when it is not covered.
static int latent_pad(int dk, int dv, int page, int* DV) {
  if (page != LT_PG || dk % 8 || dv % 8 || dv > dk || dv > 512) return 0;
  *DV = dv <= 128 ? 128 : (dv <= 256 ? 256 : 512);
  const int DK = dk <= *DV ? *DV : *DV + 64;
  return dk <= DK ? DK : 0;
}

extern "C" int mix_latent_splits(long rows, int bt_stride, int n_tiles, int H,
                                 int dk, int dv, int page) {
  int DV = 0;
  const int DK = latent_pad(dk, dv, page, &DV);
  if (!DK) return 0;
  // n_tiles > 0: tiles of 32 tokens; else single tokens
  const long blocks = n_tiles > 0
                          ? (long)n_tiles * ((32 * H + LT_ROWS - 1) / LT_ROWS)
                          : rows / H * ((H + LT_ROWS - 1) / LT_ROWS);
  // as many workgroups as run at once: LDS and registers hold one or two a CU
  const long fit = DK > 192 ? 256 : 512;
  long want = fit / blocks;
  const long most = ((long)bt_stride * page / LT_KEYS + 1) / 2;  // >= 2 steps
  if (want > most) want = most;
  if (want > 32) want = 32;
  return want < 1 ? 1 : (int)want;
}

extern "C" int mix_latent_attention(
    void* out, long ldo, int out_off, const void* q, const void* cache,
    const int* bt, int bt_stride, const int* seq_lens, const int* qlocs,
    const int* tile_seq, const int* tile_q0, int n_tiles, const int* token_seq,
    float scale, int window, int H, int dk, int dv, int page, long t0, long T,
    int nsplit, float* part_o, float* part_ml, hipStream_t s) {
  int DV = 0;
  const int DK = latent_pad(dk, dv, page, &DV);
  // (pages that do not begin at multiples of 16 bytes are not copied straight to LDS)
  if (!DK || ldo % 8 || out_off % 8 || (size_t)out % 16 || (size_t)cache % 16)
    return 0;
  if (T == 0) return 1;
  LatentArgs A;
  A.out = (u16*)out; A.ldo = ldo; A.out_off = out_off;
  A.q = (const u16*)q; A.cache = (const u16*)cache;
  A.bt = bt; A.bt_stride = bt_stride;
  A.seq_lens = seq_lens; A.qlocs = qlocs;
  A.tile_seq = tile_seq; A.tile_q0 = tile_q0; A.token_seq = token_seq;
  A.scale = scale * 1.4426950408889634f;
  A.window = window; A.H = H; A.dk = dk; A.dv = dv; A.nsplit = nsplit;
  A.t0 = t0; A.rows = T * H; A.part_o = part_o; A.part_ml = part_ml;
  A.pieces = tile_seq ? n_tiles : (int)T;
  A.n_sub = ((tile_seq ? 32 * H : H) + LT_ROWS - 1) / LT_ROWS;
  const dim3 grid((unsigned)((A.pieces + 7) / 8 * 8 * A.n_sub),
                  (unsigned)nsplit);
  const size_t smem = (size_t)2 * LT_KEYS * DK * 2 + LT_ROWS * LT_PP * 2 +
                      3 * LT_ROWS * sizeof(float);
#define LAUNCH_LT(KK, VV)                                                     \
  do {                                                                        \
    static std::atomic<unsigned long long> asked{0};                          \
    lds_limit((const void*)latent_attention_kernel<KK, VV>, (int)smem,        \
              asked);                                                         \
    hipLaunchKernelGGL((latent_attention_kernel<KK, VV>), grid, dim3(256),    \
                       smem, s, A);                                           \
  } while (0)
  if (DV == 128) {
    if (DK == 128) LAUNCH_LT(128, 128); else LAUNCH_LT(192, 128);
  } else if (DV == 256) {
    if (DK == 256) LAUNCH_LT(256, 256); else LAUNCH_LT(320, 256);
  } else {
    if (DK == 512) LAUNCH_LT(512, 512); else LAUNCH_LT(576, 512);
  }
#undef LAUNCH_LT
  if (nsplit > 1)
    hipLaunchKernelGGL(latent_join_kernel, dim3((unsigned)(T * H)), dim3(128),
                       0, s, (u16*)out, ldo, out_off, part_o, part_ml, nsplit,
                       t0, T * H, H, dv);
  return 1;
}
