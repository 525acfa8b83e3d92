// Grouped (per-expert) bf16 GEMM for dropless MoE on MI355X.
//
// Exact top-k routing with NO capacity dropping: token assignments are
// sorted by expert and laid out in per-expert segments padded to the tile
// height BM, so every workgroup tile belongs to exactly one expert and the
// grid is a STATIC upper bound (ceil(T*k/BM) + E tiles) — decode steps stay
// hipGraph-capturable; tiles past the live padded total exit early by
// reading the device-side tile-offset table.
//
//   stage 1 (gate_silu=1): act[r, 0:m]   = silu(x[tok[r]] @ Wg[e]^T)
//                                          * (x[tok[r]] @ Wu[e]^T)
//       A rows are gathered through row_tok (the padded-segment -> token
//       map; -1 = padding, clamped and discarded), B is read twice (gate
//       rows [0,m), up rows [m,2m) of the expert's weight) and the SwiGLU
//       is fused into the epilogue — the 2m-wide intermediate never exists.
//   stage 2 (gate_silu=0): out[r, 0:h]   = act[r] @ Wd[e]^T
//   ungated stage 1 (gate_silu=2): act[r, 0:m] = relu(x[tok[r]] @ Wu[e]^T)^2
//       (one B stream; experts of the form down(relu(up x)^2))
//
// Weights are stored [E, N, K] K-contiguous (torch-Linear layout per
// expert), so MFMA fragments are 8 consecutive bf16 along K for both
// operands — same verified recipe as csrc/gemm_tn.hip: BK=64 double-
// buffered direct global->LDS staging (global_load_lds dwordx4, swizzle
// mode 2), mfma_f32_16x16x32_bf16, fp32 accumulate.
//
// Two kernels by the height of the segments' tiles (the caller pads with the
// height it passes): tiles of 256 rows for prompts, tiles of 32 to 128 rows for
// fewer rows an expert and for widths the other does not take.
#include "common.h"
#include "lds_limit.h"

typedef s16x8 bf16x8;

__device__ __forceinline__ f32x4 mfma16g(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ void glds16g(const u32* g, u32* lds) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) u32*)g,
      (__attribute__((address_space(3))) u32*)lds, 16, 0, 0);
}

// swizzle mode 2 of gemm_tn.hip: row bits 1..3 XOR'd into the 16B chunk idx
__device__ __forceinline__ u32 gswz(u32 byte) {
  return byte ^ (((byte >> 8) & 7u) << 4);
}

// Tile configurations (all reuse the verified gemm_tn staging recipe):
//   BM=32,  BN=64,  4 waves 2x2  — decode steps: 40 KB of LDS for the gated
//                                  product, four workgroups a CU (64: three)
//   BM=64,  BN=64,  4 waves 2x2  — up to 72 rows an expert
//   BM=128, BN=128, 8 waves 2x4  — more rows: 4x the MFMA work per barrier, B
//                                  tiles shared across 4 M-rows of waves
//   BM=128, BN=64,  8 waves 4x2  — the same where n_cols % 128 != 0
// The segment padding (and tile_off table) is computed with the SAME BM the
// kernel is launched with; ops.expert_tile chooses it, with both sides measured.

// Stage a ROWS x 64 bf16 tile (ROWS rows of 128B) with WAVES waves; each
// wave issues ROWS/(8*WAVES) x 1KB chunks.
template <int ROWS, int WAVES>
__device__ __forceinline__ void gg_stage(u16* lds, const u16* gsrc,
                                         long row_stride_b, int wave, int lane) {
  constexpr int CH = ROWS / (8 * WAVES);
  static_assert(CH >= 1, "tile too small for wave count");
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const u32 b = (u32)(wave * CH + j) * 1024u + (u32)lane * 16u;
    const u32 lb = gswz(b);      // lane-linear LDS byte, pre-swizzled source
    glds16g((const u32*)((const char*)gsrc + (long)(lb >> 7) * row_stride_b +
                         (lb & 127u)),
            (u32*)((char*)lds + b));
  }
}

__device__ __forceinline__ const bf16x8* gg_frag(const u16* lds, int row,
                                                 int kk16) {
  u32 lb = (u32)row * 128u + (u32)kk16 * 16u;
  return (const bf16x8*)((const char*)lds + gswz(lb));
}

// the unit between the two expert matrices, on fp32 products
template <int MODE>
__device__ __forceinline__ float gg_unit(float v, float u, float limit,
                                         float rw) {
  if (MODE == 4) {
    v *= rw;
    u *= rw;
  }
  if (MODE == 1 || MODE >= 4) return v / (1.0f + __expf(-v)) * u;
  if (MODE == 3) {
    const float g = fminf(v, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g / (1.0f + __expf(-1.702f * g)) * (u + 1.0f);
  }
  if (MODE == 2) {
    v = fmaxf(v, 0.f);
    return v * v;
  }
  return v;
}

// expert e with tile_off[e] <= t < tile_off[e + 1]
__device__ __forceinline__ int gg_expert(const int* tile_off, int n, int t) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (tile_off[mid] <= t) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// MODE=1: rows gathered, B has two streams (gate/up at N-offset 0 and n_cols), output
// n_cols wide with silu(g)*u. MODE=0: plain A, plain B, plain store.
// MODE=2: rows gathered, one B stream, relu(x)^2 in the epilogue.
// MODE=3: like MODE=1 with the clamped unit g sigmoid(1.702 g) (u + 1),
// g = min(gate, limit), u = clamp(up, -limit, limit).
// MODE=4: like MODE=1 with both products of row r times row_w[r] first (the
// expert reads row_w * x).
// Waves arranged WROWS(M) x WCOLS(N); wave tile = (BM/WROWS) x (BN/WCOLS).
template <int MODE, int BM, int BN, int WROWS, int WCOLS>
__global__ __launch_bounds__(WROWS* WCOLS * 64) void grouped_gemm_kernel(
    u16* __restrict__ out,        // [rows_max, n_cols] bf16
    const u16* __restrict__ a,    // GATHER: [T, K]; else [rows_max, K]
    const u16* __restrict__ w,    // [E, N, K] bf16 (N = n_cols or 2*n_cols)
    const int* __restrict__ row_tok,    // [rows_max] or nullptr
    const int* __restrict__ tile_off,   // [E+1] padded-offset / BM
    const int* __restrict__ counts,     // [E] live rows per expert
    int n_experts, int n_cols, long K, float limit,
    const float* __restrict__ row_w) {  // [rows_max], MODE 4
  constexpr bool GATED = MODE == 1 || MODE >= 3;  // two B streams (gate, up)
  constexpr bool GATHER = MODE != 0;  // A rows come through row_tok
  constexpr int WAVES = WROWS * WCOLS;
  constexpr int WM = BM / WROWS;
  constexpr int WN = BN / WCOLS;
  constexpr int MF = WM / 16;
  constexpr int NF = WN / 16;
  const int t = blockIdx.x;
  const int n0 = blockIdx.y * BN;
  if (t >= tile_off[n_experts]) return;
  const int e = gg_expert(tile_off, n_experts, t);
  const int m0 = (t - tile_off[e]) * BM;              // within-segment row
  const int seg0 = tile_off[e] * BM;                  // segment global base
  const int rows_valid = counts[e] - m0;              // live rows this tile
  if (rows_valid <= 0) return;       // a segment longer than its rows need

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WCOLS, wn = wave % WCOLS;

  __shared__ u16 smem[2][(BM + (GATED ? 2 : 1) * BN) * 64];
  const int b_off = BM * 64;
  const int b2_off = (BM + BN) * 64;

  // Experts start at different steps of k where weight rows are multiples of 4 KB
  // apart: all in step, workgroups read the same few 128-byte columns of a hundred
  // thousand rows at a time, which lie on few memory channels. 32 experts of
  // 2048 x 2048, 128 tokens of 4 on tiles of 32: gate and up 130 -> 91 us, down 72 ->
  // 54 (5.9 TB/s and 5.0); 16 tokens 137 -> 95 and 74 -> 56; 256 tokens on tiles of 64
  // 160 -> 133 and 77 -> 55. Rows of 6 KB spread by themselves. All workgroups of an
  // expert stay in step: its column blocks share rows of x (a start for each of them
  // 65 us instead of 54, 78 instead of 55, and 12 to 27 % more than none for 60
  // experts), its tiles weights, and a row's sums come out the same in every tile.
  // Tiles of 128 rows all start at 0.
  const int KT = (int)(K >> 6);
  int ko = BM <= 64 && K % 2048 == 0 ? (int)(e * 5u) % KT * 64 : 0;
  const long Kb = K * 2;
  const u16* wa = w + (long)e * (GATED ? 2 : 1) * n_cols * K;
  const u16* wg = wa + (long)n0 * K;
  const u16* wu = wa + (long)(n_cols + n0) * K;       // up rows (stage 1)
  const u16* aa = GATHER ? a : a + (long)seg0 * K;
  const int* rt = row_tok ? row_tok + seg0 : nullptr;

  f32x4 accg[MF][NF], accu[GATED ? MF : 1][GATED ? NF : 1];
#pragma unroll
  for (int i = 0; i < MF; ++i)
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      accg[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (GATED) accu[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

  // Tiles of 64 carry their pointers along: with the offset added to the base anew
  // each step, a few workgroups take 2 to 12 % longer (4 experts of 1024 x 2560, 21
  // rows each 53.9 us, carried 47.5); tiles of 32 are 1 % faster without.
  constexpr bool CARRY = BM == 64;
  const u16 *pa = aa + ko, *pg = wg + ko, *pu = wu + ko;
  auto stage_w = [&](u16* to) {
    gg_stage<BN, WAVES>(to + b_off, CARRY ? pg : wg + ko, Kb, wave, lane);
    if (GATED)
      gg_stage<BN, WAVES>(to + b2_off, CARRY ? pu : wu + ko, Kb, wave, lane);
  };
  stage_w(smem[0]);     // (while the rows are looked up)

  // The tile's rows, 8 a chunk; chunks of rows past the live ones are left out (what the
  // LDS holds there is multiplied for rows that nobody reads: a branch around those
  // products costs 20 cycles a step). Where experts get two rows, tiles of 64 fetched
  // as much of rows as of weights: down of 28 experts of 4096 x 3072 158 -> 126 us, of
  // 2048 x 2048 on tiles of 32 50.7 -> 44.5. Rows are looked up once: at each step, the
  // wait for the table stood before the copies (16 rows an expert of 2048 x 2048 on
  // tiles of 64 139 -> 119 us, 64 of 3072 x 4096 530 -> 432, 112 of 2048 x 2048 on 128
  // 198 -> 169).
  // Only on gated tiles of 32 that wait does good where it is hidden: with all four
  // workgroups that a CU's LDS holds it takes them out of step. With fewer it is in the
  // way. So it goes by whether the last round of workgroups is over three quarters full.
  // Once and by this rule, us: 2848 workgroups of 2 x 2048 x 2048 (0.78 of a round) 267 and
  // 257, 1932 of 2 x 768 x 6144 (0.89) 545 and 529, 992 of 2 x 2048 x 2048 (0.97) 93.7 and
  // 91.6; at each step against once, 396 of 2 x 2816 x 6144 (0.39) 144 and 117, 1216 of 2 x
  // 1024 x 2880 (0.19) 202 and 174, 736 of 2 x 2048 x 6144 (0.72) 206 and 202. To ask costs
  // 0.4 us at most; the other units (six a CU) would pay 4 % for it and gain 1 to 3.
  constexpr int CHA = BM / (8 * WAVES);
  static_assert(CHA >= 1, "tile too small for wave count");
  // (from the last wave on: the first ones have the products of few rows)
  auto a_chunk = [&](int j) { return j * WAVES + WAVES - 1 - wave; };
  auto a_row = [&](int j) {
    const u32 lb = gswz((u32)a_chunk(j) * 1024u + (u32)lane * 16u);
    int row = m0 + min((int)(lb >> 7), rows_valid - 1);
    asm volatile("" : "+v"(row));       // (a look-up at a step stays there)
    return (long)(GATHER ? max(rt[row], 0) : row) * Kb + (lb & 127u);
  };
  long a_at[CHA];
#pragma unroll
  for (int j = 0; j < CHA; ++j) a_at[j] = a_row(j);
  constexpr bool AGAIN = BM == 32 && GATED;
  constexpr u32 ROUND = 256 * (160 * 1024 / sizeof(smem));
  const u32 last = (tile_off[n_experts] * gridDim.y - 1) % ROUND + 1;
  const bool again = last * 4 > ROUND * 3;

  auto stage_a = [&](u16* to) {
    const char* sa = (const char*)(CARRY ? pa : aa + ko);
#pragma unroll
    for (int j = 0; j < CHA; ++j) {
      const int c = a_chunk(j);
      if (c * 8 < rows_valid) {
        if (AGAIN && again) a_at[j] = a_row(j);
        glds16g((const u32*)(sa + a_at[j]),
                (u32*)((char*)to + c * 1024 + lane * 16));
      }
    }
  };
  stage_a(smem[0]);
  __syncthreads();

  for (int kt = 0; kt < KT; ++kt) {
    const int p = kt & 1;
    u16* aT = smem[p];
    u16* bgT = smem[p] + b_off;
    u16* buT = smem[p] + b2_off;
    if (kt + 1 < KT) {
      ko += 64;
      long step = 64;
      if (ko == (int)K) {
        ko = 0;
        step -= K;
      }
      if (CARRY) {
        pa += step;
        pg += step;
        if (GATED) pu += step;
      }
      stage_a(smem[p ^ 1]);
      stage_w(smem[p ^ 1]);
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int kk16 = kk * 4 + (lane >> 4);
      bf16x8 bg[NF], bu[GATED ? NF : 1];
#pragma unroll
      for (int j = 0; j < NF; ++j) {
        bg[j] = *gg_frag(bgT, wn * WN + j * 16 + (lane & 15), kk16);
        if (GATED)
          bu[j] = *gg_frag(buT, wn * WN + j * 16 + (lane & 15), kk16);
      }
#pragma unroll
      for (int i = 0; i < MF; ++i) {
        const bf16x8 af =
            *gg_frag(aT, wm * WM + i * 16 + (lane & 15), kk16);
#pragma unroll
        for (int j = 0; j < NF; ++j) {
          accg[i][j] = mfma16g(af, bg[j], accg[i][j]);
          if (GATED) accu[i][j] = mfma16g(af, bu[j], accu[i][j]);
        }
      }
    }
    __syncthreads();
  }

  // epilogue: D[16,16] lane l holds rows (l/16)*4+r, col l%16
  const int drow = (lane >> 4) * 4;
  const int dcol = lane & 15;
#pragma unroll
  for (int i = 0; i < MF; ++i) {
    if (wm * WM + i * 16 >= rows_valid) break;
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      const int gn = n0 + wn * WN + j * 16 + dcol;
      const int grow0 = wm * WM + i * 16 + drow;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int grow = grow0 + r;
        // Padding rows are left as they are: those of a workspace that keeps zeros or
        // results may be gathered with weight 0, and what was multiplied for them
        // need not be finite.
        if (grow >= rows_valid) continue;
        const long o = (long)(seg0 + m0 + grow) * n_cols + gn;
        const float v = gg_unit<MODE>(
            accg[i][j][r], GATED ? accu[GATED ? i : 0][GATED ? j : 0][r] : 0.f,
            limit, MODE == 4 ? row_w[seg0 + m0 + grow] : 1.f);
        out[o] = f2bf(v);
      }
    }
  }
}

// ---- tiles of 256 rows ----------------------------------------------------
// 256 rows x 256 weight rows (gated: 128 gate and 128 up rows) a tile, four waves
// of 128 x 128, one on a SIMD with all of its registers: 256 of them hold the
// sums, and a wave reads 32 KB of LDS for 2.1 MFLOP. One workgroup a CU stays for
// the whole launch and goes from tile to tile; its copies run across the tiles.
//
// Bound by the power limit and by the copies' share of the LDS: by the counters the
// matrix cores are busy 65 to 79 %, and the clock falls from 2.7 GHz in a launch of
// 44 us to 1.8 in one of 4.7 ms. What that took:
// - mfma 16x16x32 instead of 32x32x16. Both do as much a cycle, but a sum is read
//   and written half as often, and the clock the power limit leaves is higher:
//   8192^3 785 -> 727 us, the rest alike.
// - Operands of the next 32 of k are read while the products of these run (two
//   register sets), so no wave waits for the LDS behind a barrier.
// - Copies go straight to LDS by buffer loads (one address register, the step in a
//   scalar) into a ring of five units of 32 KB: three of A rows and B rows ahead
//   of those in use, A two steps and B one step before they are needed.
// At 32 experts of 2048 x 2048, gate and up / down, against eight waves of 128 x
// 64 with two buffers, in turn on one card: 4096 rows an expert 1910 / 977 -> 1595 /
// 808 us (1151 / 1125 -> 1379 / 1361 TFLOP/s), 384 rows 276 / 135 -> 224 / 117, 187
// rows 163 / 82 -> 140 / 70. A large product of the library reaches 1.65 PFLOP/s
// there (8192^3: 668 us). Cards differ by 5 to 15 % in what their power limit leaves.
//
// DENSE (modes 5 and 6) is a gated linear layer of its own, one matrix over m_rows rows,
// against the library's product and a pass of silu over its result (2 N columns
// written and read again): 2 x 3072 x 1024 at 24,000 rows 357 -> 259 us, 2 x 8192 x
// 2048 at 32,768 rows 1775 -> 1555, 2 x 12288 x 4096 4597 -> 4413, 2 x 25600 x 5120
// at 8192 rows 3280 -> 2829; the unit's inputs stay in fp32 (error against 64 bits
// 3.1e-3 -> 1.7e-3). Mode 6 is the unit with GELU by tanh; column blocks behind its own
// are 256 plain columns each, of the same input (a residual gate), so that these need no
// launch that fills the chip for itself: 2 x 8192 and 2048 columns of 2048 at 32,768
// rows 2011 -> 1814 us, at 1532 rows 112 -> 103 (119 with the product of the 2048 by the
// library); error against 64 bits 6.6e-3 -> 3.7e-3.
//
// An XCD (workgroup id % 8) takes GW_ROWS neighbouring row tiles and goes through
// all column blocks with them: its 32 workgroups share 4 row tiles and 8 column
// blocks at a time, so that four of five copies hit its L2.
#define GW_ROWS 4
#define GW_CUS 256
#define GW_UNIT (256 * 128)       // bytes of 256 rows x 64 of k
#define GW_LDS (5 * GW_UNIT)

template <int V>
struct GwFlag {
  static constexpr bool v = V != 0;
};

// What mode 7 makes of the products: columns of 128 are heads, hq of queries, hk of
// keys, hk of values (see store_heads).
struct GwHeads {
  u16* kc;                 // pages [blocks, hk, 1 << shift, 128], fewer than 2^32 tokens
  u16* vc;
  const long* pos;         // [M]
  const long* slots;       // [M]
  const float* cos_sin;    // [positions, 128]
  const u16* qw;           // [128] or null
  const u16* kw;
  float eps;
  int hq, hk, shift;
};

// an output tile: first row, first column, expert, live rows from the first on
struct GwTile {
  long seg;
  int n0, e, live;
};

// where a workgroup is: first row tile of the group, place among its XCD's share
struct GwWalk {
  int t0, place;
  bool even;       // see gw_even
};

// Next tile of the walk. Groups of 8 * GW_ROWS row tiles go through all column
// blocks, GW_ROWS rows an XCD. The rows that are left go GW_ROWS at a time, every
// eighth column block an XCD (or, of fewer than 8 column blocks, tile by tile):
// with rows of their own 1024 x 16384 x 2048 would run on one XCD of eight.
// Lanes hold tile_off and counts where experts are few; DENSE: one matrix for
// m_rows rows.
template <int BN, bool DENSE>
__device__ __forceinline__ bool gw_next(GwWalk& k, int nb, int total,
                                        int n_experts, int m_rows, int loff,
                                        int lcnt, const int* tile_off,
                                        const int* counts, GwTile& g) {
  const int xcd = blockIdx.x & 7;
  int t, col;
  for (;;) {
    const int left = total - k.t0;
    if (left >= 8 * GW_ROWS) {
      if (k.place < GW_ROWS * nb) {
        t = k.t0 + xcd * GW_ROWS + k.place % GW_ROWS;
        col = k.place / GW_ROWS;
        break;
      }
      k.place -= GW_ROWS * nb;
      k.t0 += 8 * GW_ROWS;
    } else if (left <= 0) {
      return false;
    } else if (nb >= 8 && (left > GW_ROWS || !k.even)) {
      const int rows = min(left, GW_ROWS);
      // The XCDs that get one column block more go round by as many as they are,
      // so that all end with as many tiles. Round by one, some had a tile a CU more:
      // 8 experts of 1536 x 2048 at 375 rows 84 us, now 46; 4758 rows of 2 x 6656 x
      // 3648 402 and 334.
      const int x = (xcd + k.t0 / GW_ROWS * (nb & 7)) & 7;
      const int size = rows * ((nb - x + 7) >> 3);
      if (k.place < size) {
        col = k.place / rows;
        t = k.t0 + k.place - col * rows;
        col = col * 8 + x;
        break;
      }
      k.place -= size;
      k.t0 += rows;
    } else if (nb >= 8) {
      // the last rows: as many tiles an XCD as it is short of an eighth, in one run
      const int groups = k.t0 % (8 * GW_ROWS) / GW_ROWS, e = nb & 7;
      const int all = left * nb;
      const int share = (groups * GW_ROWS * nb + all + 7) >> 3;
      int from = 0, size = 0;
      for (int y = 0; y <= xcd; ++y) {
        int has = groups * (nb >> 3);
        for (int g = 0; g < groups; ++g) has += ((y + g * e) & 7) < e;
        from += size;
        size = max(share - has * GW_ROWS, 0);
      }
      size = min(size, all - from);
      if (k.place >= size) return false;
      col = (from + k.place) / left;
      t = from + k.place - col * left + k.t0;
      break;
    } else {
      const int item = k.place * 8 + xcd;
      if (item >= left * nb) return false;
      t = item / nb;
      col = item - t * nb;
      t += k.t0;
      break;
    }
  }
  k.place += gridDim.x >> 3;
  int first, rows;
  if (DENSE) {
    g.e = first = 0;
    rows = m_rows;
  } else if (n_experts < 64) {
    g.e = __builtin_popcountll(__ballot(loff <= t)) - 1;
    first = __builtin_amdgcn_readlane(loff, g.e);
    rows = __builtin_amdgcn_readlane(lcnt, g.e);
  } else {
    g.e = gg_expert(tile_off, n_experts, t);
    first = tile_off[g.e];
    rows = counts[g.e];
  }
  g.n0 = col * BN;
  g.seg = (long)t * 256;
  g.live = rows - (t - first) * 256;
  return true;
}

// two floats to bf16 (round to nearest even), the first in the low half
typedef __bf16 gw_bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u32 gw_pack(float x, float y) {
  gw_bf16x2 p;
  p[0] = (__bf16)x;
  p[1] = (__bf16)y;
  return __builtin_bit_cast(u32, p);
}

// The gated unit of 8 sums at a time. Its operations run beside no products, with one
// wave a SIMD: a tile's 128 units a lane were a quarter of its time at a k of 1024. So
// each operation is issued for all 8 before the next, which waits for none of them
// then, and the quotient v / d is v times the reciprocal, corrected by its remainder: 10
// operations a unit instead of 15. 2 x 3072 x 1024 at 24,000 rows 260 -> 251 us, 2 x 8192 x
// 2048 at 32,768 1582 -> 1530, 2 x 12288 x 4096 4533 -> 4469, 32 experts of 2048 x 2048 at
// 4096 rows 1661 -> 1604, 187 rows 126.5 -> 123.3, in turn on one card, with 9. 1.3e9
// results were the same to the bit.
// d = 1 + exp(-v) passes 2^126 for v below -87.3, and its reciprocal, too small a number,
// is 0 then (-5e-37 for v = -88 was). So v and d are taken as quarters, which changes no
// other bit, but of v below 2^-124; it is the tenth operation (24,000 rows of k 1024 236.0
// us instead of 234.7, 32,768 of 2048 1523.5 and 1519.5, 2688 of 2 x 8064 x 320 35.8 and
// 34.5), but where the row's weight or the clamped up takes the quarter. GELU by tanh has
// long been 0 there.
template <int MODE>
__device__ __forceinline__ void gw_unit8(float (&v)[8], float (&u)[8], float limit,
                                         float rw) {
  float g[8], d[8], r[8], e[8];
  constexpr float Q = MODE == 6 ? 1.f : 0.25f;
#define GW_EACH(X)                                                          \
  _Pragma("unroll") for (int i = 0; i < 8; ++i) { X; }                      \
  __builtin_amdgcn_sched_barrier(0);
  if (MODE == 4) {
    GW_EACH(v[i] *= rw * Q)
    GW_EACH(u[i] *= rw)
  }
  if (MODE == 6) {     // 0.5 (1 + tanh z) = 1 / (1 + exp(-2 z))
    GW_EACH(d[i] = v[i] * v[i])
    GW_EACH(d[i] = fmaf(d[i], -2.302208198f * 0.044715f, -2.302208198f))
    GW_EACH(d[i] = d[i] * v[i])
  } else if (MODE == 3) {
    GW_EACH(v[i] = fminf(v[i], limit))
    GW_EACH(u[i] = fmaf(fminf(fmaxf(u[i], -limit), limit), Q, Q))   // (v stays)
    GW_EACH(d[i] = v[i] * -1.702f)
    GW_EACH(d[i] = d[i] * 1.4426950408889634f)
  } else {
    GW_EACH(d[i] = v[i] * (-1.4426950408889634f / (MODE == 4 ? Q : 1.f)))
  }
  if (MODE != 3 && MODE != 4 && MODE != 6) { GW_EACH(v[i] *= Q) }
  GW_EACH(d[i] = __builtin_amdgcn_exp2f(d[i]))
  GW_EACH(d[i] = fmaf(d[i], Q, Q))
  GW_EACH(r[i] = __builtin_amdgcn_rcpf(d[i]))
  GW_EACH(g[i] = v[i] * r[i])
  GW_EACH(e[i] = fmaf(-d[i], g[i], v[i]))
  GW_EACH(g[i] = fmaf(e[i], r[i], g[i]))
  GW_EACH(g[i] = __builtin_amdgcn_div_fixupf(g[i], d[i], v[i]))
  GW_EACH(v[i] = g[i] * u[i])
#undef GW_EACH
}

// Whether the last rows (4 or fewer) go to the XCDs by single tiles: where by column
// blocks some XCD needs a round more. 2656 rows of 2 x 5888 x 3904 (506 tiles, 66 of them
// on one XCD) 265 -> 189 us, 2 experts with 60 tiles in all 0.58 of the time. Where none
// does, runs of neighbouring tiles are up to 10 % slower (1012 rows of 2 x 8320 x 448 27.7
// and 29.9). The question itself is 0.5 % of 40 to 150 us.
__device__ __forceinline__ bool gw_even(int total, int nb) {
  const int left = total % (8 * GW_ROWS), e = nb & 7, y = threadIdx.x & 7;
  if (nb < 8 || !left) return false;
  const int groups = (left - 1) / GW_ROWS;
  int has = groups * (nb >> 3);
  for (int g = 0; g < groups; ++g) has += ((y + g * e) & 7) < e;
  const int old = has * GW_ROWS + (left - groups * GW_ROWS) *
                                      ((nb >> 3) + (((y + groups * e) & 7) < e));
  const int per = gridDim.x >> 3, before = total / (8 * GW_ROWS) * GW_ROWS * nb;
  const int rounds = (before + ((left * nb + 7) >> 3) + per - 1) / per;
  return __any(before + old > rounds * per);
}

// DENSE: see above. ANY: gathered rows of 4 GB or more in all, or operands that do
// not begin at multiples of 16 bytes; 64-bit addresses and narrow stores then.
template <int MODE, bool ANY>
__device__ __forceinline__ void gw_body(
    u16* __restrict__ out, const u16* __restrict__ a,
    const u16* __restrict__ w, const int* __restrict__ row_tok,
    const int* __restrict__ tile_off, const int* __restrict__ counts,
    int n_experts, int n_cols, long K, float limit,
    const float* __restrict__ row_w, int m_rows, const u16* __restrict__ bias,
    u16* __restrict__ rest, int n_rest, const GwHeads& H) {
  constexpr bool GATED = MODE == 1 || (MODE >= 3 && MODE < 7);
  constexpr bool DENSE = MODE >= 5, REST = MODE == 6, HEADS = MODE == 7;
  constexpr bool GATHER = MODE != 0 && !DENSE;
  constexpr int BN = GATED ? 128 : 256;   // output columns
  const int nb = n_cols / BN + (REST ? n_rest / 256 : 0);
  const int total = DENSE ? (m_rows + 255) / 256 : tile_off[n_experts];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 15, quad = lane >> 4;
  const int wm = wave >> 1, wn = wave & 1;
  extern __shared__ __attribute__((aligned(16))) char gw_smem[];

  const int loff =
      !DENSE && lane <= n_experts ? tile_off[lane] : 0x7fffffff;
  const int lcnt = !DENSE && lane < n_experts ? counts[lane] : 0;
  GwWalk walk = {0, (int)(blockIdx.x >> 3), gw_even(total, nb)};
  GwTile cur;
  auto next = [&](GwTile& g) {
    return gw_next<BN, DENSE>(walk, nb, total, n_experts, m_rows, loff, lcnt,
                              tile_off, counts, g);
  };
  if (!next(cur)) return;

  // copies: 1 KB (8 rows of 128 bytes) an instruction, pieces wave * 8 + j of
  // either operand; 16-byte chunks are XOR-swizzled by bits 1 to 3 of the row, so
  // that the 16 rows read in a cycle cover all 64 banks
  const int pr = lane >> 3;
  const int ch[2] = {((lane & 7) ^ (pr >> 1)) * 8,
                     ((lane & 7) ^ ((8 + pr) >> 1)) * 8};
  struct Source {
    __amdgpu_buffer_rsrc_t ra, rb;
    u32 va[ANY ? 1 : 8];
    const u16* pa[ANY ? 8 : 1];
    const u16* pb;
  };
  auto point = [&](const GwTile& g, Source& s) {
    const u16* base = GATHER ? a : a + g.seg * K;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = (wave * 8 + j) * 8 + pr;
      int row = DENSE ? min(r, g.live - 1) : r;
      if (GATHER)        // padding rows repeat the last (a tile may have none)
        row = max(row_tok[g.seg + min(r, max(g.live, 1) - 1)], 0);
      if (ANY)
        s.pa[ANY ? j : 0] = base + row * K + ch[j & 1];
      else
        s.va[ANY ? 0 : j] = (u32)row * (u32)(K * 2) + ch[j & 1] * 2;
    }
    const int br = wave * 64;                  // first of this wave's B rows
    long brow = (GATED && br >= 128) ? n_cols + g.n0 + br - 128 : g.n0 + br;
    if (REST && g.n0 >= n_cols) brow = 2 * g.n0 + br;   // 256 rows behind the up's
    s.pb = w + ((long)g.e * (GATED ? 2 : 1) * n_cols + brow) * K;
    s.ra = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0xffffffffu,
                                             0x00027000);
    s.rb = __builtin_amdgcn_make_buffer_rsrc((void*)s.pb, 0, 0xffffffffu,
                                             0x00027000);
  };
  const u32 vb[2] = {(u32)(pr * K + ch[0]), (u32)(pr * K + ch[1])};
  char* const mine = gw_smem + wave * 8192;
  Source src;
  auto copy_a = [&](int slot, int j, int k) {
    char* d = mine + slot + j * 1024;
    if (ANY)
      glds16g((const u32*)(src.pa[ANY ? j : 0] + k), (u32*)d);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          src.ra, (__attribute__((address_space(3))) void*)d, 16,
          src.va[ANY ? 0 : j], (u32)k * 2, 0, 0);
  };
  auto copy_b = [&](int slot, int j, int k) {
    char* d = mine + slot + j * 1024;
    if (ANY)
      glds16g((const u32*)(src.pb + k + j * 8 * K + vb[j & 1]), (u32*)d);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          src.rb, (__attribute__((address_space(3))) void*)d, 16,
          vb[j & 1] * 2, (u32)(k + j * 8 * K) * 2, 0, 0);
  };

  const int kad = ln * 128 + ((quad ^ ((ln >> 1) & 7)) << 4);
  const int arow = wm * 128 * 128;
  const int brow = wn * (GATED ? 64 : 128) * 128;
  f32x4 acc[8][8];                // gated: columns 0 to 3 gate, 4 to 7 up
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = (f32x4)(0.f);
  bf16x8 fa[2][8], fb[2][8];
  auto load_a = [&](int i, int slot, int kk) {
    fa[kk][i] = *(const bf16x8*)(gw_smem + slot + arow + i * 2048 +
                                 (kad ^ (kk << 6)));
  };
  auto load_b = [&](int j, int slot, int kk) {
    const int o = GATED ? (j >> 2) * 16384 + (j & 3) * 2048 : j * 2048;
    fb[kk][j] = *(const bf16x8*)(gw_smem + slot + brow + o + (kad ^ (kk << 6)));
  };
  auto wrap = [](int o) { return o >= GW_LDS ? o - GW_LDS : o; };

  // The sums are transposed (B rows first), so a lane has four columns of a row;
  // lanes of neighbouring column tiles swap halves: 16 bytes a lane and store.
  auto pack8 = [](const float (&x)[8]) {
    u32 p[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) p[q] = gw_pack(x[2 * q], x[2 * q + 1]);
    const auto s0 = __builtin_amdgcn_permlane16_swap(p[0], p[2], false, false);
    const auto s1 = __builtin_amdgcn_permlane16_swap(p[1], p[3], false, false);
    return u32x4{s0[0], s1[0], s0[1], s1[1]};
  };
  auto store_tile = [&](const GwTile& g) {
    const u32 off = (u32)(ln * n_cols + (quad & 1) * 16 + (quad >> 1) * 8) * 2;
    const long row = g.seg + wm * 128;
    char* at = (char*)(out + row * n_cols + g.n0 + wn * (GATED ? 64 : 128));
    const bool gate = !REST || g.n0 < n_cols;    // else plain sums, 256 columns
    u16x4 bs[REST ? 8 : 1];
    char* more = nullptr;
    if (REST) {
      const u16* bp = bias + (gate ? g.n0 : 2 * g.n0) + wn * 64 + quad * 4;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        bs[j] = bias ? *(const u16x4*)(bp + (j & 3) * 16 +
                                       (j < 4 ? 0 : gate ? n_cols : 128))
                     : (u16x4)(0);
      more = (char*)(rest + row * n_rest + 2 * (g.n0 - n_cols) + wn * 64 +
                     (long)ln * n_rest + (quad & 1) * 16 + (quad >> 1) * 8);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i, at += (long)n_cols * 32) {
      const float rw = MODE == 4 ? row_w[row + i * 16 + ln] : 1.f;
#pragma unroll
      for (int j = 0; j < (GATED ? 4 : 8); j += 2) {
        // the sums stay where the products left them until here: read all at
        // once they would need more registers than there are
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          asm volatile("" : "+a"(acc[i][j + q]));
          if (GATED) asm volatile("" : "+a"(acc[i][(j + q + 4) & 7]));
        }
        float x[8], up[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          x[q] = acc[i][j + (q >> 2)][q & 3];
          if (GATED) up[q] = acc[i][(j + (q >> 2) + 4) & 7][q & 3];
          else x[q] = gg_unit<MODE>(x[q], 0.f, limit, rw);
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {       // for the next tile
          acc[i][j + q] = (f32x4)(0.f);
          if (GATED) acc[i][(j + q + 4) & 7] = (f32x4)(0.f);
        }
        if (REST) {
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            x[q] += bf2f(bs[j + (q >> 2)][q & 3]);
            up[q] += bf2f(bs[j + 4 + (q >> 2)][q & 3]);
          }
          if (!gate) {
            u16* o = (u16*)(more + (long)i * n_rest * 32) + j * 16;
            const u32x4 pa = pack8(x), pb = pack8(up);
            if (wm * 128 + i * 16 + ln < g.live) {
              *(u32x4*)o = pa;
              *(u32x4*)(o + 128) = pb;
            }
            __builtin_amdgcn_sched_barrier(0);
            continue;
          }
        }
        if (GATED) gw_unit8<MODE>(x, up, limit, rw);
        const u32x4 pk = pack8(x);
        u16* o = (u16*)(at + off) + j * 16;
        if (DENSE && wm * 128 + i * 16 + ln >= g.live) {
        } else if (ANY) {
#pragma unroll
          for (int z = 0; z < 8; ++z)
            o[z] = (u16)(pk[z >> 1] >> ((z & 1) * 16));
        } else {
          *(u32x4*)o = pk;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  // Mode 7: a wave's 128 columns are one head, of which a lane has 32 columns of a row
  // and the lanes of equal ln the others: RMS norm (sums in registers and across four
  // lanes), rotation (columns d and d + 64 in the same lane) and the store to the
  // queries or to the token's slot, on fp32 products. By itself that pass reads and
  // writes all heads once more, at the rate of memory (78 us for 24,000 tokens of 32
  // heads, with the library's product of k 1024 267; here 198, of which 165 are the
  // product's; 32,768 of 24 heads, k 2048 383 -> 340; of 48, k 4096 1245 -> 1222).
  // Positions and slots of all rows are asked for first and each row's cosines while
  // the row before is computed, as no other wave hides them.
  auto store_heads = [&](const GwTile& g, auto plain_c) {
    constexpr bool PLAIN = decltype(plain_c)::v;
    const int hd = (g.n0 >> 7) + wn;
    const bool isq = hd < H.hq;
    const int kh = hd - H.hq - (PLAIN ? H.hk : 0);
    const long row0 = g.seg + wm * 128;
    const int live = g.live - wm * 128;     // of this wave's rows
    u32 pos[PLAIN ? 1 : 8], slot[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      // (a wave may have no live row: then the tile's last)
      const long row = g.seg + min(wm * 128 + i * 16 + ln, g.live - 1);
      if (!PLAIN) pos[PLAIN ? 0 : i] = (u32)H.pos[row];
      slot[i] = isq ? 0 : (u32)H.slots[row];
    }
    u16x4 nw[PLAIN ? 1 : 8];
    f32x4 cs[4], sn[4];
    const u16* wv = isq ? H.qw : H.kw;
    auto turn = [&](int i, int j) {
      const float* t = H.cos_sin + (long)pos[PLAIN ? 0 : i] * 128 + j * 16 + quad * 4;
      cs[j] = *(const f32x4*)t;
      sn[j] = *(const f32x4*)(t + 64);
    };
    if (!PLAIN) {
#pragma unroll
      for (int j = 0; j < 4; ++j) turn(0, j);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        nw[PLAIN ? 0 : j] =
            wv ? *(const u16x4*)(wv + j * 16 + quad * 4) : (u16x4)(0x3f80);
    }
    const int off = (quad & 1) * 16 + (quad >> 1) * 8;
    u16* const to = !PLAIN && isq ? out : PLAIN ? H.vc : H.kc;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float x[8][4];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        asm volatile("" : "+a"(acc[i][j]));
#pragma unroll
        for (int e = 0; e < 4; ++e) x[j][e] = acc[i][j][e];
        acc[i][j] = (f32x4)(0.f);
      }
      const u32 page = (slot[i] >> H.shift) * H.hk + kh;
      long at = (((long)page << H.shift) + (slot[i] & ((1u << H.shift) - 1))) * 128;
      if (!PLAIN && isq) at = ((row0 + i * 16 + ln) * H.hq + hd) * 128;
      at += off;
      float inv = 1.f;
      if (!PLAIN) {
        float q[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j] = x[j][0] * x[j][0];
#pragma unroll
        for (int e = 1; e < 4; ++e)
#pragma unroll
          for (int j = 0; j < 8; ++j) q[j] = fmaf(x[j][e], x[j][e], q[j]);
        const float sum =
            ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
        const u32 b = __float_as_uint(sum);
        const auto h = __builtin_amdgcn_permlane32_swap(b, b, false, false);
        const u32 c =
            __float_as_uint(__uint_as_float(h[0]) + __uint_as_float(h[1]));
        const auto f = __builtin_amdgcn_permlane16_swap(c, c, false, false);
        inv = rsqrtf((__uint_as_float(f[0]) + __uint_as_float(f[1])) * (1.f / 128) +
                     H.eps);
        if (!wv) inv = 1.f;
      }
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        float lo[8], hi[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const int t = j + (q >> 2), e = q & 3;
          lo[q] = x[t][e];
          hi[q] = x[t + 4][e];
          if (!PLAIN) {
            const float a = lo[q] * (inv * bf2f(nw[PLAIN ? 0 : t][e]));
            const float b = hi[q] * (inv * bf2f(nw[PLAIN ? 0 : t + 4][e]));
            lo[q] = a * cs[t][e] - b * sn[t][e];
            hi[q] = b * cs[t][e] + a * sn[t][e];
          }
        }
        if (!PLAIN && i < 7) {
          turn(i + 1, j);
          turn(i + 1, j + 1);
        }
        const u32x4 first = pack8(lo), second = pack8(hi);
        if (i * 16 + ln < live) {
          *(u32x4*)(to + at + j * 16) = first;
          *(u32x4*)(to + at + j * 16 + 64) = second;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  auto finish = [&](const GwTile& g) {
    if constexpr (HEADS) {
      if ((g.n0 >> 7) + wn >= H.hq + H.hk) store_heads(g, GwFlag<1>{});
      else store_heads(g, GwFlag<0>{});
    } else {
      store_tile(g);
    }
  };

  int sa = 0;   // LDS offset of the step's A rows; its B rows are one unit further
  // AHEAD: copies of A and B two steps on, at k2 of the source. MORE: another step
  // follows, whose operands are read at the end.
  auto step = [&](int k2, auto ahead_c, auto more_c) {
    constexpr bool AHEAD = decltype(ahead_c)::v, MORE = decltype(more_c)::v;
    const int sb = wrap(sa + GW_UNIT), na = wrap(sa + 2 * GW_UNIT),
              nbs = wrap(sa + 3 * GW_UNIT), ca = wrap(sa + 4 * GW_UNIT);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      if (kk == 1 && MORE) {
        // All reads of this step are done and the next step's operands are there
        // (behind them only the A rows of two steps on), for all four waves:
        // copies may overwrite this step's, reads may go on to the next one's.
        __builtin_amdgcn_sched_barrier(0);
        if (AHEAD)
          asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
        else
          asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int x = 0; x < 64; ++x) {
        // In squares of squares, one operand of two new at a product: what changes
        // at the matrix core's inputs is part of the power that sets the clock. Row
        // by row (the same sums): 2 x 12288 x 4096 at 32,768 rows 4458 -> 4355 us, 2
        // x 8192 x 2048 1532 -> 1512, 2 x 3072 x 1024 at 24,000 240 -> 238; with
        // zeros in all operands, far from the limit, 3572 and 3572. By columns 4421,
        // rows and columns there and back 4368 and 4376. Heads take rows there and
        // back: in squares their step has 180 moves between the sums' registers.
        const int i = HEADS ? x >> 3
                            : (x >> 1 & 1) | (x >> 3 & 1) << 1 | (x >> 5) << 2;
        const int j = HEADS ? (x & 7) ^ (x >> 3 & 1 ? 7 : 0)
                            : ((x ^ x >> 1) & 1) | (x >> 2 & 1) << 1 | (x >> 4 & 1) << 2;
        acc[i][j] = mfma16g(fb[kk][j], fa[kk][i], acc[i][j]);
        // reads behind every third product, copies behind every eighth: the LDS
        // takes both beside each other, and the cache the copies of four waves
        // (eight within the first half: down of 32 experts at 4096 rows 4 % more)
        if (x % 3 == 0 && x / 3 < 16 && (kk == 0 || MORE)) {
          const int y = x / 3;
          if (y < 8) load_b(y, kk ? nbs : sb, kk ^ 1);
          else load_a(y - 8, kk ? na : sa, kk ^ 1);
        }
        if (AHEAD && x % 8 == 1) {
          if (kk == 0) copy_a(ca, x / 8, k2);
          else copy_b(sa, x / 8, k2);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    sa = na;
  };
  // The sums in the accumulation registers wherever steps meet: with some of them
  // in the others a step has a move for every second product.
  auto keep = [&]() {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) asm volatile("" : "+a"(acc[i][j]));
  };
  constexpr GwFlag<0> no{};
  constexpr GwFlag<1> yes{};

  const int KT = (int)(K >> 6);
  const int lead = min(KT, 2);
  // Experts start at different eighths of k where rows are multiples of 4 KB long
  // (see the kernel above): gate and up / down of 32 experts of 2048 x 2048 at 187
  // rows 151 / 81 -> 129 / 67 us, at 375 rows 251 / 120 -> 224 / 117, at 4096 rows
  // 1634 / 844 and 1637 / 850. The tile's rows have no part in it: the dispatch puts
  // a token where its counter happens to stand, and the token's sums have to come
  // out the same in every place. By column blocks as well, which takes workgroups of
  // an XCD out of step: 144 / 85, 233 / 125, 1704 / 842. One matrix (DENSE) has one
  // start, 0 (whole prompts were 0 to 1.5 % faster with one for each XCD, but equal
  // rows of a batch differed).
  auto first = [&](const GwTile& g) {
    return !DENSE && K % 2048 == 0 ? (g.e * 5 & 7) * KT / 8 * 64 : 0;
  };
  int kc = first(cur);
  auto advance = [&]() {
    kc += 64;
    if (kc == (int)K) kc = 0;
  };
  // the first two steps of a tile, and the operands of its first products
  auto open = [&]() {
    for (int s = 0; s < lead; ++s) {
#pragma unroll
      for (int j = 0; j < 8; ++j) copy_a(2 * s * GW_UNIT, j, kc);
#pragma unroll
      for (int j = 0; j < 8; ++j) copy_b((2 * s + 1) * GW_UNIT, j, kc);
      advance();
    }
    if (lead == 2)
      asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    sa = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      load_b(j, GW_UNIT, 0);
      load_a(j, 0, 0);
    }
  };

  point(cur, src);
  if (!HEADS && KT < 3) {       // too short to run across tiles
    for (;;) {
      open();
      if (KT == 2) {
        step(0, no, yes);
        step(0, no, no);
      } else {
        step(0, no, no);
      }
      finish(cur);
      if (!next(cur)) return;
      point(cur, src);
      kc = first(cur);
      __syncthreads();        // the reads of this tile's operands are done
    }
  }
  open();
  for (;;) {
    GwTile nxt;
    Source after;
    const bool more = next(nxt);
    if (more) point(nxt, after);
    const int last = more ? KT : KT - 2;
    keep();
    for (int s = 0; s < last; ++s) {
      if (s == KT - 2) {      // the copies are the next tile's now
        src = after;
        kc = first(nxt);
      }
      step(kc, yes, yes);
      keep();
      advance();
    }
    if (!more) {
      step(0, no, yes);
      step(0, no, no);
    }
    finish(cur);
    if (!more) return;
    cur = nxt;
  }
}

template <int MODE, bool ANY>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
gw_kernel(u16* __restrict__ out, const u16* __restrict__ a,
          const u16* __restrict__ w, const int* __restrict__ row_tok,
          const int* __restrict__ tile_off, const int* __restrict__ counts,
          int n_experts, int n_cols, long K, float limit,
          const float* __restrict__ row_w, int m_rows,
          const u16* __restrict__ bias, u16* __restrict__ rest, int n_rest,
          GwHeads heads) {
  gw_body<MODE, ANY>(out, a, w, row_tok, tile_off, counts, n_experts, n_cols, K,
                     limit, row_w, m_rows, bias, rest, n_rest, heads);
}

// a workgroup a CU, a multiple of 8 of them
static unsigned gw_grid(long tiles, int blocks) {
  const long work = (tiles * blocks + 7) / 8 * 8;
  return (unsigned)(work < GW_CUS ? work : GW_CUS);
}

static void grouped_gemm_launch(void* out, const void* a, long a_rows,
                                const void* w,
                                const int* row_tok, const int* tile_off,
                                const int* counts, int n_experts,
                                int max_tiles, int n_cols, long K,
                                int gate_silu, int bm, float limit,
                                const float* row_w, hipStream_t stream) {
  if (max_tiles == 0) return;
#define GG_LAUNCH(GS, BM, BN, WR, WC)                                       \
  {                                                                         \
    dim3 grid((unsigned)max_tiles, (unsigned)(n_cols / BN)),                \
        block(WR* WC * 64);                                                 \
    hipLaunchKernelGGL((grouped_gemm_kernel<GS, BM, BN, WR, WC>), grid,     \
                       block, 0, stream, (u16*)out, (const u16*)a,          \
                       (const u16*)w, row_tok, tile_off, counts, n_experts, \
                       n_cols, K, limit, row_w);                            \
    return;                                                                 \
  }
#define GG_MODES(CALL)                                                      \
  {                                                                         \
    if (gate_silu == 1) CALL(1)                                             \
    else if (gate_silu == 3) CALL(3)                                        \
    else if (gate_silu == 4) CALL(4)                                        \
    else if (gate_silu == 2) CALL(2)                                        \
    else CALL(0)                                                            \
  }
#define GG_ARGS                                                             \
  (u16*)out, (const u16*)a, (const u16*)w, row_tok, tile_off, counts,       \
      n_experts, n_cols, K, limit, row_w
  const bool gated = gate_silu == 1 || gate_silu >= 3;
  if (bm == 256) {
    const dim3 grid(gw_grid(max_tiles, n_cols / (gated ? 128 : 256)));
    const bool any = (gate_silu && a_rows >= (0xf0000000l / 2) / K) ||
                     (((size_t)out | (size_t)a | (size_t)w) & 15);
#define GG_WIDE_AS(M, ANY)                                                  \
  {                                                                         \
    static std::atomic<unsigned long long> asked{0};                        \
    lds_limit((const void*)gw_kernel<M, ANY>, GW_LDS, asked);               \
    hipLaunchKernelGGL((gw_kernel<M, ANY>), grid, dim3(256), GW_LDS,        \
                       stream, GG_ARGS, 0, nullptr, nullptr, 0, GwHeads{});  \
  }
#define GG_WIDE(M)                                                          \
  {                                                                         \
    if (any) GG_WIDE_AS(M, true)                                            \
    else GG_WIDE_AS(M, false)                                               \
  }
    GG_MODES(GG_WIDE)
    return;
  }
  /* no hipGetLastError in this launcher: error-state queries are rejected
     while a stream is capturing (decode steps replay under hipGraphs) */
  if (bm == 128 && n_cols % 128 == 0) {
    if (gate_silu == 1) GG_LAUNCH(1, 128, 128, 2, 4)
    else if (gate_silu == 3) GG_LAUNCH(3, 128, 128, 2, 4)
    else if (gate_silu == 4) GG_LAUNCH(4, 128, 128, 2, 4)
    else if (gate_silu == 2) GG_LAUNCH(2, 128, 128, 2, 4)
    else GG_LAUNCH(0, 128, 128, 2, 4)
  }
  if (bm == 128) {
    if (gate_silu == 1) GG_LAUNCH(1, 128, 64, 4, 2)
    else if (gate_silu == 3) GG_LAUNCH(3, 128, 64, 4, 2)
    else if (gate_silu == 4) GG_LAUNCH(4, 128, 64, 4, 2)
    else if (gate_silu == 2) GG_LAUNCH(2, 128, 64, 4, 2)
    else GG_LAUNCH(0, 128, 64, 4, 2)
  }
  if (bm == 32) {
    if (gate_silu == 1) GG_LAUNCH(1, 32, 64, 2, 2)
    else if (gate_silu == 3) GG_LAUNCH(3, 32, 64, 2, 2)
    else if (gate_silu == 4) GG_LAUNCH(4, 32, 64, 2, 2)
    else if (gate_silu == 2) GG_LAUNCH(2, 32, 64, 2, 2)
    else GG_LAUNCH(0, 32, 64, 2, 2)
  }
  if (gate_silu == 1) GG_LAUNCH(1, 64, 64, 2, 2)
  else if (gate_silu == 3) GG_LAUNCH(3, 64, 64, 2, 2)
  else if (gate_silu == 4) GG_LAUNCH(4, 64, 64, 2, 2)
  else if (gate_silu == 2) GG_LAUNCH(2, 64, 64, 2, 2)
  else GG_LAUNCH(0, 64, 64, 2, 2)
#undef GG_LAUNCH
}

template <int MODE>
static void gw_dense(void* out, void* rest, const void* x, const void* w,
                     const void* bias, int M, int N, int n_rest, long K,
                     hipStream_t stream, const GwHeads& heads = GwHeads{}) {
  const int blocks = N / (MODE == 7 ? 256 : 128) + n_rest / 256;
  static std::atomic<unsigned long long> asked{0};
  lds_limit((const void*)gw_kernel<MODE, false>, GW_LDS, asked);
  hipLaunchKernelGGL((gw_kernel<MODE, false>),
                     dim3(gw_grid(((long)M + 255) / 256, blocks)),
                     dim3(256), GW_LDS, stream, (u16*)out, (const u16*)x,
                     (const u16*)w, nullptr, nullptr, nullptr, 0, N, K, 0.f,
                     nullptr, M, (const u16*)bias, (u16*)rest, n_rest, heads);
}

// out [M, N] = silu(x Wg^T) * (x Wu^T): w [2 N, K], the gate's rows first. x and w at
// multiples of 16 bytes, K a multiple of 64 and below 2^21 (a tile's offsets are of 32
// bits, where it begins of 64), N a multiple of 128.
extern "C" void sutro_linear_silu_mul(void* out, const void* x, const void* w,
                                      int M, int N, long K,
                                      hipStream_t stream) {
  gw_dense<5>(out, nullptr, x, w, nullptr, M, N, 0, K, stream);
}

// The same with GELU by tanh, a bias (null or at multiples of 8 bytes) and more columns
// behind them: rest [M, n_rest] = x Wr^T, w [2 N + n_rest, K], n_rest a multiple of 256.
extern "C" void sutro_linear_gelu_mul(void* out, void* rest, const void* x,
                                      const void* w, const void* bias, int M, int N,
                                      int n_rest, long K, hipStream_t stream) {
  gw_dense<6>(out, rest, x, w, bias, M, N, n_rest, K, stream);
}

// x w^T as heads of 128, w [(hq + 2 hk) 128, K] with hq even: query heads normed and
// rotated to q [M, hq, 128], key heads likewise and value heads as they are to their
// tokens' slots in pages of 1 << shift tokens, bf16. Operands at multiples of
// 16 bytes, K as above and 192 or more.
extern "C" void sutro_linear_heads(void* q, void* kc, void* vc, const void* x,
                                   const void* w, const long* pos, const long* slots,
                                   const float* cos_sin, const void* qw,
                                   const void* kw, float eps, int M, int hq, int hk,
                                   int shift, long K, hipStream_t stream) {
  const GwHeads heads = {(u16*)kc, (u16*)vc, pos, slots, cos_sin, (const u16*)qw,
                         (const u16*)kw, eps, hq, hk, shift};
  gw_dense<7>(q, nullptr, x, w, nullptr, M, (hq + 2 * hk) * 128, 0, K, stream, heads);
}

extern "C" void sutro_grouped_gemm(void* out, const void* a, long a_rows,
                                   const void* w, const int* row_tok, const int* tile_off,
                                   const int* counts, int n_experts,
                                   int max_tiles, int n_cols, long K,
                                   int gate_silu, int bm,
                                   hipStream_t stream) {
  grouped_gemm_launch(out, a, a_rows, w, row_tok, tile_off, counts, n_experts,
                      max_tiles, n_cols, K, gate_silu, bm, 0.f, nullptr,
                      stream);
}

// the clamped gated unit (mode 3) with its limit
extern "C" void sutro_grouped_gemm_glu(void* out, const void* a, long a_rows,
                                       const void* w, const int* row_tok, const int* tile_off,
                                       const int* counts, int n_experts,
                                       int max_tiles, int n_cols, long K,
                                       int bm, float limit,
                                       hipStream_t stream) {
  grouped_gemm_launch(out, a, a_rows, w, row_tok, tile_off, counts, n_experts,
                      max_tiles, n_cols, K, 3, bm, limit, nullptr, stream);
}

// the silu unit over weighted rows (mode 4)
extern "C" void sutro_grouped_gemm_weighted(
    void* out, const void* a, long a_rows, const void* w, const int* row_tok,
    const int* tile_off, const int* counts, int n_experts, int max_tiles,
    int n_cols, long K, int bm, const float* row_w, hipStream_t stream) {
  grouped_gemm_launch(out, a, a_rows, w, row_tok, tile_off, counts, n_experts,
                      max_tiles, n_cols, K, 4, bm, 0.f, row_w, stream);
}

// ---- fused MoE combine: out[t] = sum_j w[t,j] * rows[padpos[t,j]] ----
// One thread per (token, 8-element h-chunk); k reads + 1 write per thread,
// f32 accumulate, bf16 store. In the int32 layout pairs of weight 0 (experts of
// another rank) have no row to read.
template <typename P>
__global__ void __launch_bounds__(256) moe_combine_kernel(
    u16* __restrict__ out,          // [T, h] bf16
    const u16* __restrict__ rows,   // [rows_max, h] bf16
    const P* __restrict__ padpos,   // [T, k]
    const float* __restrict__ w,    // [T, k]
    int T, int h, int k) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long chunks = (long)h / 8;
  if (idx >= (long)T * chunks) return;
  const int t = (int)(idx / chunks);
  const int h0 = (int)(idx % chunks) * 8;
  float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int j = 0; j < k; ++j) {
    const float wj = w[(long)t * k + j];
    if (sizeof(P) == 4 && wj == 0.f) continue;
    const long r = padpos[(long)t * k + j];
    const u16x8 v = *(const u16x8*)(rows + r * h + h0);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += wj * bf2f(v[e]);
  }
  u16x8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = f2bf(acc[e]);
  *(u16x8*)(out + (long)t * h + h0) = o;
}

extern "C" void sutro_moe_combine(void* out, const void* rows,
                                  const void* padpos, int pos64, const float* w,
                                  int T, int h, int k, hipStream_t stream) {
  const long total = (long)T * (h / 8);
  if (total == 0) return;
  const long blocks = (total + 255) / 256;
  // no hipGetLastError here: error-state queries are rejected while a
  // stream is capturing (decode steps replay this inside hipGraphs)
  if (pos64)
    hipLaunchKernelGGL(moe_combine_kernel<long>, dim3((unsigned)blocks),
                       dim3(256), 0, stream, (u16*)out, (const u16*)rows,
                       (const long*)padpos, w, T, h, k);
  else
    hipLaunchKernelGGL(moe_combine_kernel<int>, dim3((unsigned)blocks),
                       dim3(256), 0, stream, (u16*)out, (const u16*)rows,
                       (const int*)padpos, w, T, h, k);
}
