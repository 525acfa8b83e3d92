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
template <int ROWS, int WAVES, bool GATHER>
__device__ __forceinline__ void gg_stage(
    u16* lds, const u16* gsrc, long row_stride_b, const int* row_tok,
    int m0, int rows_valid, int wave, int lane) {
  constexpr int CH = ROWS / (8 * WAVES);
  static_assert(CH >= 1, "tile too small for wave count");
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int c = wave * CH + j;
    const u32 b = (u32)c * 1024u + (u32)lane * 16u;  // lane-linear LDS byte
    const u32 lb = gswz(b);                          // pre-swizzled source
    int row = (int)(lb >> 7);
    long grow;
    if (GATHER) {
      int r = m0 + row;
      int tok = (row < rows_valid) ? row_tok[r] : 0;
      if (tok < 0) tok = 0;  // padding: deterministic garbage, discarded
      grow = (long)tok;
    } else {
      grow = (long)(m0 + min(row, rows_valid - 1));
    }
    glds16g((const u32*)((const char*)gsrc + grow * row_stride_b + (lb & 127u)),
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
  if (MODE == 1 || MODE == 4) return v / (1.0f + __expf(-v)) * u;
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

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave / WCOLS, wn = wave % WCOLS;

  __shared__ u16 smem[2][(BM + (GATED ? 2 : 1) * BN) * 64];
  const int b_off = BM * 64;
  const int b2_off = (BM + BN) * 64;

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

  // prologue
  if (GATHER)
    gg_stage<BM, WAVES, true>(smem[0], aa, Kb, rt, m0, rows_valid, wave, lane);
  else
    gg_stage<BM, WAVES, false>(smem[0], aa, Kb, nullptr, m0, BM, wave, lane);
  gg_stage<BN, WAVES, false>(smem[0] + b_off, wg, Kb, nullptr, 0, BN, wave,
                             lane);
  if (GATED)
    gg_stage<BN, WAVES, false>(smem[0] + b2_off, wu, Kb, nullptr, 0, BN, wave,
                               lane);
  __syncthreads();

  const int KT = (int)(K >> 6);
  for (int kt = 0; kt < KT; ++kt) {
    const int p = kt & 1;
    u16* aT = smem[p];
    u16* bgT = smem[p] + b_off;
    u16* buT = smem[p] + b2_off;
    if (kt + 1 < KT) {
      const long ko = (long)(kt + 1) * 64;
      if (GATHER)
        gg_stage<BM, WAVES, true>(smem[p ^ 1], aa + ko, Kb, rt, m0,
                                  rows_valid, wave, lane);
      else
        gg_stage<BM, WAVES, false>(smem[p ^ 1], aa + ko, Kb, nullptr, m0, BM,
                                   wave, lane);
      gg_stage<BN, WAVES, false>(smem[p ^ 1] + b_off, wg + ko, Kb, nullptr, 0,
                                 BN, wave, lane);
      if (GATED)
        gg_stage<BN, WAVES, false>(smem[p ^ 1] + b2_off, wu + ko, Kb, nullptr,
                                   0, BN, wave, lane);
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
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      const int gn = n0 + wn * WN + j * 16 + dcol;
      const int grow0 = wm * WM + i * 16 + drow;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int grow = grow0 + r;
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
// 256 rows x 256 weight rows (gated: 128 gate and 128 up rows) a workgroup, 8
// waves as 2 x 4, each 128 x 64 on mfma_f32_32x32x16_bf16; 64 of k a step, both
// operands copied straight into a double-buffered LDS tile (128 KB), one
// barrier a step. Bound by LDS reads and the products together: a wave reads
// 24 KB a step for 1.05 MFLOP, half of what the 64 x 32 wave tiles of the
// 128-row kernel need. At 32 experts of 2048 x 2048, gate and up / down:
// 4096 rows an expert 3187 / 2188 -> 2081 / 1086 us (690 / 502 -> 1057 / 1013
// TFLOP/s), 375 rows 422 / 249 -> 277 / 145, 187 rows 224 / 163 -> 154 / 89,
// 96 rows 142 / 67 -> 154 / 89 (the padding: the other kernel's).
//
// Row tables are looked up once, not every step. Workgroup id i runs on XCD
// i % 8: an XCD takes four neighbouring row tiles and goes through all column
// blocks with them, so what its L2 holds is used by many workgroups at a time.
#define GW_ROWS 4
template <int MODE>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
gg_wide_kernel(u16* __restrict__ out, const u16* __restrict__ a,
               const u16* __restrict__ w, const int* __restrict__ row_tok,
               const int* __restrict__ tile_off, const int* __restrict__ counts,
               int n_experts, int n_cols, long K, float limit,
               const float* __restrict__ row_w) {
  constexpr bool GATED = MODE == 1 || MODE >= 3;
  constexpr bool GATHER = MODE != 0;
  constexpr int BN = GATED ? 128 : 256;   // output columns
  constexpr int TILE = 256 * 128;         // bytes of an operand tile
  const int nb = n_cols / BN;
  const int xcd = blockIdx.x & 7, j8 = blockIdx.x >> 3;
  const int r8 = j8 % (GW_ROWS * nb);
  const int t = ((j8 / (GW_ROWS * nb)) * 8 + xcd) * GW_ROWS + r8 % GW_ROWS;
  const int n0 = r8 / GW_ROWS * BN;
  if (t >= tile_off[n_experts]) return;
  const int e = gg_expert(tile_off, n_experts, t);
  const int m0 = (t - tile_off[e]) * 256;
  const long seg = (long)tile_off[e] * 256 + m0;   // first row of the tile
  const int live = counts[e] - m0;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 31, hi = lane >> 5;
  const int wm = wave >> 2, wn = wave & 3;
  extern __shared__ __attribute__((aligned(16))) char gw_smem[];

  // copies: 1 KB (8 rows of 128 bytes) an instruction, pieces wave*4 + j of
  // either operand; 16-byte chunks are XOR-swizzled by bits 1 to 3 of the row, so
  // that the 16 rows read in a cycle cover all 64 banks (by bits 0 to 2, eight of
  // them did: down product at 4096 rows an expert 1089 -> 1058 us, the gated one
  // 2155 -> 2125)
  const int pr = lane >> 3;
  const u16* pa[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = (wave * 4 + j) * 8 + pr;
    long row;
    if (GATHER) {
      row = row_tok[seg + min(r, live - 1)];   // padding rows repeat the last
      if (row < 0) row = 0;
    } else {
      row = seg + r;
    }
    pa[j] = a + row * K + ((lane & 7) ^ (((j & 1) * 8 + pr) >> 1)) * 8;
  }
  const int br = wave * 32;                    // first of this wave's B rows
  const long brow = (GATED && br >= 128) ? n_cols + n0 + br - 128 : n0 + br;
  const u16* pb = w + ((long)e * (GATED ? 2 : 1) * n_cols + brow) * K;
  const u32 boff[2] = {(u32)(pr * K + ((lane & 7) ^ (pr >> 1)) * 8),
                       (u32)(pr * K + ((lane & 7) ^ ((8 + pr) >> 1)) * 8)};
  auto stage = [&](int buf, long k) {
    char* dst = gw_smem + buf * 2 * TILE + wave * 4096;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      glds16g((const u32*)(pa[j] + k), (u32*)(dst + j * 1024));
#pragma unroll
    for (int j = 0; j < 4; ++j)
      glds16g((const u32*)(pb + k + j * 8 * K + boff[j & 1]),
              (u32*)(dst + TILE + j * 1024));
  };

  int kad[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
    kad[kk] = ln * 128 + (((kk * 2 + hi) ^ ((ln >> 1) & 7)) << 4);
  const int arow = wm * 128 * 128;
  const int brow0 = (GATED ? wn * 32 : wn * 64) * 128 + TILE;
  const int brow1 = (GATED ? 128 + wn * 32 : wn * 64 + 32) * 128 + TILE;

  f32x16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (f32x16)(0.f);

  const int KT = (int)(K >> 6);
  stage(0, 0);
  for (int kt = 0; kt < KT; ++kt) {
    __syncthreads();
    if (kt + 1 < KT) stage((kt + 1) & 1, (long)(kt + 1) * 64);
    const char* at = gw_smem + (kt & 1) * 2 * TILE;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const bf16x8 b0 = *(const bf16x8*)(at + brow0 + kad[kk]);
      const bf16x8 b1 = *(const bf16x8*)(at + brow1 + kad[kk]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bf16x8 af = *(const bf16x8*)(at + arow + i * 4096 + kad[kk]);
        acc[i][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, b0, acc[i][0],
                                                            0, 0, 0);
        acc[i][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, b1, acc[i][1],
                                                            0, 0, 0);
      }
    }
    // ten fragments ahead of the products, then one behind each
    __builtin_amdgcn_sched_group_barrier(0x100, 10, 0);
#pragma unroll
    for (int i = 0; i < 14; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x8, 18, 0);
  }

#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const long row =
          seg + wm * 128 + i * 32 + (r & 3) + 8 * (r >> 2) + 4 * hi;
      u16* o = out + row * n_cols + n0;
      const float rw = MODE == 4 ? row_w[row] : 1.f;
      if (GATED) {
        o[wn * 32 + ln] = f2bf(
            gg_unit<MODE>(acc[i][0][r], acc[i][1][r], limit, rw));
      } else {
        o[wn * 64 + ln] = f2bf(gg_unit<MODE>(acc[i][0][r], 0.f, limit, rw));
        o[wn * 64 + 32 + ln] =
            f2bf(gg_unit<MODE>(acc[i][1][r], 0.f, limit, rw));
      }
    }
}

static void grouped_gemm_launch(void* out, const void* a, const void* w,
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
    const int nb = n_cols / (gated ? 128 : 256);
    const unsigned groups = (unsigned)((max_tiles + 8 * GW_ROWS - 1) /
                                       (8 * GW_ROWS));
    const dim3 grid(groups * 8 * GW_ROWS * nb);
#define GG_WIDE(M)                                                          \
  {                                                                         \
    static std::atomic<unsigned long long> asked{0};                        \
    lds_limit((const void*)gg_wide_kernel<M>, 4 * 256 * 128, asked);        \
    hipLaunchKernelGGL(gg_wide_kernel<M>, grid, dim3(512), 4 * 256 * 128,   \
                       stream, GG_ARGS);                                    \
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

extern "C" void sutro_grouped_gemm(void* out, const void* a, const void* w,
                                   const int* row_tok, const int* tile_off,
                                   const int* counts, int n_experts,
                                   int max_tiles, int n_cols, long K,
                                   int gate_silu, int bm,
                                   hipStream_t stream) {
  grouped_gemm_launch(out, a, w, row_tok, tile_off, counts, n_experts,
                      max_tiles, n_cols, K, gate_silu, bm, 0.f, nullptr,
                      stream);
}

// the clamped gated unit (mode 3) with its limit
extern "C" void sutro_grouped_gemm_glu(void* out, const void* a, const void* w,
                                       const int* row_tok, const int* tile_off,
                                       const int* counts, int n_experts,
                                       int max_tiles, int n_cols, long K,
                                       int bm, float limit,
                                       hipStream_t stream) {
  grouped_gemm_launch(out, a, w, row_tok, tile_off, counts, n_experts,
                      max_tiles, n_cols, K, 3, bm, limit, nullptr, stream);
}

// the silu unit over weighted rows (mode 4)
extern "C" void sutro_grouped_gemm_weighted(
    void* out, const void* a, const void* w, const int* row_tok,
    const int* tile_off, const int* counts, int n_experts, int max_tiles,
    int n_cols, long K, int bm, const float* row_w, hipStream_t stream) {
  grouped_gemm_launch(out, a, w, row_tok, tile_off, counts, n_experts,
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
