// Linear layers over 2 to 256 rows, out = x w^T (+ bias) or silu(x Wg^T) (x Wu^T), bf16
// with fp32 sums: decode steps of a batch, short prompts.
//
// Weights are read once, rows are few, so what counts is that every CU has a share of the
// weights and keeps copies on their way. One tile of the result a workgroup, the whole of
// k for it; copies go straight to LDS (buffer loads, 16 bytes a lane) into a ring of ST
// steps of BK, the next steps' on their way while one is multiplied; one barrier a step.
// KG groups of four waves share a step's k (their sums meet in LDS at the end), because
// a step of 64 x 16 or 32 x 32 is a chain of waits, not of work.
//
// Tiles: the smallest of which 256 or fewer fill the result (mid_pick), so that one round
// of the chip does it. Of larger tiles fewer bytes go from L2 to LDS (a CU takes some 28
// bytes a cycle: 64 x 64 of 256 x 4096 x 12288 are 3.1 MB a CU and 58 us), smaller ones
// leave fewer CUs idle. In a graph, weights from memory, us of the library or the
// kernel for few rows before and of this one:
//   rows of w x K     M = 2           7             16            64            128          256
//   2048 x 2048       5.6 / -         5.9 / -       6.7 /  6.0    9.5 /  6.7    9.2 /  6.9  10.3 /  8.0
//   6144 x 2048       8.5 /  6.9      8.1 /  6.9    8.7 /  6.9   10.5 /  8.4   13.3 / 10.0  24.5 / 16.0
//   8192 x 2048      11.7 /  9.6      9.6 /  9.5   10.5 /  9.7   15.0 / 11.1   17.0 / 13.5  25.4 / 17.5
//   32768 x 2048     31.5 / 25.6     32.4 / 25.7   34.3 / 25.9   37.1 / 27.6   39.1 / 31.8  43.7 / -
//   6144 x 4096      13.4 / 11.6     14.3 / 11.8   14.8 / 12.1   18.3 / 17.0   25.9 / 22.1  40.4 / 28.9
//   4096 x 4096      10.4 / 10.1     10.6 / -      12.6 / 11.2   15.5 / 13.1   24.7 / 15.9  23.0 / 20.8
//   32768 x 4096     53.5 / 45.5     56.3 / 44.9   60.6 / 44.9   62.0 / 46.5   64.2 / 55.5  76.1 / -
// and with silu_mul (rows of both halves)
//   16384 x 2048     18.0 / 13.3     17.2 / 13.9   20.8 / 13.8   22.1 / 14.9   24.8 / 18.1  34.0 / 27.5
//   24576 x 4096     40.6 / 36.5     42.4 / 36.1   46.7 / 36.2   52.1 / 38.4   55.3 / 51.2  71.6 / -
// (32768 x 4096 at 44.9 us are 6.0 TB/s.) Rings of more steps than these, steps of 64
// with more of them, and two workgroups a CU where one round is enough were no faster.
#include "common.h"
#include "lds_limit.h"

struct MidArgs {
  u16* out;           // [M, N]
  const u16* x;       // rows ldx apart
  const u16* w;       // [N, K], gated [2 N, K]: the gate's rows first
  const u16* bias;    // [N] or null
  int M, N, K;
  long ldx;
  int mt, nt;         // tiles
  int spread;
};

__device__ __forceinline__ f32x4 mid_mfma(s16x8 a, s16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
template <int N>
__device__ __forceinline__ void mid_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// BM rows of x by BN rows of w (gated: BN / 2 gate and as many up rows). In a group of
// four waves WR go over the rows of x, 4 / WR over those of w.
template <int BM, int BN, int BK, int ST, int WR, int KG, bool GATED>
__device__ __forceinline__ void mid_body(const MidArgs& A) {
  constexpr int WC = 4 / WR, GN = GATED ? BN / 2 : BN, W = 4 * KG;
  constexpr int R = 512 / BK, CPR = 64 / R;   // rows of a copy (1 KB), pieces of a row
  constexpr int LA = BM / R / W, LB = BN / R / W, LPS = LA + LB;   // copies a wave
  constexpr int UNIT = (BM + BN) * BK * 2, AB = BM * BK * 2;
  constexpr int MF = BM / WR / 16, NF = GN / WC / 16, H = GATED ? 2 : 1;
  static_assert(LA * R * W == BM && LB * R * W == BN && MF > 0 && NF > 0, "tile");
  extern __shared__ __attribute__((aligned(16))) char mid_lds[];
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // an XCD has neighbouring tiles, those of the same weights first
  int u;
  {
    const int total = A.mt * A.nt, per = total / 8, left = total % 8;
    const int x = blockIdx.x % 8;
    u = x * per + (x < left ? x : left) + blockIdx.x / 8;
  }
  const int m0 = u % A.mt * BM, n0 = u / A.mt * GN;
  const int K = A.K, KT = K / BK;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(A.x + (long)m0 * A.ldx), 0, 0xffffffffu, 0x00027000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(A.w + (long)n0 * K), 0, 0xffffffffu, 0x00027000);
  // 16-byte pieces are mixed with the row, so that those of 16 rows at the same k lie
  // on all banks; rows past the last repeat it
  auto swz = [](int row) { return BK == 64 ? (row >> 1) & 7 : row & 15; };
  const int rl = lane / CPR, cl = lane % CPR;
  u32 va[LA], vb[LB];
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const int r = (j * W + wave) * R + rl;
    va[j] = (u32)min(r, A.M - 1 - m0) * (u32)(A.ldx * 2) + ((cl ^ swz(r)) << 4);
  }
#pragma unroll
  for (int j = 0; j < LB; ++j) {
    const int r = (j * W + wave) * R + rl;
    const bool up = GATED && r >= GN;
    vb[j] = (u32)(min(up ? r - GN : r, A.N - 1 - n0) + (up ? A.N : 0)) *
                (u32)(K * 2) + ((cl ^ swz(r)) << 4);
  }
  // Tiles start at different eighths of k: where weight rows are multiples of 4 KB
  // apart, all of them in step read from few memory channels (24576 x 4096 at 64 rows
  // 43.6 us instead of 38.4, 32768 x 2048 34.5 and 26.9).
  int kn = A.spread ? u / A.mt * 5 % 8 * KT / 8 : 0, slot_n = 0;
  auto copy = [&]() {
    char* d = mid_lds + slot_n * UNIT + wave * 1024;
    const u32 ko = (u32)kn * (BK * 2);
#pragma unroll
    for (int j = 0; j < LB; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rb, (__attribute__((address_space(3))) void*)(d + AB + j * (W * 1024)), 16,
          vb[j], ko, 0, 0);
#pragma unroll
    for (int j = 0; j < LA; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          ra, (__attribute__((address_space(3))) void*)(d + j * (W * 1024)), 16,
          va[j], ko, 0, 0);
    kn = kn + 1 == KT ? 0 : kn + 1;
    slot_n = slot_n + 1 == ST ? 0 : slot_n + 1;
  };
  f32x4 acc[H][MF][NF];
#pragma unroll
  for (int h = 0; h < H; ++h)
#pragma unroll
    for (int i = 0; i < MF; ++i)
#pragma unroll
      for (int j = 0; j < NF; ++j) acc[h][i][j] = (f32x4)(0.f);
  const int kg = wave / 4;
  const int wm = wave % 4 / WC * (BM / WR), wn = wave % WC * (GN / WC);
  int slot = 0;
  // the sums are transposed (w first): a lane has four columns of a row
  auto products = [&]() {
    const char* a = mid_lds + slot * UNIT + (wm + lr) * (BK * 2);
    const char* b = mid_lds + slot * UNIT + AB + (wn + lr) * (BK * 2);
#pragma unroll
    for (int kk = 0; kk < BK / 32 / KG; ++kk) {
      const int c = (((kg * (BK / 32 / KG) + kk) * 4 + lg) ^ swz(lr)) << 4;
      s16x8 fb[H][NF], fa[MF];
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int j = 0; j < NF; ++j)
          fb[h][j] = *(const s16x8*)(b + (h * GN + j * 16) * (BK * 2) + c);
#pragma unroll
      for (int i = 0; i < MF; ++i) fa[i] = *(const s16x8*)(a + i * 16 * (BK * 2) + c);
#pragma unroll
      for (int i = 0; i < MF; ++i)
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
          for (int j = 0; j < NF; ++j)
            acc[h][i][j] = mid_mfma(fb[h][j], fa[i], acc[h][i][j]);
    }
    slot = slot + 1 == ST ? 0 : slot + 1;
  };
  // a step's copies are there for all waves, and all have read the step before it
  auto meet = []() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  const int lead = KT < ST - 1 ? KT : ST - 1;
  for (int i = 0; i < lead; ++i) copy();
  int k = 0;
  for (; k + ST - 1 < KT; ++k) {
    mid_wait<(ST - 2) * LPS>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    meet();
    copy();
    products();
  }
  for (; k < KT; ++k) {
    const int rest = KT - 1 - k;     // steps still on their way behind this one
    if (rest >= 3) mid_wait<(ST > 4 ? 3 : ST - 1) * LPS>();
    else if (rest == 2) mid_wait<2 * LPS>();
    else if (rest == 1) mid_wait<LPS>();
    else mid_wait<0>();
    meet();
    products();
  }
  if (KG > 1) {
    __syncthreads();
    f32x4* part = (f32x4*)mid_lds + (threadIdx.x & 255);
    if (kg) {
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int i = 0; i < MF; ++i)
#pragma unroll
          for (int j = 0; j < NF; ++j)
            part[(((kg - 1) * H + h) * MF * NF + i * NF + j) * 256] = acc[h][i][j];
    }
    __syncthreads();
    if (kg) return;
#pragma unroll
    for (int g = 1; g < KG; ++g)
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int i = 0; i < MF; ++i)
#pragma unroll
          for (int j = 0; j < NF; ++j)
            acc[h][i][j] += part[(((g - 1) * H + h) * MF * NF + i * NF + j) * 256];
  }
#pragma unroll
  for (int i = 0; i < MF; ++i) {
    const int m = m0 + wm + i * 16 + lr;
    if (m >= A.M) continue;
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      const int n = n0 + wn + j * 16 + lg * 4;
      if (n >= A.N) continue;        // N is a multiple of 4
      u16x4 y;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = acc[0][i][j][r];
        if (GATED) v = v / (1.0f + __expf(-v)) * acc[H - 1][i][j][r];
        else if (A.bias) v += bf2f(A.bias[n + r]);
        y[r] = f2bf(v);
      }
      *(u16x4*)(A.out + (long)m * A.N + n) = y;
    }
  }
}

template <int BM, int BN, int BK, int ST, int WR, int KG, bool GATED>
__global__ void __launch_bounds__(256 * KG) mid_kernel(const MidArgs A) {
  mid_body<BM, BN, BK, ST, WR, KG, GATED>(A);
}

template <int BM, int BN, int BK, int ST, int WR, int KG, bool GATED>
static void mid_go(MidArgs A, hipStream_t s) {
  constexpr int bytes = (BM + BN) * BK * 2 * ST, GN = GATED ? BN / 2 : BN;
  static std::atomic<unsigned long long> asked{0};
  lds_limit((const void*)mid_kernel<BM, BN, BK, ST, WR, KG, GATED>, bytes, asked);
  A.mt = (A.M + BM - 1) / BM;
  A.nt = (A.N + GN - 1) / GN;
  A.spread = BN >= 64 && A.K % 2048 == 0 && A.M <= 128;
  hipLaunchKernelGGL((mid_kernel<BM, BN, BK, ST, WR, KG, GATED>), dim3(A.mt * A.nt),
                     dim3(256 * KG), bytes, s, A);
}

// The smallest tile of which 256 or fewer make M rows by `rows` of w; of more weight
// rows than that, tiles of 128. (ops._mid_tile is the same choice: the sizes that come
// here depend on it.)
template <bool GATED, typename GO>
static void mid_pick(int M, int N, int K, GO go) {
  const long rows = GATED ? 2L * N : N;
  auto fit = [&](int bm, int bn) {
    return ((M + bm - 1) / bm) * ((rows + bn - 1) / bn) <= 256;
  };
  if constexpr (!GATED) {
    // (long rows of few weights: 4096 x 4096 at 16 rows 11.2 us on 64 x 16, 11.7)
    if (M <= 32 && !(M > 8 && K >= 4096 && fit(64, 16)) && fit(32, 32))
      return go.template tile<32, 32, 256, 4, 2, 2, false>();
    if (fit(64, 16)) return go.template tile<64, 16, 256, 4, 4, 2, false>();
  }
  if (fit(64, 32) && (GATED || M > 32))
    return go.template tile<64, 32, 256, 3, 4, 2, GATED>();
  if (M <= 32) {
    if (fit(32, 64)) return go.template tile<32, 64, 128, 3, 2, 1, GATED>();
    if (fit(32, 128)) return go.template tile<32, 128, 128, 4, 2, 2, GATED>();
    return go.template tile<32, 128, 128, 2, 2, 1, GATED>();       // two a CU
  }
  if (fit(64, 64)) return go.template tile<64, 64, 128, 5, 2, 2, GATED>();
  if (M <= 64) {
    if (fit(64, 128)) return go.template tile<64, 128, 128, 3, 2, 2, GATED>();
    return go.template tile<64, 128, 64, 3, 2, 1, GATED>();        // two a CU
  }
  if (M <= 128 || M > 192) {
    if (fit(128, 64)) return go.template tile<128, 64, 128, 3, 2, 2, GATED>();
  } else if (fit(64, 128)) {
    return go.template tile<64, 128, 128, 3, 2, 2, GATED>();
  }
  go.template tile<128, 128, 64, 5, 2, 1, GATED>();
}

struct MidLaunch {
  const MidArgs& A;
  hipStream_t s;
  template <int BM, int BN, int BK, int ST, int WR, int KG, bool GATED>
  void tile() const { mid_go<BM, BN, BK, ST, WR, KG, GATED>(A, s); }
};
struct MidSize {
  int* out;
  template <int BM, int BN, int BK, int ST, int WR, int KG, bool GATED>
  void tile() const { out[0] = BM; out[1] = BN; }
};

// rows of x and of w in a tile
extern "C" void sutro_mid_tile(int* out, int M, int N, int K, int gated) {
  if (gated) mid_pick<true>(M, N, K, MidSize{out});
  else mid_pick<false>(M, N, K, MidSize{out});
}

// x and w at multiples of 16 bytes, ldx a multiple of 8, K of 256, N of 4; offsets within
// a tile are of 32 bits: M ldx and (gated) N K below 2^30
extern "C" void sutro_linear_mid(void* out, const void* x, long ldx, const void* w,
                                 const void* bias, int M, int N, int K, int gated,
                                 hipStream_t stream) {
  const MidArgs A = {(u16*)out, (const u16*)x, (const u16*)w, (const u16*)bias,
                     M, N, K, ldx, 0, 0, 0};
  if (gated) mid_pick<true>(M, N, K, MidLaunch{A, stream});
  else mid_pick<false>(M, N, K, MidLaunch{A, stream});
}
