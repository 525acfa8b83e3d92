// Linear layers over few rows (decode steps): out[M, N] = x[M, K] W[N, K]^T (+
// bias), bf16 with fp32 sums, M up to 32, optionally with the gated unit of a
// feed-forward behind it (W: N gate rows, then N up rows).
//
// Bound by the weights, which are read once, and for the small matrices of a
// step by the time to get enough loads in flight. A workgroup owns 16 or 32
// rows of W (gated: 16 and 16) and its waves split k, each with a batch of
// fragments ahead of its products (gemm_stream.h); their sums meet in LDS.
//
// Waves, by the k-steps of a row (a batch is four). Where 4, 8 or 16 waves have
// exactly a batch each, all loads of a workgroup are in flight at once: 2048 x 512
// at 16 rows 3.4 / 3.2 / 3.7 us on 2 / 4 / 8 waves, 4104 x 1024 6.0 / 6.8 / 5.4. Else
// few waves with long runs are ahead, as one that ends after a batch or two has
// nothing in flight while its workgroup adds up: 16 rows, 6144 x 4096 on 8 waves of
// 16 rows of W 22.1 -> 14.9 us on 2 of 32, 18432 x 2048 28.0 -> 22.9, 5120 x 25600
// 111 -> 72; a router of 32 x 4096 12.0 on 16 waves, 9.2 on 2. Four of them pay up to
// 12 rows of x while a CU has no more than one workgroup (4096 x 3072 at 8 rows 8.7 on
// 2, 8.2 on 4; at 16 rows 9.1 and 9.9), not with a unit behind them, whose workgroup
// reads two blocks of weights (2 x 4096 x 3072 at 8 rows 12.2, 14.9).
#include "common.h"
#include "gemm_stream.h"

#define SETS_WAVES 4096   // most waves of a product that goes through sets of rows

struct SkinnyArgs {
  u16* out;
  const u16* x;
  const u16* w;
  const u16* bias;   // [N] or null
  long ldx, ldo;
  int M, N, K;
  int act;           // 0 none, 1 silu(gate) up (W has 2 N rows)
  // a norm in front (one row): x is norm(x + residual) * norm_w
  const u16* residual;
  u16* residual_out; // x + residual
  const u16* norm_w;
  float eps;
};

template <int NF, int MB, int WAVES, bool GATED, bool SPREAD>
__global__ void __launch_bounds__(WAVES * 64) skinny_kernel(SkinnyArgs A) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, g = lane >> 4;
  constexpr int COLS = GATED ? 16 : NF * 16;
  const int n0 = blockIdx.x * COLS;
  const int steps = A.K / GS_STEP;
  const int s0 = steps * wave / WAVES, s1 = steps * (wave + 1) / WAVES;
  const long k0 = (long)s0 * GS_STEP + g * 8;

  const u16* wp[NF];
#pragma unroll
  for (int i = 0; i < NF; ++i) {
    const int r = GATED ? min(n0 + lr, A.N - 1) + i * A.N
                        : min(n0 + i * 16 + lr, A.N - 1);
    wp[i] = A.w + (long)r * A.K + k0;
  }
  const u16* ap[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m)
    ap[m] = A.x + (long)min(m * 16 + lr, A.M - 1) * A.ldx + k0;
  f32x4 acc[NF][MB];
#pragma unroll
  for (int i = 0; i < NF; ++i)
#pragma unroll
    for (int m = 0; m < MB; ++m) acc[i][m] = (f32x4)(0.f);
  const int n = s1 - s0;
  if (n > 0)
    gs_dot<NF, MB, SPREAD>(wp, ap, n, SPREAD ? (int)(blockIdx.x * 4u) % n : 0,
                           acc);

  __shared__ f32x4 red[WAVES][NF][MB][64];
#pragma unroll
  for (int i = 0; i < NF; ++i)
#pragma unroll
    for (int m = 0; m < MB; ++m) red[wave][i][m][lane] = acc[i][m];
  __syncthreads();
  // one thread four neighbouring columns of a row
  constexpr int OUTS = (GATED ? 1 : NF) * MB;
  for (int z = threadIdx.x; z < OUTS * 64; z += WAVES * 64) {
    const int l = z & 63, m = (z >> 6) % MB, i = (z >> 6) / MB;
    const int row = m * 16 + (l & 15);
    const int col = n0 + i * 16 + (l >> 4) * 4;
    f32x4 y = red[0][i][m][l], u;
#pragma unroll
    for (int w = 1; w < WAVES; ++w) y += red[w][i][m][l];
    if (row >= A.M || col >= A.N) continue;
    if (GATED) {
      u = red[0][NF - 1][m][l];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) u += red[w][NF - 1][m][l];
    }
    if (A.bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        y[e] += bf2f(A.bias[col + e]);
        if (GATED) u[e] += bf2f(A.bias[A.N + col + e]);
      }
    }
    if (GATED) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        y[e] = y[e] / (1.f + __expf(-y[e])) * u[e];
    }
    *(u32x2*)(A.out + (long)row * A.ldo + col) = gs_pack4(y);
  }
}

// One or two rows: no matrix core, its blocks of 16 rows would be mostly empty
// and reading the fragments holds a workgroup to 16 neighbouring weight rows.
// Here a workgroup owns four (gated: two and two), the lanes of its waves lie
// along k, 1 KB of a weight row per load, and all of a wave's loads of two
// steps are in flight together. Against the library, one row: 2048 x 2048 10.9
// -> 4.8 us, 32768 x 4096 61.5 -> 48.8 (5.5 TB/s); 2 x 8192 x 2048 with the unit
// behind it 19.6 -> 14.0.
template <int MR, int WAVES, bool GATED>
__global__ void __launch_bounds__(WAVES * 64) gemv_kernel(SkinnyArgs A) {
  constexpr int R = 4, V = R * MR;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  constexpr int COLS = GATED ? R / 2 : R;
  const int n0 = blockIdx.x * COLS;
  const u16* wp[R];
#pragma unroll
  for (int i = 0; i < R; ++i)
    wp[i] = A.w + (long)(GATED ? n0 + (i & 1) + (i >> 1) * A.N : n0 + i) * A.K;
  float acc[V];
#pragma unroll
  for (int v = 0; v < V; ++v) acc[v] = 0.f;
  const int step = WAVES * 512;
  for (int k0 = threadIdx.x * 8; k0 < A.K; k0 += 2 * step) {
    u16x8 w[2][R], x[2][MR];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int k = min(k0 + b * step, A.K - 8);
#pragma unroll
      for (int i = 0; i < R; ++i) w[b][i] = *(const u16x8*)(wp[i] + k);
#pragma unroll
      for (int m = 0; m < MR; ++m)
        x[b][m] = *(const u16x8*)(A.x + (long)min(m, A.M - 1) * A.ldx + k);
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      if (k0 + b * step >= A.K) break;
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int m = 0; m < MR; ++m)
            acc[i * MR + m] = fmaf(bf2f(w[b][i][e]), bf2f(x[b][m][e]),
                                   acc[i * MR + m]);
    }
  }
  // the lanes of 64 / V neighbours end with the sum of one value: half the
  // values go to the other half of the lanes at each step
  int v0 = 0;
#pragma unroll
  for (int half = V / 2, bit = 32; half >= 1; half /= 2, bit /= 2) {
    const bool up = lane & bit;
#pragma unroll
    for (int v = 0; v < V / 2; ++v)
      if (v < half) {
        const float give = up ? acc[v] : acc[v + half];
        const float keep = up ? acc[v + half] : acc[v];
        acc[v] = keep + __shfl_xor(give, bit, 64);
      }
    v0 += up ? half : 0;
  }
#pragma unroll
  for (int bit = 32 / V; bit >= 1; bit /= 2)
    acc[0] += __shfl_xor(acc[0], bit, 64);
  __shared__ float red[WAVES][V];
  if ((lane & (64 / V - 1)) == 0) red[wave][v0] = acc[0];
  __syncthreads();
  const int m = threadIdx.x % MR, c = threadIdx.x / MR;
  if (c >= COLS || m >= A.M) return;
  auto total = [&](int i) {
    float y = red[0][i * MR + m];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) y += red[w][i * MR + m];
    const int col = GATED ? n0 + (i & 1) + (i >> 1) * A.N : n0 + i;
    return A.bias ? y + bf2f(A.bias[col]) : y;
  };
  float y = total(c);
  if (GATED) y = y / (1.f + __expf(-y)) * total(c + 2);
  A.out[(long)m * A.ldo + n0 + c] = f2bf(y);
}

// One row again, K up to WAVES * 1024: all of a weight row is loaded at once, and a
// workgroup goes through several sets of weight rows, the next one's on their way
// while a set's sums meet. Against a workgroup a set (us in a graph): 8192 x 2048
// 9.4 -> 8.4, 32768 x 2048 26.0 -> 23.9, 32768 x 4096 48.5 -> 46.0; with the unit behind
// it 2 x 8192 x 2048 14.4 -> 13.6, 2 x 12288 x 4096 37.1 -> 35.3; below 2048 sets there
// is nothing to go through, and 151936 rows lose 1 to 2 %. Twice as few or as many
// workgroups are 5 to 10 % slower, one way or the other.
//
// NORM: with the addition and RMSNorm in front of it. In a launch of its own the
// norm takes 2 to 3 us before each product of a step, all of it latency; here every
// workgroup makes the row again (three reads of it out of the L2), behind the loads
// of its first weights. Two launches and this one: 3072 x 2048 7.6 and 6.0 us, 6144 x
// 4096 14.2 and 12.2; with the unit 2 x 8192 x 2048 17.2 and 14.5, 2 x 12288 x 4096 40.9
// and 34.9.
template <int WAVES, bool GATED, bool NORM>
__global__ void __launch_bounds__(WAVES * 64) sets_gemv_kernel(SkinnyArgs A) {
  constexpr int R = 4, COLS = GATED ? R / 2 : R, T = WAVES * 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int groups = (A.N + COLS - 1) / COLS;
  __shared__ __attribute__((aligned(16))) u16 xs[NORM ? WAVES * 1024 : 8];
  __shared__ float red[WAVES][R];
  u16x8 w[2][R];
  auto load = [&](int g) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int n = g * COLS + (GATED ? i & 1 : i);
        const long row = min(n, A.N - 1) + (GATED ? (i >> 1) * (long)A.N : 0);
        w[b][i] =
            *(const u16x8*)(A.w + row * A.K + min((b * T + tid) * 8, A.K - 8));
      }
  };
  load(blockIdx.x);

  if (NORM) {
    // the squares are added in the order of the norm's own kernel (four waves a
    // row, a piece or two a lane): the two agree to the bit
    float xf[2][8], sq[2] = {0.f, 0.f};
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int k = (b * T + tid) * 8;
      if (k >= A.K) continue;
      const u16x8 xv = *(const u16x8*)(A.x + k);
      const u16x8 rv = *(const u16x8*)(A.residual + k);
      u16x8 sum;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        xf[b][e] = bf2f(xv[e]) + bf2f(rv[e]);
        sq[WAVES == 2 ? b : 0] += xf[b][e] * xf[b][e];
        sum[e] = f2bf(xf[b][e]);
      }
      if (blockIdx.x == 0) *(u16x8*)(A.residual_out + k) = sum;
    }
#pragma unroll
    for (int b = 0; b < (WAVES == 2 ? 2 : 1); ++b) {
      sq[b] = wave_sum_f32(sq[b]);
      if (lane == 0) red[wave][b] = sq[b];
    }
    __syncthreads();
    float ssq = red[0][0];
#pragma unroll
    for (int i = 1; i < 4; ++i) ssq += red[i % WAVES][i / WAVES];
    const float inv = rsqrtf(ssq / (float)A.K + A.eps);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int k = (b * T + tid) * 8;
      if (k >= A.K) continue;
      const u16x8 nv = *(const u16x8*)(A.norm_w + k);
      u16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = f2bf(xf[b][e] * inv * bf2f(nv[e]));
      *(u16x8*)(xs + k) = o;    // read by the same thread only
    }
  }

  for (int g = blockIdx.x; g < groups; g += gridDim.x) {
    float acc[R] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int k = (b * T + tid) * 8;
      if (k >= A.K) continue;
      const u16x8 xv = *(const u16x8*)((NORM ? xs : A.x) + k);
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          acc[i] = fmaf(bf2f(w[b][i][e]), bf2f(xv[e]), acc[i]);
    }
    if (g + (int)gridDim.x < groups) load(g + gridDim.x);
    // the lanes of 16 neighbours end with the sum of one value
    int v0 = 0;
#pragma unroll
    for (int half = R / 2, bit = 32; half >= 1; half /= 2, bit /= 2) {
      const bool up = lane & bit;
#pragma unroll
      for (int v = 0; v < R / 2; ++v)
        if (v < half) {
          const float give = up ? acc[v] : acc[v + half];
          const float keep = up ? acc[v + half] : acc[v];
          acc[v] = keep + __shfl_xor(give, bit, 64);
        }
      v0 += up ? half : 0;
    }
#pragma unroll
    for (int bit = 8; bit >= 1; bit /= 2)
      acc[0] += __shfl_xor(acc[0], bit, 64);
    __syncthreads();          // the sums before these have been read
    if ((lane & 15) == 0) red[wave][v0] = acc[0];
    __syncthreads();
    const int n = g * COLS + tid;
    if (tid < COLS && n < A.N) {
      auto total = [&](int i) {
        float y = red[0][i];
#pragma unroll
        for (int z = 1; z < WAVES; ++z) y += red[z][i];
        return y;
      };
      float y = total(tid);
      if (GATED) y = y / (1.f + __expf(-y)) * total(tid + 2);
      A.out[n] = f2bf(y);
    }
  }
}

// one row, K % 32 == 0, K <= 4096; residual and residual_out differ
extern "C" void sutro_norm_linear(void* out, const void* x,
                                  const void* residual, void* residual_out,
                                  const void* norm_w, float eps, const void* w,
                                  int N, int K, int act, hipStream_t s) {
  SkinnyArgs A = {};
  A.out = (u16*)out;
  A.x = (const u16*)x;
  A.w = (const u16*)w;
  A.M = 1;
  A.N = N;
  A.K = K;
  A.residual = (const u16*)residual;
  A.residual_out = (u16*)residual_out;
  A.norm_w = (const u16*)norm_w;
  A.eps = eps;
  const int groups = (N + (act ? 1 : 3)) / (act ? 2 : 4);
  const int most = SETS_WAVES / (K <= 2048 ? 2 : 4);
  const dim3 grid(groups < most ? groups : most);
#define LAUNCH_NG(WW, GG)                                                    \
  hipLaunchKernelGGL((sets_gemv_kernel<WW, GG, true>), grid, dim3(WW * 64), 0, s, A)
  if (K <= 2048) {
    if (act) LAUNCH_NG(2, true);
    else LAUNCH_NG(2, false);
  } else {
    if (act) LAUNCH_NG(4, true);
    else LAUNCH_NG(4, false);
  }
#undef LAUNCH_NG
}

template <int MR, bool GATED>
static void gemv_launch(const SkinnyArgs& A, hipStream_t s) {
  const unsigned blocks = A.N / (GATED ? 2 : 4);
  // From 2048 sets of rows on (one row, no bias), up to the largest output layers,
  // which have the same 4096 waves busy either way: see sets_gemv_kernel.
  if (MR == 1 && !A.bias && A.K > 1024 && A.K <= 4096 && blocks >= 2048 &&
      blocks < 32768) {
    if (A.K <= 2048)
      hipLaunchKernelGGL((sets_gemv_kernel<2, GATED, false>),
                         dim3(SETS_WAVES / 2), dim3(128), 0, s, A);
    else
      hipLaunchKernelGGL((sets_gemv_kernel<4, GATED, false>),
                         dim3(SETS_WAVES / 4), dim3(256), 0, s, A);
    return;
  }
#define LAUNCH_GV(WW)                                                        \
  hipLaunchKernelGGL((gemv_kernel<MR, WW, GATED>), dim3(blocks),             \
                     dim3(WW * 64), 0, s, A)
  if (A.K <= 1024) LAUNCH_GV(1);
  else if (A.K <= 2048 || blocks >= 2048) LAUNCH_GV(2);
  else if (A.K <= 4096) LAUNCH_GV(4);
  else LAUNCH_GV(8);
#undef LAUNCH_GV
}

template <int NF, int MB, bool GATED>
static void skinny_launch(const SkinnyArgs& A, hipStream_t s) {
  const unsigned blocks = (A.N + (GATED ? 16 : NF * 16) - 1) /
                          (GATED ? 16 : NF * 16);
  const int steps = A.K / GS_STEP;
#define LAUNCH_SK(WW, SPREAD)                                                \
  hipLaunchKernelGGL((skinny_kernel<NF, MB, WW, GATED, SPREAD>),             \
                     dim3(blocks), dim3(WW * 64), 0, s, A)
  // Weight rows 8 KB apart lie on few memory channels where all workgroups read
  // the same columns of them: starts are spread. 32768 x 4096 at 3 rows 62 -> 51 us,
  // 8192 x 4096 16.2 -> 14.2; rows of 4 KB or fewer than 8192 of them 0 to 10 % more.
  // Waves: see the top.
  const bool spread = A.K % 4096 == 0 && (GATED ? 2 : 1) * A.N >= 8192;
  const bool few = blocks <= 256 && !(NF == 2 && !GATED);
  if (spread) LAUNCH_SK(2, true);
  else if (steps == 16) LAUNCH_SK(4, false);
  else if (steps == 32) LAUNCH_SK(8, false);
  else if (GATED || !few || steps < 16) LAUNCH_SK(2, false);
  else if (steps == 64) LAUNCH_SK(16, false);
  else if (A.M <= 12) LAUNCH_SK(4, false);
  else LAUNCH_SK(2, false);
#undef LAUNCH_SK
}

// K % 32 == 0, N % 4 == 0, 1 <= M <= 32, 16-byte rows of x and w, 8-byte rows
// of out
extern "C" void sutro_linear_skinny(void* out, long ldo, const void* x,
                                    long ldx, const void* w, const void* bias,
                                    int M, int N, int K, int act,
                                    hipStream_t s) {
  SkinnyArgs A = {(u16*)out, (const u16*)x, (const u16*)w, (const u16*)bias,
                  ldx, ldo, M, N, K, act, nullptr, nullptr, nullptr, 0.f};
  const int mb = (M + 15) / 16;
#define SK_GEMV(MR)                                                          \
  do {                                                                       \
    if (act == 1) gemv_launch<MR, true>(A, s);                               \
    else gemv_launch<MR, false>(A, s);                                       \
    return;                                                                  \
  } while (0)
  if (M == 1) SK_GEMV(1);
  if (M == 2) SK_GEMV(2);
#undef SK_GEMV
#define SK_MB(NF, GG)                                                        \
  do {                                                                       \
    if (mb == 1) skinny_launch<NF, 1, GG>(A, s);                             \
    else skinny_launch<NF, 2, GG>(A, s);                                     \
  } while (0)
  // 32 rows of W a workgroup read half as much of x, but where they take more
  // rounds of the chip than 16 do: 10304 x 4096 at 16 rows 30.6 and 27.0 us, 6144 x
  // 4096 14.9 and 18.3. A few workgroups more than one round are none: 4104 x 3072 at
  // 3 rows 10.6 and 9.4, 4608 x 3072 10.8 and 10.8, at 16 rows 12.1 and 15.4.
  const int rounds16 = (N + 16 * 256 - 1) / (16 * 256);
  const int rounds32 = (N + 32 * 256 - 1) / (32 * 256);
  if (act == 1) SK_MB(2, true);
  else if (2 * rounds32 <= rounds16 && N >= 4352) SK_MB(2, false);
  else SK_MB(1, false);
#undef SK_MB
}
