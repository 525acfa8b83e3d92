// The inner loop of products whose weights are read once and whose rows are
// few (decode steps): weights travel from memory straight into MFMA fragments,
// a batch of k-steps ahead of their use, with no LDS, no barrier and nothing
// shared between waves, so that every wave keeps kilobytes in flight.
//
// mfma_f32_16x16x32_bf16 with the WEIGHT rows as A and the activation rows as
// B: lane l holds A[l%16][(l/16)*8 + j] and B[(l/16)*8 + j][l%16], j = 0..7,
// and D[(l/16)*4 + r][l%16], r = 0..3: four neighbouring output columns of one
// activation row, which is an 8-byte store.
#pragma once

#define GS_STEP 32   // k of one product
#define GS_BATCH 4   // k-steps loaded ahead

__device__ __forceinline__ f32x4 gs_mfma(s16x8 a, s16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

typedef __bf16 gs_bf16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2 gs_pack4(f32x4 v) {
  return __builtin_bit_cast(u32x2, __builtin_convertvector(v, gs_bf16x4));
}

// acc[i][m] += sum over k-steps [0, steps) of W_i (16 rows) x A_m (16 rows), ROUND:
// from step `first` (0 <= first < steps) on and round; wp / ap: this lane's row of
// every block at its k chunk, steps >= 1
template <int NF, int MB, bool ROUND>
__device__ __forceinline__ void gs_dot(const u16* const (&wp)[NF],
                                       const u16* const (&ap)[MB], int steps,
                                       int first,
                                       f32x4 (&acc)[NF][MB]) {
  s16x8 w[2][GS_BATCH][NF], a[2][GS_BATCH][MB];
  auto load = [&](int buf, int s0) {
#pragma unroll
    for (int u = 0; u < GS_BATCH; ++u) {
      int s = min(s0 + u, steps - 1);  // the tail repeats (not used)
      if (ROUND) s += first;
      if (ROUND && s >= steps) s -= steps;
#pragma unroll
      for (int i = 0; i < NF; ++i)
        w[buf][u][i] = *(const s16x8*)(wp[i] + s * GS_STEP);
#pragma unroll
      for (int m = 0; m < MB; ++m)
        a[buf][u][m] = *(const s16x8*)(ap[m] + s * GS_STEP);
    }
  };
  auto use = [&](int buf, int n) {
#pragma unroll
    for (int u = 0; u < GS_BATCH; ++u)
      if (u < n) {
#pragma unroll
        for (int i = 0; i < NF; ++i)
#pragma unroll
          for (int m = 0; m < MB; ++m)
            acc[i][m] = gs_mfma(w[buf][u][i], a[buf][u][m], acc[i][m]);
      }
  };
  load(0, 0);
  int s = 0;
  for (; s + 2 * GS_BATCH <= steps; s += 2 * GS_BATCH) {
    load(1, s + GS_BATCH);
    use(0, GS_BATCH);
    load(0, s + 2 * GS_BATCH);
    use(1, GS_BATCH);
  }
  if (s < steps) {
    if (s + GS_BATCH < steps) load(1, s + GS_BATCH);
    use(0, min(GS_BATCH, steps - s));
    if (s + GS_BATCH < steps) use(1, steps - s - GS_BATCH);
  }
}
