// Python bindings for the sutro-amd CDNA4 kernels.
// Tensors are validated here; raw pointers + the current HIP stream go to the
// extern "C" launchers in the .hip translation units.
#include <torch/extension.h>
#include <pybind11/numpy.h>

#include <hip/hip_runtime.h>
#include <c10/hip/HIPStream.h>

#define CHECK_CUDA(x) TORCH_CHECK((x).is_cuda(), #x " must be a GPU tensor")
#define CHECK_CONTIG(x) TORCH_CHECK((x).is_contiguous(), #x " must be contiguous")
#define CHECK_BF16(x) \
  TORCH_CHECK((x).scalar_type() == at::kBFloat16, #x " must be bf16")

static hipStream_t cur_stream() {
  return c10::hip::getCurrentHIPStream().stream();
}

extern "C" {
void sutro_rmsnorm(void*, const void*, const void*, float, long, int,
                   hipStream_t);
void sutro_fused_add_rmsnorm(void*, void*, const void*, float, long, int,
                             hipStream_t);
void sutro_silu_mul(void*, const void*, long, int, hipStream_t);
void sutro_rope_and_cache(void*, void*, const void*, const long*, const long*,
                          void*, void*, const float*, int, int, int, int, int,
                          hipStream_t);
static bool is_fp8(const torch::Tensor& t) {
  return t.scalar_type() == at::kFloat8_e4m3fn;
}
void sutro_mean_pool_normalize(float*, const void*, const int*, int, int,
                               hipStream_t);
void sutro_attn_decode(void*, const void*, const void*, const void*,
                       const int*, const int*, int, int, int, int, int, int,
                       int, float, int, float*, float*, hipStream_t);
int sutro_attn_decode_splits(int, int, int);
void sutro_attn_prefill(void*, const void*, const void*, const void*,
                        const int*, const int*, const int*, const int*,
                        const int*, int, int, int, int, int, int, int, float,
                        hipStream_t);
void sutro_mfma32_probe(float*, const void*, const void*, hipStream_t);
void sutro_gemm_tn_launch(void*, const void*, const void*, const void*, int,
                          int, long, int, int, int, int, hipStream_t);
void sutro_mfma16_probe(float*, const void*, const void*, hipStream_t);
void sutro_qkv_prep(const void*, void*, void*, void*, const long*, const long*,
                    const float*, const void*, const void*, float, int, int,
                    int, int, int, int, int, hipStream_t);
void sutro_sampler_fused(const void*, int, const float*, const float*,
                         const int*, const float*, const unsigned int*, int,
                         long, int, int, int*, float*, int, hipStream_t);
void sutro_grouped_gemm(void*, const void*, long, const void*, const int*,
                        const int*, const int*, int, int, int, long, int,
                        int, hipStream_t);
void sutro_norm_linear(void*, const void*, const void*, void*, const void*,
                       float, const void*, int, int, int, hipStream_t);
void sutro_linear_silu_mul(void*, const void*, const void*, int, int, long,
                           hipStream_t);
void sutro_linear_gelu_mul(void*, void*, const void*, const void*, const void*, int,
                           int, int, long, hipStream_t);
void sutro_linear_heads(void*, void*, void*, const void*, const void*, const long*,
                        const long*, const float*, const void*, const void*, float,
                        int, int, int, int, long, hipStream_t);
void sutro_moe_combine(void*, const void*, const void*, int, const float*, int,
                       int, int, hipStream_t);
void sutro_moe_topk(int*, float*, const void*, long, int, int, int, int,
                    hipStream_t);
void sutro_linear_mid(void*, const void*, long, const void*, const void*, int, int,
                      int, int, hipStream_t);
void sutro_mid_tile(int*, int, int, int, int);
void sutro_linear_skinny(void*, long, const void*, long, const void*,
                         const void*, int, int, int, int, hipStream_t);
long mix_moe_dispatch_scratch(long, int);
void mix_moe_dispatch(int*, int*, int*, int*, const int*, const long*, long,
                      int, int, int, long, int*, const float*, float*,
                      hipStream_t);
}

void rmsnorm(torch::Tensor out, torch::Tensor x, torch::Tensor w, double eps) {
  CHECK_CUDA(x); CHECK_CONTIG(x); CHECK_BF16(x);
  const long C = x.size(-1);
  const long rows = x.numel() / C;
  TORCH_CHECK(C % 8 == 0 && C <= 16384, "unsupported row size ", C);
  sutro_rmsnorm(out.data_ptr(), x.data_ptr(), w.data_ptr(), (float)eps, rows,
                (int)C, cur_stream());
}

void fused_add_rmsnorm(torch::Tensor x, torch::Tensor residual, torch::Tensor w,
                       double eps) {
  CHECK_CUDA(x); CHECK_CONTIG(x); CHECK_BF16(x); CHECK_CONTIG(residual);
  const long C = x.size(-1);
  const long rows = x.numel() / C;
  TORCH_CHECK(C % 8 == 0 && C <= 16384, "unsupported row size ", C);
  sutro_fused_add_rmsnorm(x.data_ptr(), residual.data_ptr(), w.data_ptr(),
                          (float)eps, rows, (int)C, cur_stream());
}

void silu_mul(torch::Tensor out, torch::Tensor x) {
  CHECK_CUDA(x); CHECK_CONTIG(x); CHECK_BF16(x);
  const long I = x.size(-1) / 2;
  const long T = x.numel() / (2 * I);
  TORCH_CHECK(I % 8 == 0, "intermediate size must be a multiple of 8");
  sutro_silu_mul(out.data_ptr(), x.data_ptr(), T, (int)I, cur_stream());
}

void rope_and_cache(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                    torch::Tensor positions, torch::Tensor slot_mapping,
                    torch::Tensor k_cache, torch::Tensor v_cache,
                    torch::Tensor cos_sin) {
  CHECK_CUDA(q); CHECK_CONTIG(q); CHECK_BF16(q);
  CHECK_CONTIG(k); CHECK_CONTIG(v); CHECK_CONTIG(k_cache);
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat, "cos_sin must be f32");
  const int T = q.size(0), Hq = q.size(1), D = q.size(2);
  const int Hk = k.size(1);
  const int bs = k_cache.size(2);
  TORCH_CHECK(D % 2 == 0 && D / 2 <= 128, "unsupported head_dim ", D);
  sutro_rope_and_cache(q.data_ptr(), k.data_ptr(), v.data_ptr(),
                       positions.data_ptr<long>(), slot_mapping.data_ptr<long>(),
                       k_cache.data_ptr(), v_cache.data_ptr(),
                       cos_sin.data_ptr<float>(), T, Hq, Hk, D, bs,
                       cur_stream());
}

void mean_pool_normalize(torch::Tensor out, torch::Tensor hidden,
                         torch::Tensor qlocs) {
  CHECK_CUDA(hidden); CHECK_CONTIG(hidden); CHECK_BF16(hidden);
  const int S = out.size(0), H = hidden.size(-1);
  TORCH_CHECK(H % 8 == 0, "hidden size must be a multiple of 8");
  sutro_mean_pool_normalize(out.data_ptr<float>(), hidden.data_ptr(),
                            qlocs.data_ptr<int>(), S, H, cur_stream());
}

void paged_attention(torch::Tensor out, torch::Tensor q, torch::Tensor k_cache,
                     torch::Tensor v_cache, torch::Tensor block_tables,
                     torch::Tensor seq_lens, torch::Tensor qlocs, double scale,
                     int64_t num_decodes, torch::Tensor tile_seq,
                     torch::Tensor tile_q0, int64_t prefill_token_count) {
  CHECK_CUDA(q); CHECK_CONTIG(q); CHECK_BF16(q); CHECK_CONTIG(k_cache);
  CHECK_CONTIG(v_cache);
  const int Hq = q.size(1), D = q.size(2);
  const int Hk = k_cache.size(1);
  const int bs = k_cache.size(2);
  const int S = seq_lens.size(0);
  TORCH_CHECK(D == 128 || D == 64,
              "attention kernels support head_dim 64/128 (got ", D, ")");
  TORCH_CHECK(bs == 32, "attention kernels require kv_block_size 32");
  TORCH_CHECK(Hq % Hk == 0 && Hq / Hk <= 8,
              "GQA group size must divide and be <= 8");
  const int bt_stride = block_tables.size(1);
  const int n_tiles = tile_seq.numel();
  if (n_tiles > 0) {
    sutro_attn_prefill(out.data_ptr(), q.data_ptr(), k_cache.data_ptr(),
                       v_cache.data_ptr(), block_tables.data_ptr<int>(),
                       seq_lens.data_ptr<int>(), qlocs.data_ptr<int>(),
                       tile_seq.data_ptr<int>(), tile_q0.data_ptr<int>(),
                       n_tiles, S - (int)num_decodes, bt_stride, Hq, Hk, D,
                       is_fp8(k_cache) ? 1 : 0, (float)scale, cur_stream());
  }
  if (num_decodes > 0) {
    const long dec_off = prefill_token_count;  // decode rows are the tail
    const int seq_offset = S - (int)num_decodes;
    const u_int16_t* qp = (const u_int16_t*)q.data_ptr();
    u_int16_t* op = (u_int16_t*)out.data_ptr();
    // partial results of contexts that are cut into runs of pages
    const int ns = sutro_attn_decode_splits((int)num_decodes, Hk, bt_stride);
    torch::Tensor po, pml;
    if (ns > 1) {
      auto o = q.options().dtype(at::kFloat);
      po = torch::empty({num_decodes * Hq * ns, D}, o);
      pml = torch::empty({num_decodes * Hq * ns, 2}, o);
    }
    sutro_attn_decode(op + dec_off * Hq * D, qp + dec_off * Hq * D,
                      k_cache.data_ptr(), v_cache.data_ptr(),
                      block_tables.data_ptr<int>(), seq_lens.data_ptr<int>(),
                      bt_stride, (int)num_decodes, Hq, Hk, D,
                      is_fp8(k_cache) ? 1 : 0, seq_offset, (float)scale, ns,
                      ns > 1 ? po.data_ptr<float>() : nullptr,
                      ns > 1 ? pml.data_ptr<float>() : nullptr, cur_stream());
  }
}

void qkv_prep(torch::Tensor qkv, torch::Tensor q_out, torch::Tensor k_cache,
              torch::Tensor v_cache, torch::Tensor positions,
              torch::Tensor slot_mapping, torch::Tensor cos_sin,
              c10::optional<torch::Tensor> q_norm_w,
              c10::optional<torch::Tensor> k_norm_w, double eps) {
  CHECK_CUDA(qkv); CHECK_CONTIG(qkv); CHECK_BF16(qkv);
  CHECK_CONTIG(q_out); CHECK_CONTIG(k_cache); CHECK_CONTIG(v_cache);
  // (pinned host memory can be read, and written, from the GPU)
  for (const auto& t : {q_out, k_cache, v_cache, positions, slot_mapping, cos_sin})
    TORCH_CHECK(t.is_cuda() || t.is_pinned(), "operands on the GPU");
  for (const auto& n : {q_norm_w, k_norm_w})
    TORCH_CHECK(!n || n->is_cuda() || n->is_pinned(), "norm weights on the GPU");
  const int T = qkv.size(0);
  const int Hq = q_out.size(1), D = q_out.size(2);
  const int Hk = k_cache.size(1);
  const int bs = k_cache.size(2);
  const int row_stride = qkv.size(1);
  TORCH_CHECK(row_stride == Hq * D + 2 * Hk * D, "qkv width mismatch");
  const void* qw = q_norm_w ? q_norm_w->data_ptr() : nullptr;
  const void* kw = k_norm_w ? k_norm_w->data_ptr() : nullptr;
  sutro_qkv_prep(qkv.data_ptr(), q_out.data_ptr(), k_cache.data_ptr(),
                 v_cache.data_ptr(), positions.data_ptr<long>(),
                 slot_mapping.data_ptr<long>(), cos_sin.data_ptr<float>(), qw,
                 kw, (float)eps, T, Hq, Hk, D, bs, row_stride,
                 is_fp8(k_cache) ? 1 : 0, cur_stream());
}

// out[M,N] = x[M,K] @ w[N,K]^T (+ res), bf16 in/out, fp32 accumulate.
// bm/bn pick the macro-tile; M%bm==0 and K%64==0 required (caller falls back
// to torch.mm otherwise). res, when given, is added to the output (fused
// residual epilogue).
torch::Tensor gemm_tn(torch::Tensor x, torch::Tensor w,
                      c10::optional<torch::Tensor> res, long bm, long bn,
                      long swz, long xcd_swz) {
  CHECK_CUDA(x); CHECK_BF16(x); CHECK_CUDA(w); CHECK_BF16(w);
  TORCH_CHECK(x.is_contiguous() && w.is_contiguous(), "contiguous required");
  const long M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(w.size(1) == K, "K mismatch");
  TORCH_CHECK(M % bm == 0 && K % 64 == 0, "shape not tile-divisible");
  auto out = torch::empty({M, N}, x.options());
  const void* rp = nullptr;
  if (res.has_value()) {
    CHECK_CUDA(*res); CHECK_BF16(*res);
    TORCH_CHECK(res->is_contiguous() && res->size(0) == M && res->size(1) == N,
                "res shape");
    rp = res->data_ptr();
  }
  sutro_gemm_tn_launch(out.data_ptr(), x.data_ptr(), w.data_ptr(), rp, (int)M,
                       (int)N, K, (int)bm, (int)bn, (int)swz, (int)xcd_swz,
                       cur_stream());
  return out;
}

torch::Tensor mfma32_probe(torch::Tensor a, torch::Tensor b) {
  CHECK_CUDA(a); CHECK_BF16(a);
  auto c = torch::zeros({32, 32}, a.options().dtype(at::kFloat));
  sutro_mfma32_probe(c.data_ptr<float>(), a.data_ptr(), b.data_ptr(),
                     cur_stream());
  return c;
}

torch::Tensor mfma16_probe(torch::Tensor a, torch::Tensor b) {
  CHECK_CUDA(a); CHECK_BF16(a);
  auto c = torch::zeros({16, 16}, a.options().dtype(at::kFloat));
  sutro_mfma16_probe(c.data_ptr<float>(), a.data_ptr(), b.data_ptr(),
                     cur_stream());
  return c;
}

static bool tile_rows_ok(long bm) {
  return bm == 32 || bm == 64 || bm == 128 || bm == 256;
}

void grouped_gemm(torch::Tensor out, torch::Tensor a, torch::Tensor w,
                  c10::optional<torch::Tensor> row_tok, torch::Tensor tile_off,
                  torch::Tensor counts, long max_tiles, bool gate_silu,
                  long bm) {
  TORCH_CHECK(tile_rows_ok(bm), "bm must be 32, 64, 128 or 256");
  CHECK_CUDA(a); CHECK_CONTIG(a); CHECK_BF16(a);
  CHECK_CUDA(w); CHECK_CONTIG(w); CHECK_BF16(w);
  CHECK_CONTIG(out); CHECK_BF16(out);
  const long E = w.size(0), N = w.size(1), K = w.size(2);
  const long n_cols = gate_silu ? N / 2 : N;
  TORCH_CHECK(K % 64 == 0 && n_cols % 64 == 0,
              "grouped_gemm needs K, n_cols multiples of 64 (K=", K,
              ", n_cols=", n_cols, ")");
  TORCH_CHECK(bm != 256 || n_cols % (gate_silu ? 128 : 256) == 0,
              "tiles of 256 rows need n_cols a multiple of 256 (gated: 128)");
  TORCH_CHECK(a.size(1) == K, "A K mismatch");
  TORCH_CHECK(out.size(1) == n_cols, "out width mismatch");
  TORCH_CHECK(tile_off.scalar_type() == at::kInt
              && counts.scalar_type() == at::kInt, "tile_off/counts int32");
  TORCH_CHECK(tile_off.numel() == E + 1 && counts.numel() == E, "seg sizes");
  const int* rt = nullptr;
  if (row_tok.has_value()) {
    TORCH_CHECK(row_tok->scalar_type() == at::kInt, "row_tok int32");
    rt = row_tok->data_ptr<int>();
  }
  sutro_grouped_gemm(out.data_ptr(), a.data_ptr(), a.size(0), w.data_ptr(), rt,
                     tile_off.data_ptr<int>(), counts.data_ptr<int>(), (int)E,
                     (int)max_tiles, (int)n_cols, K, gate_silu ? 1 : 0,
                     (int)bm, cur_stream());
}

void moe_combine(torch::Tensor out, torch::Tensor rows, torch::Tensor padpos,
                 torch::Tensor w) {
  CHECK_CUDA(rows); CHECK_CONTIG(rows); CHECK_BF16(rows);
  CHECK_CONTIG(out); CHECK_BF16(out);
  const long T = out.size(0), h = out.size(1), k = padpos.size(1);
  TORCH_CHECK(h % 8 == 0, "h must be a multiple of 8");
  const bool pos64 = padpos.scalar_type() == at::kLong;
  TORCH_CHECK(pos64 || padpos.scalar_type() == at::kInt,
              "padpos must be int64 or int32");
  TORCH_CHECK(w.scalar_type() == at::kFloat, "w must be f32");
  TORCH_CHECK(padpos.is_contiguous() && w.is_contiguous(), "contig");
  sutro_moe_combine(out.data_ptr(), rows.data_ptr(),
                    padpos.data_ptr(), pos64 ? 1 : 0, w.data_ptr<float>(),
                    (int)T, (int)h, (int)k, cur_stream());
}

// router logits bf16 [T, E] -> the top k experts of every token and their
// layout in segments of `bm` rows: weights fp32 [T, k], tile_off int32
// [segs + 1], counts int32 [segs], padpos int32 [T, k]; row_tok int32 (given)
// names the token of every row. This rank holds experts base..base+n_local-1;
// with fewer than E of them, one more segment takes the other choices.
std::vector<torch::Tensor> moe_layout(torch::Tensor logits, long k, long base,
                                      long n_local, long bm,
                                      torch::Tensor row_tok) {
  CHECK_CUDA(logits); CHECK_CONTIG(logits); CHECK_BF16(logits);
  CHECK_CUDA(row_tok); CHECK_CONTIG(row_tok);
  TORCH_CHECK(row_tok.scalar_type() == at::kInt, "row_tok int32");
  const long T = logits.size(0), E = logits.size(1);
  TORCH_CHECK(k >= 1 && k <= 64 && k <= E && E <= 1024,
              "router: up to 64 of up to 1024 experts");
  TORCH_CHECK(base >= 0 && n_local >= 1 && base + n_local <= E, "local experts");
  TORCH_CHECK(tile_rows_ok(bm), "bm must be 32, 64, 128 or 256");
  const long segs = n_local + (n_local < E ? 1 : 0);
  TORCH_CHECK(row_tok.numel() >= T * k + segs * (bm - 1), "row_tok too short");
  TORCH_CHECK(T * k + segs * bm < (1l << 31), "too many rows");
  auto i32 = row_tok.options();
  auto idx = torch::empty({T, k}, i32);
  auto wts = torch::empty({T, k}, i32.dtype(at::kFloat));
  auto tile_off = torch::empty({segs + 1}, i32);
  auto counts = torch::empty({segs}, i32);
  auto padpos = torch::empty({T, k}, i32);
  torch::Tensor scratch;
  if (const long n = mix_moe_dispatch_scratch(T * k, (int)segs))
    scratch = torch::empty({n}, i32);
  sutro_moe_topk(idx.data_ptr<int>(), wts.data_ptr<float>(), logits.data_ptr(),
                 T, (int)E, (int)k, (int)base, (int)n_local, cur_stream());
  mix_moe_dispatch(row_tok.data_ptr<int>(), tile_off.data_ptr<int>(),
                   counts.data_ptr<int>(), padpos.data_ptr<int>(),
                   idx.data_ptr<int>(), nullptr, T * k, (int)k, (int)segs,
                   (int)bm, row_tok.numel(),
                   scratch.defined() ? scratch.data_ptr<int>() : nullptr,
                   nullptr, nullptr, cur_stream());
  return {wts, tile_off, counts, padpos};
}

// out [M, N] = x [M, K] @ w [N, K]^T (+ bias), or, `gated`, silu of the first
// N rows of w [2 N, K] times the other N; bf16, up to 32 rows
torch::Tensor linear_skinny(torch::Tensor x, torch::Tensor w,
                            c10::optional<torch::Tensor> bias, bool gated) {
  TORCH_CHECK(x.is_cuda() && w.is_cuda() && x.device() == w.device(),
              "operands on one GPU");
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 &&
              w.scalar_type() == at::kBFloat16, "bf16 operands");
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && w.is_contiguous() &&
              x.stride(1) == 1, "matrix operands, rows contiguous");
  const long M = x.size(0), K = x.size(1), rows = w.size(0);
  const long N = gated ? rows / 2 : rows;
  TORCH_CHECK(w.size(1) == K && K >= 32 && K % 32 == 0 && N % 4 == 0 &&
              (!gated || rows == 2 * N) && M >= 1 && M <= 32 &&
              rows < (1l << 31) && K < (1l << 31), "unsupported sizes");
  TORCH_CHECK(x.stride(0) % 8 == 0 && (size_t)x.data_ptr() % 16 == 0 &&
              (size_t)w.data_ptr() % 16 == 0, "16-byte rows");
  const void* b = nullptr;
  if (bias.has_value()) {
    TORCH_CHECK(bias->is_cuda() && bias->scalar_type() == at::kBFloat16 &&
                bias->is_contiguous() && bias->numel() == rows, "bias");
    b = bias->data_ptr();
  }
  auto out = torch::empty({M, N}, x.options());
  sutro_linear_skinny(out.data_ptr(), N, x.data_ptr(), x.stride(0),
                      w.data_ptr(), b, (int)M, (int)N, (int)K, gated ? 1 : 0,
                      cur_stream());
  return out;
}

// linear layer over 2 to 256 rows (csrc/gemm_mid.hip), `gated` with silu_mul
torch::Tensor linear_mid(torch::Tensor x, torch::Tensor w,
                         c10::optional<torch::Tensor> bias, bool gated) {
  TORCH_CHECK(x.is_cuda() && w.is_cuda() && x.device() == w.device(),
              "operands on one GPU");
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 &&
              w.scalar_type() == at::kBFloat16, "bf16 operands");
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && w.is_contiguous() &&
              x.stride(1) == 1, "matrix operands, rows contiguous");
  const long M = x.size(0), K = x.size(1), rows = w.size(0), ld = x.stride(0);
  const long N = gated ? rows / 2 : rows;
  TORCH_CHECK(w.size(1) == K && K >= 256 && K % 256 == 0 && N >= 4 && N % 4 == 0 &&
              (!gated || rows == 2 * N) && M >= 1 && M <= 256 && K < (1l << 20) &&
              rows < (1l << 24) && ld >= K && M * ld < (1l << 30) &&
              (N + 128) * K < (gated ? 1l << 30 : 1l << 44), "unsupported sizes");
  TORCH_CHECK(ld % 8 == 0 && (size_t)x.data_ptr() % 16 == 0 &&
              (size_t)w.data_ptr() % 16 == 0, "16-byte rows");
  const void* b = nullptr;
  if (bias.has_value()) {
    TORCH_CHECK(!gated && bias->is_cuda() && bias->scalar_type() == at::kBFloat16 &&
                bias->is_contiguous() && bias->numel() == rows, "bias");
    b = bias->data_ptr();
  }
  auto out = torch::empty({M, N}, x.options());
  sutro_linear_mid(out.data_ptr(), x.data_ptr(), ld, w.data_ptr(), b, (int)M, (int)N,
                   (int)K, gated ? 1 : 0, cur_stream());
  return out;
}

// rows of x and of w (`rows` in all) in a tile of linear_mid
std::vector<long> mid_tile(long M, long rows, long K, bool gated) {
  int t[2];
  sutro_mid_tile(t, (int)M, (int)(gated ? rows / 2 : rows), (int)K, gated ? 1 : 0);
  return {t[0], t[1]};
}

// (y w^T or, `gated`, its silu unit; x + residual), y the RMSNorm of x + residual,
// one row
std::vector<torch::Tensor> norm_linear(torch::Tensor x, torch::Tensor residual,
                                       torch::Tensor norm_w, double eps,
                                       torch::Tensor w, bool gated) {
  for (const auto& t : {x, residual, norm_w, w})
    TORCH_CHECK(t.is_cuda() && t.device() == x.device() &&
                t.scalar_type() == at::kBFloat16 && t.is_contiguous() &&
                (size_t)t.data_ptr() % 16 == 0,
                "contiguous bf16 operands on one GPU, 16-byte rows");
  TORCH_CHECK(x.dim() == 2 && x.size(0) == 1 && x.sizes() == residual.sizes() &&
              w.dim() == 2, "one row");
  const long K = x.size(1), rows = w.size(0), N = gated ? rows / 2 : rows;
  TORCH_CHECK(norm_w.numel() == K && w.size(1) == K && K >= 32 &&
              K <= 4096 && K % 32 == 0 && N >= 1 && N < (1l << 30) &&
              rows == (gated ? 2 * N : N), "unsupported sizes");
  auto out = torch::empty({1, N}, x.options());
  auto sum = torch::empty_like(residual);
  sutro_norm_linear(out.data_ptr(), x.data_ptr(), residual.data_ptr(),
                    sum.data_ptr(), norm_w.data_ptr(), (float)eps, w.data_ptr(),
                    (int)N, (int)K, gated ? 1 : 0, cur_stream());
  return {out, sum};
}

static void check_gated(const torch::Tensor& x, const torch::Tensor& w, long N) {
  TORCH_CHECK(x.is_cuda() && w.is_cuda() && x.device() == w.device(),
              "operands on one GPU");
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 &&
              w.scalar_type() == at::kBFloat16, "bf16 operands");
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.is_contiguous() &&
              w.is_contiguous(), "contiguous matrices");
  const long M = x.size(0), K = x.size(1);
  TORCH_CHECK(w.size(1) == K && w.size(0) >= 2 * N && K > 0 && K % 64 == 0 &&
              N > 0 && N % 128 == 0 && M >= 1 && M * K < (1l << 30) &&
              K < (1l << 21) && w.size(0) < (1l << 25), "unsupported sizes");
  TORCH_CHECK((size_t)x.data_ptr() % 16 == 0 && (size_t)w.data_ptr() % 16 == 0,
              "16-byte rows");
}

// silu of x [M, K] times the first N rows of w [2 N, K], times x and the others
torch::Tensor linear_silu_mul(torch::Tensor x, torch::Tensor w) {
  const long N = w.size(0) / 2;
  check_gated(x, w, N);
  TORCH_CHECK(w.size(0) == 2 * N, "gate and up rows");
  auto out = torch::empty({x.size(0), N}, x.options());
  sutro_linear_silu_mul(out.data_ptr(), x.data_ptr(), w.data_ptr(),
                        (int)x.size(0), (int)N, x.size(1), cur_stream());
  return out;
}

// GELU by tanh of the first N columns of x w^T + bias times the next N, and the rest
std::vector<torch::Tensor> linear_gelu_mul(torch::Tensor x, torch::Tensor w,
                                           c10::optional<torch::Tensor> bias,
                                           long N) {
  check_gated(x, w, N);
  const long more = w.size(0) - 2 * N;
  TORCH_CHECK(more % 256 == 0, "unsupported sizes");
  if (bias.has_value())
    TORCH_CHECK(bias->scalar_type() == at::kBFloat16 && bias->is_contiguous() &&
                bias->dim() == 1 && bias->size(0) == w.size(0) &&
                bias->device() == x.device() &&
                (size_t)bias->data_ptr() % 8 == 0, "bias");
  auto out = torch::empty({x.size(0), N}, x.options());
  auto rest = torch::empty({x.size(0), more}, x.options());
  sutro_linear_gelu_mul(out.data_ptr(), rest.data_ptr(), x.data_ptr(),
                        w.data_ptr(),
                        bias.has_value() ? bias->data_ptr() : nullptr,
                        (int)x.size(0), (int)N, (int)more, x.size(1), cur_stream());
  return {out, rest};
}

// heads of 128 of x w^T: query heads normed and rotated (returned), key heads likewise
// and value heads as they are to the tokens' slots
torch::Tensor linear_heads(torch::Tensor x, torch::Tensor w, torch::Tensor k_cache,
                           torch::Tensor v_cache, torch::Tensor positions,
                           torch::Tensor slot_mapping, torch::Tensor cos_sin,
                           c10::optional<torch::Tensor> q_norm_w,
                           c10::optional<torch::Tensor> k_norm_w, double eps) {
  CHECK_CONTIG(k_cache); CHECK_CONTIG(v_cache); CHECK_CONTIG(cos_sin);
  CHECK_BF16(k_cache); CHECK_BF16(v_cache);
  CHECK_CONTIG(positions); CHECK_CONTIG(slot_mapping);
  check_gated(x, w, 128);
  for (const auto& t : {k_cache, v_cache, positions, slot_mapping, cos_sin})
    TORCH_CHECK(t.device() == x.device(), "operands on one GPU");
  for (const auto& n : {q_norm_w, k_norm_w})
    TORCH_CHECK(!n || n->device() == x.device(), "norm weights on one GPU");
  const long M = x.size(0), K = x.size(1), bs = k_cache.size(2);
  const long Hk = k_cache.size(1), Hq = w.size(0) / 128 - 2 * Hk;
  TORCH_CHECK(k_cache.dim() == 4 && k_cache.size(3) == 128 &&
              v_cache.sizes() == k_cache.sizes() && bs > 0 && (bs & (bs - 1)) == 0 &&
              k_cache.numel() >> 7 < (1l << 32) && Hk > 0 && Hq > 0 && Hq % 2 == 0 &&
              w.size(0) == (Hq + 2 * Hk) * 128 && K >= 192, "unsupported sizes");
  TORCH_CHECK(positions.numel() == M && slot_mapping.numel() == M &&
              cos_sin.dim() == 2 && cos_sin.size(1) == 128, "tokens");
  for (const auto& n : {q_norm_w, k_norm_w})
    TORCH_CHECK(!n || (n->scalar_type() == at::kBFloat16 && n->is_contiguous() &&
                       n->numel() == 128 && (size_t)n->data_ptr() % 8 == 0), "norm");
  for (const auto& t : {k_cache, v_cache, cos_sin})
    TORCH_CHECK((size_t)t.data_ptr() % 16 == 0, "16-byte rows");
  auto q = torch::empty({M, Hq, 128}, x.options());
  int shift = 0;
  while (1l << shift < bs) ++shift;
  sutro_linear_heads(q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
                     x.data_ptr(), w.data_ptr(), positions.data_ptr<long>(),
                     slot_mapping.data_ptr<long>(), cos_sin.data_ptr<float>(),
                     q_norm_w ? q_norm_w->data_ptr() : nullptr,
                     k_norm_w ? k_norm_w->data_ptr() : nullptr, (float)eps, (int)M,
                     (int)Hq, (int)Hk, shift, K, cur_stream());
  return q;
}

void sampler_fused(torch::Tensor logits, torch::Tensor temps,
                   torch::Tensor topps, torch::Tensor topks, torch::Tensor us,
                   c10::optional<torch::Tensor> mask, long vl,
                   torch::Tensor out_tok, torch::Tensor out_lp, bool greedy) {
  CHECK_CUDA(logits); CHECK_CONTIG(logits);
  const bool f32 = logits.scalar_type() == at::kFloat;
  TORCH_CHECK(f32 || logits.scalar_type() == at::kBFloat16,
              "logits must be bf16 or f32");
  const long n = logits.size(0), v_row = logits.size(1);
  TORCH_CHECK(vl <= v_row, "vocab_limit exceeds logits row");
  TORCH_CHECK(temps.numel() >= n && topps.numel() >= n && topks.numel() >= n
              && us.numel() >= n, "param tensors too small");
  TORCH_CHECK(topks.scalar_type() == at::kInt, "topks must be int32");
  const unsigned int* mptr = nullptr;
  int w_words = 0;
  if (mask.has_value()) {
    auto& mt = mask.value();
    CHECK_CUDA(mt); CHECK_CONTIG(mt);
    TORCH_CHECK(mt.scalar_type() == at::kInt, "mask must be int32 packed");
    TORCH_CHECK(mt.size(0) == n, "mask rows mismatch");
    w_words = (int)mt.size(1);
    TORCH_CHECK((long)w_words * 32 >= vl, "mask too narrow for vocab_limit");
    mptr = (const unsigned int*)mt.data_ptr();
  }
  sutro_sampler_fused(logits.data_ptr(), f32 ? 1 : 0,
                      temps.data_ptr<float>(), topps.data_ptr<float>(),
                      topks.data_ptr<int>(), us.data_ptr<float>(), mptr,
                      (int)n, v_row, (int)vl, w_words,
                      out_tok.data_ptr<int>(), out_lp.data_ptr<float>(),
                      greedy ? 1 : 0, cur_stream());
}

static uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

// len(r.prompt_token_ids) + len(r.output_token_ids), straight from the fields of a plain
// request; r.total_len of any other object
static uint64_t total_len(PyObject* r, PyObject* plain) {
  static PyObject* const prompt = PyUnicode_InternFromString("prompt_token_ids");
  static PyObject* const output = PyUnicode_InternFromString("output_token_ids");
  PyObject** fields = (PyObject*)Py_TYPE(r) == plain ? _PyObject_GetDictPtr(r) : nullptr;
  if (fields && *fields) {
    PyObject* p = PyDict_GetItemWithError(*fields, prompt);
    PyObject* o = p ? PyDict_GetItemWithError(*fields, output) : nullptr;
    const Py_ssize_t a = o ? PyObject_Size(p) : -1, b = a >= 0 ? PyObject_Size(o) : -1;
    if (b >= 0) return (uint64_t)(a + b);
    if (PyErr_Occurred()) throw py::error_already_set();
  }
  return py::cast<uint64_t>(py::handle(r).attr("total_len"));
}

// out[i] = the uniform of (seed, step) for the rows i in `rows`: 1024 rows 110 us in
// Python, most of it for the steps, and 25 here. `plain`: the class whose fields are
// read directly.
void seeded_uniforms(torch::Tensor out, py::sequence reqs,
                     py::array_t<int64_t, py::array::c_style> rows,
                     py::array_t<uint64_t, py::array::c_style> seeds,
                     c10::optional<py::array_t<int64_t, py::array::c_style>> steps,
                     py::object plain) {
  TORCH_CHECK(!out.is_cuda() && out.scalar_type() == at::kFloat && out.dim() == 1 &&
              out.is_contiguous(), "fp32 on the host");
  TORCH_CHECK(rows.ndim() == 1 && seeds.ndim() == 1 && rows.size() == seeds.size() &&
              (!steps || (steps->ndim() == 1 && steps->size() >= out.numel())),
              "a seed a row");
  const py::object fast = py::reinterpret_steal<py::object>(
      PySequence_Fast(reqs.ptr(), "a sequence of requests"));
  if (!fast) throw py::error_already_set();
  float* o = out.data_ptr<float>();
  for (py::ssize_t k = 0; k < rows.size(); ++k) {
    const int64_t i = rows.data()[k];
    TORCH_CHECK(i >= 0 && i < out.numel() &&
                i < PySequence_Fast_GET_SIZE(fast.ptr()), "row");
    const uint64_t step = steps ? (uint64_t)steps->data()[i]
                                : total_len(PySequence_Fast_GET_ITEM(fast.ptr(), i),
                                            plain.ptr());
    const uint64_t key = splitmix64(seeds.data()[k] ^ splitmix64(step));
    o[i] = (float)((double)(key >> 11) * (1.0 / (1ull << 53)));
  }
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("seeded_uniforms", &seeded_uniforms, "uniforms of (seed, step) pairs",
        py::arg("out"), py::arg("reqs"), py::arg("rows"), py::arg("seeds"),
        py::arg("steps"), py::arg("plain"));
  m.def("rmsnorm", &rmsnorm, "RMSNorm (bf16, CDNA4)");
  m.def("fused_add_rmsnorm", &fused_add_rmsnorm, "residual+=x; x=rmsnorm");
  m.def("silu_mul", &silu_mul, "fused SwiGLU");
  m.def("rope_and_cache", &rope_and_cache, "RoPE + paged KV write");
  m.def("qkv_prep", &qkv_prep, "fused qk-norm + RoPE + KV write + q gather");
  m.def("mean_pool_normalize", &mean_pool_normalize, "varlen mean pool + L2");
  m.def("paged_attention", &paged_attention, "paged prefill+decode attention");
  m.def("mfma32_probe", &mfma32_probe, "MFMA fragment-layout probe");
  m.def("mfma16_probe", &mfma16_probe, "16x16 MFMA fragment-layout probe");
  m.def("moe_combine", &moe_combine, "fused MoE weighted gather-combine");
  m.def("linear_skinny", &linear_skinny, "linear layer over few rows");
  m.def("mid_tile", &mid_tile, "tile of linear_mid");
  m.def("linear_mid", &linear_mid, "linear layer over 2 to 256 rows");
  m.def("norm_linear", &norm_linear,
        "linear layer of one row behind an addition and RMSNorm");
  m.def("linear_gelu_mul", &linear_gelu_mul,
        "linear layer with the GELU gate behind its first columns, many rows");
  m.def("linear_heads", &linear_heads,
        "QKV projection with qk-norm, RoPE and KV write behind it, many rows");
  m.def("linear_silu_mul", &linear_silu_mul,
        "linear layer with the silu gate behind it, many rows");
  m.def("moe_layout", &moe_layout, "softmax top-k router + expert segments");
  m.def("grouped_gemm", &grouped_gemm,
        "dropless MoE grouped GEMM (padded segments, static grid)");
  m.def("sampler_fused", &sampler_fused,
        "fused mask+temp+topk/topp+sample+logprob (no sort)", py::arg("logits"),
        py::arg("temps"), py::arg("topps"), py::arg("topks"), py::arg("us"),
        py::arg("mask"), py::arg("vl"), py::arg("out_tok"), py::arg("out_lp"),
        py::arg("greedy") = false);
  m.def("gemm_tn", &gemm_tn, "bf16 TN GEMM (MFMA, glds dbuf)",
        py::arg("x"), py::arg("w"), py::arg("res") = c10::nullopt,
        py::arg("bm") = 256, py::arg("bn") = 256, py::arg("swz") = 2,
        py::arg("xcd_swz") = 0);
}
