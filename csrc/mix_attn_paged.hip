// Local (chunked / windowed) paged attention of the layer-list decoders with
// bf16 pages of 32 tokens and equal key and value sizes of 64 or 128: the
// kernels of attn_paged.h with masks, kept first keys, distance bias, sinks,
// gates and an output section. Other shapes run on mix_attn_mfma.hip (prompt
// pieces) and mix_attn.hip (single tokens, fp32).
//
// Against those kernels, per call on 30-32 k prompt tokens, 16 heads, 4 kv
// heads, 128: chunk 1024 over prompts of 2 k 1165 -> 302 us (455 TFLOP/s),
// window 1024 with 64 kept keys over 2.3 k 1128 -> 378 us, window 1024 with a
// distance bias over 490 keys 455 -> 185 us. Single tokens (with the join):
// 61 rows of 490 keys 82 -> 27 us, 13 rows of 1088 keys 49 -> 16 us; 16 rows
// of a chunk that has just begun 10 -> 11 us (the join finds nothing to do).
#include "mix_common.h"
#include "attn_paged.h"

// pages that a single token sees at most
static int most_pages(int bt_stride, int chunk, int window, int keep_first) {
  long pages = bt_stride;
  if (chunk > 0) pages = min(pages, (long)(chunk + PA_PG - 1) / PA_PG + 1);
  if (window > 0)
    pages = min(pages, (long)(window + PA_PG - 1) / PA_PG + 1 +
                           (keep_first + PA_PG - 1) / PA_PG);
  return (int)pages;
}

// runs these are cut into (see attn_paged.h)
extern "C" int mix_paged_splits(long rows, int Hk, int bt_stride, int chunk,
                                int window, int keep_first) {
  return pa_splits(rows, Hk,
                   most_pages(bt_stride, chunk, window, keep_first));
}

// prompt pieces of n_tiles entries of the tile map (n_prompts of them), then the n_rows single
// tokens from row t0 on (either may be none)
extern "C" void mix_paged_attention(
    void* out, long ldo, int out_off, const void* q, const void* k_cache,
    const void* v_cache, const int* bt, int bt_stride, const int* seq_lens,
    const int* qlocs, const int* tile_seq, const int* tile_q0, int n_tiles,
    int n_prompts, const int* token_seq, long t0, int n_rows, int nsplit, float* part_o,
    float* part_ml, float scale, int chunk, int window, const void* proj,
    long ld, int gate_off, int gate_n, float out_scale, const float* bias_r1,
    const float* bias_r2, int sink, const float* sink_w, int keep_first, int H,
    int Hk, int D, hipStream_t s) {
  PagedArgs A = {};
  A.out = (u16*)out;
  A.ldo = ldo;
  A.out_off = out_off;
  A.q = (const u16*)q;
  A.kc = (const u8*)k_cache;
  A.vc = (const u8*)v_cache;
  A.bt = bt;
  A.bt_stride = bt_stride;
  A.seq_lens = seq_lens;
  A.qlocs = qlocs;
  A.Hq = H;
  A.Hk = Hk;
  A.scale = scale * PA_LOG2E;
  A.tile_seq = tile_seq;
  A.tile_q0 = tile_q0;
  A.n_tiles = n_tiles;
  A.token_seq = token_seq;
  A.t0 = t0;
  A.n_rows = n_rows;
  A.nsplit = nsplit;
  A.part_o = part_o;
  A.part_ml = part_ml;
  A.chunk = chunk;
  A.window = window;
  A.keep_first = keep_first;
  A.r1 = bias_r1;
  A.r2 = bias_r2;
  A.sink = sink;
  A.sink_w = sink_w;
  A.proj = (const u16*)proj;
  A.ld = ld;
  A.gate_off = gate_off;
  A.gate_n = gate_n;
  A.out_scale = out_scale;
  if (n_tiles > 0) {
    if (D == 128) pa_launch_prefill<128, false, true>(A, n_prompts, s);
    else pa_launch_prefill<64, false, true>(A, n_prompts, s);
  }
  if (n_rows > 0) {
    const int most = most_pages(bt_stride, chunk, window, keep_first);
    if (D == 128) pa_launch_decode<128, false, true>(A, most, s);
    else pa_launch_decode<64, false, true>(A, most, s);
  }
}
