"""Op dispatch: hand-written CDNA4 HIP kernels on GPU, torch reference on CPU.

The HIP extension (`sutro_amd._C`, built by `setup.py build_ext --inplace` or
`__graft_entry__.build()`) is REQUIRED on GPU: any op called with CUDA(HIP)
tensors raises if the extension is missing — no silent eager fallback on the
hot path.
"""

from __future__ import annotations

import functools
import os
from typing import Optional

import torch
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from . import torch_ref

_C = None
_C_ERR: Optional[str] = None
try:
    from sutro_amd import _C as _C  # type: ignore
except Exception as e:  # pragma: no cover - exercised only without built ext
    _C_ERR = f"{type(e).__name__}: {e}"


def hip_available() -> bool:
    return _C is not None


def _require_hip():
    if _C is None:
        raise RuntimeError(
            "sutro_amd HIP extension (_C) is not built but a GPU tensor was passed. "
            "Build it with `python setup.py build_ext --inplace` "
            f"(import error: {_C_ERR})"
        )
    return _C


# Env escape hatch for A/B profiling only (never the default).
_FORCE_REF = os.environ.get("SUTRO_AMD_FORCE_TORCH_REF", "0") == "1"


def _use_hip(t: torch.Tensor) -> bool:
    return t.is_cuda and not _FORCE_REF


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    if _use_hip(x):
        out = torch.empty_like(x)
        _require_hip().rmsnorm(out, x, weight, eps)
        return out
    return torch_ref.rmsnorm(x, weight, eps)


def fused_add_rmsnorm(x, residual, weight, eps: float):
    if _use_hip(x):
        # in-place: residual += x; x_out = rmsnorm(residual)
        _require_hip().fused_add_rmsnorm(x, residual, weight, eps)
        return x, residual
    return torch_ref.fused_add_rmsnorm(x, residual, weight, eps)


def silu_mul(x: torch.Tensor) -> torch.Tensor:
    if _use_hip(x):
        T, two_i = x.shape
        out = torch.empty((T, two_i // 2), dtype=x.dtype, device=x.device)
        _require_hip().silu_mul(out, x)
        return out
    return torch_ref.silu_mul(x)


def fused_qkv_prep(
    qkv: torch.Tensor,            # [T, Hq*D + 2*Hk*D] (qkv GEMM output)
    num_heads: int, num_kv_heads: int, head_dim: int,
    positions: torch.Tensor, slot_mapping: torch.Tensor,
    k_cache: torch.Tensor, v_cache: torch.Tensor,
    cos_sin: torch.Tensor,
    q_norm_w: Optional[torch.Tensor] = None,
    k_norm_w: Optional[torch.Tensor] = None,
    eps: float = 1e-6,
) -> torch.Tensor:
    """Per-head qk-RMSNorm + RoPE + paged KV write; returns contiguous q
    [T, Hq, D]. One fused kernel on GPU (reads the GEMM output in place)."""
    T = qkv.shape[0]
    if _use_hip(qkv):
        q_out = torch.empty((T, num_heads, head_dim), dtype=qkv.dtype,
                            device=qkv.device)
        _require_hip().qkv_prep(qkv, q_out, k_cache, v_cache, positions,
                                slot_mapping, cos_sin, q_norm_w, k_norm_w, eps)
        return q_out
    q_size = num_heads * head_dim
    kv_size = num_kv_heads * head_dim
    q, k, v = qkv.split([q_size, kv_size, kv_size], dim=-1)
    q = q.reshape(T, num_heads, head_dim).contiguous()
    k = k.reshape(T, num_kv_heads, head_dim).contiguous()
    v = v.reshape(T, num_kv_heads, head_dim).contiguous()
    if q_norm_w is not None:
        q = torch_ref.rmsnorm(q, q_norm_w, eps)
    if k_norm_w is not None:
        k = torch_ref.rmsnorm(k, k_norm_w, eps)
    q, k = torch_ref.apply_rope(q, k, positions, cos_sin)
    torch_ref.write_kv_cache(k, v, k_cache, v_cache, slot_mapping)
    return q


def rope_and_cache(
    q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
    positions: torch.Tensor, slot_mapping: torch.Tensor,
    k_cache: torch.Tensor, v_cache: torch.Tensor,
    cos_sin: torch.Tensor,
) -> torch.Tensor:
    """Apply RoPE to q,k (in place on GPU) and scatter k,v into the paged cache.
    Returns q (rotated)."""
    if _use_hip(q):
        _require_hip().rope_and_cache(q, k, v, positions, slot_mapping,
                                      k_cache, v_cache, cos_sin)
        return q
    q, k = torch_ref.apply_rope(q, k, positions, cos_sin)
    torch_ref.write_kv_cache(k, v, k_cache, v_cache, slot_mapping)
    return q


_EMPTY_I32: Optional[torch.Tensor] = None


def paged_attention(
    q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
    block_tables: torch.Tensor, seq_lens: torch.Tensor,
    query_start_locs: torch.Tensor, scale: float,
    num_decodes_tail: int = 0,
    tile_seq: Optional[torch.Tensor] = None,
    tile_q0: Optional[torch.Tensor] = None,
    prefill_token_count: int = 0,
) -> torch.Tensor:
    """Attention of new tokens vs full cached KV (causal within the new chunk).

    `num_decodes_tail`: trailing sequences that are single-token decodes (the
    GPU path routes them to the decode kernel). `tile_seq`/`tile_q0`: int32
    device arrays mapping prefill q-tiles of 32 rows to (seq, local row)."""
    if _use_hip(q):
        out = torch.empty_like(q)
        if tile_seq is None:
            tile_seq = torch.empty(0, dtype=torch.int32, device=q.device)
            tile_q0 = tile_seq
        _require_hip().paged_attention(out, q, k_cache, v_cache, block_tables,
                                       seq_lens, query_start_locs, scale,
                                       num_decodes_tail, tile_seq, tile_q0,
                                       prefill_token_count)
        return out
    return torch_ref.paged_attention(q, k_cache, v_cache, block_tables,
                                     seq_lens, query_start_locs, scale)


def mean_pool_normalize(hidden: torch.Tensor, query_start_locs: torch.Tensor) -> torch.Tensor:
    if _use_hip(hidden):
        S = query_start_locs.numel() - 1
        out = torch.empty((S, hidden.shape[-1]), dtype=torch.float32, device=hidden.device)
        _require_hip().mean_pool_normalize(out, hidden, query_start_locs)
        return out
    return torch_ref.mean_pool_normalize(hidden, query_start_locs)


def seeded_uniforms(out, reqs, rows, seeds, steps, plain) -> bool:
    """out[i] = the uniform of (seed, step) of request i, for i in `rows`
    (engine/sampler.py); False where there is no native code for it."""
    if _C is None:
        return False
    _C.seeded_uniforms(out, reqs, rows, seeds, steps, plain)
    return True


def sampler_fused(logits, temps, top_ps, top_ks, u, packed_mask, vocab_limit,
                  out_tok, out_lp, greedy: bool = False):
    """Fused mask+temperature+top-k/top-p+sample+logprob (csrc/sampler.hip).
    GPU-only: logits must be CUDA; raises if the extension is missing. `greedy`:
    all rows have a temperature of 0 (the result is the same, in one launch; a row of
    8192 logits takes 5 us and without the word 15)."""
    _require_hip().sampler_fused(logits, temps, top_ps, top_ks, u,
                                 packed_mask, vocab_limit, out_tok, out_lp,
                                 greedy)


_functions, _dispatches = (torch._C._len_torch_function_stack,
                           torch._C._len_torch_dispatch_stack)
_transforms = torch._C._functorch.peek_interpreter_stack
_tracing, _autocast = torch._C._is_tracing, torch._C._is_any_autocast_enabled


def _unwatched() -> bool:
    """Whether nothing of torch's has to see an operation on plain tensors:
    function and dispatch modes (counters, fake tensors, graph recorders),
    vmap and the other transforms, forward-mode derivatives, a compiler,
    autocast. (A default device is a function mode too, and minds nothing.)"""
    if _functions() and not all(isinstance(m, DeviceContext)
                                for m in _get_current_function_mode_stack()):
        return False
    return not (_dispatches() or _transforms() is not None or _autocast()
                or forward_ad._current_level >= 0
                or torch.compiler.is_compiling())


def _two_rows(rows: int, K: int, gated: bool) -> bool:
    return (rows * K <= (64 if gated else 24) << 20 or rows >= 16384
            or (rows > 8192 and K <= 5120) or (rows < 8192 and K >= 16384))


def _long_weights(M: int, rows: int, K: int) -> bool:
    """Larger matrices over 3 to 32 rows (both sides in `_few_rows`). Nearly all with a
    k that is a multiple of 256 and not above 4096 go to csrc/gemm_mid.hip before they
    come here; this decides for the others."""
    if 16384 < rows <= 24576 and rows * K <= 80 << 20 and K <= 4096:
        return M <= 16                    # the library has no good tile there
    if rows <= 8192 and K <= 4096:
        return M <= 12
    if K <= 2048 or K == 4096:
        most = 8
        # a last round of workgroups (of 32 weight rows) with many CUs idle
        if (rows > 40960 and 0 < rows % 8192 < 7782) or (
                K == 4096 and 12288 < rows < 16384):
            most = 6
        if rows * K > 1 << 28:
            most = 6 if K <= 2048 else 4
        return M <= most and (rows <= 24576 or K >= 2048)
    # nor there; of fewer than 2048 rows it has one for more than 16 of x
    return ((64 if M <= 16 else 2048) <= rows <= 5120 and K >= 16384
            and K % 4096 != 0)


def _few_rows(x, w, gated: bool = False) -> bool:
    """Whether x [M, K] w^T goes to csrc/gemm_skinny.hip. The library takes 11 us
    or more for most products; us by it and by the kernel, weights from memory:
      rows of w x K    M = 1          2             3             8             16            32
      2048 x 512                                     4.6 /  2.9     4.6 /  3.0     4.6 /  3.2     6.7 /  3.6
      2048 x 1024                                    5.8 /  3.6     5.8 /  3.8     5.8 /  4.1     8.1 /  5.0
      2048 x 2048      11.0 /  4.8    10.7 /  5.9   11.1 /  5.3   11.0 /  5.6   11.0 /  6.3   11.2 /  8.5
      4096 x 2048                                   11.6 /  6.3   11.6 /  6.4   11.6 /  7.1   11.8 /  9.2
      6144 x 2048                                   13.0 /  8.9   12.7 /  9.4   12.5 /  9.0   12.6 / 11.8
      10240 x 2048                                  16.2 / 11.9   16.0 / 13.6   14.2 / 15.3   14.2 / 21.6
      18432 x 2048                                  57.6 / 19.2   57.4 / 20.3   57.4 / 24.5   20.6 / 34.7
      32768 x 2048                                  34.0 / 30.3   31.8 / 30.2   31.7 / 33.3   34.0 / 41.1
      151936 x 2048                                  205 / 126     204 / 137     202 / 155     145 / 193
      32 x 3072                                      7.1 /  5.6     7.0 /  6.3     8.3 /  7.2     7.0 / 10.0
      2048 x 3072      12.1 /  5.2    11.9 /  6.3   12.3 /  6.8    12.3 /  7.6    12.2 /  8.6    10.3 / 11.3
      8192 x 3072                                   19.3 / 12.7   17.2 / 12.3   17.2 / 12.9   17.3 / 17.5
      16384 x 3072                                  22.5 / 22.9   21.4 / 23.4   21.5 / 26.5   21.6 / 35.1
      32 x 4096                                      8.0 /  7.1     8.1 /  7.9    10.7 /  9.0     8.4 / 12.7
      512 x 4096                                    11.0 /  7.4    11.1 /  8.3    11.1 /  9.4     8.6 / 13.0
      4096 x 4096      15.4 /  7.8    15.2 / 10.0   15.7 /  9.1   15.5 /  9.4   15.4 / 10.9   13.0 / 14.0
      6144 x 4096      15.6 / 10.9    15.3 / 13.0   15.6 / 14.5   14.5 / 13.9   14.4 / 14.8   15.2 / 20.2
      8192 x 4096      17.1 / 14.7    16.5 / 18.3   16.7 / 15.2   15.8 / 14.6   15.8 / 15.5   16.4 / 20.3
      12288 x 4096                                  27.8 / 21.5   26.7 / 23.1   26.5 / 28.5   23.1 / 39.7
      14336 x 4096                                  27.9 / 25.6    28.4 / 29.0
      20000 x 4096                                  67.2 / 34.5   67.0 / 37.6   67.1 / 46.0   38.7 / 64.9
      32768 x 4096     63.2 / 49.5    62.9 / 56.1   61.3 / 53.6   58.9 / 54.9   59.0 / 61.9   63.0 / 74.8
      21200 x 4096                                  41.6 / 38.2    40.3 / 41.0    40.6 / 45.4
      42624 x 4096                                  72.0 / 67.3    72.3 / 78.4
      59344 x 4096                                   101 / 94      96.9 / 110
      62592 x 4096                                   117 / 98       116 / 107
      65536 x 4096                                   122 / 104     120 / 107     120 / 121     122 / 178
      5120 x 5120      13.6 / 12.0    13.9 / 14.8   13.9 / 15.3   14.2 / 16.6   15.4 / 19.1   18.0 / 27.8
      12288 x 5120     26.8 / 23.9    25.9 / 25.7
      12288 x 12288    61.0 / 60.6    60.7 / 64.9
      4096 x 16384                                  30.8 / 31.3   29.8 / 31.1   29.8 / 36.6   33.7 / 46.0
      32 x 17408                                                   22.7 / 26.3    36.7 / 31.4    43.1 / 46.2
      64 x 25600                                    53.3 / 32.1    53.4 / 37.5    53.3 / 45.3    40.6 / 66.9
      1024 x 25600                                  67.0 / 32.9    67.5 / 38.9    67.2 / 46.9    65.1 / 68.6
      2048 x 25600                                  70.1 / 33.4    70.1 / 39.5    70.0 / 47.7    94.0 / 69.1
      5120 x 20000                                  70.6 / 47.5    68.9 / 50.3    69.0 / 56.8    72.4 / 75.8
      5120 x 17408                                   111 / 43      112 / 46      114 / 52      121 / 77
      5120 x 25600      135 / 51       136 / 57      134 / 60      135 / 64      137 / 72      145 / 108
    and with silu_mul behind it (rows of both halves)
      4096 x 2048      13.8 /  5.6    13.6 /  7.0   14.2 /  8.5   14.2 /  9.1   14.1 /  9.8   14.3 / 14.0
      16384 x 2048     20.8 / 14.0    20.3 / 17.6   20.7 / 15.8   19.5 / 16.1   19.5 / 18.0   19.7 / 22.9
      24576 x 4096                                  46.7 / 41.6   45.3 / 42.0   45.6 / 46.4   46.0 / 58.1
      12288 x 8192     43.9 / 42.4    43.8 / 47.5
      51200 x 5120     98.8 / 92.3    99.1 / 95.9   95.6 / 134    92.3 / 139    92.8 / 158    95.8 / 196
    Two rows lose where the library has a good tile (24 to 64 M weights of long
    rows) and one load a weight row is no longer the whole cost.

    `linear` asks `_mid_rows` first. Of the sizes above csrc/gemm_mid.hip takes those
    with a k of 512 to 4096 at 32 rows and of 1024 to 4096 at 16 (few weight rows apart),
    and at 2, 3 and 8 rows most from 4096 or 6144 weight rows on; the figures there are
    what it was measured against. With a k that is no multiple of 256 such sizes still
    come here. For those the line is on the library's side of some: beside 7 to 16 rows
    over 151936 x 2048 and 13 to 16 over 8192 x 3072."""
    if (type(x) is not torch.Tensor or _tracing()
            or type(w) not in (torch.Tensor, torch.nn.Parameter)):
        return False
    if x.dim() != 2 or not 1 <= x.shape[0] <= 32 or not _use_hip(x):
        return False
    M, K = x.shape
    rows = w.shape[0]
    fits = (M == 1 or (M == 2 and _two_rows(rows, K, gated))
            or (M <= 16 and K <= 4096 and rows * K <= 1 << 24)
            or (K <= 2048 and rows * K <= 1 << 23)
            or (M > 2 and _long_weights(M, rows, K)))
    return (fits and _unwatched() and x.dtype == torch.bfloat16
            and w.dtype == torch.bfloat16 and w.device == x.device
            and w.dim() == 2 and w.shape[1] == K and K % 32 == 0 and K > 0
            and rows % (8 if gated else 4) == 0 and rows > 0
            and w.is_contiguous() and x.stride(1) == 1
            and x.stride(0) % 8 == 0
            and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
            and not (torch.is_grad_enabled()
                     and (x.requires_grad or w.requires_grad)))


def _mid_tile(M: int, rows: int, K: int, gated: bool):
    """Rows of x and of w in a tile of csrc/gemm_mid.hip (its mid_pick), and how many
    tiles there are."""
    def tiles(m, n):
        return -(-M // m) * -(-rows // n)
    if M <= 32:
        if not gated:
            t = tiles(64, 16)
            if tiles(32, 32) <= 256 and not (M > 8 and K >= 4096 and t <= 256):
                return 32, 32, tiles(32, 32)
            if t <= 256:
                return 64, 16, t
        sizes = ((64, 32), (32, 64)) if gated else ((32, 64),)
        last = 32, 128
    else:
        sizes = ((64, 32), (64, 64)) if gated else ((64, 16), (64, 32), (64, 64))
        last = (64, 128) if M <= 64 else (128, 128)
        if M > 64:
            sizes += ((64, 128),) if 128 < M <= 192 else ((128, 64),)
    for m, n in sizes:
        if tiles(m, n) <= 256:
            return m, n, tiles(m, n)
    return *last, tiles(*last)


@functools.lru_cache(maxsize=4096)
def _mid_sizes(M: int, rows: int, K: int, gated: bool) -> bool:
    """The sizes of `_mid_rows` at which csrc/gemm_mid.hip is ahead: ranges of k and of
    weight rows, as the table there shows, and by the round: not where tiles of 128
    weight rows are a few more than the 256 CUs (or 512, two a CU), and not where larger
    tiles leave a third of the CUs without one while the library's smaller ones fit. us
    of the other side and of the kernel there:
      30 x 36512 x 3072        49.7 / 52.5      54 x 36224 x 3584        57.1 / 66.2
      48 x 39952 x 4096        70.8 / 74.9       9 x 44368 x 3584        58.2 / 61.3
       8 x 71840 x  768        26.0 / 28.0       3 x 66672 x 2048        53.4 / 58.9
      87 x  2432 x 4096        11.0 / 11.8     141 x  1472 x 3584        10.0 / 10.8
     122 x  9440 x 3072        24.1 / 25.1     240 x  4544 x 3840        25.7 / 28.5
     186 x  6224 x 3584        24.3 / 28.2     213 x 16336 x 3840 gated  48.5 / 54.0
       4 x  6528 x 3584 gated  12.3 / 12.9       6 x  2400 x 5120         8.2 /  9.7
    Of 7500 sizes drawn from those left 6 were 3 to 5 % slower than without the kernel.
    The largest output layers: 151936 x 2048 at 7 to 16 rows 204 / 112, at 32 rows 147 /
    114; 151936 x 4096 at 3 to 64 rows 244 to 266 / 217 to 229; 151936 x 1024 at 3 to 16
    rows 59 to 61 / 58 to 61."""
    bm, bn, n = _mid_tile(M, rows, K, gated)
    if K > 4096:
        return _mid_long(M, rows, K, gated, bm, bn, n)
    if M <= 16:
        return _mid_16(M, rows, K, gated, bn, n)
    if rows < 512 and K > 2048:
        return False
    if M <= 64:
        if bn < 128 or n <= 256:
            return True
        if M <= 32:                       # (two tiles a CU)
            if n <= (304 if K > 2048 else 288) and K >= 1024 and K != 2048:
                return gated and (K <= 2048 or K == 4096)
            return n <= 288 or K % 2048 == 0
        if K == 4096:
            return n > (288 if gated else 352)
        return K == 2048 or (n <= 288 and K <= (2048 if gated else 512))
    if bm == bn == 128:
        if n > 256 or K > 3072 or (K > 2560 and M > 192):
            return False
        if M <= 128:
            return M >= 96 and n >= 224 and K % 2048 == 0
        return gated and n >= (200 if M > 192 else 240) and (M > 192 or K <= 2048)
    if bn == 128 and n > 240:
        return False
    return gated or _mid_beside(M, rows, K, bm, bn, n)


def _mid_beside(M, rows, K, bm, bn, n) -> bool:
    """More than 64 rows, one round: beside the library's tiles, of which one of 32 x 32
    also takes 65 to 96, 129 to 160 or 193 to 224 rows without padding."""
    if bn == 32:
        return K <= 2560 or -(-M // 32) * -(-rows // 32) > 256
    if bm == 128:
        return K <= 2048 or n >= 192 or (M <= 96 if M <= 128 else
                                         M <= 224 and n <= 144)
    if bn == 128:
        return K <= 1536 or n >= 204 or (M <= 160 and n <= 147)
    return True


def _mid_16(M, rows, K, gated, bn, n) -> bool:
    """2 to 16 rows, a k of up to 4096."""
    if bn == 128:                         # two a CU: the beginning of a round
        if M == 2 and 256 < n <= 320 and K > 1024:
            return False
        if M > 8 and 256 < n <= 288 and 1024 <= K < 2048 and not gated:
            return False
        if M > 2 and 320 < n <= 384 and 3072 <= K < 4096 and not gated:
            return False
        if M > 2 and 512 < n <= 592 and (
                (K == 768 and not gated) or (n <= 544 and M <= 8 and (
                    K == 1024 or K > 3328 or (K == 2048 and M <= 4)))):
            return False
        if 2 < M <= 5 and n <= 160 and K <= 1280 and not gated:
            return False
    if M == 2:
        if K <= 1024:
            return rows >= (4096 if gated else 32) and rows <= 65536
        return 6144 <= rows <= 65536 and (
            K <= 2048 or (not gated and rows <= 32768 and not 8192 < rows <= 9216))
    if M <= 12:
        if gated and bn == 32 and K > 1024 and n > (
                128 if M <= 8 else 192 if K <= 1536 else 256):
            return False                  # (the other kernel for few rows)
        if K <= 1024:                     # from 513 to 1024 of k: short chains
            return K > 512 and rows >= 10240
        if K <= 1280 and 7168 < rows <= 8192:
            return False
        if K > 3072 and (rows <= 5120 or (gated and 12288 < rows <= 20480)):
            return False
        return rows >= 4096 + (K > 2048)
    if K <= 1280 and M <= 14 and rows <= 2560:
        return False
    return rows >= (10240 if K <= 512 else 8208 if K < 1024
                    else 2048 if K <= 1024 else 32)


def _mid_long(M, rows, K, gated, bm, bn, n) -> bool:
    """A k of more than 4096: one workgroup has all of it."""
    if K <= 5120:
        if M <= 16:
            if M <= 3:
                return False
            if gated or rows > 6144:
                return 16384 <= rows <= 32768
            return rows > 4096 or (M <= 8 and 512 <= rows < 2304)
        if M <= 64:
            return 512 <= rows <= 8192 or 16384 <= rows <= 32768
        if not 2048 <= rows <= (10240 if 128 < M <= 192 else 8192):
            return False
        if gated:
            return bm < 128 or n >= 192
    elif K <= 6144:
        if not (16 < M <= 128 and 4096 <= rows <= 8192):
            return False
    elif K >= 16384 and M > 32:
        return 2048 <= rows <= 6144
    else:
        if not (64 < M <= 192 and rows <= 6144) or (gated and K > 8192):
            return False
        if rows < (4096 if gated or K > 8192 else 2048):
            return False
        if bn == 128:
            return M <= 160 and (gated or n <= 147)
        if bn == 64 and (n < 176 or (K == 10240 and M > 160)):
            return False
    if gated or M <= 64:
        return True
    if bm == bn == 64 and K <= 6144 and -(-M // 32) % 2:
        return n >= (160 if M <= 96 else 145)
    return _mid_beside(M, rows, K, bm, bn, n)


def _mid_rows(x, w, gated: bool = False) -> bool:
    """Whether x [M, K] w^T goes to csrc/gemm_mid.hip, 2 to 256 rows. Against what
    it went to before (the library, or csrc/gemm_skinny.hip up to 32 rows; gated:
    and silu_mul behind it), in a graph, weights from memory, it takes this part
    of the time (the figures in us stand beside the kernel):
      rows of w x K     M = 2     4     8    16    32    64   128   192   256
      2048 x 1024       0.85  1.07  1.05  0.97  0.86  0.57  0.60  0.64  0.63
      16384 x 1024      0.82  0.89  0.84  0.77  0.61  0.69  0.77  1.09  1.06
      51200 x 1024      0.96  0.95  0.95  0.95  0.97  1.03  1.28  2.0   1.9
      2048 x 2048       1.03  1.02  0.98  0.90  0.73  0.71  0.74  0.81  0.77
      6144 x 2048       0.80  0.89  0.89  0.80  0.58  0.80  0.79  0.75  0.67
      16384 x 2048 g    0.77  0.85  0.82  0.67  0.69  0.71  0.75  0.92  0.85
      32768 x 2048      0.87  0.87  0.82  0.81  0.78  0.80  0.89  1.43  1.35
      4096 x 4096       1.00  1.10  1.02  0.89  0.80  0.85  0.64  0.63  0.91
      6144 x 4096       0.90  0.83  0.81  0.81  0.85  0.93  0.88  0.91  0.71
      16384 x 4096 g    1.07  1.12  1.05  0.92  0.93  0.95  0.92  1.01  0.88
      24576 x 4096 g    0.95  0.94  0.89  0.80  0.76  0.80  1.03  1.41  1.34
      2048 x 5120       1.23  0.66  0.67  1.23  0.96  0.85  0.91  0.84  0.86
      10240 x 5120      1.07  1.06  1.05  1.05  1.03  0.96  1.01  0.84  1.00
      4096 x 8192       1.05  1.05  1.07  1.09  0.99  0.88  0.64  0.60  1.03
      4096 x 12288      1.26  1.25  1.32  1.28  1.10  0.95  0.65  0.65  1.08
      4096 x 25600      1.25  1.23  1.13  0.98  0.74  0.44  0.64  0.77  0.66
    It loses where few weights are long rows (one workgroup has all of k), where a
    round is filled badly (`_mid_sizes`), and to the kernel for few rows where that
    one is quickest."""
    if (type(x) is not torch.Tensor or _tracing()
            or type(w) not in (torch.Tensor, torch.nn.Parameter)):
        return False
    if x.dim() != 2 or not 2 <= x.shape[0] <= 256 or not _use_hip(x):
        return False
    M, K = x.shape
    rows = w.shape[0]
    return (K % 256 == 0 and 512 <= K < 1 << 20 and rows > 0
            and _mid_sizes(M, rows, K, gated) and _unwatched()
            and x.dtype == torch.bfloat16
            and w.dtype == torch.bfloat16 and w.device == x.device
            and w.dim() == 2 and w.shape[1] == K
            and rows % (16 if gated else 4) == 0 and rows < 1 << 24
            and (not gated or (rows // 2 + 128) * K < 1 << 30)
            and w.is_contiguous() and x.stride(1) == 1
            and x.stride(0) % 8 == 0 and K <= x.stride(0) < 1 << 22
            and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
            and not (torch.is_grad_enabled()
                     and (x.requires_grad or w.requires_grad)))


def _plain_bias(bias, x, w) -> bool:
    return bias is None or (
        bias.dtype == torch.bfloat16 and bias.device == x.device
        and bias.shape == w.shape[:1] and bias.is_contiguous()
        and not (torch.is_grad_enabled() and bias.requires_grad))


def _up_to_256(x) -> bool:
    """(One look for the two kernels: eager calls on more rows pay for it.)"""
    return (type(x) is torch.Tensor and not _tracing() and x.dim() == 2
            and x.shape[0] <= 256)


def linear(x, w, bias=None):
    """x w^T (+ bias): the library's product, or over up to 256 rows (decode
    steps, short prompts) csrc/gemm_mid.hip or csrc/gemm_skinny.hip."""
    if _up_to_256(x):
        if _mid_rows(x, w) and _plain_bias(bias, x, w):
            return _require_hip().linear_mid(x, w, bias, False)
        if _few_rows(x, w) and _plain_bias(bias, x, w):
            return _require_hip().linear_skinny(x, w, bias, False)
    return F.linear(x, w, bias)


def _many_rows(x, w) -> bool:
    """Whether csrc/grouped_gemm.hip makes silu_mul(x w^T) in one launch. Its
    tiles are 256 rows by 128 columns of the result, one a CU at a time. Far
    below 256 of them the library's smaller tiles are ahead, and from there on
    where the last round leaves a quarter of all places empty (us of both,
    tiles):
      2 x 3072 x 1024    1024 rows  25.1 /  26.7 ( 96)   2048   36.2 / 29.2 (192)
                         2600 rows  51.6 /  54.3 (264)   3328   58.6 / 53.6 (312)
      2 x 6144 x 2048     512 rows  33.4 /  42.6 ( 96)   1024   53.6 / 48.9 (192)
                         2816 rows   138 /   141 (528)   3328    156 /  145 (624)
      2 x 8192 x 2048     512 rows  39.7 /  45.5 (128)   1024   66.5 / 54.2 (256)
                         1280 rows  86.9 /  89.4 (320)   1536   96.7 / 93.1 (384)
      2 x 12288 x 4096    768 rows   150 /   161 (288)   1024    173 /  170 (384)
    or where a row tile that is nearly empty does (of all rows that the places
    have, those of x):
      2 x 25344 x 2048    274 rows  77.4 /  93.4 (0.41)
      2 x 26496 x 5120    363 rows   224 /   239 (0.57)
      2 x 21248 x 4096   1027 rows   339 /   364 (0.65)
      2 x 23168 x 512     775 rows  83.2 /  51.2 (0.71)
      2 x 12544 x 256     938 rows  36.8 /  25.8 (0.70)
    Otherwise it is 2 to 50 % faster, or as fast (the figures at many rows stand
    beside the kernel). Short k, which the library does worst at, still gains
    with two fifths of the places empty. (192 to 255 tiles would gain where they
    were tried; they stay with the library.)"""
    if (type(x) is not torch.Tensor or _tracing()
            or type(w) not in (torch.Tensor, torch.nn.Parameter)):
        return False
    if x.dim() != 2 or w.dim() != 2:
        return False
    M, K = x.shape
    rows = w.shape[0]
    tiles = -(-M // 256) * (rows // 256)
    if tiles < 256:
        return False
    places = -(-tiles // 256) * 256
    filled, live = (0.6, 0.5) if K <= 1024 else (0.75, 0.67)
    return (tiles >= places * filled and M * (rows // 256) >= 256 * places * live
            and rows % 256 == 0 and K % 64 == 0 and 0 < K < 1 << 21
            and M * K < 1 << 30 and rows < 1 << 24 and w.shape[1] == K
            and _use_hip(x) and _unwatched()
            and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
            and w.device == x.device and x.is_contiguous()
            and w.is_contiguous()
            and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
            and not (torch.is_grad_enabled()
                     and (x.requires_grad or w.requires_grad)))


def linear_silu_mul(x, w):
    """silu_mul(x w^T), w the gate's rows and then the up's."""
    if _up_to_256(x):
        if _mid_rows(x, w, gated=True):
            return _require_hip().linear_mid(x, w, None, True)
        if _few_rows(x, w, gated=True):
            return _require_hip().linear_skinny(x, w, None, True)
    if _many_rows(x, w):
        return _require_hip().linear_silu_mul(x, w)
    return silu_mul(F.linear(x, w))


def linear_gelu_mul(x, w, bias, ff: int):
    """(gelu_tanh(gate) * up, the rest) of x w^T + bias, whose first 2 ff columns are
    gate and up: where one launch makes all of it (prompts), else None. us of the
    library and the unit's launch, and of this one, columns 2 ff + the rest:
      16384 + 2048 x 2048   32768 rows  2011 / 1814    8192   529 / 464
      17408 + 2048 x 2048    1532 rows   112 /  103
      20992 + 4096 x 4096    5298 rows   878 /  801
       6144 + 1024 x 1024   26243 rows   444 /  333
       2560 +  512 x  512   11279 rows    97 /   58
      12288 + 4096 x 4096   26526 rows  2437 / 2471
    With a long k and few gated columns the unit's pass is small beside the product,
    which the library makes 2 % faster."""
    if not (_many_rows(x, w) and ff % 128 == 0 and 0 < 2 * ff <= w.shape[0]
            and w.shape[0] % 256 == 0
            and (x.shape[1] < 4096 or 2 * ff * 5 >= w.shape[0] * 4)
            and _plain_bias(bias, x, w)
            and (bias is None or bias.data_ptr() % 8 == 0)):
        return None
    return _require_hip().linear_gelu_mul(x, w, bias, ff)


def linear_silu_rows(x, w):
    """silu_mul(x w^T) where one launch makes it (prompts), else None. Against the
    library and the unit's launch 0.86 to 0.95 of the time at 16384 x 2048 and 24576
    x 4096, 0.45 to 0.8 with a k of 1024 and less."""
    return _require_hip().linear_silu_mul(x, w) if _many_rows(x, w) else None


def _heads_pay(M: int, K: int, rows: int) -> bool:
    """Whether the QKV projection of M rows pays in one launch, of the sizes that
    `_many_rows` takes. Up to a k of 2048 by the share that x's rows are of all rows in
    its rounds of 256 tiles of 256 x 256; lowest quotient of the library's time with
    the pass by the launch's from a share on, 700 sizes:
      share         0.58   0.62   0.66   0.70   0.72   0.74   0.76   0.80
      k up to 512   1.28   1.19   1.19   1.24   1.26   1.26   1.22
      640 .. 1024   0.89   0.93   0.92   0.96   1.03   0.99   1.10
      .. 2048                            0.97   0.95   0.96   1.00   1.01
    Above, where the library's product is 4 to 7 % faster than this one and the pass small
    beside it, where 0.95 of the places have a tile: 0.99 up to a k of 6144, 0.96 at
    8192 (200 sizes)."""
    tiles = -(-M // 256) * (rows // 256)
    places = -(-tiles // 256) * 256
    if K > 2048:
        return K <= 6144 and tiles >= 0.95 * places
    return K <= 512 or M * (rows // 256) >= 256 * places * (0.72 if K <= 1024 else 0.76)


def linear_qkv_prep(x, w, num_heads: int, num_kv_heads: int, head_dim: int,
                    positions, slot_mapping, k_cache, v_cache, cos_sin,
                    q_norm_w=None, k_norm_w=None, eps: float = 1e-6):
    """fused_qkv_prep of x w^T where one launch makes it (prompts), else None. us of the
    library's product with the pass over its result, and of this one, by rows (* not
    taken: fewer than 256 tiles, or by `_heads_pay`):
       4096 x  512    4096   35.5 /  27.9     6000   62.5 /  46.1    24000  203 / 136
       4096 x 1024   *3000   36.3 /  34.3     4096   44.6 /  38.0    24000  267 / 198
       3072 x 2048   *6000   99.1 / 101.3    *8192  108.7 / 106.6    32768  383 / 340
       6144 x 4096   *6000    257 /  281      8192    310 /  304     32768 1245 / 1222
      10240 x 5120   *3000    241 /  246     *6000    517 /  481     16384 1290 / 1244
    e4m3 pages keep the pass: nothing here rounds to them."""
    caches = (k_cache, v_cache)
    norms = tuple(n for n in (q_norm_w, k_norm_w) if n is not None)
    if not (head_dim == 128 and num_heads % 2 == 0 and _many_rows(x, w)
            and x.shape[1] >= 192 and _heads_pay(*x.shape, w.shape[0])
            and all(t.dtype == torch.bfloat16 and t.is_contiguous()
                    and t.data_ptr() % 16 == 0 for t in caches)
            and w.shape[0] == (num_heads + 2 * num_kv_heads) * 128
            and k_cache.dim() == 4 and k_cache.shape == v_cache.shape
            and k_cache.shape[1] == num_kv_heads and k_cache.shape[3] == 128
            and k_cache.shape[2] & (k_cache.shape[2] - 1) == 0
            and k_cache.numel() >> 7 < 1 << 32
            and cos_sin.is_contiguous() and cos_sin.data_ptr() % 16 == 0
            and cos_sin.dtype == torch.float32 and cos_sin.shape[1:] == (128,)
            and all(t.is_contiguous() and t.numel() == x.shape[0]
                    for t in (positions, slot_mapping))
            and all(n.dtype == torch.bfloat16 and n.is_contiguous()
                    and n.numel() == 128 and n.data_ptr() % 8 == 0 for n in norms)
            and all(t.device == x.device for t in
                    caches + norms + (positions, slot_mapping, cos_sin))):
        return None
    return _require_hip().linear_heads(x, w, k_cache, v_cache, positions,
                                       slot_mapping, cos_sin, q_norm_w, k_norm_w,
                                       eps)


def _one_row(x, residual, norm_w, w, gated: bool) -> bool:
    """Whether csrc/gemm_skinny.hip makes the norm of one row inside the product
    behind it. Up to 4096 waves make it, each workgroup for itself, and with short
    rows most of their lanes have no weights to read meanwhile: of two launches
    it takes 0.65 to 0.95 up to 12288 rows of weights; at 65536 0.92 to 0.98 from
    a k of 768 on, 1.00 at 640, 1.2 to 1.4 at 512 and less; at 131072 1.0 to 1.7."""
    return (x.shape[0] == 1 and _few_rows(x, w, gated) and x.shape[1] <= 4096
            and w.shape[0] <= (65536 if x.shape[1] > 640 else 12288)
            and x.is_contiguous()
            and type(residual) is torch.Tensor
            and type(norm_w) in (torch.Tensor, torch.nn.Parameter)
            and residual.shape == x.shape and norm_w.shape == x.shape[1:]
            and residual.dtype == torch.bfloat16
            and norm_w.dtype == torch.bfloat16
            and residual.device == x.device and norm_w.device == x.device
            and residual.is_contiguous() and norm_w.is_contiguous()
            and residual.data_ptr() % 16 == 0
            and norm_w.data_ptr() % 16 == 0
            and not (torch.is_grad_enabled()
                     and (residual.requires_grad or norm_w.requires_grad)))


def norm_linear(x, residual, norm_w, eps: float, w, gated: bool = False):
    """(y w^T, r) for r = x + residual and y = rmsnorm(r), `gated`: (silu_mul(y
    w^T), r). x and residual may be overwritten."""
    if _one_row(x, residual, norm_w, w, gated):
        return _require_hip().norm_linear(x, residual, norm_w, eps, w, gated)
    x, residual = fused_add_rmsnorm(x, residual, norm_w, eps)
    return (linear_silu_mul(x, w) if gated else linear(x, w)), residual


def expert_tile(n_rows: int, experts: int, inner: int, width: int,
                gated: bool = True, local: Optional[int] = None) -> int:
    """Rows that the segments of both expert GEMMs of a layer are padded to,
    for `n_rows` (token, expert) pairs in bf16 on the matrix cores (K and N
    multiples of 64), by the rows an expert gets on average. Taller tiles do
    more work per byte but pad more; both products together, at 32 experts of
    2048 x 2048: at 72 rows 240 / 221 / 208 us on tiles of 64 / 128 / 256, at 96
    rows 243 / 226 / 209, at 192 rows 366 / 314 / 204, at 384 rows 890 / 465 /
    332. (So tiles of 256 would already pay at 72 rows there, and the lines below
    were drawn when their kernel was a slower one; they have not been moved.)

    They also leave fewer workgroups: one of 256 rows takes 128 columns of the
    gated product or 256 of the other, and with few of them in either product
    the chip idles: the rule wants 128. 8 experts of 1024 x 512, 192 / 512 / 1024
    rows an expert (24 / 64 / 128 of either) 28 / 43 / 52 us on 64, 29 / 35 / 53 on
    128, 43 / 46 / 48 on 256. 8 of 2048 x 2048 are past the crossing with 64 to 96
    of the second, 192 / 384 / 512 rows: 74 / 115 / 136 us on 128, 85 / 101 / 102 on
    256. Tiles of 128 want 96.

    Up to 16 rows, where the weights are all there is to read, tiles of 32: four
    workgroups of the gated product fit a CU instead of three. They are taken
    unless their number then fills the rounds worse: 1024 workgroups (2048 wide)
    156 -> 144 us, 1536 (3072 wide, K 4096) 427 -> 447.

    `local`: the experts whose products this rank makes (all by default); its
    workgroups are counted."""
    local = experts if local is None else local
    avg = n_rows / experts
    rows = avg * local
    if avg <= 16:
        blocks = min(local, max(1, round(rows))) * (inner // 64)
        if blocks <= 768 or -(-blocks // 1024) * 4 <= -(-blocks // 768) * 3:
            return 32
    cols = 128 if gated else 256
    if (avg >= 144 and inner % cols == 0 and width % 256 == 0
            and rows / 256 * min(inner // cols, width // 256) >= 128):
        return 256
    return 128 if avg >= 72 and rows / 128 * (inner // 128) >= 96 else 64


def grouped_gemm(out, a, w, row_tok, tile_off, counts, max_tiles, gate_silu,
                 bm=64):
    """Dropless-MoE grouped GEMM: csrc/grouped_gemm.hip on GPU, torch
    reference on CPU (same padded-segment layout). bm = segment tile height
    (see expert_tile; the host pads with the same value)."""
    if _use_hip(a):
        _require_hip().grouped_gemm(out, a, w, row_tok, tile_off, counts,
                                    max_tiles, gate_silu, bm)
        return out
    return torch_ref.grouped_gemm(out, a, w, row_tok, tile_off, counts,
                                  max_tiles, gate_silu, bm)


def moe_layout(logits, k: int, base: int, n_local: int, bm: int, row_tok):
    """Softmax top-k router and expert layout of one rank (csrc/moe_topk.hip,
    csrc/moe_dispatch.hip), GPU only: bf16 logits [T, E] -> (weights fp32
    [T, k], tile_off, counts, padpos int32 [T, k]); `row_tok` (int32) receives
    the token of every padded row. The rank holds the experts base .. base +
    n_local - 1; other choices share one more segment, with weight 0."""
    return _require_hip().moe_layout(logits, k, base, n_local, bm, row_tok)


def moe_combine(out, rows, padpos, w):
    """out[t] = sum_j w[t,j] * rows[padpos[t,j]]: fused bf16 gather-combine
    (csrc/grouped_gemm.hip) on GPU, deterministic torch gather on CPU."""
    if _use_hip(rows):
        _require_hip().moe_combine(out, rows, padpos, w)
        return out
    contrib = rows[padpos].float()          # [T, k, h]
    out.copy_((contrib * w.unsqueeze(-1)).sum(dim=1).to(out.dtype))
    return out
