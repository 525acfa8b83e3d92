"""The expert GEMMs on tiles of 32, 64 and 256 rows against the torch
reference: empty experts, segments one row short of, at and past a tile, one
and several steps of k, every unit between the two matrices."""

import pytest
import torch

from sutro_amd.ops import hybrid as hops
from sutro_amd.ops import torch_ref as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _segments(counts, bm):
    pad = [(c + bm - 1) // bm * bm for c in counts]
    off = torch.tensor([0] + pad).cumsum(0) // bm
    return off.to(torch.int32), torch.tensor(counts, dtype=torch.int32)


@pytest.mark.parametrize("K", [64, 320, 1024])   # 64: a single step
@pytest.mark.parametrize("bm,counts", [
    (32, [1, 31, 0, 32, 33, 70]), (64, [1, 63, 0, 64, 65, 130]), (256, [1, 255, 0, 256, 257, 600])])
@pytest.mark.parametrize("act", [hops.ACT_NONE, hops.ACT_SILU_GATE,
                                 hops.ACT_RELU2, hops.ACT_GLU_CLAMPED,
                                 "weighted"])
def test_tiles(K, bm, counts, act):
    g = torch.Generator().manual_seed(K + bm)
    row_w = None
    weighted = act == "weighted"
    if weighted:
        act = hops.ACT_SILU_GATE
    gated = act in (hops.ACT_SILU_GATE, hops.ACT_GLU_CLAMPED)
    ff = 256
    off, cnt = _segments(counts, bm)
    rows = int(off[-1]) * bm + bm          # one tile nobody owns
    T = 97
    N = 2 * ff if gated else ff
    w = (torch.randn(len(counts), N, K, generator=g) * K ** -0.5).bfloat16()
    row_tok = torch.full((rows,), -1, dtype=torch.int32)
    live = torch.zeros(rows, dtype=torch.bool)
    for e, c in enumerate(counts):
        a = int(off[e]) * bm
        row_tok[a:a + c] = torch.randint(T, (c,), generator=g).int()
        live[a:a + c] = True
    if act == hops.ACT_NONE:
        x, tok = torch.randn(rows, K, generator=g).bfloat16(), None
    else:
        x, tok = torch.randn(T, K, generator=g).bfloat16(), row_tok
    if weighted:
        row_w = torch.rand(rows, generator=g)
    out = torch.full((rows, ff), 7.0, dtype=torch.bfloat16, device=DEV)
    d = [None if t is None else t.to(DEV) for t in (x, w, tok, off, cnt, row_w)]
    hops.expert_gemm(out, *d[:5], act, bm, 1.5, d[5])
    want = torch.zeros(rows, ff)
    if gated:
        R.glu_grouped_gemm(want, x, w, tok, off, cnt, bm, 1.5,
                           silu=act == hops.ACT_SILU_GATE, row_w=row_w)
    else:
        R.grouped_gemm(want, x, w, tok, off, cnt, rows // bm, act, bm)
    got = out.float().cpu()
    # one rounding of the result to bf16 (2^-9) over fp32 sums of K products
    torch.testing.assert_close(got[live], want[live], rtol=2 ** -7,
                               atol=2 ** -7)
    # the tile that belongs to no segment is left alone
    assert (got[int(off[-1]) * bm:] == 7.0).all()


@pytest.mark.parametrize("n_rows,want", [
    (1, 32), (128, 32), (129, 64), (575, 64), (576, 128), (1151, 128), (1152, 256), (99999, 256)])
def test_tile_rule(n_rows, want):
    from sutro_amd.ops import expert_tile

    assert expert_tile(n_rows, 8, 128, 256) == want
    # widths the wide kernel does not take
    assert expert_tile(n_rows, 8, 192, 256) <= 128
    assert expert_tile(n_rows, 8, 128, 320) <= 128
    assert expert_tile(n_rows, 8, 128, 256, gated=False) <= 128
    # 1536 workgroups: two rounds of three a CU, but one and a half of four
    assert expert_tile(512, 32, 3072, 4096) == 64
