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

    # wide enough that every tile leaves enough workgroups
    assert expert_tile(n_rows, 8, 16384, 16384) == want
    # widths the wide kernel does not take
    assert expert_tile(n_rows, 8, 16384 + 64, 16384) <= 128
    assert expert_tile(n_rows, 8, 16384, 16384 + 64) <= 128
    assert expert_tile(n_rows, 8, 16384 + 128, 16384, gated=False) <= 128
    # 1536 workgroups: two rounds of three a CU, but one and a half of four
    assert expert_tile(512, 32, 3072, 4096) == 64


@pytest.mark.parametrize("experts,inner,width,avg,want", [
    (8, 512, 1024, 128, 64), (8, 512, 1024, 192, 64), (8, 512, 1024, 512, 128),
    (8, 512, 1024, 1024, 256), (8, 2048, 2048, 96, 128),
    (8, 2048, 2048, 192, 128), (8, 2048, 2048, 384, 128),
    (8, 2048, 2048, 512, 256), (8, 1024, 512, 1024, 128),
    (4, 512, 512, 512, 64), (32, 2048, 2048, 192, 256)])
def test_tiles_that_leave_the_chip_busy(experts, inner, width, avg, want):
    """Few experts of small matrices: tiles by the workgroups they leave (the
    figures, and sizes past the crossing, stand with the rule)."""
    from sutro_amd.ops import expert_tile

    n = avg * experts
    assert expert_tile(n, experts, inner, width) == want
    # one of four ranks, with the same experts and rows of its own
    assert expert_tile(4 * n, 4 * experts, inner, width, local=experts) == want


@pytest.mark.parametrize("act,weighted,dtype", [
    (hops.ACT_GLU_CLAMPED, True, torch.bfloat16),
    (hops.ACT_RELU2, True, torch.bfloat16),
    (hops.ACT_SILU_GATE, False, torch.float32)])
def test_plain_kernel_takes_every_tile(act, weighted, dtype):
    """Units that the matrix-core kernel does not have over weighted rows, and
    float32, on the tile that `expert_gemm_tile` names for a few tokens and on
    the others."""
    g = torch.Generator().manual_seed(11)
    E, K, ff, T, k = 8, 128, 64, 9, 2
    gated = act in (hops.ACT_SILU_GATE, hops.ACT_GLU_CLAMPED)
    w = (torch.randn(E, ff * (2 if gated else 1), K, generator=g)
         * K ** -0.5).to(dtype)
    x = torch.randn(T, K, generator=g).to(dtype)
    idx = torch.stack([torch.randperm(E, generator=g)[:k]
                       for _ in range(T)]).int()
    wts = torch.rand(T, k, generator=g)
    xd, wd = x.to(DEV), w.to(DEV)
    for bm in {hops.expert_gemm_tile(xd, wd, T * k, gated), 32, 64, 128, 256}:
        rt, off, cnt, pos, rw = hops.moe_dispatch(idx.to(DEV), E, bm,
                                                  wts.to(DEV))
        out = torch.zeros(rt.shape[0], ff, dtype=dtype, device=DEV)
        hops.expert_gemm(out, xd, wd, rt, off, cnt, act, bm, 1.5,
                         rw if weighted else None)
        got = out[pos.long()].float().cpu()
        for t in range(T):
            for j in range(k):
                y = x[t].double() @ w[idx[t, j]].double().T
                if weighted:
                    y = y * float(wts[t, j])
                if act == hops.ACT_RELU2:
                    y = y.clamp(min=0) ** 2
                else:
                    a, u = y[:ff], y[ff:]
                    if act == hops.ACT_GLU_CLAMPED:
                        a, u = a.clamp(max=1.5), u.clamp(-1.5, 1.5)
                        y = a * torch.sigmoid(1.702 * a) * (u + 1)
                    else:
                        y = a * torch.sigmoid(a) * u
                # one rounding to the type over sums of 128 products
                tol = 2 ** -8 if dtype == torch.bfloat16 else 1e-5
                torch.testing.assert_close(got[t, j].double(), y, rtol=tol,
                                           atol=tol)
