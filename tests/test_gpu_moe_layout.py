"""The softmax top-k router with its expert layout, against the torch router:
expert counts around the lanes of a wave, one and many runs of pairs, the
experts of one rank out of several, ties and logits that are not finite."""

import pytest
import torch

from sutro_amd import ops
from sutro_amd.ops import torch_ref as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _layout(logits, k, base, n_local, bm):
    T, E = logits.shape
    rows = T * k + (n_local + 1) * bm
    row_tok = torch.full((rows,), -7, dtype=torch.int32, device=DEV)
    w, off, cnt, pos = ops.moe_layout(logits.to(DEV), k, base, n_local, bm,
                                      row_tok)
    return [x.cpu() for x in (row_tok, w, off, cnt, pos.long())]


@pytest.mark.parametrize("T,E,k,base,n_local,bm", [
    (1, 3, 1, 0, 3, 64), (5, 3, 3, 0, 3, 64), (70, 64, 8, 0, 64, 64),
    (129, 65, 4, 0, 65, 64), (33, 130, 8, 65, 65, 64),
    (2048, 32, 4, 0, 32, 128),           # 8192 pairs: the three-launch layout
    (2500, 300, 6, 100, 100, 64), (3, 1024, 64, 0, 1024, 64)])
def test_layout(T, E, k, base, n_local, bm):
    g = torch.Generator().manual_seed(E * 7 + k)
    # distinct logits in every row: the choice is unique
    logits = torch.stack([torch.randperm(E, generator=g) for _ in range(T)])
    logits = ((logits - E / 2) * (6.0 / E)).bfloat16()
    if E > 200:  # more values than bf16 holds in that range: keep them apart
        logits = torch.stack([torch.randperm(E, generator=g)
                              for _ in range(T)]).bfloat16()
        # integers up to 256 are exact; larger ones may tie with a neighbour
    row_tok, w, off, cnt, pos = _layout(logits, k, base, n_local, bm)
    rw, ri = R.topk_softmax_router(logits.float(), k)
    lf = logits.float()
    for t in range(T):
        kept = sorted(lf[t, ri[t]].tolist())
        # which expert owns the row of every pair
        seg = torch.searchsorted(off * bm, pos[t], right=True) - 1
        mine = seg < n_local
        assert len(set(pos[t].tolist())) == k
        assert (row_tok[pos[t]] == t).all()
        e = seg + base
        if n_local == E:
            assert sorted(lf[t, e].tolist()) == kept      # ties may swap
            order = lf[t, e].argsort(descending=True, stable=True)
            torch.testing.assert_close(w[t][order], rw[t], atol=1e-6, rtol=1e-5)
        else:
            inside = ((ri[t] >= base) & (ri[t] < base + n_local)).sum()
            if E <= 256:
                assert mine.sum() == inside
        assert (w[t][~mine] == 0).all()
    assert int(cnt.sum()) == T * k
    for s in range(cnt.numel()):
        a, b = int(off[s]) * bm, int(off[s + 1]) * bm
        assert (row_tok[a:b] >= 0).sum() == cnt[s] <= b - a
        assert b - a - cnt[s] < bm


def test_ties_and_non_finite():
    logits = torch.tensor([[1.0, 1.0, 1.0, 1.0],
                           [float("-inf"), 0.0, float("-inf"), float("-inf")],
                           [float("inf"), 0.0, 1.0, 2.0],
                           [float("nan"), 0.0, 1.0, 2.0]]).bfloat16()
    row_tok, w, off, cnt, pos = _layout(logits, 2, 0, 4, 64)
    seg = torch.searchsorted(off * 64, pos.reshape(-1), right=True) - 1
    seg = seg.view(4, 2)
    assert seg[0].tolist() == [0, 1]                # the lower index first
    assert seg[1].tolist() == [1, 0] and w[1].tolist() == [1.0, 0.0]
    # as the torch router: a row with inf or NaN has NaN weights
    assert w[2].isnan().any() and w[3].isnan().all()
    assert ((seg >= 0) & (seg < 4)).all()


@pytest.mark.parametrize("E,k", [(8, 2), (70, 8)])
def test_masks_of_the_lowest_value(E, k):
    """Logits masked with the type's lowest value are ordinary numbers: a token
    with nothing else shares its weight among them, and beside others they
    weigh nothing."""
    lowest = torch.finfo(torch.bfloat16).min
    logits = torch.full((4, E), lowest)
    logits[1, 3] = 0.0
    logits[2, 3:3 + k] = 1.0
    logits[3, 5] = lowest * (1 - 2.0 ** -7)       # the next number above it
    logits = logits.bfloat16()
    row_tok, w, off, cnt, pos = _layout(logits, k, 0, E, 64)
    want, _ = R.topk_softmax_router(logits, k)
    assert torch.isfinite(w).all()
    torch.testing.assert_close(w.sort(1)[0], want.sort(1)[0])
    assert int(cnt.sum()) == 4 * k
