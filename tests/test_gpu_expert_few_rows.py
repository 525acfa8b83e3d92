"""The expert GEMMs on tiles of 32 to 128 rows where the last tile of an expert has few
rows: what lies in padding rows is not seen in the others, and nothing is put there."""

import pytest
import torch

from sutro_amd.ops import hybrid as hops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("bm", [32, 64, 128])
@pytest.mark.parametrize("act", [hops.ACT_NONE, hops.ACT_SILU_GATE, hops.ACT_RELU2])
@pytest.mark.parametrize("K,ff,more", [(64, 64, 0), (320, 192, 0), (2048, 1024, 24),
                                       (4096, 1024, 24), (1024, 1024, 55)])
def test_live_rows(K, ff, more, act, bm):
    """Counts around chunks of 8 rows and blocks of 16; with 24 experts more 816
    workgroups of tiles of 32, a round nearly full (gated ones look their rows up at each
    step then), with 55 more a second round of few."""
    counts = [1, 0, 7, 8, 9, 15, 16, 17, 31, 32, 33, 2, 63, 65, 127, 129, 0, 3]
    counts += [5] * more
    g = torch.Generator(device=DEV).manual_seed(K + bm)
    gated, gather = act == hops.ACT_SILU_GATE, act != hops.ACT_NONE
    tiles = [(c + bm - 1) // bm for c in counts]
    off = torch.tensor([0] + tiles, device=DEV).cumsum(0).int()
    cnt = torch.tensor(counts, device=DEV, dtype=torch.int32)
    rows, T = sum(tiles) * bm, 50
    w = torch.randn(len(counts), 2 * ff if gated else ff, K, generator=g, device=DEV)
    w = (w * K ** -0.5).bfloat16()
    x = torch.randn(T if gather else rows, K, generator=g, device=DEV).bfloat16()
    live = torch.zeros(rows, dtype=torch.bool, device=DEV)
    tok = torch.full((rows,), -1, device=DEV, dtype=torch.int32)
    for e, c in enumerate(counts):
        a = int(off[e]) * bm
        live[a:a + c] = True
        tok[a:a + c] = torch.randint(1, T, (c,), generator=g, device=DEV).int()
    if gather:
        x[0] = float("nan")            # what a row without a token would read
    else:
        x[~live] = float("nan")
    out = torch.zeros(rows, ff, device=DEV, dtype=torch.bfloat16)
    hops.expert_gemm(out, x, w, tok if gather else None, off, cnt, act, bm, 0.0, None)
    assert (out[~live] == 0).all()
    for e, c in enumerate(counts):
        a = int(off[e]) * bm
        xe = (x[tok[a:a + c].long()] if gather else x[a:a + c]).float()
        y = xe @ w[e].float().T
        if gated:
            y = torch.nn.functional.silu(y[:, :ff]) * y[:, ff:]
        elif act == hops.ACT_RELU2:
            y = y.relu() ** 2
        # one rounding to bf16 (2^-8) and fp32 sums of K products in other orders
        torch.testing.assert_close(out[a:a + c].float(), y, rtol=2 ** -7,
                                   atol=2 ** -7)


@pytest.mark.parametrize("bm", [32, 64, 128, 256])
@pytest.mark.parametrize("act", [hops.ACT_NONE, hops.ACT_SILU_GATE])
def test_segments_longer_than_their_rows(act, bm):
    """Two tiles for every expert, however many rows it has: none, a few, one more than
    a tile. Tiles without rows are not asked for the row in front of them."""
    counts = [0, 3, bm + 1, 0, bm, 2 * bm]
    g = torch.Generator(device=DEV).manual_seed(bm)
    gated, gather = act == hops.ACT_SILU_GATE, act != hops.ACT_NONE
    K, ff, E = 128, 256, len(counts)
    off = torch.arange(E + 1, device=DEV, dtype=torch.int32) * 2
    cnt = torch.tensor(counts, device=DEV, dtype=torch.int32)
    w = torch.randn(E, 2 * ff if gated else ff, K, generator=g, device=DEV)
    w = (w * K ** -0.5).bfloat16()
    rows, T = 2 * E * bm, 40
    x = torch.randn(T if gather else rows, K, generator=g, device=DEV).bfloat16()
    tok = torch.randint(0, T, (rows,), generator=g, device=DEV).int()
    for e, c in enumerate(counts):
        tok[2 * e * bm + c:2 * (e + 1) * bm] = -1
    out = torch.zeros(rows, ff, device=DEV, dtype=torch.bfloat16)
    hops.expert_gemm(out, x, w, tok if gather else None, off, cnt, act, bm, 0.0, None)
    for e, c in enumerate(counts):
        a = 2 * e * bm
        y = (x[tok[a:a + c].long()] if gather else x[a:a + c]).float() @ w[e].float().T
        if gated:
            y = torch.nn.functional.silu(y[:, :ff]) * y[:, ff:]
        torch.testing.assert_close(out[a:a + c].float(), y, rtol=2 ** -7,
                                   atol=2 ** -7)
