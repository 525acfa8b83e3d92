"""The expert GEMMs on tiles of 256 rows where a workgroup goes through several
tiles: more tiles than workgroups, one to several steps of k, few and many experts
(their table in lanes, or searched), operands off 16-byte boundaries."""

import pytest
import torch

from sutro_amd.ops import hybrid as hops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _run(counts, K, ff, act, shift=0):
    g = torch.Generator(device=DEV).manual_seed(K + len(counts))

    def rnd(*shape):
        n = 1
        for s in shape:
            n *= s
        flat = torch.randn(n + shift, generator=g, device=DEV).bfloat16()
        return flat[shift:].view(*shape)

    gated = act == hops.ACT_SILU_GATE
    tiles = [(c + 255) // 256 for c in counts]
    off = torch.tensor([0] + tiles, device=DEV).cumsum(0).int()
    cnt = torch.tensor(counts, device=DEV, dtype=torch.int32)
    rows = sum(tiles) * 256
    w = rnd(len(counts), 2 * ff if gated else ff, K).mul_(K ** -0.5)
    T = 300
    x = rnd(T, K) if gated else rnd(rows, K)
    tok = None
    if gated:
        tok = torch.full((rows,), -1, device=DEV, dtype=torch.int32)
        for e, c in enumerate(counts):
            a = int(off[e]) * 256
            tok[a:a + c] = torch.randint(T, (c,), generator=g,
                                         device=DEV).int()
    out = rnd(rows, ff)
    hops.expert_gemm(out, x, w, tok, off, cnt, act, 256, 0.0, None)
    for e, c in enumerate(counts):
        a = int(off[e]) * 256
        xe = (x[tok[a:a + c].long()] if gated else x[a:a + c]).float()
        y = xe @ w[e].float().T
        if gated:
            y = torch.nn.functional.silu(y[:, :ff]) * y[:, ff:]
        # one rounding to bf16 (2^-9) over fp32 sums of K products
        torch.testing.assert_close(out[a:a + c].float(), y, rtol=2 ** -7,
                                   atol=2 ** -7)


@pytest.mark.parametrize("K", [64, 128, 192, 256, 448])
@pytest.mark.parametrize("act", [hops.ACT_NONE, hops.ACT_SILU_GATE])
def test_more_tiles_than_workgroups(K, act):
    # 8 tiles of a group, 5 column blocks (gated: 10) and a last group in part
    _run([300, 0, 1, 256, 257, 9000, 2500], K, 1280, act)


@pytest.mark.parametrize("experts", [63, 64, 130])
def test_many_experts(experts):
    _run([(i * 37) % 300 for i in range(experts)], 192, 256,
         hops.ACT_SILU_GATE)


@pytest.mark.parametrize("act", [hops.ACT_NONE, hops.ACT_SILU_GATE])
def test_operands_off_boundaries(act):
    _run([600, 5, 300], 320, 512, act, shift=8 + 2)


@pytest.mark.parametrize("K", [1024, 2048, 4096])
@pytest.mark.parametrize("act", [hops.ACT_NONE, hops.ACT_SILU_GATE])
@pytest.mark.parametrize("bm", [32, 64, 128, 256])
def test_place_of_a_row(K, act, bm):
    """The dispatch puts tokens where its counters stand: a token's result is the
    same to the bit in every tile of its expert, on every XCD."""
    g = torch.Generator(device=DEV).manual_seed(K)
    gated = act == hops.ACT_SILU_GATE
    counts, ff, T = [9000, 300, 5000], 512, 7
    tiles = [(c + bm - 1) // bm for c in counts]
    off = torch.tensor([0] + tiles, device=DEV).cumsum(0).int()
    cnt = torch.tensor(counts, device=DEV, dtype=torch.int32)
    rows = sum(tiles) * bm
    x = torch.randn(T, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(3, 2 * ff if gated else ff, K, generator=g, device=DEV)
         * K ** -0.5).bfloat16()
    which = torch.arange(rows, device=DEV) * 5 % T
    out = torch.empty(rows, ff, device=DEV, dtype=torch.bfloat16)
    if gated:
        hops.expert_gemm(out, x, w, which.int(), off, cnt, act, bm, 0.0, None)
    else:
        hops.expert_gemm(out, x[which], w, None, off, cnt, act, bm, 0.0, None)
    for e, c in enumerate(counts):
        a = int(off[e]) * bm
        for t in range(T):
            same = out[a:a + c][which[a:a + c] == t]
            assert torch.equal(same, same[:1].expand_as(same)), (e, t)


@pytest.mark.parametrize("bm", [32, 64])
@pytest.mark.parametrize("K", [2048, 4096])
@pytest.mark.parametrize("act", [hops.ACT_NONE, hops.ACT_SILU_GATE])
def test_starts_of_small_tiles(bm, K, act):
    """Rows of 4 KB: experts that begin at all steps of k, some without rows,
    some with several tiles, against 64 bits."""
    g = torch.Generator(device=DEV).manual_seed(K + bm)
    counts = [(i * 23) % 70 for i in range(40)]
    gated = act == hops.ACT_SILU_GATE
    ff, T = 128, 50
    tiles = [(c + bm - 1) // bm for c in counts]
    off = torch.tensor([0] + tiles, device=DEV).cumsum(0).int()
    cnt = torch.tensor(counts, device=DEV, dtype=torch.int32)
    rows = sum(tiles) * bm
    w = (torch.randn(40, 2 * ff if gated else ff, K, generator=g, device=DEV)
         * K ** -0.5).bfloat16()
    x = torch.randn(T, K, generator=g, device=DEV).bfloat16()
    which = torch.arange(rows, device=DEV) * 7 % T
    out = torch.empty(rows, ff, device=DEV, dtype=torch.bfloat16)
    if gated:
        hops.expert_gemm(out, x, w, which.int(), off, cnt, act, bm, 0.0, None)
    else:
        hops.expert_gemm(out, x[which], w, None, off, cnt, act, bm, 0.0, None)
    for e, c in enumerate(counts):
        a = int(off[e]) * bm
        y = x[which[a:a + c]].double() @ w[e].double().T
        if gated:
            y = torch.nn.functional.silu(y[:, :ff]) * y[:, ff:]
        # fp32 sums of K products of size K^-1/2, one rounding to bf16
        torch.testing.assert_close(out[a:a + c].double(), y, rtol=2 ** -8,
                                   atol=2 ** -12)


@pytest.mark.parametrize("K", [2048, 4096])
@pytest.mark.parametrize("act", [hops.ACT_NONE, hops.ACT_SILU_GATE])
@pytest.mark.parametrize("shift", [0, 8 + 2])
def test_rows_of_4_kb(K, act, shift):
    """Experts start at steps of their own, and a workgroup goes from a tile of
    one to a tile of the next: more tiles than workgroups, 64-bit addresses too."""
    _run([3000, 0, 257, 2900, 1, 520, 256, 700], K, 2304, act, shift)


def test_gathered_rows_past_4_gb():
    """1,100,000 rows of 4 KB: more than 32-bit offsets reach."""
    K, ff, R = 2048, 256, 1_100_000
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.zeros(R, K, device=DEV, dtype=torch.bfloat16)
    used = torch.cat([torch.arange(0, 40), torch.arange(1048576 - 40, 1048576 + 40),
                      torch.arange(R - 40, R)]).to(DEV)
    x[used] = torch.randn(len(used), K, generator=g, device=DEV).bfloat16()
    counts = [300, 70]
    off = torch.tensor([0, 2, 3], device=DEV, dtype=torch.int32)
    cnt = torch.tensor(counts, device=DEV, dtype=torch.int32)
    tok = used[torch.arange(768, device=DEV) * 7 % len(used)]
    w = (torch.randn(2, 2 * ff, K, generator=g, device=DEV)
         * K ** -0.5).bfloat16()
    out = torch.empty(768, ff, device=DEV, dtype=torch.bfloat16)
    hops.expert_gemm(out, x, w, tok.int(), off, cnt, hops.ACT_SILU_GATE, 256,
                     0.0, None)
    for e, a, c in ((0, 0, 300), (1, 512, 70)):
        y = x[tok[a:a + c]].double() @ w[e].double().T
        y = torch.nn.functional.silu(y[:, :ff]) * y[:, ff:]
        # fp32 sums of K products, one rounding to bf16
        torch.testing.assert_close(out[a:a + c].double(), y, rtol=2 ** -8,
                                   atol=2 ** -12)
