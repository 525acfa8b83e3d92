"""Linear layers over 2 to 256 rows: the kernel against float64 at the edges of its
tiles, with every tile it chooses from, and what ops.linear sends to it.

The sums are fp32 over K products of bf16 (exact in fp32): off by at most K 2**-24 of
the sum of the magnitudes, in any order; the result is rounded to bf16, 2**-8 of
itself (with the gated unit, of the unit: silu's slope is below 1.1, and its
exponential is good to 2**-20)."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from sutro_amd import _C, ops


def rand(*shape, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return torch.randn(*shape, generator=g).to(torch.bfloat16).cuda()


def check(M, K, N, gated):
    w = rand(2 * N if gated else N, K) * K ** -0.5
    x = rand(M, K + 8, seed=1)[:, :K]          # rows with a gap between them
    exact = x.double() @ w.double().t()
    mag = x.double().abs() @ w.double().abs().t()
    if gated:
        got = _C.linear_mid(x, w, None, True).double()
        g, u = exact[:, :N], exact[:, N:]
        err = (K + 2) * 2.0**-24 * mag
        want = F.silu(g) * u
        bound = want.abs() * (2.0**-8 + 2.0**-19) \
            + 1.1 * err[:, :N] * u.abs() + err[:, N:] * g.abs() + 1e-9
        assert ((got - want).abs() <= bound).all()
        return
    bias = rand(N, seed=3)
    for b in (None, bias):
        want = exact + (b.double() if b is not None else 0)
        got = _C.linear_mid(x, w, b, False).double()
        bound = want.abs() * 2.0**-8 + (K + 2) * 2.0**-24 * (mag + 4)
        assert ((got - want).abs() <= bound).all()


# the tile follows from rows and weight rows: one tile and less, its edges, more tiles
# than a round; K of one step, of less steps than the ring, of many
@pytest.mark.parametrize("M", [2, 31, 32, 33, 64, 65, 127, 129, 200, 256])
@pytest.mark.parametrize("N", [4, 20, 1000, 3080])
@pytest.mark.parametrize("K", [256, 768, 2048])
def test_kernel(M, N, K):
    check(M, K, N, False)
    check(M, K, N, True)


@pytest.mark.parametrize("M,N,K", [
    (9, 4100, 4096), (16, 8200, 2048), (30, 16400, 512), (32, 33000, 256),
    (40, 8300, 1024), (64, 16500, 768), (50, 33000, 512), (100, 8300, 1024),
    (128, 16600, 512), (90, 33000, 256), (180, 12000, 512), (250, 16000, 512),
    # starts at eighths of k
    (20, 16400, 2048), (31, 33000, 2048), (60, 9000, 4096), (64, 33000, 2048),
    (100, 9000, 2048), (128, 16600, 2048), (128, 33000, 4096)])
def test_larger_tiles(M, N, K):
    check(M, K, N, False)
    check(M, K, N // 8 * 4, True)


@pytest.mark.parametrize("M,N,K,gated", [(60, 2048, 2048, False),
                                         (250, 4096, 2048, True),
                                         (20, 32768, 2048, False)])
def test_place_of_a_row(M, N, K, gated):
    """Equal rows of a batch have equal results, in whichever tile they are."""
    x, w = rand(5, K), rand(N, K, seed=1)
    which = torch.arange(M, device="cuda") * 3 % 5
    got = _C.linear_mid(x[which], w, None, gated)
    for t in range(5):
        same = got[which == t]
        assert torch.equal(same, same[:1].expand_as(same)), t


def test_replays():
    """In a graph, several times, between other work."""
    x, w, out = rand(48, 2048), rand(3072, 2048, seed=2), None
    want = ops.linear(x, w)
    assert ops._mid_rows(x, w)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = ops.linear(x, w)
    for i in range(3):
        out.zero_()
        g.replay()
        (x @ x.t()).sum().item()
        assert torch.equal(out, want)


def test_refused():
    x, w = rand(8, 512), rand(256, 512)
    for a, b, gated in ((rand(257, 512), w, False), (rand(8, 320), rand(256, 320), False),
                        (x, rand(254, 512), False), (x.float(), w, False),
                        (x, rand(512, 256).t(), False), (rand(8, 516)[:, :512], w, False),
                        (x[:, :256], w, False)):
        with pytest.raises(RuntimeError):
            _C.linear_mid(a, b, None, gated)
