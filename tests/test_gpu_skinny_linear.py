"""Linear layers over few rows: the kernel against float64 at the edges of its
tiles, and what ops.linear sends to it.

The sums are fp32 over K products of bf16 (exact in fp32): off by at most
K 2**-24 of the sum of the magnitudes, in any order; the result is rounded to
bf16, 2**-8 of itself (with the gated unit, of the unit: silu's slope is below
1.1, and its exponential is good to 2**-20)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from sutro_amd import _C, ops
    from sutro_amd.models.linear import Linear


def rand(*shape, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return torch.randn(*shape, generator=g).to(torch.bfloat16).cuda()


# rows: one, two (lanes along k), 16 and 32 (blocks of the matrix core) and
# around; K: one step, less than a wave's share, no multiple of a batch
@pytest.mark.parametrize("M", [1, 2, 3, 15, 16, 17, 32])
@pytest.mark.parametrize("K,N", [(32, 8), (96, 40), (512, 64), (1024, 2056),
                                 (1056, 24), (2080, 136), (4096, 8200),
                                 (6176, 96)])
def test_against_float64(M, K, N):
    w = rand(N, K) * K ** -0.5
    bias = rand(N, seed=3)
    # rows with a gap between them
    x = rand(M, K + 8, seed=1)[:, :K]
    exact = x.double() @ w.double().t()
    mag = x.double().abs() @ w.double().abs().t()
    for b in (None, bias):
        want = exact + (b.double() if b is not None else 0)
        got = _C.linear_skinny(x, w, b, False).double()
        bound = want.abs() * 2.0**-8 + (K + 2) * 2.0**-24 * (mag + 4)
        assert ((got - want).abs() <= bound).all()
    got = _C.linear_skinny(x, w, None, True).double()
    g, u = exact[:, :N // 2], exact[:, N // 2:]
    err = (K + 2) * 2.0**-24 * mag
    want = F.silu(g) * u
    bound = want.abs() * (2.0**-8 + 2.0**-19) \
        + 1.1 * err[:, :N // 2] * u.abs() + err[:, N // 2:] * g.abs() + 1e-9
    assert ((got - want).abs() <= bound).all()


def test_route():
    """What the kernel does not take stays with the library."""
    w = rand(256, 512)
    x = rand(8, 512)
    assert ops._few_rows(x, w) and ops._few_rows(x[:1], w)
    no = [(rand(33, 512), w), (x.float(), w.float()), (rand(8, 500), rand(256, 500)),
          (x, rand(254, 512)), (x, rand(512, 256).t()),
          (rand(512, 8).t(), w), (rand(8, 516)[:, :512], w),
          (rand(8 * 512 + 1)[1:].view(8, 512), w), (x[None], w),
          (rand(8, 8192), rand(2048, 8192)), (rand(0, 512), w)]
    for a, b in no:
        assert not ops._few_rows(a, b)
    layer = Linear(512, 256, bias=True, dtype=torch.bfloat16).cuda()
    y = layer(x)                                 # records a graph: library
    assert y.requires_grad
    with torch.no_grad():
        z = layer(x)
    ref = F.linear(x.double(), layer.weight.double(), layer.bias.double())
    assert (z.double() - ref).abs().max() < 2.0**-7
    seen = []
    layer.register_forward_hook(lambda m, a, o: seen.append(o))
    with torch.no_grad():
        layer(x)
    assert len(seen) == 1
