"""One row's addition and RMSNorm inside the product behind it: widths below, at
and past what a pass of a workgroup takes, more sets of weight rows than
workgroups, ragged last sets; and what torch has to see goes the old way."""

import pytest
import torch
import torch.nn.functional as F

from sutro_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _operands(N, K, gated):
    g = torch.Generator(device=DEV).manual_seed(N + K)

    def rnd(*s):
        return torch.randn(*s, generator=g, device=DEV).bfloat16()

    return (rnd(1, K), rnd(1, K), (1 + 0.1 * rnd(K).float()).bfloat16(),
            (rnd(2 * N if gated else N, K).float() * K ** -0.5).bfloat16())


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("N,K", [
    (4, 32), (3072, 1024), (4100, 2016), (8192, 2048), (1028, 2080),
    (6144, 4096), (12288, 2560)])
def test_kernel(N, K, gated):
    x, res, nw, w = _operands(N, K, gated)
    before = (x.clone(), res.clone())
    got, total = ops._require_hip().norm_linear(x, res, nw, 1e-6, w, gated)
    assert torch.equal(x, before[0]) and torch.equal(res, before[1])
    s = x.double() + res.double()
    assert torch.equal(total, s.float().bfloat16())
    y = (s * torch.rsqrt(s.pow(2).mean() + 1e-6) * nw.double()).bfloat16()
    y = y.double() @ w.double().T
    if gated:
        y = F.silu(y[:, :N]) * y[:, N:]
    # a norm rounded the other way in places (2^-9 of a term of K), fp32 sums,
    # one rounding to bf16
    torch.testing.assert_close(got.double(), y, rtol=2 ** -7, atol=2 ** -8)


def test_route():
    x, res, nw, w = _operands(512, 2048, False)
    assert ops._one_row(x, res, nw, w, False)
    got, total = ops.norm_linear(x.clone(), res.clone(), nw, 1e-6, w)
    x2, r2 = ops.fused_add_rmsnorm(x.clone(), res.clone(), nw, 1e-6)
    assert torch.equal(total, r2)
    torch.testing.assert_close(got, ops.linear(x2, w), rtol=2 ** -7,
                               atol=2 ** -8)
    assert not ops._one_row(x.expand(2, 2048), res, nw, w, False)
    assert not ops._one_row(x, res.float(), nw, w, False)
    assert not ops._one_row(x, res, nw.float(), w, False)
    p = torch.nn.Parameter(nw)
    assert not ops._one_row(x, res, p, w, False)
    with torch.no_grad():
        assert ops._one_row(x, res, p, w, False)


@pytest.mark.parametrize("K", [512, 1024, 2048, 2560, 4096])
def test_norm_to_the_bit(K):
    """Through the unit matrix: the row the norm's own kernel makes."""
    eye = torch.eye(K, device=DEV).bfloat16()
    for seed in range(20):
        torch.manual_seed(seed)
        x, res = (torch.randn(1, K, device=DEV).bfloat16() for _ in range(2))
        nw = (1 + 0.1 * torch.randn(K, device=DEV)).bfloat16()
        got, total = ops._require_hip().norm_linear(x, res, nw, 1e-6, eye,
                                                    False)
        want, r2 = ops.fused_add_rmsnorm(x.clone(), res.clone(), nw, 1e-6)
        assert torch.equal(got, want) and torch.equal(total, r2)


@pytest.mark.parametrize("N,K,gated", [
    (8188, 2048, False), (8200, 2080, False), (20000, 4096, False),
    (4100, 2048, True), (12288, 3104, True)])
def test_one_row_through_sets(N, K, gated):
    """2047 and more sets of weight rows, without a norm."""
    x, _, _, w = _operands(N, K, gated)
    got = ops._require_hip().linear_skinny(x, w, None, gated).double()
    y = x.double() @ w.double().T
    if gated:
        y = F.silu(y[:, :N]) * y[:, N:]
    # fp32 sums of K products of size 1, one rounding to bf16 at the end
    torch.testing.assert_close(got, y, rtol=2 ** -8, atol=2 ** -12)
