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
