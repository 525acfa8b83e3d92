"""The gated residual norm at the widths and row counts where its launch changes,
against float64 (a sum of W squares in fp32 in any order: W 2**-24 of it; sigmoid
good to 2**-21)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from sutro_amd.ops import hybrid as hops


@pytest.mark.parametrize("T,W", [(1, 2048), (2047, 2048), (2049, 2048),
                                 (2050, 1032), (3, 4096), (2, 8192), (5, 72)])
def test_gated_norm_residual(T, W):
    g = torch.Generator().manual_seed(T + W)
    x = torch.randn(T, W, generator=g)
    y = torch.randn(T, W, generator=g).to(torch.bfloat16)
    proj = torch.randn(T, W + 16, generator=g).to(torch.bfloat16)
    gain = torch.tensor([1.3])
    h = torch.empty(T, W, dtype=torch.bfloat16, device="cuda")
    xd = x.cuda()
    hops.gated_norm_residual(xd, y.cuda(), proj.cuda(), 8, gain.cuda(), 2e-5,
                             0.75, h)
    z = y.double() * proj[:, 8:8 + W].double().sigmoid()
    step = 0.75 * gain.double() * z * (z.square().mean(-1, keepdim=True)
                                       + 2e-5).rsqrt()
    bound = step.abs() * (W * 2.0**-24 + 2.0**-20) + 2.0**-23 * (1 + x.abs())
    assert ((xd.cpu().double() - x.double() - step).abs() <= bound).all()
    assert torch.equal(h.cpu(), xd.cpu().to(torch.bfloat16))
