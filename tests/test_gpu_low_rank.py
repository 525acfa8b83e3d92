"""The low-rank gates on the matrix cores against float64, at the edges of their
tiles (16 tokens, 128 a wave, 512 a workgroup; 16 channels) and for every rank
they take. W2 is split exactly, the products are exact and the sums fp32: the
pre-activation is off by at most (3 rank + 2) 2**-24 of the sum of the
magnitudes, and gates have a slope below 1 (decay: below exp(a_log) / e + 1)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from sutro_amd.ops import hybrid as hops


def rand(*shape, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return torch.randn(*shape, generator=g)


@pytest.mark.parametrize("T", [1, 15, 17, 128, 129, 513])
@pytest.mark.parametrize("rank,dk,dv", [(8, 64, 64), (32, 128, 128),
                                        (24, 192, 128), (16, 128, 64)])
def test_low_rank_gates(T, rank, dk, dv):
    H = 3
    qo, ko, vo = 0, H * dk, 2 * H * dk
    bo = vo + H * dv
    ao = bo + 8
    go = ao + rank
    proj = rand(T, go + rank).to(torch.bfloat16)
    proj[0, ao], proj[-1, go] = float("inf"), float("-inf")
    a2, g2 = rand(H * dk, rank, seed=1), rand(H * dv, rank, seed=2)
    a2[:, 0], g2[:, 0] = 0.5, 0.25       # two of the three terms are zero there
    dt_bias, a_log = rand(H * dk, seed=3), rand(H, seed=4) * 0.3
    C = 2 * H * dk + H * dv
    i32 = dict(dtype=torch.int32, device="cuda")
    _, _, _, decay, beta = hops.delta_prep(
        proj.cuda(), qo, ko, vo, bo, ao, H, H, dk, dv, rand(C, 4).cuda(),
        a2.cuda(), dt_bias.cuda(), a_log.cuda(),
        torch.zeros(1, 3, C, device="cuda"), torch.zeros(1, **i32),
        torch.tensor([0, T], **i32), torch.tensor([T], **i32),
        token_seq=torch.zeros(T, **i32))
    x = proj[:, ao:ao + rank].double()
    x[0, 0] = 3.38953139e38
    pre = x @ a2.double().t() + dt_bias.double()
    mag = x.abs() @ a2.double().abs().t() + dt_bias.double().abs()
    rate = a_log.double().exp()[:, None]
    want = torch.exp(-rate * torch.nn.functional.softplus(pre).view(T, H, dk))
    err = (3 * rank + 2) * 2.0**-24 * mag.view(T, H, dk)
    got = decay.cpu().double()
    assert ((got - want).abs() <= (rate / 2.718 + 1) * err + 1e-6)[1:].all()
    assert (got[0] == 0).all()
    torch.testing.assert_close(beta.cpu(), proj[:, bo:bo + H].float().sigmoid(),
                               rtol=1e-6, atol=1e-6)
    o, nw = rand(T, H, dv, seed=5), rand(dv, seed=6)
    out = torch.zeros(T, H * dv + 16, dtype=torch.bfloat16, device="cuda")
    hops.delta_out(o.cuda(), nw.cuda(), proj.cuda(), go, g2.cuda(), 2e-5, out,
                   8, 0.45)
    x = proj[:, go:go + rank].double()
    x[-1, 0] = -3.38953139e38
    pre = (x @ g2.double().t()).view(T, H, dv)
    mag = (x.abs() @ g2.double().abs().t()).view(T, H, dv)
    n = o.double() * (o.double().square().mean(-1, keepdim=True) + 2e-5).rsqrt()
    n = 0.45 * n * nw.double()
    want = n * pre.sigmoid()
    bound = want.abs() * 2.0**-8 + n.abs() * ((3 * rank + 2) * 2.0**-24 * mag
                                              + 1e-6)
    got = out.cpu().double()
    assert (got[:, :8] == 0).all() and (got[:, 8 + H * dv:] == 0).all()
    got = got[:, 8:8 + H * dv].view(T, H, dv)
    ok = (got - want).abs() <= bound
    assert ok[:-1].all() and (got[-1] == 0).all()


@pytest.mark.parametrize("T", [1400, 8191, 60000])   # 16, 32, 128 tokens a wave
def test_tokens_of_a_wave(T):
    """A token's gate does not depend on how many tokens its wave takes."""
    H, dv, rank = 16, 64, 16
    g = torch.Generator(device="cuda").manual_seed(T)
    o = torch.randn(T, H, dv, generator=g, device="cuda")
    proj = torch.randn(T, rank, generator=g, device="cuda").bfloat16()
    g2 = torch.randn(H * dv, rank, generator=g, device="cuda")
    norm_w = torch.randn(dv, generator=g, device="cuda")

    def gate(rows):
        out = torch.full((rows.stop - rows.start, H * dv), 7.0, device="cuda",
                         dtype=torch.bfloat16)
        hops.delta_out(o[rows], norm_w, proj[rows], 0, g2, 1e-5, out, 0, 1.0)
        return out

    whole = gate(slice(0, T))
    for a in (0, 100, T // 2, T - 90):
        rows = slice(a, min(a + 90, T))
        assert torch.equal(whole[rows], gate(rows))
    assert (whole != 7.0).any(1).all()
