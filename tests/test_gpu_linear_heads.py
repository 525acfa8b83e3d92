"""QKV projections of prompts with qk-norm, rotation and the store to pages in the
same launch: edges of row tiles, few and many heads, short k, tokens out of order."""

import pytest
import torch

from sutro_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(M, Hq, Hk, K, bs=32, seed=0, norm=True):
    g = torch.Generator(device=DEV).manual_seed(seed + M + K)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn((Hq + 2 * Hk) * 128, K, generator=g, device=DEV)
         * K ** -0.5).bfloat16()
    pos = torch.randint(0, 500, (M,), generator=g, device=DEV)
    blocks = -(-M // bs) + 3
    slots = torch.randperm(blocks * bs, generator=g, device=DEV)[:M]
    kc, vc = (torch.full((blocks, Hk, bs, 128), 7., device=DEV).bfloat16()
              for _ in range(2))
    cos_sin = torch.randn(500, 128, generator=g, device=DEV)
    n = [torch.rand(128, generator=g, device=DEV).bfloat16() if norm else None
         for _ in range(2)]
    return x, w, kc, vc, pos, slots, cos_sin, *n


def _exact(x, w, kc, vc, pos, slots, cos_sin, qw, kw, eps):
    Hk, bs = kc.shape[1:3]
    y = (x.double() @ w.double().T).view(x.shape[0], -1, 128)
    Hq = y.shape[1] - 2 * Hk
    c, s = (cos_sin[pos].double()[:, None, a:a + 64] for a in (0, 64))

    def turned(h, n):
        if n is not None:
            h = h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + eps) * n.double()
        a, b = h[..., :64], h[..., 64:]
        return torch.cat([a * c - b * s, b * c + a * s], -1)

    kc, vc = kc.double().clone(), vc.double().clone()
    kc[slots // bs, :, slots % bs] = turned(y[:, Hq:Hq + Hk], kw)
    vc[slots // bs, :, slots % bs] = y[:, Hq + Hk:]
    return turned(y[:, :Hq], qw), kc, vc


@pytest.mark.parametrize("M,Hq,Hk,K,norm", [
    (1, 2, 1, 192, True), (255, 2, 1, 256, True), (257, 4, 2, 320, False),
    (1000, 16, 4, 1024, True), (8193, 8, 8, 192, True), (2600, 16, 8, 2048, True),
    (777, 6, 1, 4096, True)])
@pytest.mark.parametrize("bs", [32, 16])
def test_kernel(M, Hq, Hk, K, norm, bs):
    ops_in = _case(M, Hq, Hk, K, bs, norm=norm)
    x, w, kc, vc, *rest = ops_in
    want = _exact(*ops_in, 1e-6)
    q = ops._require_hip().linear_heads(x, w, kc, vc, *rest, 1e-6)
    # fp32 sums, norm and rotation: one rounding to bf16 at the end
    for got, ref in zip((q, kc, vc), want):
        torch.testing.assert_close(got.double(), ref, rtol=2 ** -8, atol=2 ** -12)


def test_route():
    """Both ways agree; what the one launch does not take goes the other way."""
    M, Hq, Hk, K = 4096, 16, 8, 512
    x, w, kc, vc, pos, slots, cos_sin, qw, kw = _case(M, Hq, Hk, K)
    args = (Hq, Hk, 128, pos, slots)
    k2, v2 = kc.clone(), vc.clone()
    one = ops.linear_qkv_prep(x, w, *args, kc, vc, cos_sin, qw, kw, 1e-6)
    two = ops.fused_qkv_prep(ops.linear(x, w), *args, k2, v2, cos_sin, qw, kw, 1e-6)
    # (two roundings to bf16 there, rotated into each other)
    for a, b in ((one, two), (kc, k2), (vc, v2)):
        torch.testing.assert_close(a.float(), b.float(), rtol=2 ** -7, atol=2 ** -5)
    f8 = torch.float8_e4m3fn
    for a, k, v in ((args, kc.to(f8), vc.to(f8)),
                    ((2 * Hq, 2 * Hk, 64) + args[3:], kc.view(-1, 16, 32, 64),
                     vc.view(-1, 16, 32, 64))):
        assert ops.linear_qkv_prep(x, w, *a, k, v, cos_sin, qw, kw, 1e-6) is None
    assert ops.linear_qkv_prep(x[:64], w, *args, kc, vc, cos_sin, qw, kw,
                               1e-6) is None


@pytest.mark.parametrize("which", range(2, 9))
def test_operands_on_the_host(which):
    """An error, by either way, and not an address of the host's on the GPU."""
    M, Hq, Hk, K = 4096, 16, 8, 512
    host = list(_case(M, Hq, Hk, K))
    host[which] = host[which].cpu()
    x, w, kc, vc, pos, slots, cos_sin, qw, kw = host
    args = (Hq, Hk, 128, pos, slots, kc, vc, cos_sin, qw, kw, 1e-6)
    assert ops.linear_qkv_prep(x, w, *args) is None
    with pytest.raises(RuntimeError, match="GPU"):
        ops._require_hip().linear_heads(*host, 1e-6)
    with pytest.raises(RuntimeError, match="GPU"):
        ops.fused_qkv_prep(ops.linear(x, w), *args)


def test_longer_positions():
    """Positions and slots of the largest batch, of which the first are used."""
    M, Hq, Hk, K = 4096, 16, 8, 512
    x, w, kc, vc, pos, slots, cos_sin, qw, kw = _case(M, Hq, Hk, K)
    qkv, outs = ops.linear(x, w), []
    for p, s in ((pos, slots), (pos.repeat(2), slots.repeat(2))):
        k, v = kc.clone(), vc.clone()
        args = (Hq, Hk, 128, p, s, k, v, cos_sin, qw, kw, 1e-6)
        assert (ops.linear_qkv_prep(x, w, *args) is None) == (p is not pos)
        outs.append((ops.fused_qkv_prep(qkv, *args), k, v))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
