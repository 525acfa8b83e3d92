"""RMSNorm over wide rows and the step after the QKV projection, at the sizes
where their launches change: rows of one and of four waves, one workgroup a
token and a part of its heads. Results are bf16: within one of its steps
(2**-7 of the value, fp32 arithmetic in another order may round the other way);
rotated values are sums of two products, each of up to the larger operand."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from sutro_amd import ops


def rand(*shape, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return torch.randn(*shape, generator=g).to(torch.bfloat16)


def close(got, want, slack=0.0):
    got, want = got.float().cpu(), want.float()
    assert ((got - want).abs() <= want.abs() * 2.0**-7 + slack).all()


@pytest.mark.parametrize("rows", [1, 2047, 2048, 2051])
@pytest.mark.parametrize("C", [264, 1024, 1032, 2048, 4096, 4104, 6144])
def test_rmsnorm(rows, C):
    x, r, w = rand(rows, C), rand(rows, C, seed=1), rand(C, seed=2)

    def norm(s):
        return s * (s.square().mean(-1, keepdim=True) + 1e-6).rsqrt() * w.double()

    close(ops.rmsnorm(x.cuda(), w.cuda(), 1e-6), norm(x.double()), 1e-6)
    s = x.double() + r.double()
    y, res = ops.fused_add_rmsnorm(x.cuda(), r.cuda(), w.cuda(), 1e-6)
    close(y, norm(s), 1e-6)
    assert torch.equal(res.cpu(), s.float().to(torch.bfloat16))


@pytest.mark.parametrize("T", [1, 3, 1023, 1024])
@pytest.mark.parametrize("Hq,Hk,D", [(16, 8, 128), (5, 1, 128), (32, 3, 64),
                                     (40, 8, 128)])
@pytest.mark.parametrize("normed", [False, True])
def test_after_qkv(T, Hq, Hk, D, normed):
    bs, nb = 16, T // 16 + 3
    qkv = rand(T, (Hq + 2 * Hk) * D)
    pos = torch.arange(T) * 7 % 501
    slots = torch.randperm(nb * bs, generator=torch.Generator().manual_seed(T))
    slots = slots[:T]
    inv = 1.0 / 10000 ** (torch.arange(0, D, 2) / D)
    ang = torch.arange(501)[:, None] * inv
    table = torch.cat([ang.cos(), ang.sin()], 1).float()
    qw, kw = (rand(D, seed=4), rand(D, seed=5)) if normed else (None, None)
    out = []
    for dev in ("cuda", "cpu"):
        k = torch.zeros(nb, Hk, bs, D, dtype=torch.bfloat16, device=dev)
        v = torch.zeros_like(k)
        f = (lambda t: None if t is None else t.to(dev)) if dev == "cuda" \
            else (lambda t: t)
        q = ops.fused_qkv_prep(f(qkv), Hq, Hk, D, f(pos), f(slots), k, v,
                               f(table), f(qw), f(kw))
        out.append((q, k, v))
    (q, k, v), (rq, rk, rv) = out
    big = float(qkv.float().abs().max()) * (4 if normed else 1)
    # the reference rounds the normed value to bf16 before it rotates
    close(q, rq, big * 2.0**-7)
    close(k, rk, big * 2.0**-7)
    assert torch.equal(v.cpu(), rv)
