"""Embedding sums with their norm, queries and keys of tied attention and the read-out
of the mLSTM against float64, at the widths where their vector forms begin, end and
change the number of vectors a thread (others take the general kernels).

Rounding to bf16 (8 significant bits) is off by up to 2**-8 of a value, sums of n
squares in any order by fewer than n 2**-24 of themselves and by half as much below a
root; ten more operations of 2**-24 each are allowed for."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from sutro_amd.ops import hybrid as hops
    from sutro_amd.ops import torch_ref

TYPES = [torch.bfloat16, torch.float32]


def rand(*shape, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return torch.randn(*shape, generator=g)


def close(got, want, n, extra=0.0):
    rel = (n / 2 + 10) * 2.0 ** -24
    if got.dtype == torch.bfloat16:
        rel += 2.0 ** -8
    err = (got.double().cpu() - want).abs()
    assert bool((err <= rel * want.abs() + extra).all()), float(err.max())


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("W", [4, 15, 124, 128, 1020, 1024, 1028, 2048, 4100, 8192, 8196])
@pytest.mark.parametrize("bigram,sine", [(True, True), (False, True), (False, False)])
def test_token_embed_norm(dtype, W, bigram, sine):
    T, V, buckets = 9, 33, 7
    emb, big = rand(V, W).to(dtype), rand(buckets + 1, W, seed=1).to(dtype)
    g = torch.Generator().manual_seed(W)
    ids = torch.randint(0, V, (T,), generator=g)
    prev = torch.cat([torch.tensor([-1]), ids[:-1]])
    pos = torch.arange(T) * 1000 + 3
    w = 1 + rand(W, seed=2) / 10
    freq = hops.sinusoid_inv_freq(W, 10000.0) if sine else None
    want = 0.5 * emb[ids].double()
    size = want.abs()
    if bigram:
        row = torch.where(prev < 0, buckets, (prev * 5 + ids * 9) % buckets)
        want = want + big[row].double()
        size = size + big[row].double().abs()
    if sine:
        ang = (pos.float()[:, None] * freq[None]).double()
        want = want + torch.stack([ang.sin(), ang.cos()], -1).reshape(T, -1)[:, :W]
        size = size + 1
    dev = lambda t: None if t is None else t.cuda()
    h = torch.empty(T, W, dtype=dtype, device="cuda")
    x = hops.token_embed(ids.cuda(), dev(prev), pos.cuda(), emb.cuda(),
                         big.cuda() if bigram else None, buckets if bigram else 0,
                         5, 9, dev(freq), scale=0.5, norm_w=w.cuda(), eps=1e-5, h_out=h)
    # (a sine is good to four units of its last place)
    err = (x.double().cpu() - want).abs()
    assert bool((err <= 6 * 2.0 ** -23 * size).all()), float(err.max())
    plain = hops.token_embed(ids.cuda(), dev(prev), pos.cuda(), emb.cuda(),
                             big.cuda() if bigram else None, buckets if bigram else 0,
                             5, 9, dev(freq), scale=0.5)
    assert torch.equal(x, plain)
    x = x.double().cpu()
    close(h, x / (x.square().mean(-1, keepdim=True) + 1e-5).sqrt() * w.double(), W)


@pytest.mark.parametrize("dtype,other", [TYPES, TYPES[::-1]])
def test_token_embed_norm_of_another_type(dtype, other):
    """Activations need not be of the embeddings' type."""
    emb, w = rand(33, 64).to(dtype).cuda(), (1 + rand(64, seed=2) / 10).cuda()
    ids = torch.arange(9, device="cuda")
    h = torch.empty(9, 64, dtype=other, device="cuda")
    x = hops.token_embed(ids, None, ids, emb, None, 0, 0, 0, None, norm_w=w, eps=1e-5,
                         h_out=h)
    assert torch.equal(x, emb[:9].float())
    assert torch.equal(h, hops.weighted_rmsnorm(x, w, 1e-5, other))


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("H,G,dk", [(16, 4, 128), (3, 1, 8), (1, 2, 12), (17, 1, 128),
                                    (32, 2, 128), (33, 3, 128), (8, 8, 256), (2, 2, 7),
                                    (4, 3, 64), (13, 1, 32), (55, 1, 8)])
def test_tied_attn_prep(dtype, H, G, dk):
    T, page, temp = 5, 4, 3
    q0, k0 = 8, 8 + H * dk
    proj = rand(T, k0 + G * dk + (-(G + H) * dk) % 8).to(dtype)
    qw, kw = 1 + rand(H * dk, seed=1) / 10, 1 + rand(G * dk, seed=2) / 10
    pos, slots = torch.tensor([0, 1, 2, 7, 500]), torch.tensor([3, 4, 11, 0, 9])
    kc = torch.zeros(3, G, page, dk, dtype=dtype, device="cuda")
    vc = torch.zeros_like(kc)
    q = hops.tied_attn_prep(proj.cuda(), q0, k0, H, G, dk, qw.cuda(), kw.cuda(), 1e-5,
                            pos.cuda(), 0.2, temp, slots.cuda(), kc, vc)
    p = proj.double()
    unit = lambda v: v / (v.square().mean(-1, keepdim=True) + 1e-5).sqrt()
    grow = 1 + 0.2 * torch.log(((pos + 1) // temp).double() + 1)
    close(q.reshape(T, -1), unit(p[:, q0:k0]) * qw.double() * grow[:, None], H * dk)
    raw = proj[:, k0:k0 + G * dk]
    close(kc[slots // page, :, slots % page].reshape(T, -1),
          unit(raw.double()) * kw.double(), G * dk)
    assert torch.equal(vc[slots // page, :, slots % page].reshape(T, -1).cpu(), raw)


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("H,dv", [(8, 128), (3, 1), (2, 65), (1, 129), (2, 256), (2, 257)])
def test_mlstm_out(dtype, H, dv):
    T = 7
    o, em = rand(T, H, dv + 1), rand(T, H, seed=1).exp()
    proj, w = rand(T, H * dv + 3, seed=2).to(dtype), 1 + rand(H * dv, seed=3) / 10
    out = torch.zeros(T, H * dv + 5, dtype=dtype, device="cuda")
    hops.mlstm_out(o.cuda(), em.cuda(), w.cuda(), proj.cuda(), 3, 1e-5, out, 2)
    x = o.double()
    h = x[..., :dv] / (torch.maximum(x[..., dv].abs(), em.double()) + 1e-6)[..., None]
    h = (h / (h.square().mean(-1, keepdim=True) + 1e-5).sqrt()).reshape(T, -1)
    want = h * w.double() * torch.sigmoid(proj[:, 3:].double())
    close(out[:, 2:2 + H * dv], want, dv)
    assert not out[:, :2].any() and not out[:, 2 + H * dv:].any()


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("m", [260, 520, 1024, 1028, 2048, 2052, 2056, 4096, 4104])
@pytest.mark.parametrize("parts,shared", [(1, False), (3, True), (2, None)])
def test_gated_norm_of_long_parts(dtype, m, parts, shared):
    T, n = 3, m * parts
    o, proj = rand(T, n), rand(T, n + 16, seed=1).to(dtype)
    w = None if shared is None else 1 + rand(m if shared else n, seed=2) / 10
    z = proj[:, 8:8 + n].double()
    for first, silu in ((True, False), (False, True), (False, False)):
        out = torch.zeros(T, n + 16, dtype=dtype, device="cuda")
        hops.gated_group_norm(o.cuda(), proj.cuda(), 8, None if w is None else w.cuda(),
                              1e-5, parts, first, out, 8, silu)
        gate = torch.sigmoid(z) * (z if first or silu else 1)
        y = (o.double() * gate if first else o.double()).reshape(T, parts, m)
        y = (y / (y.square().mean(-1, keepdim=True) + 1e-5).sqrt()).reshape(T, n)
        if w is not None:
            y = y * (w.double().repeat(parts) if shared else w.double())
        close(out[:, 8:8 + n], y if first else y * gate, m)
        assert not out[:, :8].any() and not out[:, 8 + n:].any()


@pytest.mark.parametrize("T", [1, 16, 17, 2048, 2049, 2117])
@pytest.mark.parametrize("E,W", [(1, 32), (4, 64), (15, 544), (28, 2048), (65, 96), (256, 512)])
def test_router_scores(T, E, W):
    """Exact products of three terms a weight, fp32 sums: off by at most 3 W 2**-24 of
    the sum of the magnitudes; sums that are not finite as one product a number has them."""
    h, w = rand(T, W).to(torch.bfloat16), rand(E, W, seed=1)
    scores = hops._mix().router_scores      # (also where a rule prefers the library)
    got = scores(h.cuda(), w.cuda()).double().cpu()
    want = h.double() @ w.double().T
    size = h.double().abs() @ w.double().abs().T
    assert bool(((got - want).abs() <= 3 * W * 2.0 ** -24 * size).all())
    h[0, 1], h[-1, W - 1], w[E - 1, 2] = float("inf"), float("nan"), 3.4e38
    w[0, 1] = abs(w[0, 1]) + 1
    got = scores(h.cuda(), w.cuda()).cpu()
    assert torch.equal(torch.isnan(got[-1]), torch.ones(E, dtype=torch.bool))
    if T > 1:
        assert float(got[0, 0]) == float("inf") and not torch.isnan(got[0]).any()
        assert torch.isfinite(got[1:-1, :E - 1]).all()
        near = 3.4e38 * h[1:-1, 2].double().abs() < 3e38
        assert torch.isfinite(got[1:-1, E - 1][near]).all()


@pytest.mark.parametrize("make", [lambda h, w: (h.float(), w), lambda h, w: (h[:, 8:], w[:, 8:]),
                                  lambda h, w: (h[:, :40], w[:, :40]),
                                  lambda h, w: (h[:, 1:33], w[:, 1:33]),
                                  lambda h, w: (h.t()[:9].t(), w.t()[:9].t())])
def test_router_scores_elsewhere(make):
    h, w = make(rand(70, 96).to(torch.bfloat16).cuda(), rand(300, 96, seed=1)[:20].cuda())
    want = h.double() @ w.double().T
    got = hops.router_scores(h, w).double()
    size = h.double().abs() @ w.double().abs().T
    assert bool(((got - want).abs() <= 3 * 96 * 2.0 ** -24 * size).all())


@pytest.mark.parametrize("T", [13, 2117])
@pytest.mark.parametrize("E,W", [(4, 32), (28, 544), (32, 2048)])
def test_router_scores_beyond_bf16(T, E, W):
    """Weights whose first bf16 number is infinite, and sums of which a part is: what
    64 bits give, rounded once."""
    h, w = rand(T, W).to(torch.bfloat16), rand(E, W, seed=1)
    h[:, 0], h[:, 1], h[:, W - 1] = 2.0, -1.5, -0.25
    w[:, 0], w[:, 1], w[1, W - 1] = 3.4e38, 3.4e38, float("inf")
    h[T // 2, 2:] = float("nan")
    got = hops._mix().router_scores(h.cuda(), w.cuda()).double().cpu()
    assert torch.isnan(got[T // 2]).all()
    sure = torch.arange(T) != T // 2
    assert (got[sure, 1] == -float("inf")).all()
    cols = torch.arange(E) != 1
    got, want = (x[sure][:, cols] for x in (got, h.double() @ w.double().T))
    assert bool(((got - want).abs() <= 2.0 ** -24 * want.abs()).all())


@pytest.mark.parametrize("T,E,W,kernel", [
    (13, 256, 2048, 1), (256, 256, 2048, 1), (257, 65, 2048, 0), (257, 64, 2048, 1),
    (30001, 64, 2048, 1), (13, 257, 2048, 0), (1024, 48, 8192, 1), (1025, 48, 8192, 0),
    (1536, 48, 5120, 1), (2999, 16, 6144, 0), (3000, 16, 6144, 1), (13, 32, 2040, 0)])
def test_router_rule(T, E, W, kernel):
    h = torch.empty(T, W, dtype=torch.bfloat16, device="cuda")      # (never read)
    assert hops._router_kernel(h, torch.empty(E, W, device="cuda")) == bool(kernel)
