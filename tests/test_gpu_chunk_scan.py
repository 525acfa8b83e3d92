"""Recurrences with one decay per head, and the gated delta rule, in chunks of 32
tokens, beside sequences too short for them, against the recurrence in float64: sizes around the chunk, the key and
value tiles and the last column group, grouped keys, strided rows, old and new states."""

import pytest
import torch

from sutro_amd.ops import hybrid as hops
from sutro_amd.ops import torch_ref as ref

pytestmark = pytest.mark.gpu

DEV = "cuda"
LENS = [33, 1, 95, 0, 32, 31, 64, 200, 7]
OLD = [0, 5, 3, 2, 0, 9, 40, 0, 0]       # tokens a sequence had before


def _batch():
    q = torch.tensor([0] + LENS).cumsum(0).int()
    total = torch.tensor([n + o for n, o in zip(LENS, OLD)], dtype=torch.int32)
    slots = torch.tensor([4, 9, 0, 7, 2, 1, 8, 3, 6], dtype=torch.int32)
    return q, total, slots


def _recur(q, k, v, a, b, skip, state, qlocs, total, slots):
    """In float64: [T, G, dk], [T, H, dv], [T, H] -> o, states by slot."""
    rep = v.shape[1] // k.shape[1]
    q, k = (x.double().repeat_interleave(rep, 1) for x in (q, k))
    v, a, b, state = v.double(), a.double(), b.double(), state.double().clone()
    o = torch.zeros(v.shape, dtype=torch.float64)
    for s in range(len(total)):
        lo, hi = int(qlocs[s]), int(qlocs[s + 1])
        if lo == hi:
            continue
        S = state[slots[s]] * (1.0 if int(total[s]) > hi - lo else 0.0)
        for t in range(lo, hi):
            S = (S * a[t][:, None, None]
                 + k[t][:, :, None] * (b[t][:, None] * v[t])[:, None, :])
            o[t] = (S * q[t][:, :, None]).sum(1) + skip.double()[:, None] * v[t]
        state[slots[s]] = S
    return o, state


def _off(got, want):
    return float((got.double().cpu() - want).norm() / want.norm())


# fp32 sums of up to dk + 32 products, a few roundings each: below 32 units of 2^-24
TOL = 32 * 2.0 ** -24


@pytest.mark.parametrize("H,G,dk,dv,kind", [
    (2, 2, 128, 128, "constant"), (4, 2, 128, 130, "token"),
    (2, 1, 100, 20, "token"), (3, 3, 64, 256, "constant"), (2, 2, 36, 72, "token"),
    (2, 2, 8, 300, "constant"), (2, 2, 128, 16, "zero")])
def test_decay_chunks(H, G, dk, dv, kind):
    g = torch.Generator().manual_seed(dk + dv)
    qlocs, total, slots = _batch()
    T = int(qlocs[-1])
    # rows of one buffer, as the mixers hand them over
    buf = torch.randn(T, 2 * G * dk + H * dv + 4, generator=g)
    q = buf[:, :G * dk].view(T, G, dk)
    k = buf[:, G * dk:2 * G * dk].view(T, G, dk)
    v = buf[:, 2 * G * dk:2 * G * dk + H * dv].view(T, H, dv)
    state = torch.randn(11, H, dk, dv, generator=g)
    if kind == "constant":
        a = 1.0 - 2.0 ** torch.linspace(-2.0, -9.0, H)
        gain = skip = None
    else:
        a = torch.rand(T, H, generator=g)
        if kind == "zero":              # decays that forget everything, and growth
            a[::5] = 0.0
            a[3::7] = 1.25
        gain, skip = torch.rand(T, H, generator=g), torch.randn(H, generator=g)
    want, end = _recur(
        q, k, v, a.expand(T, H) if a.dim() == 1 else a,
        torch.ones(T, H) if gain is None else gain,
        torch.zeros(H) if skip is None else skip, state, qlocs, total, slots)
    d = buf.to(DEV)
    st = state.to(DEV)
    o = hops.decay_scan(
        d[:, :G * dk].unflatten(1, (G, dk)),
        d[:, G * dk:2 * G * dk].unflatten(1, (G, dk)),
        d[:, 2 * G * dk:2 * G * dk + H * dv].unflatten(1, (H, dv)), a.to(DEV),
        None if gain is None else gain.to(DEV),
        None if skip is None else skip.to(DEV), st, slots.to(DEV),
        qlocs.to(DEV), total.to(DEV))
    assert _off(o, want) < TOL
    assert _off(st, end) < TOL
    for s in (5, 10):                   # slots of no sequence, and of an empty one
        assert torch.equal(st[s].cpu(), state[s])
    assert torch.equal(st[7].cpu(), state[7])


@pytest.mark.parametrize("which", ["q", "k", "v", "windows"])
def test_rows_less_than_a_head_apart(which):
    """One row for all tokens, and rows that overlap: token by token, as ever."""
    g = torch.Generator().manual_seed(12)
    H, dk, dv = 2, 64, 48
    qlocs, total, slots = _batch()
    T = int(qlocs[-1])
    x = {"q": torch.randn(T, 1, dk, generator=g), "k": torch.randn(T, 1, dk, generator=g),
         "v": torch.randn(T, H, dv, generator=g)}
    dev = {n: t.to(DEV) for n, t in x.items()}
    if which == "windows":
        buf = torch.randn(4 * T + dk, generator=g)
        x["k"] = buf.as_strided((T, 1, dk), (4, dk, 1))
        dev["k"] = buf.to(DEV).as_strided((T, 1, dk), (4, dk, 1))
    else:
        x[which], dev[which] = (t[which][:1].expand(T, -1, -1) for t in (x, dev))
    a = torch.rand(T, H, generator=g)
    state = torch.randn(11, H, dk, dv, generator=g)
    want, end = _recur(*x.values(), a, torch.ones(T, H), torch.zeros(H), state, qlocs,
                       total, slots)
    st = state.to(DEV)
    o = hops.decay_scan(*dev.values(), a.to(DEV), None, None, st, slots.to(DEV),
                        qlocs.to(DEV), total.to(DEV))
    assert _off(o, want) < TOL
    assert _off(st, end) < TOL


@pytest.mark.parametrize("H,dk,dv", [(2, 128, 128), (3, 64, 40), (1, 12, 144),
                                     (2, 100, 143)])
def test_mlstm_chunks(H, dk, dv):
    g = torch.Generator().manual_seed(dk + dv)
    qlocs, total, slots = _batch()
    T = int(qlocs[-1])
    cols = 2 * H * dk + H * dv
    cols += -cols % 4
    proj = torch.randn(T, cols + 2 * H + 8, generator=g)
    proj = proj[:, :(cols + 2 * H + 3) // 4 * 4].contiguous().bfloat16()
    offs = (0, H * dk, 2 * H * dk, cols, cols + H)
    ib, fb = torch.randn(H, generator=g), torch.randn(H, generator=g) + 2
    mem = torch.randn(11, H, dk, dv + 1, generator=g)
    m0 = torch.randn(11, H, generator=g)
    args = (H, dk, dv, ib, fb, 5.0)
    want_m, want_ms = mem.clone(), m0.clone()
    want, em = ref.mlstm_scan(proj, *offs, *args, want_m, want_ms, slots, qlocs,
                              total)
    md, ms = mem.to(DEV), m0.to(DEV)
    o, got_em = hops.mlstm_scan(proj.to(DEV), *offs, H, dk, dv, ib.to(DEV),
                                fb.to(DEV), 5.0, md, ms, slots.to(DEV),
                                qlocs.to(DEV), total.to(DEV))
    # the reference is fp32 as well: its roundings and its gates' beside the kernel's
    assert _off(o, want.double()) < 4 * TOL
    assert _off(md, want_m.double()) < 4 * TOL
    assert _off(got_em, em.double()) < 4 * TOL


def _delta(q, k, v, d, beta, state, qlocs, total, slots):
    """The gated delta rule in float64; d [T, H, dk]."""
    rep = v.shape[1] // k.shape[1]
    q, k = (x.double().repeat_interleave(rep, 1) for x in (q, k))
    v, d, beta = v.double(), d.double(), beta.double()
    state = state.double().clone()
    o = torch.zeros(v.shape, dtype=torch.float64)
    for s in range(len(total)):
        lo, hi = int(qlocs[s]), int(qlocs[s + 1])
        if lo == hi:
            continue
        S = state[slots[s]] * (1.0 if int(total[s]) > hi - lo else 0.0)
        for t in range(lo, hi):
            S = S * d[t][:, :, None]
            u = beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
            S = S + k[t][:, :, None] * u[:, None, :]
            o[t] = (S * q[t][:, :, None]).sum(1)
        state[slots[s]] = S
    return o, state


@pytest.mark.parametrize("H,G,dk,dv,kind", [
    (2, 2, 128, 128, "channel"), (4, 2, 128, 130, "head"), (2, 1, 100, 20, "channel"),
    (3, 3, 64, 72, "head"), (2, 2, 36, 144, "channel"), (2, 2, 8, 16, "head"),
    (2, 2, 128, 48, "zero"), (2, 2, 128, 128, "one"), (17, 17, 64, 128, "channel"),
    (16, 16, 128, 128, "channel"), (16, 4, 128, 128, "head"), (17, 17, 64, 72, "head"),
    (8, 8, 96, 200, "channel"), (8, 2, 128, 260, "head"), (15, 5, 60, 136, "head")])
def test_delta_chunks(H, G, dk, dv, kind):
    g = torch.Generator().manual_seed(dk + dv + H)
    lens = [65, 1, 95, 0, 64, 63, 96, 200, 7]
    if H >= 8:              # above 128 groups of up to 128 columns: eight tiles in each
        assert 9 * H * -(-dv // 128) > 128 and dv > 64
        lens = [64 + i for i in range(9)]
    qlocs = torch.tensor([0] + lens).cumsum(0).int()
    total = torch.tensor([n + o for n, o in zip(lens, OLD)], dtype=torch.int32)
    _, _, slots = _batch()
    T = int(qlocs[-1])
    unit = torch.nn.functional.normalize
    q = unit(torch.randn(T, G, dk, generator=g), dim=-1) * dk ** -0.5
    k = unit(torch.randn(T, G, dk, generator=g) + 0.2, dim=-1)
    v = torch.randn(T, H, dv, generator=g)
    shape = (T, H) if kind == "head" else (T, H, dk)
    d = torch.exp(-0.5 * torch.nn.functional.softplus(
        torch.randn(shape, generator=g) * 2))
    if kind == "zero":                  # memory that ends, and strong decays
        d[::5] = 0.0
        d[3::7, :, ::2] = 1e-30
    if kind == "one":                   # no decay at all
        d[:] = 1.0
    beta = torch.sigmoid(torch.randn(T, H, generator=g))
    state = torch.randn(11, H, dk, dv, generator=g)
    want, end = _delta(q, k, v, d[..., None].expand(T, H, dk) if kind == "head" else d,
                       beta, state, qlocs, total, slots)
    st = state.to(DEV)
    o = hops.delta_scan(*(x.to(DEV) for x in (q, k, v, d, beta)), st, slots.to(DEV),
                        qlocs.to(DEV), total.to(DEV))
    assert _off(o, want) < TOL
    assert _off(st, end) < TOL
    for s in (5, 10) + ((7,) if H < 8 else ()):
        assert torch.equal(st[s].cpu(), state[s])


@pytest.mark.parametrize("bad", [float("inf"), float("nan"), 3e38])
@pytest.mark.parametrize("which", ["q", "k", "v", "d", "beta", "state"])
def test_delta_numbers_that_are_not_finite(bad, which):
    g = torch.Generator().manual_seed(5)
    H, dk, dv, T = 2, 64, 48, 170
    qlocs = torch.tensor([0, 90, 170], dtype=torch.int32)
    total = torch.tensor([94, 84], dtype=torch.int32)
    slots = torch.tensor([1, 0], dtype=torch.int32)
    x = {"q": torch.randn(T, H, dk, generator=g) * dk ** -0.5,
         "k": torch.nn.functional.normalize(torch.randn(T, H, dk, generator=g), dim=-1),
         "v": torch.randn(T, H, dv, generator=g),
         "d": torch.rand(T, H, dk, generator=g) * 0.5 + 0.5,
         "beta": torch.rand(T, H, generator=g)}
    state = torch.randn(2, H, dk, dv, generator=g)
    if which == "state":
        state[1, 0, 5, 7] = bad
    elif which == "beta":
        x["beta"][41, 1] = bad
    else:
        x[which][41, 1, 9] = bad
    want_s = state.clone()
    want = ref.delta_scan(*x.values(), want_s, slots, qlocs, total)
    st = state.to(DEV)
    got = hops.delta_scan(*(y.to(DEV) for y in x.values()), st, slots.to(DEV),
                          qlocs.to(DEV), total.to(DEV)).cpu()
    # every other head and sequence is as it was, and so are the tokens before
    mine = torch.zeros_like(want, dtype=torch.bool)
    head = 0 if which == "state" else 1
    mine[0 if which == "state" else 41:90, head] = True
    torch.testing.assert_close(got[~mine], want[~mine], rtol=2e-4, atol=2e-4)
    assert torch.equal(torch.isfinite(got), torch.isfinite(want))
    fine = torch.isfinite(want_s)
    assert torch.equal(torch.isfinite(st.cpu()), fine)
    # and what is finite is right; numbers of 3e38 that cancel leave 2^-20 of themselves
    off = 2e-4 + 2.0 ** -20 * torch.where(fine, want_s, 0).abs().amax(2, True)
    diff = torch.where(fine, st.cpu() - want_s, 0).abs()
    assert (diff <= off + 2e-4 * torch.where(fine, want_s, 0).abs()).all()


@pytest.mark.parametrize("bad", [float("inf"), float("nan"), 3e38])
@pytest.mark.parametrize("which", ["q", "k", "v", "decay", "state"])
def test_numbers_that_are_not_finite(bad, which):
    """They reach what the recurrence lets them reach: no earlier token, no other
    sequence, and in a value no other column."""
    g = torch.Generator().manual_seed(3)
    H, dk, dv = 2, 64, 48
    lens, old = [70, 40], [4, 4]
    qlocs = torch.tensor([0, 70, 110], dtype=torch.int32)
    total = torch.tensor([74, 44], dtype=torch.int32)
    slots = torch.tensor([1, 0], dtype=torch.int32)
    T = 110
    q, k = (torch.randn(T, H, dk, generator=g) for _ in "qk")
    v = torch.randn(T, H, dv, generator=g)
    a = torch.rand(T, H, generator=g) * 0.5 + 0.5
    state = torch.randn(2, H, dk, dv, generator=g)
    where = {"q": q, "k": k, "v": v}
    if which == "decay":
        a[41, 1] = bad
    elif which == "state":
        state[1, 0, 5, 7] = bad
    else:
        where[which][41, 1, 9] = bad
    want_s = state.clone()
    want = ref.decay_scan(q, k, v, a, None, None, want_s, slots, qlocs, total)
    st = state.to(DEV)
    got = hops.decay_scan(q.to(DEV), k.to(DEV), v.to(DEV), a.to(DEV), None, None,
                          st, slots.to(DEV), qlocs.to(DEV), total.to(DEV)).cpu()
    for x, y in ((got, want), (st.cpu(), want_s)):
        fine = torch.isfinite(y)
        assert torch.equal(torch.isfinite(x), fine)
        torch.testing.assert_close(x[fine], y[fine], rtol=2e-4, atol=2e-4)


# (What overflows in the order of one sum only, 3e38 times a gain, may be finite in the
# other: not compared.)
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("which", ["v", "gain", "skip", "decay"])
def test_gain_and_skip_beside_numbers_that_are_not_finite(bad, which):
    g = torch.Generator().manual_seed(4)
    H, G, dk, dv, T = 2, 1, 100, 40, 110
    qlocs = torch.tensor([0, 70, 110], dtype=torch.int32)
    total = torch.tensor([74, 40], dtype=torch.int32)
    slots = torch.tensor([1, 0], dtype=torch.int32)
    q, k = (torch.randn(T, G, dk, generator=g) for _ in "qk")
    x = {"v": torch.randn(T, H, dv, generator=g),
         "decay": torch.rand(T, H, generator=g) * 0.5 + 0.5,
         "gain": torch.rand(T, H, generator=g), "skip": torch.randn(H, generator=g)}
    x[which][{"v": (41, 1, 9), "skip": (1,)}.get(which, (41, 1))] = bad
    state = torch.randn(2, H, dk, dv, generator=g)
    want_s = state.clone()
    want = ref.decay_scan(q, k, *x.values(), want_s, slots, qlocs, total)
    st = state.to(DEV)
    got = hops.decay_scan(*(y.to(DEV) for y in (q, k, *x.values())), st,
                          slots.to(DEV), qlocs.to(DEV), total.to(DEV)).cpu()
    for y, z in ((got, want), (st.cpu(), want_s)):
        fine = torch.isfinite(z)
        assert torch.equal(torch.isfinite(y), fine)
        torch.testing.assert_close(y[fine], z[fine], rtol=2e-4, atol=2e-4)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("which", ["q", "k", "v", "memory", "ones"])
def test_mlstm_numbers_that_are_not_finite(bad, which):
    g = torch.Generator().manual_seed(6)
    H, dk, dv, T = 2, 64, 48, 110
    qlocs = torch.tensor([0, 70, 110], dtype=torch.int32)
    total = torch.tensor([74, 40], dtype=torch.int32)
    slots = torch.tensor([1, 0], dtype=torch.int32)
    cols = 2 * H * dk + H * dv
    offs = (0, H * dk, 2 * H * dk, cols, cols + H)
    proj = torch.randn(T, cols + 2 * H, generator=g)
    mem = torch.randn(2, H, dk, dv + 1, generator=g)
    if which in "qkv":
        i = "qkv".index(which)
        proj[41, offs[i] + (dv if which == "v" else dk) + 9] = bad     # of head 1
    else:                                # a column of the memory, or its normaliser
        mem[1, 0, 5, 7 if which == "memory" else dv] = bad
    proj = proj.bfloat16()
    ib, fb = torch.randn(H, generator=g), torch.randn(H, generator=g) + 2
    m0 = torch.randn(2, H, generator=g)
    want_m, want_ms = mem.clone(), m0.clone()
    want, em = ref.mlstm_scan(proj, *offs, H, dk, dv, ib, fb, 5.0, want_m, want_ms,
                              slots, qlocs, total)
    md, ms = mem.to(DEV), m0.to(DEV)
    got, got_em = hops.mlstm_scan(proj.to(DEV), *offs, H, dk, dv, ib.to(DEV),
                                  fb.to(DEV), 5.0, md, ms, slots.to(DEV),
                                  qlocs.to(DEV), total.to(DEV))
    for y, z in ((got.cpu(), want), (md.cpu(), want_m), (got_em.cpu(), em)):
        fine = torch.isfinite(z)
        assert torch.equal(torch.isfinite(y), fine)
        torch.testing.assert_close(y[fine], z[fine], rtol=2e-4, atol=2e-4)


@pytest.mark.parametrize("front", [31, 100, 1000])
@pytest.mark.parametrize("delta", [False, True])
def test_tokens_in_front_of_the_first_sequence(front, delta):
    """Rows that no sequence has, before the first one: the same results to the bit as
    without them."""
    g = torch.Generator().manual_seed(front)
    H, dk, dv, T = 2, 64, 48, 170
    qlocs = torch.tensor([0, 90, 170], dtype=torch.int32)
    total = torch.tensor([94, 80], dtype=torch.int32).to(DEV)
    slots = torch.tensor([1, 0], dtype=torch.int32).to(DEV)
    n = front + T
    q, k = (torch.nn.functional.normalize(torch.randn(n, H, dk, generator=g), dim=-1)
            for _ in "qk")
    v = torch.randn(n, H, dv, generator=g)
    a = torch.rand(n, H, generator=g) * 0.5 + 0.5
    b = torch.rand(n, H, generator=g)
    state = torch.randn(2, H, dk, dv, generator=g)

    def run(lo, locs):
        x = [y[lo:].contiguous().to(DEV) for y in (q, k, v, a, b)]
        st = state.to(DEV)
        f = hops.delta_scan if delta else hops.decay_scan
        more = () if delta else (None,)
        return f(*x, *more, st, slots, locs.to(DEV), total), st

    got, st = run(0, qlocs + front)
    want, end = run(front, qlocs)
    assert torch.equal(got[front:], want)
    assert torch.equal(st, end)


@pytest.mark.parametrize("head", [False, True])
def test_delta_decays_that_stay_the_same(head):
    """The rounding of a product of decays is the same in every chunk then, and must not
    add up: 128 chunks whose products are off by a third of 2^-24 each, one way, are
    8e-6 off for keys that resemble each other and a small beta. Roundings both ways
    stay below TOL."""
    g = torch.Generator().manual_seed(8)
    H, dk, dv, T = 2, 64, 16, 4096
    unit = torch.nn.functional.normalize
    q = unit(torch.randn(T, H, dk, generator=g), dim=-1) * dk ** -0.5
    k = unit(torch.randn(1, H, dk, generator=g)
             + 0.3 * torch.randn(T, H, dk, generator=g), dim=-1)
    v = torch.randn(T, H, dv, generator=g)
    d = torch.full((T, H) if head else (T, H, dk), 0.9987654)
    beta = torch.full((T, H), 0.02)
    state = torch.randn(1, H, dk, dv, generator=g)
    qlocs = torch.tensor([0, T], dtype=torch.int32)
    total, slots = torch.tensor([T + 1]).int(), torch.tensor([0]).int()
    want, end = _delta(q, k, v, d[..., None].expand(T, H, dk) if head else d, beta,
                       state, qlocs, total, slots)
    st = state.to(DEV)
    o = hops.delta_scan(*(x.to(DEV) for x in (q, k, v, d, beta)), st, slots.to(DEV),
                        qlocs.to(DEV), total.to(DEV))
    assert _off(o, want) < TOL
    assert _off(st, end) < TOL


@pytest.mark.parametrize("decay", [0.9987654, 0.99987])
def test_decays_that_stay_the_same(decay):
    g = torch.Generator().manual_seed(9)
    H, dk, dv, T = 2, 64, 16, 8192
    q, k = (torch.randn(T, H, dk, generator=g) * dk ** -0.5 for _ in "qk")
    v = torch.randn(T, H, dv, generator=g)
    a = torch.full((H,), decay)
    state = torch.randn(1, H, dk, dv, generator=g)
    qlocs = torch.tensor([0, T], dtype=torch.int32)
    total, slots = torch.tensor([T + 1]).int(), torch.tensor([0]).int()
    want, end = _recur(q, k, v, a.expand(T, H), torch.ones(T, H), torch.zeros(H), state,
                       qlocs, total, slots)
    st = state.to(DEV)
    o = hops.decay_scan(q.to(DEV), k.to(DEV), v.to(DEV), a.to(DEV), None, None, st,
                        slots.to(DEV), qlocs.to(DEV), total.to(DEV))
    assert _off(o, want) < TOL
    assert _off(st, end) < TOL


@pytest.mark.parametrize("front", [0, 75])
@pytest.mark.parametrize("kind", ["decay", "delta", "deltah", "mlstm"])
def test_long_sequences_among_many(kind, front):
    """150 sequences, a few of them long: the chunks find those by their rank, 64
    sequences at a time, whatever lies between them (none, one token, pieces)."""
    g = torch.Generator().manual_seed(front + 1)
    H, dk, dv = 2, 64, 48
    lens = [(0, 1, 1, 3, 1)[i % 5] for i in range(150)]
    for i, n in {0: 70, 62: 97, 63: 64, 64: 131, 65: 65, 127: 66, 128: 96, 149: 100}.items():
        lens[i] = n
    qlocs = torch.tensor([0] + lens).cumsum(0).int() + front
    T = int(qlocs[-1])
    total = torch.tensor([n + i % 2 for i, n in enumerate(lens)], dtype=torch.int32)
    slots = torch.randperm(151, generator=g)[:150].int()
    meta = (slots.to(DEV), qlocs.to(DEV), total.to(DEV))
    if kind == "mlstm":
        cols = 2 * H * dk + H * dv
        offs = (0, H * dk, 2 * H * dk, cols, cols + H)
        proj = torch.randn(T, cols + 2 * H, generator=g).bfloat16()
        ib, fb = torch.randn(H, generator=g), torch.randn(H, generator=g) + 2
        state, m0 = torch.randn(151, H, dk, dv + 1, generator=g), torch.randn(151, H, generator=g)
        end, want_m = state.clone(), m0.clone()
        want, _ = ref.mlstm_scan(proj, *offs, H, dk, dv, ib, fb, 5.0, end, want_m, slots,
                                 qlocs, total)
        st = state.to(DEV)
        o, _ = hops.mlstm_scan(proj.to(DEV), *offs, H, dk, dv, ib.to(DEV), fb.to(DEV),
                               5.0, st, m0.to(DEV), *meta)
        tol = 4 * TOL                   # the reference is fp32 as well
    else:
        unit = torch.nn.functional.normalize
        q, k = (unit(torch.randn(T, H, dk, generator=g), dim=-1) for _ in "qk")
        v = torch.randn(T, H, dv, generator=g)
        a, b = torch.rand(T, H, generator=g), torch.rand(T, H, generator=g)
        state = torch.randn(151, H, dk, dv, generator=g)
        st = state.to(DEV)
        if kind == "decay":
            want, end = _recur(q, k, v, a, b, torch.zeros(H), state, qlocs, total, slots)
            o = hops.decay_scan(*(x.to(DEV) for x in (q, k, v, a, b)), None, st, *meta)
        else:
            d = a if kind == "deltah" else torch.rand(T, H, dk, generator=g)
            want, end = _delta(q, k, v, d[..., None].expand(T, H, dk)
                               if kind == "deltah" else d, b, state, qlocs, total, slots)
            o = hops.delta_scan(*(x.to(DEV) for x in (q, k, v, d, b)), st, *meta)
        tol = TOL
    assert _off(o[front:], want[front:].double()) < tol
    assert _off(st, end.double()) < tol
    # the longest of them makes no difference but to the kernels that are taken
    for longest in (131, 1):
        again = state.to(DEV)
        if kind == "mlstm":
            o, _ = hops.mlstm_scan(proj.to(DEV), *offs, H, dk, dv, ib.to(DEV), fb.to(DEV),
                                   5.0, again, m0.to(DEV), *meta, longest)
        elif kind == "decay":
            o = hops.decay_scan(*(x.to(DEV) for x in (q, k, v, a, b)), None, again, *meta,
                                longest)
        else:
            o = hops.delta_scan(*(x.to(DEV) for x in (q, k, v, d, b)), again, *meta, longest)
        assert _off(o[front:], want[front:].double()) < tol
        assert _off(again, end.double()) < tol
    for s, n in zip(slots.tolist(), lens):
        if not n:
            assert torch.equal(st[s].cpu(), state[s])


@pytest.mark.parametrize("dk,dv,H,S,n", [
    (128, 32, 16, 40, 70), (128, 32, 16, 4, 200), (16, 64, 16, 80, 40), (16, 16, 4, 3, 40),
    (64, 64, 16, 33, 50), (64, 128, 16, 33, 26), (128, 128, 16, 17, 66), (96, 96, 16, 40, 97)])
def test_both_sides_of_the_rule(dk, dv, H, S, n):
    """A round of workgroups and more of them: sequences of n tokens on either side, and
    one that is longer than all others can be."""
    g = torch.Generator().manual_seed(n)
    lens = [n] * (S - 1) + [n * 3]
    qlocs = torch.tensor([0] + lens).cumsum(0).int()
    T = int(qlocs[-1])
    total, slots = torch.tensor(lens).int() + 1, torch.arange(S).int()
    unit = torch.nn.functional.normalize
    q, k = (unit(torch.randn(T, H, dk, generator=g), dim=-1) for _ in "qk")
    v = torch.randn(T, H, dv, generator=g)
    a, b = torch.rand(T, H, generator=g), torch.rand(T, H, generator=g)
    state = torch.randn(S, H, dk, dv, generator=g)
    meta = [x.to(DEV) for x in (slots, qlocs, total)]
    x = [y.to(DEV) for y in (q, k, v, a, b)]
    for delta in (False, True):
        st = state.to(DEV)
        want = torch.zeros(T, H, dv, dtype=torch.float64, device=DEV)
        end = state.to(DEV).double()
        for t in range(3 * n):          # all sequences side by side, on the GPU
            live = [s for s in range(S) if t < lens[s]]
            at = (qlocs[:-1][live].long() + t).to(DEV)
            live = torch.tensor(live, device=DEV)
            P = end[live] * a.to(DEV).double()[at][:, :, None, None]
            kk, vv, bb = (y.double()[at] for y in (x[1], x[2], x[4]))
            u = vv - (P * kk[..., None]).sum(2) if delta else vv
            P = P + kk[..., None] * (bb[..., None] * u)[:, :, None, :]
            want[at] = (P * x[0].double()[at][..., None]).sum(2)
            end[live] = P
        f = hops.delta_scan if delta else hops.decay_scan
        o = f(*x, *(() if delta else (None,)), st, *meta)
        assert float((o.double() - want).norm() / want.norm()) < TOL
        assert float((st.double() - end).norm() / end.norm()) < TOL
