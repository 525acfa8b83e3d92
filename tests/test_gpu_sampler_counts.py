"""The sampler's counting kernel (bf16 rows) at the rows where its bookkeeping
can go wrong, against the same arithmetic in whole numbers: q = floor(p 2**32)
of float32 exponentials, whose sums are exact. The kernel's exponential takes
exp2 of a rounded product, so p is off by up to (1 + |s|) 2**-24 of itself;
weighted with p that is below 2**-22 of a sum, of the sum up to a token and of
the whole: a token must hold u within 2**-21. Logprobs: 1e-5, which is 40 ulp
of a sum of float32 exponentials in another order."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from sutro_amd import ops

DEV = "cuda"


def pack(keep):
    n, v = keep.shape
    words = (v + 31) // 32
    bits = torch.zeros(n, words * 32, dtype=torch.int64)
    bits[:, :v] = keep.long().cpu()
    w = (bits.view(n, words, 32) << torch.arange(32)).sum(-1)
    return torch.where(w >= 2**31, w - 2**32, w).to(torch.int32).to(DEV)


def check(logits, vl, temp, top_p, top_k, u, keep=None):
    n = logits.shape[0]
    temps = torch.full((n,), temp, device=DEV)
    top_ps = torch.full((n,), top_p, device=DEV)
    top_ks = torch.full((n,), top_k or vl, dtype=torch.int32, device=DEV)
    us = torch.full((n,), u, device=DEV)
    tok = torch.empty(n, dtype=torch.int32, device=DEV)
    lp = torch.empty(n, device=DEV)
    ops.sampler_fused(logits, temps, top_ps, top_ks, us,
                      pack(keep) if keep is not None else None, vl, tok, lp)
    tok, lp = tok.long().cpu(), lp.cpu()
    for r in range(n):
        v = logits[r, :vl].cpu().float()
        alive = torch.ones(vl, dtype=torch.bool) if keep is None \
            else keep[r, :vl].cpu()
        m = v[(alive & (v == v[alive].max())).nonzero()[0, 0]]   # its sign too
        t = int(tok[r])
        s = (v - m) * (1.0 if temp == 0 else 1.0 / torch.tensor(temp))
        p = torch.where(alive, s.exp(), 0.0)
        want = s[t] - p.double().sum().log()
        assert abs(float(lp[r]) - float(want)) < 1e-5, (r, temp)
        if temp == 0:
            assert t == int(torch.where(alive & (v == m))[0][0])
            continue
        q = (p.double() * 2**32).floor().long()
        s = torch.where(alive, s, -torch.inf)
        # scaled logits rank by their bits: -0.0 below 0.0
        s = torch.where((s == 0) & s.signbit(), -1e-45, s)
        order = s.argsort(descending=True, stable=True)
        ss, above = s[order], q[order].cumsum(0) - q[order]
        first = torch.searchsorted(-ss, -ss)        # of the values that tie
        ok = (first < (top_k or vl)) & \
            (above[first].double() < max(1.0, top_p * float(q.sum())))
        kept = torch.zeros(vl, dtype=torch.bool)
        kept[order] = ok
        kept &= alive
        c = torch.where(kept, q, 0).cumsum(0).double() / \
            float(q[kept].sum())
        eps = 2.0**-21
        assert kept[t], (r, temp, top_p, top_k)
        assert u < c[t] + eps and u >= (c[t - 1] if t else 0.0) - eps, \
            (r, temp, top_p, top_k, t)
    return tok, lp


# one chunk, tails of a chunk, a full tile (19 chunks of 8192) and more
@pytest.mark.parametrize("row,vl", [(2048, 2048), (8192, 8191), (8200, 8193),
                                    (16384, 9001), (155648, 155648),
                                    (155656, 155649), (200000, 199999)])
@pytest.mark.parametrize("masked", [False, True])
def test_sizes(row, vl, masked):
    g = torch.Generator().manual_seed(row + masked)
    n = 3
    # nine values, spread so that every boundary is far from any u here
    lg = (torch.randint(-4, 5, (n, row), generator=g) * 0.75)
    lg = lg.to(torch.bfloat16).to(DEV)
    keep = torch.rand(n, row, generator=g) < 0.4 if masked else None
    for temp, top_p, top_k, u in ((0.7, 0.83, 0, 0.313), (1.3, 1.0, 0, 0.777),
                                  (1.0, 1.0, 40, 0.5), (0.0, 1.0, 0, 0.5),
                                  (1.0, 1e-9, 0, 0.9)):
        check(lg, vl, temp, top_p, top_k, u, keep)
    # the last token alone alive
    if masked:
        keep = torch.zeros(n, row, dtype=torch.bool)
        keep[:, vl - 1] = True
        tok, lp = check(lg, vl, 0.9, 0.9, 3, 0.99, keep)
        assert (tok == vl - 1).all() and lp.abs().max() == 0


def test_values_that_repeat_beyond_a_counter():
    """65,535 to 131,072 tokens of one value: the 16-bit counters overflow and
    the rows are sampled all the same."""
    v = 140000
    for value in (0.0, -2.5, 3.0):
        for reps in (65535, 65536, 65537, 131072):
            lg = torch.full((1, v), value - 1.0)
            lg[0, 500:500 + reps] = value
            lg[0, 500 + reps:] = float("-inf")
            lg = lg.to(torch.bfloat16).to(DEV)
            for temp, top_k, u in ((1.0, 0, 0.37), (0.8, 7, 0.99), (0.0, 0, 0.)):
                check(lg, v, temp, 1.0, top_k, u)


def test_extreme_rows():
    v = 4096
    ninf = float("-inf")
    base = torch.full((8, v), ninf)
    base[1, 77] = 1.0                                  # one finite logit
    base[2, :] = torch.linspace(-1.5e38, 1.5e38, v)    # the whole range
    base[3, 10], base[3, 20] = -0.0, 0.0               # zeros, -0 first
    base[4, 10], base[4, 20] = 0.0, -0.0               # zeros, +0 first
    base[5, :] = torch.arange(v) * 1e-20               # keys that coincide:
    base[5, 7] = 9.0                                   # all but one at -9
    base[6, 100:200] = -torch.logspace(-38, 1, 100)    # subnormal steps
    base[7, :] = -1.0
    lg = base.to(torch.bfloat16).to(DEV)
    for temp, top_p, top_k, u in ((1.0, 1.0, 0, 0.4), (0.5, 0.9, 2, 0.9),
                                  (0.0, 1.0, 0, 0.0), (2.0, 1.0, 1, 0.6)):
        check(lg[1:], v, temp, top_p, top_k, u)
    # nothing alive, by the logits or by the mask: token 0, logprob -inf
    one = torch.ones(1, device=DEV)
    for row, mask in ((0, None), (1, torch.zeros(1, v, dtype=torch.bool))):
        tok = torch.full((1,), 9, dtype=torch.int32, device=DEV)
        lp = torch.zeros(1, device=DEV)
        ops.sampler_fused(lg[row:row + 1], one, one, (one * v).int(), one * 0.5,
                          None if mask is None else pack(mask), v, tok, lp)
        assert tok.item() == 0 and lp.item() == ninf


def same_as_general(logits, temp, top_p, top_k, us, keep=None):
    """bf16 rows against the same values in float32, which the kernel without
    counters samples: the tokens are equal, as both sum whole numbers."""
    v = logits.shape[1]
    mask = None if keep is None else pack(keep)
    for u in us:
        res = []
        for lg in (logits, logits.float()):
            n = lg.shape[0]
            tok = torch.full((n,), -7, dtype=torch.int32, device=DEV)
            lp = torch.zeros(n, device=DEV)
            ops.sampler_fused(
                lg, torch.full((n,), temp, device=DEV),
                torch.full((n,), top_p, device=DEV),
                torch.full((n,), top_k or v, dtype=torch.int32, device=DEV),
                torch.full((n,), u, device=DEV), mask, v, tok, lp)
            res.append((tok.cpu(), lp.cpu()))
        assert torch.equal(res[0][0], res[1][0]), (temp, top_p, top_k, u)
        torch.testing.assert_close(res[0][1], res[1][1], rtol=0, atol=1e-5,
                                   equal_nan=True)


@pytest.mark.parametrize("temp,top_p,top_k", [
    (0.0, 1.0, 0), (1.0, 1.0, 1), (0.7, 1.0, 2), (1.0, 1e-9, 0), (3.0, 0.9, 0)])
def test_values_that_round_to_the_maximum(temp, top_p, top_k):
    """Values whose exponential is 1 although they are not the largest: only
    those that are kept have a mass."""
    v = 4096
    rows = torch.full((6, v), -1.0)
    rows[0, 10], rows[0, 20] = -1e-9, 0.0
    rows[1, 5:205] = -torch.logspace(-6, -30, 200)       # rising towards zero
    rows[2, 5:205] = torch.logspace(-30, -9, 200)        # rising from zero
    rows[3, 700:900] = torch.logspace(-30, -9, 200)
    rows[3, 3000:3200] = -torch.logspace(-9, -30, 200)
    rows[4, :] = torch.linspace(1e-12, 1e-9, v)
    rows[5, 600], rows[5, 601], rows[5, 4000] = 1e-9, 2e-9, 3e-9
    same_as_general(rows.to(torch.bfloat16).to(DEV), temp, top_p, top_k,
                    (0.0, 0.3, 0.999))


@pytest.mark.parametrize("temp,top_p,top_k", [
    (0.0, 1.0, 0), (1.0, 1.0, 0), (0.7, 0.9, 0), (1.0, 1.0, 3)])
def test_infinities_and_nans(temp, top_p, top_k):
    v = 4096
    inf, nan = float("inf"), float("nan")
    rows = torch.randn(8, v, generator=torch.Generator().manual_seed(5))
    rows[0, 70], rows[0, 3000] = inf, inf         # greedy: the first of them
    rows[1, 9] = inf
    rows[2, 70:90] = -inf
    rows[3, 5], rows[3, 4000] = nan, nan
    rows[4, 5], rows[4, 4000], rows[4, 6] = nan, inf, -inf
    rows[5, :] = inf
    rows[6, :] = nan
    rows[7, 1:] = nan
    same_as_general(rows.to(torch.bfloat16).to(DEV), temp, top_p, top_k,
                    (0.0, 0.4, 0.999))
    bits = rows.to(torch.bfloat16).view(torch.int16)
    bits[3, 5], bits[3, 4000] = -1, -1            # the NaN of all bits
    same_as_general(bits.view(torch.bfloat16).to(DEV), temp, top_p, top_k,
                    (0.0, 0.4, 0.999))


@pytest.mark.parametrize("temp,top_p,top_k", [
    (0.8, 0.95, 0), (1.0, 1.0, 5), (2.0, 0.5, 0), (3.0, 1.0, 0), (30.0, 0.9, 0)])
def test_ends_of_the_short_range(temp, top_p, top_k):
    """Rows at the edges of what is counted by magnitudes from 2^-24 to 255, among
    more rows than there are workgroups, and greedy rows between them."""
    v = 4096
    rows = torch.randn(600, v, generator=torch.Generator().manual_seed(7)) * 3
    rows[0] = rows[0].clamp(max=1.5)              # below 2
    rows[1] = rows[1].clamp(max=2.0)
    rows[2, 9], rows[3, 9], rows[4, 9], rows[5, 9] = 254., 255., 256., 1e30
    rows[6, ::3], rows[7, ::3], rows[8, ::3] = -255., -256., -1e30
    rows[9, ::2], rows[10, ::2] = -float("inf"), 0.
    tiny = 2.0 ** -torch.arange(20, 30).repeat_interleave(2)
    tiny[::2] *= -1
    rows[11, :20], rows[12, :20], rows[12, 20:] = tiny, tiny, 3.
    rows[13, :], rows[13, :20] = -5., tiny
    rows[14, :] = 2.5
    rows[15, :], rows[15, 4000] = -300., 100.
    lg = rows.to(torch.bfloat16).to(DEV)
    same_as_general(lg, temp, top_p, top_k, (0.0, 0.3, 0.999))
    # the last of several pieces of 512 is not full, and not all of a wave's have one
    wide = torch.randn(3, 70008, generator=torch.Generator().manual_seed(8)) * 2.5
    same_as_general(wide.to(torch.bfloat16).to(DEV), temp, top_p, top_k,
                    (0.0, 0.5, 0.999))


@pytest.mark.parametrize("temp,top_p,top_k", [
    (0.8, 0.95, 0), (1.0, 1.0, 5), (3.0, 1.0, 0), (30.0, 0.9, 0), (1e9, 1.0, 0)])
def test_rows_that_are_small_or_negative(temp, top_p, top_k):
    """Flat rows and log-probabilities: a largest logit of 2 and less, with and
    without others of 2^-24 and less, zeros and negative zeros, and all of them negative."""
    v = 4096
    rows = torch.randn(28, v, generator=torch.Generator().manual_seed(9)) * 0.2
    tiny = 2.0 ** -torch.arange(20, 30).repeat_interleave(2)
    tiny[::2] *= -1
    rows[1, 50], rows[2, 50], rows[3, 50] = 0.0, -0.0, 1e-9
    rows[4:8] -= torch.tensor([0.5, 2.0, 20.0, 253.0])[:, None]
    rows[8] = rows[8].clamp(max=0.0)
    rows[9], rows[10] = -rows[9].abs() - 2.0 ** -24, -rows[10].abs() - 2.0 ** -23
    rows[11] = torch.log_softmax(rows[11] * 10, -1)
    rows[12] = torch.log_softmax(rows[12] * 100, -1)
    rows[13], rows[13, 7] = -30.0, 0.0
    rows[14], rows[14, 7] = -30.0, -1e-3
    rows[15, :20], rows[15, 20:] = tiny, -3.0
    rows[16, :20], rows[16, 20:] = -tiny.abs(), -3.0
    rows[17, :20], rows[17, 20] = tiny, 1.9921875
    rows[24:, :20] = tiny
    rows[24:, 20] = torch.tensor([1.0078125, 1.0, 0.99609375, 2.0])
    rows[18], rows[18, ::3], rows[18, 5] = -200.0, -255.0, -254.0
    rows[19], rows[19, ::3], rows[19, 5] = -254.0, -256.0, -255.0
    rows[20], rows[21] = -255.0, -300.0
    rows[22, ::2] = -float("inf")
    rows[23], rows[23, ::2] = -float("inf"), -2.0
    same_as_general(rows.to(torch.bfloat16).to(DEV), temp, top_p, top_k,
                    (0.0, 0.3, 0.999))


@pytest.mark.parametrize("temp,top_p,top_k", [
    (0.8, 0.95, 0), (1.0, 1.0, 5), (6.0, 1.0, 0), (6.5, 1.0, 0), (9.0, 0.9, 3000),
    (30.0, 0.9, 0)])
def test_masked_ends_of_the_short_range(temp, top_p, top_k):
    """Under a mask what lies at -255 and below is not counted, and rows are left
    where (255 + the largest) / temperature is 40 or less: from a temperature of 6.4 on
    at a largest of 1.5, of 8.9 at 100. What is masked is no number, infinite, or larger."""
    v = 4096
    g = torch.Generator().manual_seed(11)
    rows = torch.randn(300, v, generator=g) * 3
    keep = torch.rand(300, v, generator=g) < 0.5
    rows[0] = rows[0].clamp(max=1.5)
    rows[1, 9], rows[2, 9], rows[3, 9] = 100.0, 254.0, 255.0
    for r, low in ((4, -254.0), (5, -255.0), (6, -256.0), (7, -1e30),
                   (8, -float("inf"))):
        rows[r, ::3] = low
        rows[r + 5, ::3] = low
        rows[r + 5, 9] = 100.0
    rows[14] = rows[14] / 20 - 20.0
    rows[15] = torch.log_softmax(rows[15], -1)
    rows[16] /= 10
    rows[17, 5:], rows[17, 5] = -255.0, 1.5
    rows[18], rows[18, 5:8] = -300.0, 2.5
    rows[19] = -255.0
    for r in (1, 2, 3, *range(9, 14)):
        keep[r, 9] = True
    keep[17, :], keep[18, 5:8], keep[18, 100:] = True, True, True
    for i, odd in enumerate((float("nan"), float("inf"), 250.0, 300.0)):
        rows[20 + i] = torch.where(keep[20 + i], rows[20 + i], odd)
    keep[24, :] = False
    keep[24, 4000] = True
    same_as_general(rows.to(torch.bfloat16).to(DEV), temp, top_p, top_k,
                    (0.0, 0.3, 0.999), keep)


@pytest.mark.parametrize("row,vl", [(2048, 2048), (8200, 8193), (70008, 70005),
                                    (155648, 155648)])
@pytest.mark.parametrize("masked", [False, True])
def test_greedy_rows_among_others(row, vl, masked):
    """More rows than workgroups, every third of them greedy: to the bit what two calls
    make of them, ties, numbers that are none and rows without a live logit among them."""
    n = 300
    g = torch.Generator().manual_seed(vl)
    lg = (torch.randn(n, row, generator=g) * 3).to(torch.bfloat16)
    inf, nan = float("inf"), float("nan")
    lg[0, 40], lg[0, vl - 1] = 30.0, 30.0
    lg[3, vl - 1], lg[6, :], lg[9, 5], lg[12, 7] = 30.0, -inf, inf, nan
    lg[15, ::2], lg[18, 3] = nan, -inf
    lg[0:n:3, vl:] = 100.0
    bits = lg.view(torch.int16)
    bits[21, 5] = -1                              # the NaN of all bits
    keep = torch.rand(n, row, generator=g) < 0.3
    keep[[0, 3], vl - 1], keep[24, :], keep[27, :] = True, False, False
    keep[27, vl - 1] = True
    lg, mask = lg.to(DEV), pack(keep) if masked else None
    temps = torch.full((n,), 0.8, device=DEV)
    temps[::3] = 0.0
    rest = (torch.full((n,), 0.9, device=DEV),
            torch.full((n,), vl, dtype=torch.int32, device=DEV),
            torch.rand(n, generator=g).to(DEV))

    def sample(rows, **kw):
        k = len(range(n)[rows])
        tok, lp = torch.empty(k, dtype=torch.int32, device=DEV), torch.empty(k, device=DEV)
        ops.sampler_fused(lg[rows].contiguous(), temps[rows].contiguous(),
                          *(t[rows].contiguous() for t in rest),
                          None if mask is None else mask[rows].contiguous(), vl, tok, lp,
                          **kw)
        return tok, lp.view(torch.int32)

    tok, lp = sample(slice(None))
    for rows, kw in ((slice(0, n, 3), dict(greedy=True)), (slice(1, n, 3), {}),
                     (slice(2, n, 3), {})):
        one = sample(rows, **kw)
        assert torch.equal(tok[rows], one[0])
        assert torch.equal(lp[rows], one[1])
