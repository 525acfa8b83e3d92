"""Keys and values that a query must not see (what an earlier request left
behind the context, keys before a window or between the kept first keys and the
window, later tokens of the same prompt) may be infinite or NaN: results are
the same to the bit as with zeros in their place."""

import math

import pytest
import torch

from sutro_amd import ops
from sutro_amd.ops import hybrid as hops

pytestmark = pytest.mark.gpu
DEV = "cuda"
INF, NAN = float("inf"), float("nan")


class Pages:
    """Random pages for sequences of `lens` keys; every sequence's table has a
    page more than it needs."""

    def __init__(self, lens, Hk, D, fp8=False, seed=0):
        g = torch.Generator().manual_seed(seed)
        need = [n // 32 + 2 for n in lens]
        perm = torch.randperm(sum(need), generator=g).int()
        self.bt = torch.zeros(len(lens), max(need), dtype=torch.int32)
        at = 0
        for s, n in enumerate(need):
            self.bt[s, :n] = perm[at:at + n]
            at += n
        shape = (sum(need), Hk, 32, D)
        self.k, self.v = (torch.randn(shape, generator=g) for _ in range(2))
        self.fp8 = fp8
        self.g = g

    def with_unseen(self, unseen, value):
        """(keys, values) with `value` in the rows of the (sequence, position)
        pairs."""
        k, v = self.k.clone(), self.v.clone()
        for s, p in unseen:
            page = int(self.bt[s, p // 32])
            k[page, :, p % 32] = value
            v[page, :, p % 32] = value
        kind = torch.float8_e4m3fn if self.fp8 else torch.bfloat16
        return k.to(kind).to(DEV), v.to(kind).to(DEV)


def _same(run, pages, unseen):
    want = run(*pages.with_unseen(unseen, 0.0))
    assert torch.isfinite(want.float()).all()
    for value in ((NAN,) if pages.fp8 else (INF, -INF, NAN)):
        got = run(*pages.with_unseen(unseen, value))
        assert torch.equal(got, want), value


def _behind(lens):
    return [(s, p) for s, n in enumerate(lens)
            for p in range(n, (n // 32 + 2) * 32)]


@pytest.mark.parametrize("Hq,Hk,D,fp8", [(8, 2, 128, False), (5, 1, 64, False),
                                         (8, 4, 128, True), (4, 2, 64, True)])
def test_behind_the_context(Hq, Hk, D, fp8):
    lens = [1, 31, 32, 33, 700, 63, 95, 97, 130]
    new = [1, 1, 1, 1, 1, 63, 40, 97, 2]
    order = [5, 6, 7, 8, 0, 1, 2, 3, 4]                # prompts, then tokens
    lens, new = [lens[i] for i in order], [new[i] for i in order]
    pg = Pages(lens, Hk, D, fp8, seed=Hq)
    q = torch.randn(sum(new), Hq, D, generator=pg.g).bfloat16().to(DEV)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    ql = torch.tensor([0] + new).cumsum(0).int().to(DEV)
    bt = pg.bt.to(DEV)
    ts = [s for s in range(4) for _ in range(0, new[s], 32)]
    tq = [j for s in range(4) for j in range(0, new[s], 32)]
    ts, tq = (torch.tensor(x, dtype=torch.int32, device=DEV) for x in (ts, tq))

    def run(k, v):
        return ops.paged_attention(
            q, k, v, bt, sl, ql, 1.0 / math.sqrt(D), num_decodes_tail=5,
            tile_seq=ts, tile_q0=tq, prefill_token_count=sum(new[:4]))

    _same(run, pg, _behind(lens))


@pytest.mark.parametrize("Hq,Hk", [(8, 2), (2, 1), (3, 3)])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("start", [0, 7, 45])
def test_later_tokens_of_a_prompt(Hq, Hk, D, start):
    """Rows of a 32-row block never read what lies 16 or more keys behind its
    last one."""
    n = 200
    pg = Pages([start + n], Hk, D, seed=3)
    q = torch.randn(n, Hq, D, generator=pg.g).bfloat16().to(DEV)
    sl = torch.tensor([start + n], dtype=torch.int32, device=DEV)
    ql = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    ts = torch.zeros(7, dtype=torch.int32, device=DEV)
    tq = torch.arange(0, n, 32, dtype=torch.int32, device=DEV)
    bt = pg.bt.to(DEV)
    for blocks in (1, 2, 3, 5):
        rows = blocks * 32

        def run(k, v):
            out = ops.paged_attention(
                q, k, v, bt, sl, ql, D ** -0.5, num_decodes_tail=0,
                tile_seq=ts, tile_q0=tq, prefill_token_count=n)
            return out[:rows]

        _same(run, pg, [(0, p) for p in range((start + rows + 15) // 16 * 16,
                                              start + n)])


@pytest.mark.parametrize("Hq,Hk,D", [(8, 2, 128), (4, 4, 64), (6, 2, 64)])
@pytest.mark.parametrize("chunk,window,keep", [
    (0, 0, 0), (100, 0, 0), (0, 45, 0), (0, 300, 70), (0, 33, 5)])
@pytest.mark.parametrize("prompt", [False, True])
def test_layer_list_attention(Hq, Hk, D, chunk, window, keep, prompt):
    lens = [1, 40, 333, 900, 96]
    new = [1, 25, 140, 64, 33] if prompt else [1] * 5
    pg = Pages(lens, Hk, D, seed=window + D)
    T = sum(new)
    q = torch.randn(T, Hq, D, generator=pg.g).bfloat16().to(DEV)
    proj = torch.randn(T, 16, generator=pg.g).bfloat16().to(DEV)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    ql = torch.tensor([0] + new).cumsum(0).int().to(DEV)
    bt = pg.bt.to(DEV)
    seq = torch.repeat_interleave(torch.arange(5), torch.tensor(new)).int().to(DEV)
    kw = {}
    if prompt:
        kw = dict(
            tile_seq=torch.tensor([s for s in range(5)
                                   for _ in range(0, new[s], 32)],
                                  dtype=torch.int32, device=DEV),
            tile_q0=torch.tensor([j for c in new for j in range(0, c, 32)],
                                 dtype=torch.int32, device=DEV),
            prefill_rows=T)
    unseen = []
    for s, n in enumerate(lens):
        seen = torch.zeros((n // 32 + 2) * 32, dtype=torch.bool)
        for p in range(n - new[s], n):
            lo = p // chunk * chunk if chunk else 0
            kept = lo
            if window:
                lo = max(lo, p - window + 1)
            seen[lo:p + 1] = True
            seen[kept:max(kept, min(keep, p + 1))] = True
        unseen += [(s, p) for p in range(seen.numel()) if not seen[p]]

    def run(k, v):
        out = torch.zeros(T, Hq * D, dtype=torch.bfloat16, device=DEV)
        hops.local_attention(q, k, v, bt, sl, ql, D ** -0.5, chunk, window,
                             proj, -1, out, 0, 1.0, token_seq=seq,
                             keep_first=keep, **kw)
        return out

    _same(run, pg, unseen)


@pytest.mark.parametrize("Hq,Hk,chunk,window,keep", [
    (8, 8, 32, 0, 0), (8, 8, 0, 40, 9), (6, 2, 64, 0, 0), (4, 1, 32, 0, 0)])
def test_many_narrow_prompts(Hq, Hk, chunk, window, keep):
    """Enough prompts with heads of 64 and a narrow chunk or window to leave the
    kernel of 128 rows a workgroup: against the reference, and with what no
    32-row block sees poisoned."""
    from sutro_amd.ops import torch_ref as R

    D, S = 64, 140
    g = torch.Generator().manual_seed(Hq)
    new = torch.randint(33, 97, (S,), generator=g).tolist()
    lens = [n + int(c) for n, c in
            zip(new, torch.randint(0, 40, (S,), generator=g))]
    if keep:
        lens[3] = new[3] + 200
    pg = Pages(lens, Hk, D, seed=1)
    T = sum(new)
    q = torch.randn(T, Hq, D, generator=g).bfloat16()
    proj = torch.randn(T, 16, generator=g).bfloat16()
    sl = torch.tensor(lens, dtype=torch.int32)
    ql = torch.tensor([0] + new).cumsum(0).int()
    ts = torch.tensor([s for s in range(S) for _ in range(0, new[s], 32)]).int()
    tq = torch.tensor([j for c in new for j in range(0, c, 32)]).int()
    seq = torch.repeat_interleave(torch.arange(S), torch.tensor(new)).int()
    hpb = 4 if Hq // Hk % 4 == 0 else (2 if Hq // Hk % 2 == 0 else 1)
    assert ts.numel() * Hq // hpb >= (2048 if window else 1024) or Hq // Hk == 4
    unseen = []
    for s, n in enumerate(lens):
        seen = torch.zeros((n // 32 + 2) * 32, dtype=torch.bool)
        for p in range(n - new[s], n):
            lo = p // chunk * chunk if chunk else 0
            kept = lo
            if window:
                lo = max(lo, p - window + 1)
            seen[lo:p + 1] = True
            seen[kept:max(kept, min(keep, p + 1))] = True
        unseen += [(s, p) for p in range(seen.numel()) if not seen[p]]
    d = [x.to(DEV) for x in (q, pg.bt, sl, ql, proj, seq, ts, tq)]

    def run(k, v):
        out = torch.zeros(T, Hq * D, dtype=torch.bfloat16, device=DEV)
        hops.local_attention(d[0], k, v, d[1], d[2], d[3], D ** -0.5, chunk,
                             window, d[4], -1, out, 0, 1.0, token_seq=d[5],
                             tile_seq=d[6], tile_q0=d[7], prefill_rows=T,
                             keep_first=keep)
        return out

    _same(run, pg, unseen)
    k, v = (x.cpu().float() for x in pg.with_unseen([], 0.0))
    want = torch.zeros(T, Hq * D)
    R.local_attention(q.float(), k, v, pg.bt, sl, ql, D ** -0.5, chunk, window,
                      proj, -1, want, 0, 1.0, keep_first=keep)
    got = run(*pg.with_unseen([], 0.0)).float().cpu()
    # weights and results are rounded to bf16 once each
    bound = 2.0 ** -8 * v.abs().max().item() + 1e-3
    assert (got - want).abs().max().item() < bound
