"""The paged attention kernels at the sizes where their splits change: run
borders of the decode kernel, tile and workgroup borders of the prompt
kernel."""

import math

import pytest
import torch

from sutro_amd import ops
from sutro_amd.ops import torch_ref as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _paged(lens, new, Hq, Hk, D, fp8, spare=0, seed=0):
    """Random queries and shuffled pages; block tables `spare` columns wider
    than the longest sequence needs."""
    g = torch.Generator().manual_seed(seed)
    pages = [(n + 31) // 32 for n in lens]
    perm = torch.randperm(sum(pages) + 3, generator=g).tolist()
    bt = torch.zeros(len(lens), max(pages) + spare, dtype=torch.int32)
    at = 0
    for s, n in enumerate(pages):
        bt[s, :n] = torch.tensor(perm[at:at + n])
        at += n
    shape = (len(perm), Hk, 32, D)
    kc, vc = (torch.randn(shape, generator=g).bfloat16() for _ in range(2))
    if fp8:
        kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
    q = torch.randn(sum(new), Hq, D, generator=g).bfloat16()
    ql = torch.tensor([0] + new).cumsum(0).to(torch.int32)
    return q, kc, vc, bt, torch.tensor(lens, dtype=torch.int32), ql


def _check(args, got):
    """Weights p and results are rounded to bf16 once each, 2^-8 of sum(p |v|)
    at most, element by element; 2^-12 is for scores of up to 20 in 32 bits."""
    q, kc, vc, bt, sl, ql = args
    ref, size = (R.paged_attention(q.float(), kc.float(), v, bt, sl, ql,
                                   1.0 / math.sqrt(q.shape[2]))
                 for v in (vc.float(), vc.float().abs()))
    bound = (2.0 ** -7 + 2.0 ** -12) * size
    err = (got.float().cpu() - ref).abs()
    assert (err <= bound).all(), (err / bound).max().item()
    return ref, bound


RUN = 256    # keys of a run


def _plant(args):
    """A key of weight exp(14) in every run of every sequence (single tokens),
    for one head of each group that has another, so that no run can be left out
    or counted twice unseen."""
    q, kc, vc, bt, sl, ql = args
    Hk, D = kc.shape[1], kc.shape[3]
    G = q.shape[1] // Hk
    for s, n in enumerate(sl.tolist()):
        runs = (n + RUN - 1) // RUN
        for r in range(runs):
            p = min(r * RUN + 37 * r % RUN, n - 1)
            head = q[s].view(Hk, G, D)[:, r % max(min(G, runs // 2), 1)].float()
            key = head * (14 * math.sqrt(D) / head.square().sum(-1, keepdim=True))
            kc[int(bt[s, p // 32]), :, p % 32] = key.to(kc.dtype)


def _assert_runs_show(args, ref, bound):
    """Leaving out or doubling any run moves the reference past the bound."""
    q, kc, vc, bt, sl, ql = args
    Hk, D = kc.shape[1], kc.shape[3]
    G = q.shape[1] // Hk
    for s, n in enumerate(sl.tolist()):
        runs = (n + RUN - 1) // RUN
        if runs < 2:
            continue
        pages = bt[s, :(n + 31) // 32].long()
        k, v = (x[pages].float().transpose(0, 1).reshape(Hk, -1, D)[:, :n]
                for x in (kc, vc))
        z = q[s].float().view(Hk, G, D) @ k.transpose(1, 2) / math.sqrt(D)
        p = (z - z.amax(-1, keepdim=True)).exp()
        for r in range(runs):
            for times in (0.0, 2.0):
                w = p.clone()
                w[:, :, r * RUN:(r + 1) * RUN] *= times
                o = (w @ v / w.sum(-1, keepdim=True)).view(Hk * G, D)
                assert ((o - ref[s]).abs() > 2 * bound[s]).any(), (s, r, times)


@pytest.mark.parametrize("Hq,Hk,D,fp8", [
    (16, 4, 128, False), (5, 1, 128, False), (8, 1, 64, False),
    (8, 8, 128, True), (14, 2, 64, True)])
@pytest.mark.parametrize("lens,spare", [
    ([1, 32, 33], 0),              # one run each
    ([255, 256, 257, 3], 40),      # 8 pages = one run; wide tables
    ([2049, 40, 8191], 5),         # many runs beside a single one
])
@pytest.mark.parametrize("planted", [False, True])
def test_decode_runs(Hq, Hk, D, fp8, lens, spare, planted):
    args = _paged(lens, [1] * len(lens), Hq, Hk, D, fp8, spare, seed=D + Hq)
    if planted:
        _plant(args)
    q, kc, vc, bt, sl, ql = (x.to(DEV) for x in args)
    got = ops.paged_attention(q, kc, vc, bt, sl, ql, 1.0 / math.sqrt(D),
                              num_decodes_tail=len(lens))
    ref, bound = _check(args, got)
    if planted:
        _assert_runs_show(args, ref, bound)


def _tiles(new):
    return ([s for s, c in enumerate(new) for _ in range(0, c, 32)],
            [j for c in new for j in range(0, c, 32)])


def _prefill(args, D, tiles):
    q, kc, vc, bt, sl, ql = (x.to(DEV) for x in args)
    ts, tq = (torch.tensor(x, dtype=torch.int32, device=DEV) for x in tiles)
    return ops.paged_attention(q, kc, vc, bt, sl, ql, 1.0 / math.sqrt(D),
                               num_decodes_tail=0, tile_seq=ts, tile_q0=tq,
                               prefill_token_count=q.shape[0])


# every split of query heads and row blocks over the waves of a workgroup
@pytest.mark.parametrize("Hq,Hk", [(3, 3), (4, 2), (6, 2), (8, 2), (10, 2),
                                   (6, 1), (7, 1), (8, 1)])
@pytest.mark.parametrize("D,fp8", [(128, False), (64, True)])
def test_prompt_tiles(Hq, Hk, D, fp8):
    # whole prompts and continued ones around borders of pages, key steps
    # and row blocks
    new = [1, 31, 32, 33, 64, 65, 128, 129, 40, 96]
    ctx = [0, 0, 0, 0, 0, 0, 0, 0, 25, 352]
    lens = [a + b for a, b in zip(new, ctx)]
    args = _paged(lens, new, Hq, Hk, D, fp8, seed=Hq)
    _check(args, _prefill(args, D, _tiles(new)))


# enough prompts of one and of two blocks for workgroups of four and of two heads
# of any group
@pytest.mark.parametrize("Hq,Hk", [(3, 1), (14, 2), (5, 1), (6, 1)])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("longest", [32, 64])
def test_many_short_prompts(Hq, Hk, D, longest):
    n = 1600 // Hq
    g = torch.Generator().manual_seed(Hq)
    new = torch.randint(longest - 31, longest + 1, (n,), generator=g).tolist()
    ctx = torch.randint(0, 70, (n,), generator=g).tolist()
    args = _paged([a + b for a, b in zip(new, ctx)], new, Hq, Hk, D, False, seed=D)
    _check(args, _prefill(args, D, _tiles(new)))


# heads of 64, several steps a prompt: four workgroups a CU
@pytest.mark.parametrize("Hq,Hk", [(8, 8), (14, 2), (16, 8), (16, 4)])
@pytest.mark.parametrize("fp8", [False, True])
def test_many_prompts_of_several_steps(Hq, Hk, fp8):
    g = torch.Generator().manual_seed(Hq)
    new = torch.randint(90, 257, (130,), generator=g).tolist()
    ctx = torch.randint(0, 150, (130,), generator=g).tolist()
    args = _paged([a + b for a, b in zip(new, ctx)], new, Hq, Hk, 64, fp8, seed=3)
    tiles = _tiles(new)
    assert 512 <= len(tiles[0]) <= 8 * 130
    _check(args, _prefill(args, 64, tiles))


# one block and several a workgroup, two workgroups a CU and four
@pytest.mark.parametrize("Hq,Hk,D,prompts", [
    (8, 2, 128, 1), (5, 1, 128, 1), (4, 1, 64, 1), (3, 3, 64, 1), (8, 8, 64, 30),
    (16, 4, 64, 60)])
@pytest.mark.parametrize("k_at,v_at", [(1, 0), (0, 4), (3, 7)])
def test_pages_at_other_places(Hq, Hk, D, prompts, k_at, v_at):
    """Pages that begin elsewhere than at multiples of 16 bytes (a part of a larger
    buffer): the same results to the bit, values behind the context not a number."""
    new = [1, 33, 63, 64, 65, 130, 40] * prompts
    ctx = [0, 0, 70, 0, 5, 31, 352] * prompts
    lens = [a + b for a, b in zip(new, ctx)]
    args = _paged(lens, new, Hq, Hk, D, False, seed=Hq)
    q, kc, vc, bt, sl, ql = args
    tiles = _tiles(new)
    assert prompts == 1 or 512 <= len(tiles[0]) * Hk <= 8 * len(new) * Hk
    want = _prefill(args, D, tiles)
    if prompts == 1:
        _check(args, want)
    for s, n in enumerate(lens):
        if n % 32:
            vc[int(bt[s, n // 32]), :, n % 32:] = float("nan")

    def shifted(c, at):
        flat = torch.empty(c.numel() + at, dtype=c.dtype, device=DEV)
        part = flat[at:].view(c.shape)
        part.copy_(c)
        assert part.data_ptr() % 16 == at * 2
        return part

    moved = (q, shifted(kc, k_at), shifted(vc, v_at), bt, sl, ql)
    assert torch.equal(_prefill(moved, D, tiles), want)


@pytest.mark.parametrize("which", [1, 2])
def test_pages_with_gaps_are_refused(which):
    args = list(_paged([40], [40], 2, 1, 64, False))
    c = args[which]
    args[which] = torch.cat([c, c], -1).to(DEV)[..., :64]
    with pytest.raises(RuntimeError, match="contiguous"):
        _prefill(args, 64, _tiles([40]))


@pytest.mark.parametrize("Hq,Hk", [(2, 2), (4, 2), (4, 1)])
def test_prompt_tiles_in_any_order(Hq, Hk):
    # a tile map need not list a sequence's tiles in order, nor at all
    new = [200, 130]
    args = _paged(new, new, Hq, Hk, 128, False, seed=9)
    ts, tq = _tiles(new)
    whole = _prefill(args, 128, (ts, tq))
    _check(args, whole)
    for order in (list(range(len(ts)))[::-1], [3, 0, 9, 1, 4, 5, 7]):
        part = _prefill(args, 128, ([ts[i] for i in order],
                                    [tq[i] for i in order]))
        for i in order:
            a = (0 if ts[i] == 0 else 200) + tq[i]
            b = min(a + 32, 200 if ts[i] == 0 else 330)
            assert torch.equal(part[a:b], whole[a:b])


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("delta", [0.375, 0.6, 0.65, 0.9, 1.05, 1.25])
def test_sum_of_many_weights(D, delta):
    """The denominator of a prompt's row over 40,000 keys, a first one above all
    others and the rest alike, so that results are (rounded weights x values) /
    (weights). Every page holds the same 32 values a column. The roundings of
    the results to bf16 (up to 2^-8 of a value between 1 and 2) are 0 on
    average: the mean of 64 D of them is within 4 * 2^-8 / sqrt(3 * 64 D)."""
    n, H, new = 40000, 64, 32
    pages = (n + 31) // 32
    g = torch.Generator().manual_seed(2)
    u = torch.randn(D, generator=g).sign().to(DEV)
    v = (1 + torch.rand(H, 32, D, generator=g)).bfloat16().to(DEV)
    vc = v.expand(pages, H, 32, D).contiguous()
    top = torch.tensor(8.0 / D).bfloat16().item()
    low = torch.tensor((8.0 - delta) / D).bfloat16().item()
    kc = (u * low).bfloat16().expand(pages, H, 32, D).contiguous()
    kc[0, :, 0] = (u * top).bfloat16()
    q = u.bfloat16().expand(new, H, D).contiguous()
    i32 = dict(dtype=torch.int32, device=DEV)
    one = torch.zeros(1, **i32)
    out = ops.paged_attention(
        q, kc, vc, torch.arange(pages, **i32)[None], torch.tensor([n], **i32),
        torch.tensor([0, new], **i32), 1.0, num_decodes_tail=0, tile_seq=one,
        tile_q0=one, prefill_token_count=new)
    p = math.exp(D * low - D * top)
    b = torch.tensor(p).bfloat16().item()
    last = new - 1                                   # its row sees every key
    total = v.double().sum(1) * pages - v[:, 0].double()
    want = (v[:, 0].double() + b * total) / (1 + (n - 1) * p)
    ratio = (out[last].double() / want).mean().item()
    assert abs(ratio - 1) < 4 * 2.0 ** -8 / math.sqrt(3 * H * D)


@pytest.mark.parametrize("Hq,Hk,rows", [(2, 1, 1026), (6, 3, 343), (16, 8, 129)])
@pytest.mark.parametrize("D,fp8", [(128, False), (64, True)])
@pytest.mark.parametrize("longest", [192, 420])
def test_decode_many_rows(Hq, Hk, rows, D, fp8, longest):
    """1026 to 1032 (row, kv head) pairs: four of them share a workgroup where
    none has more than six pages; the last four are not whole, and fours of
    one and of three heads a row span rows of different lengths."""
    g = torch.Generator().manual_seed(rows)
    choice = torch.tensor([1, 20, 32, 33, 100, 160, 192, 193, 260, 420])
    choice = choice[choice <= longest]
    lens = choice[torch.randint(len(choice), (rows,), generator=g)]
    lens[:40] = torch.where(lens[:40] > 192, 192, lens[:40])
    lens[-1] = longest
    args = _paged(lens.tolist(), [1] * rows, Hq, Hk, D, fp8, seed=rows)
    got = ops.paged_attention(*(x.to(DEV) for x in args), 1.0 / math.sqrt(D),
                              num_decodes_tail=rows)
    _check(args, got)
