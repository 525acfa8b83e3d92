"""Layer-list attention on the paged kernels (bf16, pages of 32, keys and values
of 64 or 128): sinks, kept first keys, distance bias, gates and output sections
over contexts of many runs and over prompt pieces, against a 64-bit oracle; and
equal head sizes that the paged kernels do not take."""

import math

import pytest
import torch

from sutro_amd.ops import hybrid as hops

pytestmark = pytest.mark.gpu
DEV = "cuda"
RUN = 256      # visible keys of a run, where contexts are cut


def _case(lens, new, H, G, D, chunk, window, keep, seed):
    """Keys whose scores are about -9 +- 1, but about 0 for one key in every
    run's worth of visible ones and one head of the group (as in _visible for
    the last row of each sequence): weights of runs, of the keys planted in them
    and of a sink of score 0 are all of one size."""
    g = torch.Generator().manual_seed(seed)
    need = [(n + 31) // 32 for n in lens]
    perm = torch.randperm(sum(need) + 2, generator=g)
    bt = torch.zeros(len(lens), max(need) + 3, dtype=torch.int32)
    at = 0
    for s, n in enumerate(need):
        bt[s, :n] = perm[at:at + n].int()
        at += n
    common = torch.randn(G, D, generator=g).sign()
    T = sum(new)
    q = torch.randn(T, G, H // G, D, generator=g)
    q = (q + 2 * common[:, None]).bfloat16()
    kc = torch.randn(len(perm), G, 32, D, generator=g) / 2.5
    kc = (kc - common[:, None] * 4.5 / math.sqrt(D)).bfloat16()
    vc = torch.randn(len(perm), G, 32, D, generator=g).bfloat16()
    ends = torch.tensor([0] + new).cumsum(0).tolist()
    for s, n in enumerate(lens):
        seen = _visible(n - 1, n, chunk, window, keep).nonzero().flatten()
        runs = (len(seen) + RUN - 1) // RUN
        for r in range(runs):
            p = int(seen[min(r * RUN + 37 * (r + 1) % RUN, len(seen) - 1)])
            head = q[ends[s + 1] - 1, :, r % max(min(H // G, runs // 2), 1)].float()
            mate = common * math.sqrt(D) / D * (head * common).sum(-1, keepdim=True)
            kc[bt[s, p // 32], :, p % 32] = (
                (head * math.sqrt(D) - mate) / D / 4).bfloat16()
    return (q.view(T, H, D), kc, vc, bt, torch.tensor(lens, dtype=torch.int32),
            torch.tensor(ends, dtype=torch.int32),
            torch.repeat_interleave(torch.arange(len(lens)),
                                    torch.tensor(new)).int())


def _visible(p, n, chunk, window, keep):
    k = torch.arange(n)
    seen = k <= p
    if chunk:
        seen &= k >= p // chunk * chunk
    if window:
        seen &= (k > p - window) | (k < keep)
    return seen


def _oracle(args, t, chunk, window, keep, bias, sink, sink_w):
    """Row t in 64 bits, in parts: sum(p v), sum(p |v|) and sum(p) of each run's
    worth of visible keys ([runs, H, D] and [runs, H, 1]) and the sink's weight
    [H, 1]."""
    q, kc, vc, bt, sl, ql, seq = args
    s = int(seq[t])
    n = int(sl[s])
    p = n - int(ql[s + 1]) + t
    G, D = kc.shape[1], kc.shape[3]
    H = q.shape[1]
    seen = _visible(p, n, chunk, window, keep)
    pages = bt[s, :(n + 31) // 32].long()
    k, v = (x[pages].double().transpose(0, 1).reshape(G, -1, D)[:, :n][:, seen]
            for x in (kc, vc))
    z = (q[t].double().view(G, H // G, D) @ k.transpose(1, 2)).view(H, -1)
    z = z / math.sqrt(D)
    if bias is not None:
        r1, r2 = (x.double()[:, None] for x in bias)
        far = (p - torch.arange(n)[seen]).double()
        z = z - r1 * torch.log(1 + r2 * far)
    w = z.exp().view(G, H // G, -1).split(RUN, 2)
    extra = torch.zeros(H, 1, dtype=torch.double)
    if sink:
        extra += 1.0 if sink_w is None else sink_w.double()[:, None].exp()
    val, mag = (torch.stack([(x @ y).view(H, D)
                             for x, y in zip(w, u.split(RUN, 1))])
                for u in (v, v.abs()))
    return val, mag, torch.stack([x.sum(-1).view(H, 1) for x in w]), extra


_KINDS = {
    "plain": dict(),
    "zero sink": dict(sink=True),
    "learned sinks": dict(sink=True, learned=True, gate=1),
    "bias": dict(bias=True, gate=1),
    "element gate": dict(gate=64),
    "all": dict(sink=True, learned=True, bias=True, gate=64),
}


def _run(kind, H, G, D, chunk, window, keep, lens, new, n_prompts, seed,
         out_off=8):
    opt = _KINDS[kind]
    args = _case(lens, new, H, G, D, chunk, window, keep, seed)
    g = torch.Generator().manual_seed(seed + 1)
    T = sum(new)
    gate_n = {0: 0, 1: 1, 64: D}[opt.get("gate", 0)]
    proj = torch.randn(T, 8 + H * max(gate_n, 1), generator=g).bfloat16()
    bias = sink_w = None
    if opt.get("bias"):
        bias = (torch.rand(H, generator=g) * 0.4 - 0.1,
                torch.rand(H, generator=g) * 0.05)
    if opt.get("learned"):
        sink_w = torch.randn(H, generator=g)
    kw = {}
    if n_prompts:
        kw = dict(
            tile_seq=torch.tensor([s for s in range(n_prompts)
                                   for _ in range(0, new[s], 32)]).int().to(DEV),
            tile_q0=torch.tensor([j for c in new[:n_prompts]
                                  for j in range(0, c, 32)]).int().to(DEV),
            prefill_rows=sum(new[:n_prompts]))
    if bias is not None:
        kw.update(bias_r1=bias[0].to(DEV), bias_r2=bias[1].to(DEV))
    if sink_w is not None:
        kw.update(sink_w=sink_w.to(DEV))
    out = torch.full((T, out_off + H * D + 4), 7.0, dtype=torch.bfloat16,
                     device=DEV)
    q, kc, vc, bt, sl, ql, seq = (x.to(DEV) for x in args)
    hops.local_attention(q, kc, vc, bt, sl, ql, D ** -0.5, chunk, window,
                         proj.to(DEV), 8 if gate_n else -1, out, out_off, 0.75,
                         token_seq=seq, sink=opt.get("sink", False),
                         keep_first=keep, gate_n=max(gate_n, 1), **kw)
    out = out.float().cpu()
    assert (out[:, :out_off] == 7).all() and (out[:, out_off + H * D:] == 7).all()
    got = out[:, out_off:out_off + H * D].view(T, H, D).double()
    for t in range(T):
        val, mag, den, extra = _oracle(args, t, chunk, window, keep, bias,
                                       opt.get("sink", False), sink_w)
        total = den.sum(0) + extra
        want, size = val.sum(0) / total, mag.sum(0) / total
        f = torch.full((H, 1), 0.75, dtype=torch.double)
        if gate_n:
            f = f * torch.sigmoid(proj[t, 8:].double()).view(H, gate_n)
        # the result is rounded to bf16, 2^-8 of it; prompts round their weights
        # as well; 2^-12 is for scores of up to 20 in 32 bits
        low = t < sum(new[:n_prompts])
        bound = ((2.0 ** -7 if low else 2.0 ** -8) + 2.0 ** -12) * size * f
        err = (got[t] - want * f).abs()
        assert (err <= bound).all(), (t, (err / bound).max().item())
        # single tokens: every run and the sink count once
        if low:
            continue
        wrong = [(val.sum(0) + x * val[r]) / (total + x * den[r])
                 for r in range(len(val)) for x in (-1, 1) if len(val) > 1]
        if opt.get("sink"):
            wrong += [val.sum(0) / (total + x * extra) for x in (-1, 1)]
        for i, bad in enumerate(wrong):
            assert ((bad - want).abs() * f > 2 * bound).any(), (t, i)


@pytest.mark.parametrize("kind", _KINDS)
@pytest.mark.parametrize("H,G,D", [(8, 2, 128), (5, 1, 64)])
@pytest.mark.parametrize("chunk,window,keep", [
    (0, 0, 0), (0, 700, 400), (2048, 0, 0)])
def test_single_tokens_over_many_runs(kind, H, G, D, chunk, window, keep):
    lens = [300, 3000, 1025, 31, 2049]
    _run(kind, H, G, D, chunk, window, keep, lens, [1] * 5, 0, seed=D + window)


@pytest.mark.parametrize("kind", _KINDS)
@pytest.mark.parametrize("H,G,D", [(8, 2, 128), (3, 3, 64), (2, 1, 128)])
@pytest.mark.parametrize("chunk,window,keep", [(0, 0, 0), (0, 70, 40)])
def test_prompt_pieces(kind, H, G, D, chunk, window, keep):
    new = [70, 33, 130, 1, 1]
    lens = [270, 33, 161, 500, 65]
    _run(kind, H, G, D, chunk, window, keep, lens, new, 3, seed=H)


@pytest.mark.parametrize("H,G,D,out_off", [
    (8, 2, 128, 2),      # results at an odd place: both on the other kernels
    (4, 4, 64, 6),
    (17, 1, 64, 8),      # more than 16 heads a kv head: single tokens only
    (40, 2, 128, 8)])
@pytest.mark.parametrize("kind", ["plain", "all"])
def test_beside_the_paged_kernels(H, G, D, out_off, kind):
    new = [70, 33, 1, 1]
    lens = [270, 33, 400, 65]
    _run(kind, H, G, D, 0, 150, 20, lens, new, 2, seed=H, out_off=out_off)


@pytest.mark.parametrize("H,G,D,prompts", [
    (8, 8, 64, 126), (16, 8, 64, 126),    # fill the chip: the other kernel
    (3, 1, 128, 175), (14, 2, 64, 40)])   # four heads of an odd group a workgroup
@pytest.mark.parametrize("kind", ["plain", "all"])
@pytest.mark.parametrize("window,keep", [(0, 0), (24, 3)])
def test_many_prompts_of_one_block(H, G, D, prompts, kind, window, keep):
    g = torch.Generator().manual_seed(H)
    new = torch.randint(1, 7, (prompts,), generator=g).tolist()
    new[0] = 32
    lens = [n + int(c) for n, c in
            zip(new, torch.randint(0, 50, (prompts,), generator=g))]
    _run(kind, H, G, D, 0, window, keep, lens, new, prompts, seed=H)
