"""Attention over one shared latent a token: prompt pieces and single tokens of
uneven sequences, at every padded size of the kernel, against 64 bits."""

import pytest
import torch

from sutro_amd.ops import hybrid as hops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("window", [0, 50, 128])
@pytest.mark.parametrize("H,dk,dv", [
    (5, 24, 16), (3, 136, 120), (2, 256, 256), (9, 264, 136), (16, 320, 256),
    (3, 392, 392), (1, 512, 512), (7, 520, 264), (32, 576, 512)])
def test_uneven_sequences(H, dk, dv, window):
    """Sequences of one key to seven steps of 64, with and without cached tokens
    in front, tiles with fewer than 64 rows, and decoded tokens whose keys may be
    cut into runs. A weight is rounded to bf16, at most 2^-8 of itself, and so is
    the result: 2^-7 of the largest value, and 2^-12 more for scores in 32 bits."""
    dev = "cuda"
    g = torch.Generator().manual_seed(dk * H + window)
    new = [1, 63, 64, 65, 33, 2, 130, 200]       # prompt pieces
    old = [0, 0, 31, 64, 300, 95, 0, 201]        # tokens in front of them
    new += [1, 1, 1, 1]                          # decoded tokens
    old += [0, 64, 127, 420]
    P, T = sum(new[:8]), sum(new)
    S = len(new)
    per = 16
    blocks = S * per + 1
    table = (torch.randperm(blocks - 1, generator=g) + 1)[:S * per]
    table = table.int().view(S, per).contiguous()
    cache = torch.randn(blocks, 1, 32, dk, generator=g).bfloat16()
    q = torch.randn(T, H, dk, generator=g).bfloat16()
    locs = [0]
    for n in new:
        locs.append(locs[-1] + n)
    tiles = [(i, a) for i in range(8) for a in range(0, new[i], 32)]
    scale = dk ** -0.5
    off, wide = 8, H * dv + 24                   # a section of longer rows
    out = torch.full((T, wide), 7.0, dtype=torch.bfloat16, device=dev)
    c = cache.to(dev)
    hops.local_attention(
        q.to(dev), c, c[..., :dv], table.to(dev),
        torch.tensor([a + b for a, b in zip(new, old)], dtype=torch.int32,
                     device=dev),
        torch.tensor(locs, dtype=torch.int32, device=dev), scale, 0, window,
        torch.empty(T, 8, dtype=torch.bfloat16, device=dev), -1, out, off, 1.0,
        token_seq=torch.tensor([i for i in range(S) for _ in range(new[i])],
                               dtype=torch.int32, device=dev),
        tile_seq=torch.tensor([t[0] for t in tiles], dtype=torch.int32,
                              device=dev),
        tile_q0=torch.tensor([t[1] for t in tiles], dtype=torch.int32,
                             device=dev), prefill_rows=P)
    out = out.cpu().double()
    assert (out[:, :off] == 7).all() and (out[:, off + H * dv:] == 7).all()
    got = out[:, off:off + H * dv].view(T, H, dv)
    for i in range(S):
        n = new[i] + old[i]
        kv = cache[table[i].long()].reshape(-1, dk)[:n].double()
        qs = q[locs[i]:locs[i + 1]].double()
        s = torch.einsum("thd,kd->htk", qs, kv) * scale
        at = old[i] + torch.arange(new[i])[:, None] - torch.arange(n)[None]
        seen = (at >= 0) & ((at < window) if window else (at >= 0))
        s.masked_fill_(~seen, float("-inf"))
        want = torch.einsum("htk,kd->thd", s.softmax(-1), kv[:, :dv])
        err = (got[locs[i]:locs[i + 1]] - want).abs().max()
        assert err <= (2 ** -7 + 2 ** -12) * float(kv[:, :dv].abs().max())


@pytest.mark.parametrize("start", [1, 4])
def test_pages_at_other_places(start):
    """Pages that begin at 2 or 8 bytes past a multiple of 16 (a part of a larger
    buffer): the general kernel's, one rounding of weights and results from the other."""
    dev = "cuda"
    H, dk, dv, S = 4, 72, 64, 3
    g = torch.Generator().manual_seed(start)
    flat = torch.randn(start + 5 * 32 * dk, generator=g).bfloat16().to(dev)
    cache = flat[start:].view(5, 1, 32, dk)
    q = torch.randn(S, H, dk, generator=g).bfloat16().to(dev)
    i32 = dict(dtype=torch.int32, device=dev)
    table = torch.tensor([[1, 2], [3, 0], [4, 0]], **i32)
    lens, locs = torch.tensor([50, 32, 3], **i32), torch.arange(S + 1, **i32)
    rest = (table, lens, locs, dk ** -0.5, 0, 0,
            torch.empty(S, 8, dtype=torch.bfloat16, device=dev), -1)
    outs = []
    for c in (cache, cache.clone()):
        out = torch.zeros(S, H * dv, dtype=torch.bfloat16, device=dev)
        hops.local_attention(q, c, c[..., :dv], *rest, out, 0, 1.0,
                             token_seq=torch.arange(S, **i32))
        outs.append(out.double())
    assert (outs[0] - outs[1]).abs().max() <= 2 ** -6 * float(cache.abs().max())
