"""Delta-rule inputs over runs of tokens: a batch large enough for them against
the same sequences in batches too small for them. Both sum the taps in one
order: equal to the bit, filter histories too."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from sutro_amd.ops import hybrid as hops


@pytest.mark.parametrize("G,H,dk,dv,head_gates", [
    (2, 2, 128, 128, False), (2, 4, 128, 64, True), (4, 4, 64, 40, True)])
def test_runs_of_tokens(G, H, dk, dv, head_gates):
    g = torch.Generator().manual_seed(G + dv)
    # new tokens and earlier ones: runs start inside, end inside and span
    # sequences; single tokens with and without a history; long pieces
    new = [1, 1, 2, 3, 1, 7, 8, 9, 1, 5, 1, 1, 1, 6] + [37] * 60
    new += [14000 // (G * dk // 256) - sum(new)]
    old = [0, 5, 0, 2, 1, 0, 9, 1, 2, 3, 0, 0, 40, 1] + [0, 2, 3] * 20 + [4]
    T, S = sum(new), len(new)
    C = 2 * G * dk + H * dv
    ncol = C + 3 * H + (-3 * H) % 8
    proj = torch.randn(T, ncol, generator=g).to(torch.bfloat16).cuda()
    conv_w = torch.randn(C, 4, generator=g).cuda()
    a2 = None if head_gates else torch.randn(H * dk, H, generator=g).cuda()
    n_dt = H if head_gates else H * dk
    dt_bias = torch.randn(n_dt, generator=g).cuda()
    a_log = torch.randn(H, generator=g).cuda()
    state = torch.randn(S, 3, C, generator=g).cuda()

    def part(first, last, state):
        lens = torch.tensor(new[first:last])
        t0 = sum(new[:first])
        q = torch.cat([torch.zeros(1, dtype=torch.long), lens.cumsum(0)]).int()
        total = (lens + torch.tensor(old[first:last])).int()
        seq = torch.repeat_interleave(torch.arange(len(lens)), lens).int()
        return hops.delta_prep(
            proj[t0:t0 + int(lens.sum())].contiguous(), 0, G * dk, 2 * G * dk,
            C, C + H, H, G, dk, dv, conv_w, a2, dt_bias, a_log, state,
            torch.arange(first, last).int().cuda(), q.cuda(), total.cuda(),
            token_seq=seq.cuda())

    whole_state, part_state = state.clone(), state.clone()
    whole = part(0, S, whole_state)
    cut = S - 1
    small = [part(0, 14, part_state), part(14, 44, part_state),
             part(44, cut, part_state)]
    # the last sequence alone is large: its first tokens are compared by hand
    n = sum(new[:cut])
    for w, *p in zip(whole, *small):
        assert torch.equal(w[:n], torch.cat(p))
    assert torch.equal(whole_state[:cut], part_state[:cut])
    # and its tokens against the filter itself, in float64
    x = proj[n:, :C].double()
    x = torch.cat([state[cut].double(), x])
    y = sum(conv_w[:, k].double() * x[k:k + T - n] for k in range(4))
    y = (y * y.sigmoid())[:, 2 * G * dk:].view(T - n, H, dv)
    assert (whole[2][n:].double() - y).abs().max() < 1e-4
