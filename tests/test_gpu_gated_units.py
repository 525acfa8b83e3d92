"""The gated units of the products on tiles of 256 rows, for sums chosen one by one:
steep and flat parts, both ends of the exponential, infinities and NaN."""

import math

import pytest
import torch

from sutro_amd import ops
from sutro_amd.ops import hybrid as hops

pytestmark = pytest.mark.gpu
DEV = "cuda"
K, N, M = 64, 128, 256
GATES = [0.0, -0.0, 1e-30, 1e-3, 0.5, 1.0, 1.5, 3.0, 7.0, 11.0, 52.0, 87.0, 88.0, 88.5,
         20.0, 100.0, 1e4, 1e30, 3e38, math.inf, math.nan]
UPS = [0.0, 1.0, -1.0, 0.3, 7.5, -9.0, 1e-20, 1e20]


def _operands():
    """x [M, K], w [2 N, K] whose product has gate GATES (either sign) and up UPS
    in all pairs: a row of x is one column of w."""
    g = torch.tensor(GATES + [-v for v in GATES])
    pairs = torch.cartesian_prod(g, torch.tensor(UPS)).bfloat16()
    w = torch.zeros(2 * N, K, dtype=torch.bfloat16)
    n = len(pairs)
    cols = -(-n // N)
    for c in range(cols):
        part = pairs[c * N:(c + 1) * N]
        w[:len(part), c], w[N:N + len(part), c] = part[:, 0], part[:, 1]
    x = torch.zeros(M, K, dtype=torch.bfloat16)
    x[torch.arange(M), torch.arange(M) % cols] = 1
    return x, w


def _want(x, w, unit):
    y = x.double() @ w.double().T
    return unit(y[:, :N], y[:, N:])


def _check(got, want, power):
    """One rounding to bf16 (2^-8 / (1 + 2^-8), below 2^-126 half of 2^-133), the unit in
    fp32 far below it; where e^power is infinite in fp32 (2^128) the quotient, under
    2^-121 of the up's 1e20, is 0."""
    got, past = got.double().cpu(), torch.exp(power.float()).isinf()
    assert torch.equal(got.isnan(), want.isnan())
    ok = ~want.isnan()
    big = want.abs() > 3.4e38                       # past bf16's largest: infinite
    assert torch.equal(got[ok & big], want[ok & big].sign() * math.inf)
    ok &= ~big
    err = (got[ok] - want[ok]).abs()
    lost = past[ok].double() * 2.0 ** -121 * 1e20
    assert (err <= want[ok].abs() * 2 ** -8 + 2.0 ** -134 + lost).all()


def silu(g, u):
    return g / (1 + torch.exp(-g)) * u


def gelu(g, u):
    z = 2 * math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3)
    return torch.where(g.abs() > 1e4, g * (g > 0), g / (1 + torch.exp(-z))) * u


def clamped(g, u, limit=7.0):
    lim = torch.tensor(limit, dtype=g.dtype)        # (of a NaN the limit)
    g, u = torch.fmin(g, lim), torch.fmin(torch.fmax(u, -lim), lim)
    return g / (1 + torch.exp(-1.702 * g)) * (u + 1)


def test_one_matrix():
    x, w = _operands()
    got = ops._require_hip().linear_silu_mul(x.to(DEV), w.to(DEV))
    _check(got, _want(x, w, silu), _want(x, w, lambda g, u: -g))


def test_gelu():
    x, w = _operands()
    x, w = x[:, :3], w[:, :3]           # (an infinite gate: 0 or the gate itself)
    w[w.isinf()] = 0
    x, w = (torch.nn.functional.pad(t, (0, K - 3)) for t in (x, w))
    got = ops._require_hip().linear_gelu_mul(x.to(DEV), w.to(DEV), None, N)[0]
    _check(got, _want(x, w, gelu), torch.full_like(got.double().cpu(), math.inf))


@pytest.mark.parametrize("biased", [True, False])
@pytest.mark.parametrize("rows,ff,k,more", [(1, 128, 64, 0), (255, 256, 192, 256),
                                            (257, 384, 1024, 2048),
                                            (3000, 1152, 320, 512)])
def test_columns_behind(rows, ff, k, more, biased):
    """GELU with a bias, and plain columns behind gate and up: the fp32 sum (and
    unit) rounded once, 2^-8, and the sum's own error of k products in fp32."""
    g = torch.Generator().manual_seed(rows + k)
    x = torch.randn(rows, k, generator=g).bfloat16()
    w = (torch.randn(2 * ff + more, k, generator=g) * 2 * k ** -0.5).bfloat16()
    b = torch.randn(2 * ff + more, generator=g).bfloat16() if biased else None
    act, rest = ops._require_hip().linear_gelu_mul(
        x.to(DEV), w.to(DEV), None if b is None else b.to(DEV), ff)
    y = x.double() @ w.double().T + (0 if b is None else b.double())
    gate, up, more_y = y[:, :ff], y[:, ff:2 * ff], y[:, 2 * ff:]
    sums = k * 2.0 ** -22
    want = gelu(gate, up)
    assert ((act.double().cpu() - want).abs() <= want.abs() * 2 ** -8
            + sums * (1 + gate.abs()) * (1 + up.abs())).all()
    assert rest.shape == more_y.shape
    assert ((rest.double().cpu() - more_y).abs() <= more_y.abs() * 2 ** -8
            + sums).all()


@pytest.mark.parametrize("kind", ["silu", "clamped", "weighted"])
def test_experts(kind):
    x, w = _operands()
    off = torch.tensor([0, 1], dtype=torch.int32, device=DEV)
    cnt = torch.tensor([M], dtype=torch.int32, device=DEV)
    tok = torch.arange(M, dtype=torch.int32, device=DEV)
    out = torch.zeros(M, N, dtype=torch.bfloat16, device=DEV)
    rw = torch.rand(M, generator=torch.Generator().manual_seed(1)) * 0.5 + 0.25
    rw[::7] = 1.0
    act = hops.ACT_GLU_CLAMPED if kind == "clamped" else hops.ACT_SILU_GATE
    hops.expert_gemm(out, x.to(DEV), w.to(DEV)[None], tok, off, cnt, act, 256, 7.0,
                     rw.to(DEV) if kind == "weighted" else None)
    y = rw[:, None].double() if kind == "weighted" else 1.0
    unit, c = (clamped, 1.702) if kind == "clamped" else (silu, 1.0)
    _check(out, _want(x, w, lambda g, u: unit(g * y, u * y)),
           _want(x, w, lambda g, u: -c * y * g))


@pytest.mark.parametrize("tiles,blocks", [
    (5, 8), (5, 9), (5, 15), (6, 9), (11, 46), (13, 39), (9, 29), (35, 11), (33, 60), (7, 8)])
@pytest.mark.parametrize("gated", [False, True])
def test_every_tile_once(tiles, blocks, gated):
    """Row tiles by column blocks at which the last rows go to the XCDs by single tiles, or
    not: whole numbers come out as they are."""
    M, N, K = tiles * 256 - 5, blocks * (128 if gated else 256), 64
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randint(-2, 3, (M, K), generator=g, device=DEV).bfloat16()
    w = torch.randint(-2, 3, (2 * N if gated else N, K), generator=g, device=DEV).bfloat16()
    y = x.float() @ w.float().T
    if gated:
        got = ops._require_hip().linear_silu_mul(x, w)
        want = torch.nn.functional.silu(y[:, :N]) * y[:, N:]
        assert ((got.float() - want).abs() <= want.abs() * 2 ** -8).all()
        return
    off = torch.tensor([0, tiles], dtype=torch.int32, device=DEV)
    cnt = torch.tensor([M], dtype=torch.int32, device=DEV)
    a = torch.zeros(tiles * 256, K, dtype=torch.bfloat16, device=DEV)
    a[:M] = x
    out = torch.zeros(tiles * 256, N, dtype=torch.bfloat16, device=DEV)
    hops.expert_gemm(out, a, w[None], None, off, cnt, hops.ACT_NONE, 256)
    assert torch.equal(out[:M].float(), y.bfloat16().float())
