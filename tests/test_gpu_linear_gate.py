"""Gated linear layers over many rows in one launch: edges of row tiles, column
blocks that do not divide among the XCDs, few and many tiles, one to many steps."""

import pytest
import torch
import torch.nn.functional as F

from sutro_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _operands(M, N, K, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed + M + K)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(2 * N, K, generator=g, device=DEV) * K ** -0.5).bfloat16()
    return x, w


def _exact(x, w):
    y = x.double() @ w.double().T
    n = y.shape[1] // 2
    return F.silu(y[:, :n]) * y[:, n:]


@pytest.mark.parametrize("M,N,K", [
    (1, 128, 64), (255, 128, 128), (256, 384, 192), (257, 1152, 256),
    (1000, 1280, 2048), (2304, 896, 320), (8193, 256, 192), (9000, 1024, 448),
    (300, 17 * 128, 4096)])
def test_kernel(M, N, K):
    x, w = _operands(M, N, K)
    got = ops._require_hip().linear_silu_mul(x, w).double()
    want = _exact(x, w)
    # fp32 sums of K products of size 1, one rounding to bf16 at the end
    torch.testing.assert_close(got, want, rtol=2 ** -8, atol=2 ** -12)


@pytest.mark.parametrize("M,N,K", [
    (9000, 1024, 2048), (8500, 1152, 4096), (2300, 4096, 2048)])
def test_more_tiles_than_workgroups(M, N, K):
    test_kernel(M, N, K)


@pytest.mark.parametrize("M", [1025, 2900, 8193 + 1800])
@pytest.mark.parametrize("blocks", [9, 12, 15])
def test_leftover_row_tiles(M, blocks):
    """Row tiles past the last group of 32, four at a time on all XCDs, with
    column blocks that do not divide among these."""
    test_kernel(M, blocks * 128, 192)


def test_route():
    """The one launch and the library's two passes agree, and what torch has to
    see still goes through torch."""
    x, w = _operands(4096, 2048, 256)
    assert ops._many_rows(x, w)
    one = ops.linear_silu_mul(x, w).double()
    two = ops.silu_mul(F.linear(x, w)).double()
    want = _exact(x, w)
    err = ((one - want).norm() / want.norm(), (two - want).norm() / want.norm())
    assert err[0] <= err[1]
    assert not ops._many_rows(x[:, :192], w[:, :192])     # strided
    assert not ops._many_rows(x[:3000], w)                # too few tiles
    more = x.repeat(3, 1)
    assert ops._many_rows(more[:5632], w)                 # 352 of 512 places
    assert not ops._many_rows(more[:4608], w)             # 288
    assert not ops._many_rows(x.float(), w.float())
    wide = torch.empty(2, 4096, 256, device=DEV, dtype=torch.bfloat16)
    assert not ops._many_rows(wide, w)
    p = torch.nn.Parameter(w)
    assert not ops._many_rows(x, p)
    with torch.no_grad():
        assert ops._many_rows(x, p)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not ops._many_rows(x, w)


@pytest.mark.parametrize("K", [1024, 2048, 4096])
def test_place_of_a_row(K):
    """Equal rows of a batch have equal results, in whichever tile they are."""
    x, w = _operands(5, 1024, K)
    which = torch.arange(9000, device=DEV) * 3 % 5
    got = ops._require_hip().linear_silu_mul(x[which], w)
    for t in range(5):
        same = got[which == t]
        assert torch.equal(same, same[:1].expand_as(same)), t
