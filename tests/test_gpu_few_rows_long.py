"""Linear layers over few rows with larger matrices: 16 and 32 weight rows a
workgroup, two to sixteen waves, starts of k that differ between workgroups."""

import pytest
import torch
import torch.nn.functional as F

from sutro_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("M", [3, 16, 17, 32])
@pytest.mark.parametrize("N,K,gated", [
    (4096, 64, False), (4100, 2080, False), (6144, 2048, False),
    (8272, 2048, False), (8192, 4096, False), (8196, 4096, False),
    (18432, 96, False), (4096, 8192, True), (8200, 4096, True),
    (512, 4096, True), (1024, 12288, False), (520, 2048, True)])
def test_kernel(N, K, gated, M):
    g = torch.Generator(device=DEV).manual_seed(N + K + M)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).bfloat16()
    got = ops._require_hip().linear_skinny(x, w, None, gated).double()
    y = x.double() @ w.double().T
    if gated:
        y = F.silu(y[:, :N // 2]) * y[:, N // 2:]
    # fp32 sums of K products of size 1, one rounding to bf16 at the end
    torch.testing.assert_close(got, y, rtol=2 ** -8, atol=2 ** -12)


@pytest.mark.parametrize("M", [3, 12, 13, 17])
@pytest.mark.parametrize("N,K,gated", [
    (64, 448, False), (4096, 512, False), (9216, 512, False),
    (12, 1024, False), (8272, 1024, False), (2048, 1056, False),
    (4096, 2048, False), (4112, 2048, False), (4348, 640, False),
    (4352, 640, False), (4096, 2080, False), (40, 512, True), (8208, 512, True),
    (1024, 1024, True), (256, 2048, True), (8192, 1536, True)])
def test_waves(N, K, gated, M):
    """A batch each for 4, 8 and 16 waves, one k-step less and more; a round of
    workgroups and some more."""
    test_kernel(N, K, gated, M)


@pytest.mark.parametrize("M,rows,K,want", [
    (3, 20000, 2048, True), (16, 24576, 2048, True), (16, 24576, 4096, False),
    (17, 20000, 2048, False), (12, 8192, 4096, True), (13, 8192, 4096, False),
    (8, 65536, 4096, True), (8, 151936, 2048, False), (6, 151936, 2048, True),
    (8, 30000, 1024, False), (32, 5120, 25600, True), (3, 4096, 16384, False),
    (3, 5120, 5120, False), (8, 16384, 3072, False)])
def test_rule(M, rows, K, want):
    assert ops._long_weights(M, rows, K) == want
