"""Where a linear layer over 2 to 256 rows leaves the library: by its sizes, and never
where something of torch's has to see the product."""

import pytest
import torch

from sutro_amd import ops


@pytest.fixture
def on_gpu(monkeypatch):
    monkeypatch.setattr(ops, "_use_hip", lambda t: True)


def bf(*shape):
    return torch.empty(*shape, dtype=torch.bfloat16)      # (never read)


@pytest.mark.parametrize("M,K,rows,gated,kernel", [
    (1, 2048, 8192, False, 0), (2, 2048, 8192, False, 1), (2, 2048, 4096, False, 0),
    (2, 4096, 16384, True, 0), (8, 1024, 4096, False, 0), (8, 1024, 16384, False, 1),
    (8, 4096, 4096, False, 0), (16, 4096, 4096, False, 1), (16, 512, 4096, False, 0),
    (32, 512, 64, False, 1), (32, 4096, 32, False, 0), (64, 1024, 51200, False, 0),
    (64, 2048, 51200, False, 1), (128, 2048, 16384, True, 1),
    (128, 2048, 24576, False, 0), (128, 2048, 32768, False, 1),
    (192, 4096, 10240, False, 1), (192, 4096, 16384, True, 0),
    (256, 4096, 8192, False, 1), (256, 4096, 10240, False, 0),
    (256, 2048, 16384, True, 1), (257, 2048, 4096, False, 0),
    (6, 5120, 5120, False, 1), (16, 5120, 2048, False, 0), (128, 8192, 2048, False, 1),
    (48, 8192, 2048, False, 0), (200, 25600, 5120, False, 1),
    (128, 25600, 5120, True, 1), (128, 12288, 4096, True, 0)])
def test_sizes(on_gpu, M, K, rows, gated, kernel):
    assert ops._mid_rows(bf(M, K), bf(rows, K), gated) == bool(kernel)


def test_operands(on_gpu):
    x, w = bf(48, 2048), bf(3072, 2048)
    assert ops._mid_rows(x, w) and ops._mid_rows(bf(48, 2056)[:, :2048], w)
    for a, b in ((x.float(), w.float()), (x[None], w), (bf(2048, 48).t(), w),
                 (bf(48, 2052)[:, :2048], w), (bf(1, 2048).expand(48, 2048), w),
                 (x, bf(2048, 3072).t()), (x, bf(3070, 2048)), (bf(48, 2000), bf(3072, 2000)),
                 (x, bf(3072, 2304)), (bf(48 * 2048 + 1)[1:].view(48, 2048), w)):
        assert not ops._mid_rows(a, b)
    assert ops._mid_rows(x, bf(4096, 2048), True)
    assert not ops._mid_rows(x, bf(4104, 2048), True)     # an odd number of eights
    w.requires_grad_()
    assert not ops._mid_rows(x, w)
    with torch.no_grad():
        assert ops._mid_rows(x, w)
        with torch.autocast("cpu", dtype=torch.float16):
            assert not ops._mid_rows(x, w)
        seen = []
        torch.func.vmap(lambda v: seen.append(ops._mid_rows(v, w)) or v)(x[None])
    assert seen == [False]


@pytest.mark.parametrize("M,K,rows,gated", [
    (20, 2048, 0, False), (100, 2048, 0, False), (256, 2048, 0, False),
    (20, 2048, 0, True), (100, 2048, 0, True), (48, 1 << 20, 2048, False),
    (100, 1 << 20, 4096, True)])
def test_sizes_the_kernel_refuses(on_gpu, M, K, rows, gated):
    """No weights at all, and rows of a million numbers: the library's. (Meta tensors
    stand in for them: the rule does not read.)"""
    x = torch.empty(M, K, dtype=torch.bfloat16, device="meta")
    w = torch.empty(rows, K, dtype=torch.bfloat16, device="meta")
    assert not ops._mid_rows(x, w, gated)
