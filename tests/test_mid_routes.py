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


def test_the_rule_knows_the_kernels_tiles():
    if ops._C is None:
        pytest.skip("extension not built")
    for M in (2, 8, 9, 16, 31, 32, 33, 64, 65, 96, 128, 129, 150, 192, 193, 256):
        for K in (512, 2048, 4096, 5120):
            for rows in (16, 1024, 1040, 2048, 2064, 4096, 4112, 5456, 5472, 8192,
                         8208, 10880, 10896, 16384, 16400, 32768, 32784, 151936):
                for gated in (False, True):
                    m, n, tiles = ops._mid_tile(M, rows, K, gated)
                    assert [m, n] == ops._C.mid_tile(M, rows, K, gated)
                    assert tiles == -(-M // m) * -(-rows // n)


@pytest.mark.parametrize("M,K,rows,gated,kernel", [
    (30, 3072, 36512, False, 0), (30, 3072, 32768, False, 1),
    (54, 3584, 36224, False, 0), (54, 3584, 32768, False, 1),
    (48, 4096, 39952, False, 0), (48, 4096, 51200, False, 1),
    (9, 3584, 44368, False, 0), (9, 4096, 44368, False, 1),
    (8, 768, 71840, False, 0), (8, 768, 65536, False, 1), (3, 2048, 66672, False, 0),
    (87, 4096, 2432, False, 0), (87, 4096, 2752, False, 1), (87, 4096, 2432, True, 1),
    (97, 4096, 2432, False, 1), (171, 3584, 1472, False, 1), (141, 3584, 1472, False, 0),
    (122, 3072, 9440, False, 0), (122, 3072, 12288, False, 1), (90, 3072, 9440, False, 1),
    (240, 3840, 4544, False, 0), (240, 3840, 6144, False, 1), (186, 3584, 6224, False, 0),
    (150, 3584, 6224, False, 1), (186, 3584, 6224, True, 1),
    (213, 3840, 16336, True, 0), (213, 2048, 16336, True, 1),
    (6, 5120, 2288, False, 1), (6, 5120, 4096, False, 0), (14, 768, 4096, False, 0),
    (4, 3584, 6528, True, 0), (80, 8192, 5056, False, 0), (80, 8192, 5696, False, 1)])
def test_rounds(on_gpu, M, K, rows, gated, kernel):
    """Tiles that begin a round with few of them, or leave a third of the CUs without
    one, where the library's tiles fit."""
    assert ops._mid_rows(bf(M, K), bf(rows, K), gated) == bool(kernel)
