"""Where a gated layer of a layer list may leave its product and unit for one launch:
the sizes it takes, and never where something has to see the product."""

import pytest
import torch

from sutro_amd import ops
from sutro_amd.models import prenorm, vodinex
from sutro_amd.models.layers import SectionedLinear


class _Kernels:
    def __init__(self):
        self.calls = 0

    def linear_gelu_mul(self, x, w, bias, ff):
        self.calls += 1
        return [x.new_zeros(x.shape[0], ff),
                x.new_zeros(x.shape[0], w.shape[0] - 2 * ff)]

    def linear_silu_mul(self, x, w):
        self.calls += 1
        return x.new_zeros(x.shape[0], w.shape[0] // 2)


@pytest.fixture
def kernels(monkeypatch):
    k = _Kernels()
    monkeypatch.setattr(ops, "_use_hip", lambda t: True)
    monkeypatch.setattr(ops, "_require_hip", lambda: k)
    return k


def _bf(*shape):
    return torch.empty(*shape, dtype=torch.bfloat16)       # (never read)


@pytest.mark.parametrize("rows,k,ff,more,one", [
    (32768, 2048, 8192, 2048, 1), (1532, 2048, 8704, 2048, 1),
    (255, 2048, 8192, 2048, 0),          # few rows
    (8192, 2048, 8192, 136, 0),          # columns behind: not whole tiles
    (8192, 2048, 8128, 2048, 0),         # nor the gate's
    (26526, 4096, 6144, 4096, 0), (5298, 4096, 10496, 4096, 1)])
def test_gelu_sizes(kernels, rows, k, ff, more, one):
    n = 2 * ff + more
    with torch.no_grad():
        made = ops.linear_gelu_mul(_bf(rows, k), _bf(n, k), _bf(n), ff)
    assert (made is not None) == bool(one) == bool(kernels.calls)


def test_gelu_operands(kernels):
    x, w, b = _bf(8192, 512), _bf(4608, 512), _bf(4608)
    f = ops.linear_gelu_mul
    with torch.no_grad():
        assert f(x, w, b, 2048) is not None and f(x, w, None, 2048) is not None
        assert f(x, w, b.float(), 2048) is None
        assert f(x, w, _bf(9216)[::2], 2048) is None
        assert f(x.float(), w, b, 2048) is None
        assert f(x, w, _bf(4609)[1:], 2048) is None
        assert f(_bf(512, 8192).T, w, b, 2048) is None
    assert f(x, w.requires_grad_(), b, 2048) is None
    assert kernels.calls == 2


@pytest.mark.parametrize("model", [vodinex, prenorm])
def test_hooked_layers_see_their_input(model):
    """Blocks ask whether the layer is the plain one that nothing watches."""
    lin = SectionedLinear(64, [("gate", 64, False), ("up", 64, False)],
                          torch.bfloat16)
    assert model.unhooked(lin)
    h = lin.register_forward_hook(lambda m, a, y: None)
    assert not model.unhooked(lin)
    h.remove()
    lin.forward = lambda x: x
    assert not model.unhooked(lin)
