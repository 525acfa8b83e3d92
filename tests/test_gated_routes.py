"""Where a gated layer of a layer list may leave its product and unit for one launch:
the sizes it takes, and never where something has to see the product."""

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from sutro_amd import ops
from sutro_amd.models import prenorm, vodinex
from sutro_amd.models.hybrid_spec import (AttnMixerSpec, HybridLayerSpec,
                                          HybridSpec)
from sutro_amd.models.layers import SectionedLinear
from sutro_amd.ops import hybrid as hops


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


W, T = 256, 3


class _Computed(_Kernels):
    """What the two launches make, by the operations they stand for."""

    def linear_gelu_mul(self, x, w, bias, ff):
        self.calls += 1
        y = F.linear(x, w, bias)
        return [hops.gelu_tanh_mul(y, 0, ff, ff), y[:, 2 * ff:].contiguous()]

    def linear_silu_mul(self, x, w):
        self.calls += 1
        ff = w.shape[0] // 2
        return hops.glu_mul(F.linear(x, w), 0, ff, ff, hops.GLU_SILU)


class _Mixer(nn.Module):
    def forward(self, proj, off, tag, fb, kv, out, at, scale, **kw):
        out.copy_(proj[:, :out.shape[1]])


class _Derived(SectionedLinear):
    pass


def _block(kind, ff):
    torch.manual_seed(0)
    mixer = AttnMixerSpec(heads=4, kv_heads=4, dim=64, vdim=64, scale=0.125)
    layer = HybridLayerSpec("attention", mixer, ff=ff, ff_kind="swiglu")
    spec = HybridSpec(name="block", arch="", hidden_size=W, vocab_size=8,
                      layers=(layer,))
    if kind == "vodinex":
        block = vodinex.HybridBlock(spec, layer, 0, torch.bfloat16)
        block.mixers[0] = _Mixer()
    else:
        block = prenorm.PreNormBlock(spec, layer, 0, torch.bfloat16)
        block.mixer = _Mixer()
    with torch.no_grad():
        for p in block.parameters():
            p.normal_(0, 0.1)
    return block


def _run(kind, block):
    g = torch.Generator().manual_seed(1)
    x = torch.randn(T, W, generator=g)
    h = x.bfloat16()
    more = () if kind == "vodinex" else (torch.ones(W),)
    with torch.no_grad():
        block(x, h, None, None, *more)
    return x, h


@pytest.fixture
def computed(monkeypatch):
    k = _Computed()
    monkeypatch.setattr(ops, "_require_hip", lambda: k)
    monkeypatch.setattr(ops, "_many_rows", lambda x, w: True)
    return k


@pytest.mark.parametrize("kind", ["vodinex", "prenorm"])
def test_blocks_take_the_launch(computed, monkeypatch, kind):
    """With it a block computes what it computes without it; the residual gate is then
    read where the launch leaves it."""
    block = _block(kind, 128)
    got = _run(kind, block)
    assert computed.calls == 1
    monkeypatch.setattr(ops, "_many_rows", lambda x, w: False)
    want = _run(kind, block)
    assert computed.calls == 1
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("how", ["hook", "pre_hook", "forward", "class", "offsets"])
@pytest.mark.parametrize("kind", ["vodinex", "prenorm"])
def test_blocks_call_a_layer_that_is_not_plain(computed, monkeypatch, kind, how):
    """Watched, replaced, derived, or with sections that are not two halves: the layer
    sees its input and the block its result."""
    block = _block(kind, 124 if how == "offsets" else 128)
    lin, seen = block.ff_in, []
    if how == "hook":
        lin.register_forward_hook(lambda m, a, y: seen.append(a[0].shape))
    elif how == "pre_hook":
        lin.register_forward_pre_hook(lambda m, a: seen.append(a[0].shape))
    elif how == "forward":
        def forward(x, call=lin.forward):
            seen.append(x.shape)
            return call(x)
        lin.forward = forward
    elif how == "class":
        lin.__class__ = _Derived
    got = _run(kind, block)
    assert computed.calls == 0
    assert seen == [(T, W)] or how in ("class", "offsets")
    monkeypatch.setattr(ops, "_many_rows", lambda x, w: False)
    for a, b in zip(got, _run(kind, block)):
        assert torch.equal(a, b)
