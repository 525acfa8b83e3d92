"""Decoder blocks whose attention or feed-forward was replaced, subclassed or
hooked: every module is called with its own input, as it is in a plain block."""

import pytest
import torch
import torch.nn as nn

from sutro_amd import ops
from sutro_amd.models import linear
from sutro_amd.models.qwen3 import Qwen3Attention, Qwen3Block
from sutro_amd.models.registry import tiny_spec_for_tests

WIDTH = 64


class Plain(nn.Module):
    """No projection of the usual name."""

    def __init__(self):
        super().__init__()
        self.mix = nn.Linear(WIDTH, WIDTH, bias=False)

    def forward(self, x, fb, kv, cos_sin):
        return self.mix(x)


class Own(nn.Module):
    """The usual projection, a forward of its own."""

    def __init__(self):
        super().__init__()
        self.qkv_proj = linear.Linear(WIDTH, WIDTH, bias=False)

    def forward(self, x, fb, kv, cos_sin):
        return self.qkv_proj(x) + x


class Derived(Qwen3Attention):
    def forward(self, x, fb, kv, cos_sin):
        return self.o_proj(self.qkv_proj(x)[:, :self.q_size])


def _block(kind):
    torch.manual_seed(0)
    spec = tiny_spec_for_tests()
    block = Qwen3Block(spec, torch.float32, 0)
    if kind is Derived:
        block.self_attn = Derived(spec, torch.float32, 0)
    else:
        block.self_attn = kind()
    with torch.no_grad():
        for p in block.parameters():
            p.normal_(0, 0.1)
    return block


def _expected(block, x, residual):
    r = x + residual
    n = block.input_layernorm
    x = block.self_attn(ops.torch_ref.rmsnorm(r, n.weight, n.eps), None, None,
                        None)
    r = r + x
    n = block.post_attention_layernorm
    return block.mlp(ops.torch_ref.rmsnorm(r, n.weight, n.eps)), r


@pytest.mark.parametrize("kind", [Plain, Own, Derived])
@pytest.mark.parametrize("rows", [1, 3])
def test_other_attention(kind, rows):
    block = _block(kind)
    x, residual = torch.randn(rows, WIDTH), torch.randn(rows, WIDTH)
    with torch.no_grad():
        want = _expected(block, x.clone(), residual.clone())
        got = block(x, residual, None, None, None)
    # the same fp32 operations in the same order
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b)


HOOKS = ["register_forward_hook", "register_forward_pre_hook",
         "register_full_backward_hook", "register_full_backward_pre_hook"]


@pytest.mark.parametrize("hook", HOOKS)
def test_hooked_modules_are_watched(hook):
    layer = linear.Linear(8, 8, bias=False)
    assert linear.bare(layer) and linear.unhooked(layer)
    handle = getattr(layer, hook)(lambda *a: None)
    assert not linear.bare(layer) and not linear.unhooked(layer)
    handle.remove()
    assert linear.bare(layer) and linear.unhooked(layer)


@pytest.mark.parametrize("inner", [False, True])
def test_backward_hook_of_the_feed_forward(inner):
    """On the whole of it, and on its first layer."""
    block = _block(Plain)
    seen = []
    module = block.mlp.gate_up_proj if inner else block.mlp
    module.register_full_backward_hook(
        lambda m, gin, gout: seen.append((gin, gout)))
    x = torch.randn(1, WIDTH, requires_grad=True)
    y, _ = block(x, torch.randn(1, WIDTH), None, None, None)
    y.sum().backward()
    (gin, gout), = seen
    assert [tuple(g.shape) for g in gin] == [(1, WIDTH)]
    assert gout[0].shape == (1, module.weight.shape[0] if inner else WIDTH)


@pytest.mark.parametrize("rows,calls", [(1, 1), (2, 0), (18, 0)])
def test_only_one_row_asks_for_the_norm_inside(monkeypatch, rows, calls):
    """The checks of that call cost small eager batches 5 us a layer."""
    block, seen = _block(Plain), []
    whole = ops.norm_linear
    monkeypatch.setattr(ops, "norm_linear",
                        lambda *a, **k: seen.append(1) or whole(*a, **k))
    with torch.no_grad():
        block(torch.randn(rows, WIDTH), torch.randn(rows, WIDTH), None, None,
              None)
    assert len(seen) == calls
