"""Where a linear layer may leave torch's product for the kernel over few rows:
never where something of torch's has to see the product."""

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from sutro_amd import ops
from sutro_amd.models import linear as L
from sutro_amd.models.qwen3 import Qwen3MLP
from sutro_amd.parallel.tp import TPContext


class _Kernels:
    """Stands in for the extension: counts the calls that reach it."""

    def __init__(self):
        self.calls = 0

    def linear_skinny(self, x, w, bias, gated):
        self.calls += 1
        y = F.linear(x, w, bias)
        if gated:
            a, b = y.chunk(2, -1)
            y = F.silu(a) * b
        return y


@pytest.fixture
def kernels(monkeypatch):
    k = _Kernels()
    monkeypatch.setattr(ops, "_use_hip", lambda t: True)
    monkeypatch.setattr(ops, "_require_hip", lambda: k)
    return k


def _operands(rows=4, n=8, k=32):
    g = torch.Generator().manual_seed(1)
    return (torch.randn(rows, k, generator=g).bfloat16(),
            torch.randn(n, k, generator=g).bfloat16())


def test_plain_call_takes_the_kernel(kernels):
    x, w = _operands()
    with torch.no_grad():
        ops.linear(x, w)
    assert kernels.calls == 1


def test_gradients(kernels):
    x, w = _operands()
    w.requires_grad_()
    ops.linear(x, w).sum().backward()
    assert kernels.calls == 0 and w.grad is not None


def test_forward_mode(kernels):
    x, w = _operands()
    t = torch.ones_like(x)
    with torch.no_grad(), forward_ad.dual_level():
        y = ops.linear(forward_ad.make_dual(x, t), w)
        tangent = forward_ad.unpack_dual(y).tangent
    assert kernels.calls == 0
    torch.testing.assert_close(tangent, F.linear(t, w))


def test_vmap(kernels):
    x, w = _operands()
    xs = torch.stack([x, 2 * x])
    with torch.no_grad():
        y = torch.func.vmap(lambda v: ops.linear(v, w))(xs)
    assert kernels.calls == 0
    torch.testing.assert_close(y, F.linear(xs, w))


def test_modes_see_the_product(kernels):
    x, w = _operands()
    seen = []

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with torch.no_grad():
        with Functions():
            ops.linear(x, w)
        assert "linear" in seen
        del seen[:]
        with Dispatch():
            ops.linear(x, w)
        assert seen
    assert kernels.calls == 0


def test_trace(kernels):
    x, w = _operands()
    with torch.no_grad():
        f = torch.jit.trace(lambda v: ops.linear(v, w), (x,),
                            check_trace=False)
        assert kernels.calls == 0
        torch.testing.assert_close(f(3 * x), F.linear(3 * x, w))


def test_autocast(kernels):
    x, w = _operands()
    with torch.no_grad(), torch.autocast("cpu", dtype=torch.float16):
        y = ops.linear(x, w)
    assert kernels.calls == 0 and y.dtype == torch.float16


def test_hooks_on_every_module():
    mlp = Qwen3MLP(32, 16, torch.bfloat16, TPContext())
    called = []
    handles = [
        nn.modules.module.register_module_forward_hook(
            lambda m, a, y: called.append(m)),
        nn.modules.module.register_module_forward_pre_hook(
            lambda m, a: called.append(m))]
    try:
        assert not L.bare(mlp.gate_up_proj)
        with torch.no_grad():
            mlp(torch.zeros(2, 32, dtype=torch.bfloat16))
        assert called.count(mlp.gate_up_proj) == 2
    finally:
        for h in handles:
            h.remove()
    assert L.bare(mlp.gate_up_proj)


@pytest.mark.parametrize("rows,k,n,gated,kernel", [
    (1, 5120, 5120, False, 1), (2, 5120, 5120, False, 0),
    (2, 4096, 6144, False, 1), (2, 4096, 8192, False, 0),
    (2, 5120, 10240, False, 1), (2, 16384, 4096, False, 1),
    (2, 8192, 6144, True, 1), (2, 8192, 12288, True, 0)])
def test_one_and_two_rows(kernels, rows, k, n, gated, kernel):
    """Two rows over matrices where the library is the faster one."""
    w = torch.empty(n, k, dtype=torch.bfloat16)      # (never read)
    assert ops._few_rows(torch.empty(rows, k, dtype=torch.bfloat16), w,
                         gated) == bool(kernel)


@pytest.mark.parametrize("rows,k,n,kernel", [
    (3, 25600, 5120, 1), (32, 25600, 2048, 1), (17, 25600, 1024, 0),
    (32, 17408, 128, 0), (16, 25600, 64, 1), (8, 17408, 32, 0),
    (3, 25600, 16, 0)])
def test_long_rows_of_few(kernels, rows, k, n, kernel):
    """Long rows of weights, but so few that the library is ahead: 64 x 25600 at
    32 rows 41 us by it and 67 by the kernel, at 16 rows 53 and 45."""
    w = torch.empty(n, k, dtype=torch.bfloat16)      # (never read)
    assert ops._few_rows(torch.empty(rows, k, dtype=torch.bfloat16),
                         w) == bool(kernel)


@pytest.mark.parametrize("rows,k,n,kernel", [
    (274, 2048, 50688, 0), (363, 5120, 52992, 0), (512, 2048, 50688, 1),
    (1027, 4096, 42496, 0), (1280, 4096, 42496, 1), (775, 512, 46336, 1),
    (300, 1024, 34816, 0), (2048, 1024, 8192, 1), (2047, 1024, 7936, 0)])
def test_gated_layers_of_many_rows(kernels, rows, k, n, kernel):
    """A row tile with few rows in it counts by its rows."""
    x = torch.empty(rows, k, dtype=torch.bfloat16)
    w = torch.empty(n, k, dtype=torch.bfloat16)      # (never read)
    assert ops._many_rows(x, w) == bool(kernel)


@pytest.mark.parametrize("k,n,inside", [
    (128, 12288, 1), (128, 35296, 0), (640, 16384, 0), (672, 65536, 1),
    (2048, 65536, 1), (2048, 131072, 0), (4096, 24576, 1), (4128, 4096, 0)])
def test_norm_in_front_of_one_row(kernels, k, n, inside):
    """Many short rows of weights: the norm has a launch of its own."""
    def bf(*shape):
        return torch.empty(*shape, dtype=torch.bfloat16)
    assert ops._one_row(bf(1, k), bf(1, k), bf(k), bf(n, k),
                        False) == bool(inside)


@pytest.mark.parametrize("rows,k,n,kernel", [
    (16, 4096, 20480, 1), (16, 4096, 20720, 0), (8, 4096, 20720, 1),
    (8, 4096, 14336, 0), (6, 4096, 14336, 1), (8, 4096, 40960, 1),
    (8, 4096, 59344, 0), (6, 4096, 59344, 1), (8, 4096, 65536, 1),
    (5, 4096, 113184, 0), (6, 2048, 151936, 1), (8, 2048, 59424, 0)])
def test_larger_matrices(kernels, rows, k, n, kernel):
    """Where the library has a good tile, or the last round of workgroups leaves
    CUs idle, for as many rows as the kernel is still ahead."""
    w = torch.empty(n, k, dtype=torch.bfloat16)      # (never read)
    assert ops._few_rows(torch.empty(rows, k, dtype=torch.bfloat16),
                         w) == bool(kernel)


class _Names(_Kernels):
    """The same, with the name of the kernel instead of its result."""

    def linear_skinny(self, x, w, bias, gated):
        return "few"

    def linear_mid(self, x, w, bias, gated):
        return "mid"


@pytest.mark.parametrize("rows,k,n,kernel", [
    # the sizes above
    (16, 4096, 20480, "mid"), (16, 4096, 20720, "mid"), (8, 4096, 20720, "mid"),
    (8, 4096, 14336, "mid"), (6, 4096, 14336, "mid"), (8, 4096, 40960, "mid"),
    (8, 4096, 59344, "mid"), (6, 4096, 59344, "mid"), (8, 4096, 65536, "mid"),
    (5, 4096, 113184, "mid"), (6, 2048, 151936, "mid"), (8, 2048, 59424, "mid"),
    (2, 5120, 10240, "few"), (2, 4096, 6144, "mid"), (3, 25600, 5120, "few"),
    (32, 25600, 2048, "few"), (32, 17408, 128, "lib"), (16, 25600, 64, "few"),
    # where the first kernel is not ahead, and a k that it does not take
    (8, 4096, 66560, "lib"), (6, 4096, 66560, "lib"), (4, 4096, 66560, "few"),
    (8, 2048, 4080, "few"), (8, 4096, 4096, "few"), (32, 4096, 32, "lib"),
    (12, 4064, 4096, "few"), (13, 4064, 4096, "few"), (13, 4064, 8192, "lib"),
    (8, 1600, 59424, "lib"), (8, 2016, 20000, "few"), (8, 2016, 151936, "lib"),
    (33, 4064, 4096, "lib"), (33, 4096, 4096, "mid"), (257, 4096, 4096, "lib")])
def test_the_kernel_that_is_called(monkeypatch, rows, k, n, kernel):
    """Both rules one behind the other, as ops.linear asks them."""
    monkeypatch.setattr(ops, "_use_hip", lambda t: True)
    monkeypatch.setattr(ops, "_require_hip", _Names)
    monkeypatch.setattr(F, "linear", lambda x, w, bias=None: "lib")
    with torch.no_grad():
        assert ops.linear(torch.empty(rows, k, dtype=torch.bfloat16),
                          torch.empty(n, k, dtype=torch.bfloat16)) == kernel
