"""The decoders' linear layer: torch's, with the product of ops.linear."""

from __future__ import annotations

import torch
import torch.nn as nn
from torch.nn.modules import module

from .. import ops


class Linear(nn.Linear):
    def forward(self, input: torch.Tensor) -> torch.Tensor:
        return ops.linear(input, self.weight, self.bias)


def unhooked(block: nn.Module) -> bool:
    """Whether nothing sees what goes into a module and comes out of it (or
    their gradients) but the module: no hooks, its own or every module's, and
    no forward of the object's own."""
    return (not block._forward_hooks and not block._forward_pre_hooks
            and not block._backward_hooks and not block._backward_pre_hooks
            and not module._has_any_global_hook()
            and "forward" not in block.__dict__)


def bare(layer: nn.Module) -> bool:
    """Whether a caller may fuse this layer's product with what follows it: a
    Linear without bias that nothing watches."""
    return type(layer) is Linear and layer.bias is None and unhooked(layer)
