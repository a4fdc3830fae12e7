"""When a product on a module's weight and bias is all that calling the module does."""
from __future__ import annotations

import torch
import torch.nn as nn


def unhooked(mod: nn.Module) -> bool:
    """Calling mod runs its class's forward and nothing else."""
    return not mod._forward_hooks and not mod._forward_pre_hooks


def plain_linear(mod: nn.Module, x: torch.Tensor) -> bool:
    """Whether the hand-written products may read mod's weight and bias in mod(x)'s place: torch.nn.Linear itself, without hooks, no
    autocast, a bias of x's dtype.  What a caller has put around the module sees it called as ever."""
    return (type(mod) is nn.Linear and unhooked(mod) and not torch.is_autocast_enabled()
            and (mod.bias is None or (mod.bias.dtype == x.dtype and mod.bias.is_contiguous() and mod.bias.data_ptr() % 16 == 0)))
