"""When a product on a module's weight and bias is all that calling the module does."""
from __future__ import annotations

import torch
import torch.nn as nn
from torch.nn.modules import module as _module


def unhooked(mod: nn.Module) -> bool:
    """Calling mod runs its class's forward and nothing else: no hooks, of its own or of all modules, and no forward of the object's own
    (what libraries that move or cast weights put in its place)."""
    return not (mod._forward_hooks or mod._forward_pre_hooks or _module._global_forward_hooks or _module._global_forward_pre_hooks
                or "forward" in mod.__dict__)


def plain_linear(mod: nn.Module, x: torch.Tensor) -> bool:
    """Whether the hand-written products may read mod's weight and bias in mod(x)'s place: torch.nn.Linear itself, without hooks, a
    plain tensor as its weight, no autocast, a bias of x's dtype.  What a caller has put around the module sees it called as ever."""
    own = lambda t: type(t) in (nn.Parameter, torch.Tensor)
    return (type(mod) is nn.Linear and unhooked(mod) and own(mod.weight) and not torch.is_autocast_enabled()
            and (mod.bias is None or (own(mod.bias) and mod.bias.dtype == x.dtype and mod.bias.is_contiguous() and mod.bias.data_ptr() % 16 == 0)))
