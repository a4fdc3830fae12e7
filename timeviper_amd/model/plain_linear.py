"""When a product on a module's weight and bias is all that calling the module does."""
from __future__ import annotations

import torch
import torch.nn as nn
from torch.nn.modules import module as _module


def unhooked(mod: nn.Module) -> bool:
    """Calling mod runs its class's forward and nothing else: no hooks, of its own or of all modules, and no forward of the object's own
    (what libraries that move or cast weights put in its place)."""
    own = mod.__dict__
    return not (own["_forward_hooks"] or own["_forward_pre_hooks"] or "forward" in own or _module._global_forward_hooks
                or _module._global_forward_pre_hooks)


def plain_linear(mod: nn.Module, x: torch.Tensor) -> bool:
    """Whether the hand-written products may read mod's weight and bias in mod(x)'s place: torch.nn.Linear itself, without hooks, a
    plain tensor as its weight, no autocast, a bias of x's dtype.  What a caller has put around the module sees it called as ever."""
    if type(mod) is not nn.Linear or not unhooked(mod) or torch.is_autocast_enabled():
        return False
    own = mod._parameters                    # (half of this function's time otherwise: nn.Module.__getattr__)
    w, b = own.get("weight"), own.get("bias")
    if (type(w) is not nn.Parameter and type(w) is not torch.Tensor) or "bias" not in own:
        return False
    return b is None or ((type(b) is nn.Parameter or type(b) is torch.Tensor) and b.dtype == x.dtype and b.is_contiguous() and b.data_ptr() % 16 == 0)
