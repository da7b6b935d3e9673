"""Whether modules may be passed by: a fused pass that reads a module's
parameters instead of calling it would leave out its forward hooks."""

from __future__ import annotations

from torch.nn.modules import module as _module


def hooked(*modules) -> bool:
    """True where calling one of the modules runs forward hooks, its own
    or those registered for all modules."""
    if _module._global_forward_hooks or _module._global_forward_pre_hooks:
        return True
    for m in modules:
        if m._forward_hooks or m._forward_pre_hooks:
            return True
    return False
