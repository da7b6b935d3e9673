"""Whether modules may be passed by: a fused pass that reads a module's
parameters instead of calling it would leave out its forward hooks, and a
forward that somebody has put in the place of its class's."""

from __future__ import annotations

from torch.nn.modules import module as _module

_forwards: dict = {}


def passed_by(cls):
    """Marks a class of modules for which fused passes stand in: they do what
    its forward does now."""
    _forwards[cls] = cls.forward
    return cls


def hooked(*modules) -> bool:
    """True where calling one of the modules runs forward hooks, its own
    or those registered for all modules, or another forward than its class
    was written with."""
    if _module._global_forward_hooks or _module._global_forward_pre_hooks:
        return True
    for m in modules:
        cls = type(m)
        if (m._forward_hooks or m._forward_pre_hooks
                or "forward" in m.__dict__
                or cls.forward is not _forwards.get(cls, cls.forward)):
            return True
    return False
