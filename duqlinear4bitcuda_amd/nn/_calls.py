"""What the native ``__call__`` of the module classes (``csrc/duq_host.cpp``) stands for.

It runs a call past ``torch.nn.Module.__call__`` and the class's ``forward`` only where these are the functions they
were written as.  Which functions those are is taken down here, where a class is defined and where this package is
imported, and not when the native module is loaded at the first call: a function that a program put in their place
before that (with ``functools.wraps`` it looks like the original in every attribute) is a replaced function too.
"""
from __future__ import annotations

from torch.nn.modules import module as _module

# in the order of `enum Kind` in csrc/duq_host.cpp; LOOKED_AT: no call of its own, only part of a product's
KINDS = ("sym_quantizer", "sym_layer", "own_layer", "eight_bit", "sym_product", "asym_product")
LOOKED_AT = "looked_at"

classes = []   # (class, number of its kind or -1, its forward)


def native_call(kind):
    """Class decorator: calls of that class may be run natively, as that kind, while its forward is the one it has now."""
    number = -1 if kind == LOOKED_AT else KINDS.index(kind)

    def register(cls):
        classes.append((cls, number, cls.__dict__["forward"]))
        return cls
    return register


def _torchs_own(name):
    """The function of that name of torch.nn.Module, None where another one had been put in its place (``__globals__`` is what
    no wrapper can take over)."""
    f = _module.Module.__dict__.get(name)
    return f if getattr(f, "__globals__", None) is vars(_module) else None


module_call, module_call_impl = _torchs_own("__call__"), _torchs_own("_call_impl")
