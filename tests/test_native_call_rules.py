"""When the native ``__call__`` of the module classes (csrc/duq_host.cpp) may stand for a module's call, and what comes next
where it may not.  Each case has a process of its own: what counts is what was put in place BEFORE the first call of the
package, which loads the native module."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# every kind of class; x runs through none of them on the CPU, where the ops refuse it: what is looked at is who was called
HEAD = """
import functools, torch
seen = []
def wrapped(real):
    @functools.wraps(real)
    def f(*a, **k):
        seen.append(f)
        return real(*a, **k)
    return f
def modules():
    from duqlinear4bitcuda_amd import nn as qnn
    lin = torch.nn.Linear(128, 64)
    sq = qnn.Linear4bitSQ(128, 64)
    four = [c(128, 64) for c in (qnn.Linear4bitDUSQ, qnn.Linear4bitASQ, qnn.LinearQuant4bitDUASQ, qnn.Linear4bitASQRowSum,
                                 qnn.LinearQuant4bitDUASQRowSum, qnn.LinearQuant8bitASQ)]
    return [qnn.SymQuantizer(), sq, *four, qnn.SymQuantMatMul(), qnn.AsymQuantMatMul()]
def call(m):
    x = torch.zeros(2, 128, dtype=torch.float16)
    try:
        m(x, x) if hasattr(m, "quantizer_B") else m(x)
    except (RuntimeError, AssertionError):
        pass
def plain():
    from duqlinear4bitcuda_amd import _lib
    return [_lib.host().plain_call(m) for m in modules()]
"""

CASES = {
    "nothing replaced": "assert all(plain()), plain()",
    "forward of the classes": """
from duqlinear4bitcuda_amd import nn as qnn
mods = modules()
for m in mods:
    type(m).forward = wrapped(type(m).forward)
qnn.AsymQuantizer.forward = wrapped(qnn.AsymQuantizer.forward)
assert not any(plain())
from duqlinear4bitcuda_amd import _lib
assert not _lib.host().plain_call(qnn.AsymQuantizer())
for m in mods:
    seen.clear()
    call(m)
    assert seen and seen[0] is type(m).forward, type(m)
""",
    "__call__ of the classes": """
mods = modules()
calls = {type(m): wrapped(torch.nn.Module.__call__) for m in mods}
for cls, f in calls.items():
    cls.__call__ = f
assert not any(plain())
for m in mods:
    seen.clear()
    call(m)
    assert type(m).__call__ is calls[type(m)] and seen and seen[0] is calls[type(m)], type(m)
""",
    "torch's call before the import": """
real, put = torch.nn.Module.__call__, wrapped(torch.nn.Module.__call__)
torch.nn.Module.__call__ = put
assert not any(plain())
for m in modules():
    seen.clear()
    call(m)
    assert seen and seen[0] is put
torch.nn.Module.__call__ = real
""",
    "torch's _call_impl before the first call": """
mods = modules()
put = torch.nn.Module._call_impl = wrapped(torch.nn.Module._call_impl)
assert not any(plain())
for m in mods:
    seen.clear()
    call(m)
    assert seen and seen[0] is put
""",
    "tracing, hooks of every module, hooks of an instance": """
plain()
from duqlinear4bitcuda_amd import _lib
for m in modules():
    seen.clear()
    torch.jit.trace(lambda x: (seen.append(_lib.host().plain_call(m)), x + 1)[1], torch.zeros(2), check_trace=False)
    assert seen == [False] and _lib.host().plain_call(m)
    for register in (torch.nn.modules.module.register_module_forward_hook, torch.nn.modules.module.register_module_forward_pre_hook,
                     torch.nn.modules.module.register_module_full_backward_hook,
                     torch.nn.modules.module.register_module_full_backward_pre_hook, m.register_forward_hook,
                     m.register_forward_pre_hook, m.register_full_backward_hook, m.register_full_backward_pre_hook):
        handle = register(lambda *a: None)
        assert not _lib.host().plain_call(m), register
        handle.remove()
        assert _lib.host().plain_call(m)
""",
}


def run(body):
    r = subprocess.run([sys.executable, "-c", HEAD + body], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("what", CASES)
def test_what_was_replaced_before_the_first_call_is_called(what):
    run(CASES[what])


# put in place before or after the first call: what a call does must not depend on that
METHOD_ORDER = {
    "a class behind in the method order": """
class Mixin(torch.nn.Module):
    def __call__(self, *a, **k):
        seen.append("mixin")
        return super().__call__(*a, **k)
for m in modules():
    cls = type(m)
    sub = type("Sub", (cls, Mixin), {})
    s = sub(128, 64) if hasattr(m, "in_features") else sub()
    seen.clear()
    call(s)
    assert seen == ["mixin"], (cls, seen)
""",
    "a base class": """
from duqlinear4bitcuda_amd.nn.linear import _Linear4bitBase as base
base.__call__ = wrapped(torch.nn.Module.__call__)
for m in modules():
    below = isinstance(m, base)
    seen.clear()
    call(m)
    assert (seen == [base.__call__]) == below and (first or host.plain_call(m) != below), type(m)
del base.__call__
base._call_impl = wrapped(torch.nn.Module._call_impl)
for m in modules():
    below = isinstance(m, base)
    seen.clear()
    call(m)
    assert (seen == [base._call_impl]) == below and (first or host.plain_call(m) != below), type(m)
del base._call_impl
""",
    "an instance": """
for m in modules():
    m._call_impl = wrapped(m._call_impl)
    seen.clear()
    call(m)
    assert seen == [m._call_impl] and (first or not host.plain_call(m)), type(m)
    del m._call_impl
    m.compile(backend=lambda g, x: g)
    assert first or not host.plain_call(m)
""",
    "a callable that is no function": """
class Next:
    def __call__(self, *a, **k):
        seen.append(a)
class Binds:
    def __get__(self, obj, cls):
        return lambda *a, **k: seen.append((obj, *a))
for behind in (Next(), Binds(), staticmethod(lambda *a, **k: seen.append(a))):
    Mixin = type("Mixin", (torch.nn.Module,), {"__call__": behind})
    for m in modules():
        sub = type("Sub", (type(m), Mixin), {})
        s = sub(128, 64) if hasattr(m, "in_features") else sub()
        seen.clear()
        s(5)
        assert seen == [(s, 5)] if isinstance(behind, Binds) else seen == [(5,)], (type(m), behind)
""",
    "calls through the class": """
import inspect
for m in modules():
    cls = type(m)
    for bad in ((), (5,)):
        try:
            cls.__call__(*bad)
        except (TypeError, AttributeError):
            pass
        else:
            raise AssertionError(bad)
    other = torch.nn.Identity()
    assert cls.__call__(other, 3) == 3 and cls.__call__(other, input=4) == 4
    assert str(inspect.signature(cls.__call__)) == "(self, *args, **kwargs)" and str(inspect.signature(m)) == "(*args, **kwargs)"
    assert cls.__call__.__name__ in ("__call__", "_wrapped_call_impl")
""",
}


@pytest.mark.parametrize("first", (True, False), ids=("before the first call", "after it"))
@pytest.mark.parametrize("what", METHOD_ORDER)
def test_the_next_call_in_the_method_order(what, first):
    loaded = "" if first else "from duqlinear4bitcuda_amd import _lib\nhost = _lib.host()\n"
    run(f"first = {first}\n" + loaded + METHOD_ORDER[what])
