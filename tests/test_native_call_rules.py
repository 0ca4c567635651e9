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
        m(x, x) if "MatMul" in type(m).__name__ else m(x)
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
}


def run(body):
    r = subprocess.run([sys.executable, "-c", HEAD + body], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("what", CASES)
def test_what_was_replaced_before_the_first_call_is_called(what):
    run(CASES[what])
