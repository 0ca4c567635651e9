"""The native host module (csrc/duq_host.cpp): it answers None for what it does not take, and where it does, the bits are
those of the Python code that stands behind it."""
import pytest
import torch


def test_declines_what_is_not_the_plain_case():
    from duqlinear4bitcuda_amd import _lib

    host = _lib.host()
    x = torch.zeros(2, 128, dtype=torch.float16)                       # on the CPU
    assert host.defer(x, 1024, False, 96, 1.0, 6) is None and host.defer(None, 1024, False, 96, 1.0, 6) is None
    assert host.quantize_rows(x, 0, True, False, 1.0, 6, 0) is None
    assert host.linear4(0, x, x, None, x, x, None, None, None, None, None, None, False, 0) is None
    assert host.linear4_batched(0, x, x, None, x, x, None, None, None, None, 0) is None
    assert host.linear8(x, None, None, x, None, x, x, None, 2, 0) is None and host.quantize_rows_8bit(x, 0) is None
    w = torch.zeros(4, 64, dtype=torch.uint8)
    call = host.FusedCall(0, 4, 128, 0, 1024, (w.data_ptr(),) + (None,) * 7, ("weight",), (w,))
    assert call.take({"weight": w}, x) is None and call.take_rows({"weight": w}, x) is None
    with pytest.raises(ValueError):
        host.FusedCall(0, 4, 128, 0, 1024, (None,), ("weight",), (w,))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 9, 65, 1025])
def test_native_and_python_host_code_give_the_same_bits(dev, monkeypatch, rows):
    """The same module steps once natively and once with every library function replaced by a Python one."""
    from duqlinear4bitcuda_amd import _lib
    from duqlinear4bitcuda_amd import nn as qnn

    K, N = 256, 96
    gen = torch.Generator().manual_seed(rows)
    lin = torch.nn.Linear(K, N, bias=True).half().to(dev).requires_grad_(False)
    sw = lin.weight.abs().amax(1, keepdim=True) / 7
    x = torch.randn(rows, K, generator=gen).half().to(dev)
    b = torch.randn(3, 17, K, generator=gen).half().to(dev)

    def steps():
        sq = torch.nn.Sequential(qnn.SymQuantizer(0.95), qnn.Linear4bitSQ.from_float(lin, sw).to(dev))
        fp6 = torch.nn.Sequential(qnn.SymQuantizer(shadow="only", shadow_min_rows=1), qnn.Linear4bitSQ.from_float(lin, sw).to(dev).enable_fp6())
        fp6[1].fp6_min_tiles = 0
        mods = [sq, fp6] + [c.from_linear(lin).to(dev) for c in (qnn.Linear4bitASQ, qnn.Linear4bitASQRowSum, qnn.LinearQuant4bitDUASQRowSum)]
        out = [m(x) for m in mods for _ in range(2)]
        l8 = qnn.LinearQuant8bitASQ.from_linear(lin.float()).to(dev)
        lin.half()
        for tiled in (True, False):
            l8.tiled = tiled
            out.append(l8(x.float()))
        return out + [qnn.SymQuantMatMul()(b, b), qnn.AsymQuantMatMul()(b, b)]

    native = steps()
    lib, calls = _lib.load(), []
    for name in _lib.PROTOTYPES:
        if not name.endswith("_bytes"):
            real = getattr(lib, name)
            monkeypatch.setattr(lib, name, (lambda *a, _r=real, _n=name: (calls.append(_n), _r(*a))[1]), raising=False)
    python = steps()
    assert len(calls) >= len(python) and len(python) == len(native)
    for p, n in zip(python, native):
        assert p.dtype == n.dtype and p.shape == n.shape and torch.equal(p, n)


BROKEN = {
    "missing": "_lib.HOST_PATH = '/nonexistent/_duq_host.so'",
    "another torch": "torch.__version__ = torch.torch_version.TorchVersion('2.99.0+x')",
}


@pytest.mark.parametrize("what", BROKEN)
def test_the_package_runs_without_the_native_module(what):
    """Without it the calls reach the Python code behind them (here: its refusal of tensors on the CPU), after one warning."""
    import os
    import subprocess
    import sys
    code = f"""
import warnings, torch
from duqlinear4bitcuda_amd import _HIP, _lib, nn as qnn
{BROKEN[what]}
x = torch.zeros(2, 128, dtype=torch.float16)
mods = [qnn.SymQuantizer(), qnn.Linear4bitASQ(128, 64), qnn.SymQuantMatMul(), qnn.AsymQuantMatMul()]
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    for m in mods:
        try:
            m(x, x) if hasattr(m, "quantizer_B") else m(x)
        except RuntimeError as e:
            assert "to be on a GPU device" in str(e), e
        else:
            raise AssertionError(m)
seen = [w for w in seen if "_duq_host" in str(w.message)]
assert len(seen) == 1 and seen[0].category is RuntimeWarning, seen
assert _lib.host() is None and _HIP._host_for("duq_linear4bit_forward") is None
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", code], cwd=root, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.gpu
def test_prepared_calls_without_the_native_module(dev, monkeypatch):
    from duqlinear4bitcuda_amd import _lib
    from duqlinear4bitcuda_amd import nn as qnn
    lin = torch.nn.Linear(256, 96).half().to(dev).requires_grad_(False)
    x = torch.randn(5, 256, device=dev).half()
    want = qnn.Linear4bitASQ.from_linear(lin).to(dev)(x)
    monkeypatch.setattr(_lib, "host", lambda: None)
    layer = qnn.Linear4bitASQ.from_linear(lin).to(dev)
    for _ in range(2):
        assert torch.equal(layer(x), want) and layer._decode.native is None


def test_first_calls_from_several_threads():
    """The library and the native module are loaded once, whoever comes first."""
    import os
    import subprocess
    import sys
    code = """
import sys, threading
sys.setswitchinterval(1e-6)
from duqlinear4bitcuda_amd import _lib, nn
start, got, errors = threading.Barrier(8), [], []
def first():
    start.wait()
    try:
        got.append((_lib.host(), _lib.load()))
    except BaseException as e:
        errors.append(e)
threads = [threading.Thread(target=first) for _ in range(8)]
[t.start() for t in threads]
[t.join() for t in threads]
assert not errors, errors
assert len(got) == 8 and len({id(h) for h, _ in got}) == 1 and len({id(lib) for _, lib in got}) == 1
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    for _ in range(3):
        r = subprocess.run([sys.executable, "-c", code], cwd=root, capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("called", [False, pytest.param(True, marks=pytest.mark.gpu)])
def test_a_layer_with_a_prepared_call_is_copied_and_saved(called):
    """The prepared call holds addresses of this process and stays behind: a copy prepares its own."""
    import copy
    import io

    from duqlinear4bitcuda_amd import _lib
    from duqlinear4bitcuda_amd import nn as qnn
    lin = torch.nn.Linear(256, 96).half().requires_grad_(False)
    sq = qnn.Linear4bitSQ.from_float(lin, lin.weight.abs().amax(1, keepdim=True) / 7)
    for layer, model in ((sq, torch.nn.Sequential(qnn.SymQuantizer(), sq)), (a := qnn.Linear4bitASQ.from_linear(lin), a)):
        if called:
            model.to("cuda:0")
            x = torch.randn(3, 256, device="cuda:0").half()
            want = model(x)
            assert layer._decode is not None
        else:
            layer._decode = _lib.load()
        file = io.BytesIO()
        torch.save(model, file)
        file.seek(0)
        for other in (copy.deepcopy(model), torch.load(file, weights_only=False)):
            new = other[1] if isinstance(other, torch.nn.Sequential) else other
            assert new._decode is None and layer._decode is not None
            assert torch.equal(new.weight, layer.weight) and new.weight.data_ptr() != layer.weight.data_ptr()
            if called:
                assert torch.equal(other(x), want)
                new.weight.zero_()
                assert not torch.equal(other(x), want) and torch.equal(model(x), want)


@pytest.mark.parametrize("what", ["weight_tiled", "weight_shadow"])
def test_copies_of_a_weight_made_by_two_threads_at_once(monkeypatch, what):
    """A thread that is behind with the copy of an older weight must not leave it in the place of the newer one."""
    import threading

    from duqlinear4bitcuda_amd import nn as qnn
    from duqlinear4bitcuda_amd.nn import linear
    monkeypatch.setattr(linear.tensor_utils, "weight_tile_8bit", lambda w: w.clone())
    monkeypatch.setattr(linear.tensor_utils, "weight_shadow", lambda w: w.clone())
    if what == "weight_tiled":
        layer = qnn.LinearQuant8bitASQ(128, 64)
        make = layer._tiled_weight
    else:
        layer = qnn.Linear4bitASQ(128, 64)
        monkeypatch.setattr(torch.Tensor, "is_cuda", True)
        layer.enable_fp6()
        make = layer._fp6_ready
    layer.weight.fill_(1)
    real, older_made, newer_put, older_done = layer.register_buffer, threading.Event(), threading.Event(), threading.Event()

    def put(name, t, persistent):
        if threading.current_thread() is older:
            older_made.set()
            newer_put.wait(1)
        real(name, t, persistent=persistent)
        if threading.current_thread() is newer:
            newer_put.set()
            older_done.wait(1)

    def first():
        make()
        older_done.set()

    older, newer = threading.Thread(target=first), threading.Thread(target=make)
    layer.register_buffer = put
    older.start()
    older_made.wait()
    layer.weight.fill_(2)
    newer.start()
    older.join()
    newer.join()
    make()
    assert (layer._buffers[what] == 2).all()
