"""The native calls of a quantizer that writes 6-bit float shadows and of the symmetric layer behind it: the same objects and bits
as from the Python code, which takes whatever is more than the plain case."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _pair(dev, dual, bias, K=384, N=96, seed=0, **settings):
    from duqlinear4bitcuda_amd import nn as qnn
    torch.manual_seed(seed)
    lin = torch.nn.Linear(K, N, bias=bias).half().to(dev).requires_grad_(False)
    w = lin.weight.abs()
    s = (w[:, :10].amax(1, keepdim=True) / 7, w[:, 10:].amax(1, keepdim=True) / 7) if dual else (w.amax(1, keepdim=True) / 7,)
    layer = (qnn.Linear4bitDUSQ if dual else qnn.Linear4bitSQ).from_float(lin, *s).to(dev).enable_fp6()
    return qnn.SymQuantizer(**settings), layer


@pytest.mark.parametrize("dual", [False, True])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("rows", [1, 95, 96, 1100])
@pytest.mark.parametrize("shadow", [True, "only", "".join(("on", "ly")), False])
def test_same_as_the_python_code(dev, dual, bias, rows, shadow):
    print("shadow calls", dual, bias, rows, shadow, flush=True)
    quantizer, layer = _pair(dev, dual, bias, input_clip_ratio=0.9, qmax=7, shadow=shadow)
    x = torch.randn(1, rows, 384, device=dev).half()
    for lead in (x, x[0]):
        p = quantizer(lead)
        y = layer(p)
        q = type(quantizer).forward(quantizer, lead)
        want = type(layer).forward(layer, q)
        assert y.shape == want.shape and torch.equal(y, want)
        for name in ("_q", "_s", "shadow_x", "_src", "zeros_x", "rowsum_x", "_staged"):
            a, b = getattr(p, name), getattr(q, name)
            assert (a is None) == (b is None) or name == "_staged"
            if isinstance(a, torch.Tensor):
                assert a.shape == b.shape and torch.equal(a, b)


@pytest.mark.parametrize("dual", [False, True])
def test_what_is_more_than_the_plain_case(dev, dual, monkeypatch):
    from duqlinear4bitcuda_amd import _lib
    quantizer, layer = _pair(dev, dual, False, shadow="only", shadow_min_rows=1)
    x = torch.randn(100, 384, device=dev).half()
    want = layer(quantizer(x))
    # the shadow of the weight follows changes in place, of its memory and of the tensor
    other = layer.weight.flip(0).contiguous()
    for change in (lambda: layer.weight.copy_(other), lambda: setattr(layer.weight, "data", other.flip(0).contiguous()),
                   lambda: layer._buffers.update(weight=other.clone())):
        before = layer(quantizer(x))
        change()
        got = layer(quantizer(x))
        fresh = _pair(dev, dual, False)[1]
        fresh.weight.copy_(layer.weight)
        assert torch.equal(got, type(fresh).forward(fresh, quantizer(x))) and not torch.equal(got, before)
    # a bias that appears later, as a buffer and as a parameter
    bias = torch.ones(96, device=dev, dtype=torch.float16)
    before = layer(quantizer(x))
    for put in (lambda: layer.register_buffer("bias", bias), lambda: layer.register_parameter("bias", torch.nn.Parameter(bias, requires_grad=False))):
        layer.__dict__.pop("bias", None), layer._buffers.pop("bias", None)
        put()
        assert torch.equal(layer(quantizer(x)), before + bias)
    # settings that are refused, and a layer without its shadow
    quantizer.qmax = 9
    with pytest.raises((RuntimeError, ValueError)):
        quantizer(x)
    quantizer.qmax = 6
    layer._buffers["weight_shadow"] = None
    with pytest.raises(AssertionError, match="enable_fp6"):
        layer(quantizer(x))
    # a tracer's functions see the calls
    quantizer, layer = _pair(dev, dual, False, shadow="only", shadow_min_rows=1)
    lib, seen = _lib.load(), []
    for name in ("duq_quantize_rows_sym_bf6", "duq_linear4bit_forward_bf6"):
        real = getattr(lib, name)
        monkeypatch.setattr(lib, name, (lambda *a, _r=real, _n=name: (seen.append(_n), _r(*a))[1]), raising=False)
    assert torch.equal(layer(quantizer(x)), want) and len(seen) == 2


def test_recorded(dev):
    quantizer, layer = _pair(dev, False, True, shadow="only", shadow_min_rows=1)
    x = torch.randn(200, 384, device=dev).half()
    layer(quantizer(x))
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = layer(quantizer(x))
    for i in range(3):
        x.copy_(torch.randn(200, 384, device=dev).half())
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, layer(quantizer(x)))
