"""The native ``__call__`` of the module classes (csrc/duq_host.cpp): same bits as torch.nn.Module.__call__ with the
class's forward, which it leaves to torch wherever a call is more than that."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,M,N,K", [((1,), 1, 1, 64), ((3,), 1, 65, 64), ((2, 3), 7, 33, 128), ((5,), 129, 64, 512),
                                         ((2,), 31, 130, 576), ((1,), 1, 257, 4160), ((9,), 400, 300, 192), ((2,), 3, 5, 16448)],
                         ids=str)
def test_products_of_activations_in_one_call(dev, monkeypatch, batch, M, N, K):
    """Both operands quantized by one launch (rows of both kinds of row kernel, in and beyond the register cache) against
    the module's separate steps, and settings of the two quantizers that differ."""
    from duqlinear4bitcuda_amd import _HIP as ops
    from duqlinear4bitcuda_amd import nn as qnn
    print("product", batch, M, N, K, flush=True)
    g = torch.Generator(device=dev).manual_seed(N)
    a, b = (torch.randn(*batch, r, K, generator=g, device=dev).half() for r in (M, N))
    asym, sym, other = qnn.AsymQuantMatMul(), qnn.SymQuantMatMul(), qnn.SymQuantMatMul()
    other.quantizer_A.input_clip_ratio, other.quantizer_B.qmax = 0.8, 7
    calls = ((asym, a, b), (sym, a, b), (other, a, b), (sym, a, b.view(-1, K)[:N].contiguous()))
    asym(a, b)
    steps = []
    real = ops._launch
    with monkeypatch.context() as m:
        m.setattr(ops, "_launch", lambda *x: (steps.append(x[1]), real(*x))[1])
        got = [f(x, y) for f, x, y in calls]
        assert len(steps) == 3 * len(calls)
    for (f, x, y), want in zip(calls, got):
        out = f(x, y)
        assert out.shape == want.shape and torch.equal(out, want)


def test_calls_that_are_more_than_the_forward(dev, monkeypatch):
    from duqlinear4bitcuda_amd import nn as qnn
    K, N = 256, 96
    lin = torch.nn.Linear(K, N).half().to(dev).requires_grad_(False)
    sw = lin.weight.abs().amax(1, keepdim=True) / 7
    x = torch.randn(5, K, device=dev).half()
    l8 = qnn.LinearQuant8bitASQ.from_linear(lin.float()).to(dev)
    lin.half()
    pairs = [(torch.nn.Sequential(qnn.SymQuantizer(), qnn.Linear4bitSQ.from_float(lin, sw).to(dev)), (x,)),
             (qnn.Linear4bitASQ.from_linear(lin).to(dev), (x,)), (l8, (x.float(),)),
             (qnn.SymQuantMatMul(), (x, x)), (qnn.AsymQuantMatMul(), (x[None], x[None]))]
    for mod, args in pairs:
        inner = list(mod) if isinstance(mod, torch.nn.Sequential) else [mod]
        mod(*args)
        want = mod(*args)
        seen = []
        for m in inner:                                      # hooks of the instance
            handle = m.register_forward_hook(lambda *a: seen.append(a))
            assert torch.equal(mod(*args), want) and len(seen) == 1
            handle.remove()
            seen.clear()
        handle = torch.nn.modules.module.register_module_forward_pre_hook(lambda *a: seen.append(a))   # of every module
        assert torch.equal(mod(*args), want) and len(seen) >= len(inner)
        handle.remove()
        seen.clear()
        for m in inner:                                      # a replaced forward, of the class and of the instance
            real = type(m).forward
            with monkeypatch.context() as c:
                c.setattr(type(m), "forward", lambda self, *a: (seen.append(1), real(self, *a))[1])
                assert torch.equal(mod(*args), want) and seen == [1]
            seen.clear()
            m.forward = lambda *a, _m=m, _r=real: (seen.append(1), _r(_m, *a))[1]
            assert torch.equal(mod(*args), want) and seen == [1]
            del m.forward
            seen.clear()
        assert torch.equal(mod(*args), want) and not seen
    # the copy of an 8-bit weight follows changes in place; a layer's prepared call follows its buffers
    before = l8(x.float())
    l8.weight.add_(1)
    assert not torch.equal(l8(x.float()), before)
    l8.weight.sub_(1)
    assert torch.equal(l8(x.float()), before)
    sq = pairs[0][0]
    before = sq(x)
    sq[1].weight_scales = sq[1].weight_scales * 2
    assert not torch.equal(sq(x), before)
    # operands that do not fit raise what the steps raise
    with pytest.raises(RuntimeError, match="same leading dimensions"):
        qnn.SymQuantMatMul()(torch.zeros(2, 4, K, device=dev).half(), torch.zeros(3, 4, K, device=dev).half())
    with pytest.raises(AssertionError, match="Batch dimensions"):
        qnn.AsymQuantMatMul()(torch.zeros(2, 4, K, device=dev).half(), torch.zeros(3, 4, K, device=dev).half())


def test_tensors_without_memory_of_their_own(dev):
    """What has no address (a vmap wrapper, a sparse tensor) is refused with a Python error by modules and ops, as by the Python
    code that the native calls stand for."""
    from duqlinear4bitcuda_amd import _HIP as hip, nn as qnn
    x = torch.randn(3, 4, 128, device=dev).half()
    lin = torch.nn.Linear(128, 64, bias=False, device=dev, dtype=torch.float16)
    with torch.device(dev):
        layer = qnn.Linear4bitASQ.from_linear(lin)
    layer = layer.to(dev)
    product = qnn.AsymQuantMatMul()
    layer(x[0]), product(x, x)   # (the plain case, prepared)
    refused = (RuntimeError, ValueError, TypeError, NotImplementedError)
    for f in (layer, hip.quantize_rows_sym, lambda v: product(v, v)):
        with pytest.raises(refused):
            torch.func.vmap(lambda v: (f(v), v)[1])(x)
        with pytest.raises(refused):
            f(x[0].to_sparse())


def test_eight_bit_call_holds_its_tensors(dev):
    """What the layer's buffers held when a call was made lives until the library has returned, whoever replaces it meanwhile:
    looked at from inside the call, at the status of a copy of the weight that the library refuses unlaunched (misaligned)."""
    import weakref

    from duqlinear4bitcuda_amd import _lib, nn as qnn
    from duqlinear4bitcuda_amd.tools.tensor_utils import PackedQuantizedTensor
    K, N = 256, 96
    layer = qnn.LinearQuant8bitASQ.from_linear(torch.nn.Linear(K, N)).to(dev)
    x = torch.randn(8, K, device=dev)
    want = layer(x)
    copy = layer._buffers["weight_tiled"]
    layer._buffers["weight_tiled"] = torch.empty(copy.numel() + 1, dtype=copy.dtype, device=dev)[1:]
    names = ("weight_tiled", "weight_scales", "weight_zeros", "bias")
    saved = {n: layer._buffers[n].clone() for n in names[1:]}
    there = []

    class Refused(Exception):
        pass

    def status(code, name):
        refs = [weakref.ref(layer._buffers.pop(n)) for n in names]
        there.extend(r() is not None for r in refs)
        raise Refused(name)

    host = _lib.host()
    host.setup(PackedQuantizedTensor, status)
    try:
        with pytest.raises(Refused, match="quantize_linear8bit_forward"):
            layer(x)
    finally:
        host.setup(PackedQuantizedTensor, _lib.check)
    assert there == [True] * 4
    layer._buffers.update(saved, weight_tiled=copy)
    assert torch.equal(layer(x), want)


def test_quantizer_settings_replaced_by_a_finalizer(dev):
    """The object that hands the rows on is allocated with the settings in hand; the garbage collector may run there."""
    import gc

    from duqlinear4bitcuda_amd import nn as qnn
    q = qnn.SymQuantizer(float("0.75"))
    x = torch.randn(2, 256, device=dev).half()
    q(x)
    there = []

    def replaced(phase, info):
        q.input_clip_ratio = float("0.5")
        there.append([float(i) for i in range(1000)])   # (what was freed is in use again)

    before = gc.get_threshold()
    gc.callbacks.append(replaced)
    gc.set_threshold(1)
    try:
        for _ in range(20):
            q.input_clip_ratio = float("0.75")
            p = q(x)
            assert p._clip in (0.5, 0.75)
    finally:
        gc.set_threshold(*before)
        gc.callbacks.remove(replaced)
    assert there


@pytest.mark.parametrize("native", [True, False])
def test_buffers_given_other_memory(dev, monkeypatch, native):
    """An assignment to a buffer's .data leaves the tensor and changes its memory: the prepared call must not keep the old."""
    from duqlinear4bitcuda_amd import _lib, nn as qnn
    if not native:
        monkeypatch.setattr(_lib, "host", lambda: None)
    gen = torch.Generator(device=dev).manual_seed(3)
    lin = torch.nn.Linear(256, 96, bias=True, device=dev, dtype=torch.float16).requires_grad_(False)
    x = torch.randn(5, 256, generator=gen, device=dev).half()
    for cls in (qnn.Linear4bitASQ, qnn.LinearQuant4bitDUASQ, qnn.Linear4bitASQRowSum, qnn.LinearQuant4bitDUASQRowSum):
        layer, fresh = (cls.from_linear(lin).to(dev) for _ in range(2))
        layer(x)
        assert (layer._decode.native is not None) == native
        for name, buf in layer._buffers.items():
            before = layer(x)
            other = torch.flip(buf, (0,)) if name == "weight" else buf + 1
            buf.data = other.clone()
            fresh._buffers[name] = other
            got = layer(x)
            fresh._decode = None
            same, changed = torch.equal(got, fresh(x)), not torch.equal(got, before)
            assert same and changed, (cls, name)


@pytest.mark.parametrize("most", [10 ** 30, 2 ** 62, -10 ** 30, 0])
def test_settings_of_any_size(dev, most):
    """Row counts that a C integer does not hold, or whose product with the row length it does not, and layers of no columns."""
    from duqlinear4bitcuda_amd import nn as qnn
    K, N = 256, 96
    lin = torch.nn.Linear(K, N).half().to(dev).requires_grad_(False)
    x = torch.randn(70, K, device=dev).half()
    sq = torch.nn.Sequential(qnn.SymQuantizer(), qnn.Linear4bitSQ.from_float(lin, lin.weight.abs().amax(1, keepdim=True) / 7).to(dev))
    asq = qnn.Linear4bitASQ.from_linear(lin).to(dev)
    l8 = qnn.LinearQuant8bitASQ.from_linear(lin.float()).to(dev)
    want = [sq(x), asq(x), l8(x.float())]
    sq[0].defer_rows = most
    assert (sq[0](x)._src is not None) == (most > 0)
    asq.enable_fp6().fp6_min_tiles = most
    l8.one_call_rows = most
    for _ in range(2):
        assert all(torch.equal(m(a), w) for m, a, w in zip((sq, asq, l8), (x, x, x.float()), want))
    sq[0].shadow, sq[0].shadow_min_rows = True, most
    assert torch.equal(sq(x), want[0])
    empty = qnn.LinearQuant8bitASQ(0, 8).to(dev)
    with pytest.raises((RuntimeError, IndexError, ZeroDivisionError)):
        empty(torch.zeros(3, 0, device=dev))
