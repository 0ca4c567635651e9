"""The modules under ``torch.inference_mode()``, how a server calls them: what is made there are tensors that count no
versions.  Same bits as outside, with layers built outside and inside."""
import pytest
import torch

pytestmark = pytest.mark.gpu
K, N = 256, 96


def models(dev):
    """(model, takes float32) of every kind of layer, the symmetric ones with and without the 6-bit float path."""
    from duqlinear4bitcuda_amd import nn as qnn
    gen = torch.Generator(device=dev).manual_seed(7)
    lin = torch.nn.Linear(K, N, bias=True, device=dev, dtype=torch.float16).requires_grad_(False)
    lin.weight.copy_(torch.randn(N, K, generator=gen, device=dev) * 0.02)
    lin.bias.copy_(torch.randn(N, generator=gen, device=dev))
    w = lin.weight.abs()
    s = (w.amax(1, keepdim=True) / 7,)
    s2 = (w[:, :10].amax(1, keepdim=True) / 7, w[:, 10:].amax(1, keepdim=True) / 7)
    out = [torch.nn.Sequential(qnn.SymQuantizer(0.95), qnn.Linear4bitSQ.from_float(lin, *s).to(dev)),
           torch.nn.Sequential(qnn.SymQuantizer(), qnn.Linear4bitDUSQ.from_float(lin, *s2).to(dev))]
    out += [c.from_linear(lin).to(dev) for c in (qnn.Linear4bitASQ, qnn.LinearQuant4bitDUASQ, qnn.Linear4bitASQRowSum,
                                                 qnn.LinearQuant4bitDUASQRowSum)]
    if not torch.is_inference_mode_enabled():
        for m in (torch.nn.Sequential(qnn.SymQuantizer(shadow="only", shadow_min_rows=65), qnn.Linear4bitSQ.from_float(lin, *s).to(dev)),
                  qnn.Linear4bitASQ.from_linear(lin).to(dev)):
            layer = m[1] if isinstance(m, torch.nn.Sequential) else m
            layer.enable_fp6().fp6_min_tiles = 0
            out.append(m)
    eight = [qnn.LinearQuant8bitASQ.from_linear(lin.float()).to(dev) for _ in range(2)]
    eight[1].fused = False
    return out, eight


@pytest.mark.parametrize("rows", [1, 9, 65, 1025])
def test_inference_mode_gives_the_same_bits(dev, rows):
    from duqlinear4bitcuda_amd import nn as qnn
    x = torch.randn(rows, K, generator=torch.Generator(device=dev).manual_seed(rows), device=dev)
    four, eight = models(dev)
    products = [qnn.SymQuantMatMul(), qnn.AsymQuantMatMul()]
    want = [m(x.half()) for m in four], [m(x) for m in eight], [p(x.half()[None], x.half()[None]) for p in products]
    fresh = models(dev)                            # (no call of them yet)
    with torch.inference_mode():
        for f, e in ((four, eight), fresh, models(dev)):
            for a in (x, x.clone()):
                assert a.is_inference() == (a is not x)
                h = a.half()
                for _ in range(2):
                    got = [m(h) for m in f], [m(a) for m in e], [p(h[None], h[None]) for p in products]
                    for g, w in zip(got, want):
                        assert all(torch.equal(a, b) for a, b in zip(g, w)) and len(g) in (len(w), len(w) - 2)
    for f, e in ((four, eight), fresh):            # and outside again
        assert all(torch.equal(m(x.half()), w) for m, w in zip(f, want[0])) and all(torch.equal(m(x), w) for m, w in zip(e, want[1]))


def test_changes_in_inference_mode_are_seen(dev):
    from duqlinear4bitcuda_amd import nn as qnn
    with torch.inference_mode():
        four, (eight, _) = models(dev)
        x = torch.randn(9, K, device=dev)
        before = eight(x)
        eight.weight.add_(1)                       # (a weight that counts no versions)
        assert not torch.equal(eight(x), before)
        with pytest.raises(AssertionError, match="inference_mode"):
            four[0][1].enable_fp6()
        h = x.half()
        want, p = four[0](h), four[0][0](h)
        h.zero_()                                  # between the quantizer and the layer
        assert torch.equal(four[0][1](p), want)
    four, (eight, _) = models(dev)
    x = torch.randn(9, K, device=dev)
    before = eight(x)
    with torch.inference_mode():
        eight.weight.add_(1)
        assert not torch.equal(eight(x), before)


def test_recorded_in_inference_mode(dev):
    from duqlinear4bitcuda_amd.tools.graphs import GraphedForward
    x = [torch.randn(1, K, device=dev).half() for _ in range(4)]
    model = models(dev)[0][0]
    want = [model(v) for v in x]
    with torch.inference_mode():
        g = GraphedForward(model, x[0].clone())
        for v, w in zip(x, want):
            assert torch.equal(g(v.clone()), w)
    for v, w in zip(x, want):
        assert torch.equal(g(v), w)
