"""Several symmetric layers behind one quantizer, where each call is a quantizer launch and a GEMM launch: the first layer leaves
codes and scales in the packed tensor, the next ones on its stream and in its recording run their GEMM alone.  Same bits as layers
that quantize for themselves."""
import copy
import pickle

import pytest
import torch

pytestmark = pytest.mark.gpu


def _layers(dev, K, outs, seed=0):
    from duqlinear4bitcuda_amd import nn as qnn
    g = torch.Generator(device=dev).manual_seed(seed)
    layers = []
    for i, N in enumerate(outs):
        lin = torch.nn.Linear(K, N, bias=bool(i % 2), dtype=torch.float16).to(dev)
        with torch.no_grad():
            lin.weight.copy_(torch.randn(N, K, generator=g, device=dev) * 0.02)
        s = lin.weight.detach().abs().amax(-1, keepdim=True) / 7
        layers.append((qnn.Linear4bitSQ.from_float(lin, s) if i != 1 else qnn.Linear4bitDUSQ.from_float(lin, s, s)).to(dev))
    return layers


def _alone(layers, quantizer, x):
    return [m(quantizer(x)) for m in layers]


def _equal(got, want):
    for a, b in zip(got, want):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


# eight rows and sixteen short ones are one launch, with nothing to leave
@pytest.mark.parametrize("M,K,shares", [(8, 512, False), (16, 512, False), (17, 512, True), (9, 8192, True), (77, 1088, True), (1024, 512, True),
                                        (1025, 512, False)])
def test_same_bits(dev, M, K, shares):
    from duqlinear4bitcuda_amd import nn as qnn
    layers, q = _layers(dev, K, (320, 513, 64)), qnn.SymQuantizer(0.9, 7)
    for rep in range(2):   # (the first calls of a layer prepare it)
        x = torch.randn(M, K, device=dev, dtype=torch.float16)
        want = _alone(layers, q, x)
        p = q(x)
        got = [layers[0](p)]
        left = p._staged
        got += [m(p) for m in layers[1:]]
        assert p._staged is left
        if rep:
            assert (left is not None) == shares
        _equal(got, want)
    _equal([m(p) for m in layers], want)   # read by something else in between
    codes, scales = p.quantized_x, p.scales_x
    assert p._staged is None
    _equal([m(p) for m in layers], want)
    assert codes.shape == (M, K // 2) and scales.numel() == M


def test_other_streams_and_recordings_quantize_for_themselves(dev):
    from duqlinear4bitcuda_amd import nn as qnn
    layers, q = _layers(dev, 1024, (256, 384)), qnn.SymQuantizer()
    x = torch.randn(40, 1024, device=dev, dtype=torch.float16)
    want = _alone(layers, q, x)
    p = q(x)
    _equal([m(p) for m in layers], want)
    first, side = p._staged, torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = layers[1](p)
        assert p._staged is not first
    torch.cuda.current_stream().wait_stream(side)
    _equal([y], want[1:])
    static, graph = x.clone(), torch.cuda.CUDAGraph()
    p = q(static)
    _equal([layers[0](p)], want[:1])
    outside = p._staged
    with torch.cuda.graph(graph):
        out = [m(p) for m in layers]
        inside = p._staged
    assert inside is not outside
    _equal([m(p) for m in layers], want)      # (nothing of the recording has run)
    for seed in range(3):
        x2 = torch.randn(40, 1024, device=dev, dtype=torch.float16)
        want2 = _alone(layers, q, x2)
        static.copy_(x2)
        graph.replay()
        torch.cuda.synchronize()
        _equal(out, want2)


def test_rows_that_change_are_refused_and_copies_go_without(dev):
    from duqlinear4bitcuda_amd import nn as qnn
    layers, q = _layers(dev, 512, (128, 256)), qnn.SymQuantizer()
    x = torch.randn(33, 512, device=dev, dtype=torch.float16)
    want = _alone(layers, q, x)
    p = q(x)
    layers[0](p)
    for other in (copy.deepcopy(p), pickle.loads(pickle.dumps(p))):
        assert other._staged is None
        assert torch.equal(other._src, x)
    _equal([copy.copy(p) and layers[1](copy.copy(p))], want[1:])
    x.add_(1)
    with pytest.raises(RuntimeError, match="modified in place"):
        layers[1](p)


@pytest.mark.parametrize("rounds", [1, 2])   # (2: the second rows may come to lie where the first ones were)
def test_rows_given_other_memory_are_quantized(dev, rounds):
    """An assignment to .data between two layers keeps the tensor's version: the second layer takes the rows that are there now."""
    from duqlinear4bitcuda_amd import nn as qnn
    layers, q = _layers(dev, 512, (128, 256)), qnn.SymQuantizer()
    x = torch.randn(33, 512, device=dev, dtype=torch.float16)
    _alone(layers, q, x)
    p = q(x)
    layers[0](p)
    for _ in range(rounds):
        x.data = torch.randn(33, 512, device=dev, dtype=torch.float16)
    want = _alone(layers, q, x.clone())
    _equal([layers[1](p)], want[1:])
    _equal([m(p) for m in layers], want)
    codes, scales = tuple(t.clone() for t in (p.quantized_x, p.scales_x))
    other = q(x.clone())
    assert torch.equal(codes, other.quantized_x) and torch.equal(scales, other.scales_x)
