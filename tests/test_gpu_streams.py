"""Layers called on several streams, and while a graph is recorded: the copy of the weight that a first call makes is made
on one of the streams, unknown to the caller."""
import pytest
import torch

pytestmark = pytest.mark.gpu
K, N = 4096, 1024


def layers(dev, seed=1):
    from duqlinear4bitcuda_amd import nn as qnn
    gen = torch.Generator(device=dev).manual_seed(seed)
    lin = torch.nn.Linear(K, N, bias=False, device=dev, dtype=torch.float16).requires_grad_(False)
    lin.weight.copy_(torch.randn(N, K, generator=gen, device=dev) * 0.02)
    x = torch.randn(128, K, generator=gen, device=dev)
    fp6 = qnn.Linear4bitASQ.from_linear(lin).to(dev).enable_fp6()
    fp6.fp6_min_tiles = 0
    return [(qnn.LinearQuant8bitASQ.from_linear(lin.float()).to(dev), x), (fp6, x.half())]


@pytest.mark.parametrize("k", [0, 1], ids=["tiled copy", "6-bit float shadow"])
def test_a_copy_made_on_one_stream_is_read_on_another(dev, k):
    layer, x = layers(dev)[k]
    layer.weight.mul_(1)                                    # (the copy has to be made again)
    fused, layer.fused = layer.fused, False
    want = layer(x)                                         # without any copy
    layer.fused = fused
    one, other = torch.cuda.Stream(dev), torch.cuda.Stream(dev)
    for stream in (one, other):                             # (memory for each stream, so that no call has to wait for it,
        with torch.cuda.stream(stream):                     # with another weight's copy in it)
            warm, y = layers(dev, 2)[k]
            warm.weight.mul_(1)
            warm(y), warm(y), torch.empty(1 << 24, device=dev)
            del warm, y
    torch.cuda.synchronize()
    with torch.cuda.stream(one):
        torch.cuda._sleep(20_000_000)                       # some ms of work in front of what makes the copy
        first = layer(x)
    with torch.cuda.stream(other):
        second = layer(x)
    torch.cuda.synchronize()
    assert torch.equal(second, want) and torch.equal(first, want)


@pytest.mark.parametrize("k", [0, 1], ids=["tiled copy", "6-bit float shadow"])
def test_a_copy_made_while_recording_stays_in_the_recording(dev, k):
    layer, x = layers(dev)[k]
    want = layer(x)
    layer.weight.mul_(1)                                    # (the same values, another version)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        recorded = layer(x)
    assert torch.equal(layer(x), want)                      # before any replay
    for _ in range(3):
        recorded.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded, want) and torch.equal(layer(x), want)
    changed = layer.weight.clone().add_(1)
    layer.weight.copy_(changed)
    now = layer(x)
    assert not torch.equal(now, want)
    graph.replay()                                          # (a recording reads the weight as it is)
    torch.cuda.synchronize()
    assert torch.equal(recorded, now)
