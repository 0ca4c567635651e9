"""Layers on their way to the GPU: through pinned memory where torch's own move is asked for, the same buffers either way."""
import pytest
import torch

from duqlinear4bitcuda_amd import nn as qnn
from duqlinear4bitcuda_amd.nn import linear as impl


def _layer(bias=True, n=1500, k=2048):
    torch.manual_seed(n)
    return qnn.Linear4bitASQ.from_linear(torch.nn.Linear(k, n, bias=bias).half())


def test_what_counts_as_a_move():
    seen = []

    class Probe(torch.nn.Module):
        def _apply(self, fn, recurse=True):
            seen.append(impl._is_move(fn))
            return self

    p = Probe()
    p.to("cpu"), p.to(torch.float16), p.cuda(), p.half(), p.share_memory()
    p._apply(lambda t: t)
    assert seen == [True, True, True, False, False, False]


def test_other_functions_see_the_buffers_themselves():
    m = _layer()
    before = {k: t for k, t in m.state_dict(keep_vars=True).items()}
    seen = []
    m._apply(lambda t: (seen.append(id(t)), t)[1])
    assert set(seen) == {id(t) for t in before.values()}
    assert m.to("cpu") is m and all(m.state_dict(keep_vars=True)[k] is t for k, t in before.items())


@pytest.mark.gpu
@pytest.mark.parametrize("stage", [1 << 24, 1 << 20, 768 * 256])
def test_moves(dev, stage, monkeypatch):
    """One piece, several, and pieces that end inside a buffer."""
    monkeypatch.setattr(impl, "_STAGE_BYTES", stage)
    want = {k: t.clone() for k, t in _layer().state_dict().items()}
    for move in (lambda m: m.to(dev), lambda m: m.cuda(), lambda m: torch.nn.Sequential(m, torch.nn.ReLU()).to("cuda")[0],
                 lambda m: m.to(dev, non_blocking=True)):
        m = move(_layer())
        assert all(t.device == dev for t in m.state_dict().values())
        assert all(torch.equal(t.cpu(), want[k]) and t.dtype == want[k].dtype for k, t in m.state_dict().items())
    m = _layer().to(dev, torch.float32)   # (the codes stay bytes, floats are cast)
    assert m.weight.dtype == torch.uint8 and m.bias.dtype == torch.float32 and m.weight.is_cuda and m.bias.is_cuda
    assert torch.equal(m.weight.cpu(), want["weight"]) and torch.equal(m.bias.cpu(), want["bias"].float())
    m = _layer().to(dev).to("cpu")
    assert torch.equal(m.weight, want["weight"])
    tied = _layer()
    tied.register_buffer("again", tied.weight, persistent=False)
    tied.to(dev)
    assert tied.again is tied.weight or torch.equal(tied.again, tied.weight)
    with torch.inference_mode():
        m = _layer()
        assert torch.equal(m.to(dev).weight.cpu(), want["weight"])


def test_a_default_device_is_not_asked():
    """Where a move leads is told by a host tensor, whatever device a caller has made the default one."""
    t, seen = torch.zeros(4, 8), []
    with torch.device("meta"):
        assert impl._fetch([t], lambda t: (seen.append(t.device.type), t)[1]) == {}
    assert seen == ["cpu"]


@pytest.mark.gpu
@pytest.mark.parametrize("stage", [1 << 24, 768 * 256])
def test_moves_under_a_default_device(dev, stage, monkeypatch):
    """The device of the pinned buffers and of the probe is named: under torch.device("cuda") and set_default_device layers
    move as they do without, and a cast of a layer on the host stays there."""
    monkeypatch.setattr(impl, "_STAGE_BYTES", stage)
    want = {k: t.clone() for k, t in _layer().state_dict().items()}
    same = lambda m: all(torch.equal(t.cpu(), want[k]) for k, t in m.state_dict().items())

    def check():
        for move in (lambda m: m.to("cuda"), lambda m: m.cuda()):
            m = move(hosts.pop())
            assert all(t.is_cuda for t in m.state_dict().values()) and same(m)
        m = hosts.pop().to(torch.float16)
        assert all(t.device.type == "cpu" for t in m.state_dict().values()) and same(m)
        back = [torch.empty_like(t) for t in want.values()]   # (device results into host tensors, as a conversion stores them)
        impl._store(*((d, t.to(dev)) for d, t in zip(back, want.values())))
        assert all(not d.is_cuda and torch.equal(d, t) for d, t in zip(back, want.values()))

    hosts = [_layer() for _ in range(6)]
    with torch.device("cuda"):
        check()
    torch.set_default_device("cuda")
    try:
        check()
    finally:
        torch.set_default_device(None)
