"""Output rows that are not whole cache lines: larger outputs than the L2s hold are stored another way.  The same rows of a call on
either side of that line, and of the two kinds of width, agree."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# N: whole lines, 16-byte rows, others; M: 16 Mi outputs at most, and more, in every kind of tile
@pytest.mark.parametrize("N,fp6", [(8192, False), (8208, False), (8200, False), (8196, False), (2049, False), (8192, True), (8208, True)])
@pytest.mark.parametrize("K", [128, 640])
def test_either_side_of_the_line(dev, N, K, fp6):
    from duqlinear4bitcuda_amd import nn as qnn
    print("output stores", N, K, fp6, flush=True)
    g = torch.Generator(device=dev).manual_seed(N)
    lin = torch.nn.Linear(K, N, device=dev, dtype=torch.float16).requires_grad_(False)
    layer = qnn.Linear4bitSQ.from_float(lin, lin.weight.abs().amax(1, keepdim=True) / 7).to(dev)
    quantizer = qnn.SymQuantizer(shadow="only", shadow_min_rows=1) if fp6 else qnn.SymQuantizer()
    if fp6:
        layer.enable_fp6().fp6_min_tiles = 0
    most = (16 << 20) // N
    x = torch.randn(most + 300, K, generator=g, device=dev).half()
    large = layer(quantizer(x))
    for part in (slice(0, 64), slice(most - 130, most), slice(most + 170, most + 300)):
        assert torch.equal(layer(quantizer(x[part])), large[part])
    assert torch.equal(layer(quantizer(x[:most])), large[:most])
