"""Products with one row of A: one launch that quantizes the rows of B and multiplies them at once, against the
separate steps (quantizers, int32 GEMM, dequantization), same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# every class of lengths, the first length beyond; rows of B that fill no workgroup, and that take two per group of lanes
@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("batch,N,K", [(3, 65, 64), (2, 31, 128), (1, 257, 192), (40, 1, 256), (1, 33000, 256), (3, 5501, 320), (2, 17, 512), (5, 3, 576),
                                       (1, 130, 1024), (2, 9, 1088), (1, 33, 2048), (3, 5, 2112), (40, 205, 4096), (1, 4, 4160)], ids=str)
def test_against_the_steps(dev, M, batch, N, K):
    from duqlinear4bitcuda_amd import nn as qnn
    print("product of few rows", M, batch, N, K, flush=True)
    g = torch.Generator(device=dev).manual_seed(N + K)
    a, b = (torch.randn(batch, r, K, generator=g, device=dev).half() * 3 for r in (M, N))
    b[0, 0] = 0
    b[-1, -1, 0] = 60000
    if N > 8:
        b[0, 3, 5], b[0, 4, 6], b[0, 5] = float("inf"), float("nan"), -0.25
        b[0, 6] = 2.0 ** -24
    asym, sym, other = qnn.AsymQuantMatMul(), qnn.SymQuantMatMul(), qnn.SymQuantMatMul()
    other.quantizer_A.input_clip_ratio, other.quantizer_B.qmax = 0.8, 7
    for f in (asym, sym, other):
        got = f(a, b)
        f.fused = False
        want = f(a, b)
        assert got.shape == want.shape == (batch, M, N)
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(1.0), want.nan_to_num(1.0))


def test_more_products_than_a_grid_dimension(dev):
    from duqlinear4bitcuda_amd import nn as qnn
    g = torch.Generator(device=dev).manual_seed(1)
    a, b = (torch.randn(65537, r, 64, generator=g, device=dev).half() for r in (1, 2))
    f = qnn.AsymQuantMatMul()
    got = f(a, b)
    assert torch.equal(got[-3:], f(a[-3:].contiguous(), b[-3:].contiguous())) and torch.equal(got[:5], f(a[:5], b[:5]))
