"""Products of short rows in one launch (csrc/duq_product.hip): rows, columns and runs of tiles that end anywhere, every length of row,
clips and code ranges of either operand, rows of zeros, infinities and NaN; against the oracle, and on larger ones against quantizers and
product as launches of their own."""
import numpy as np
import pytest
import torch

from oracle import duq_oracle as orc

pytestmark = pytest.mark.gpu


def _inputs(n, M, N, K, dev, special):
    g = torch.Generator(device=dev).manual_seed(n + M + N + K)
    a, b = (torch.randn(n, r, K, device=dev, generator=g) * (1 + 3 * torch.rand(n, r, 1, device=dev, generator=g)) for r in (M, N))
    a, b = a.half(), b.half()
    if special:
        for x in (a, b):
            x[0, 0] = 0
            x[0, -1] = 1.5
            x[-1, x.shape[1] // 2, K - 1] = float("inf")
            x[-1, x.shape[1] // 3, 0] = float("nan")
            x[0, x.shape[1] // 2] = 65504
            x[0, x.shape[1] // 2, ::2] = -65504
            x[0, x.shape[1] // 3] = torch.linspace(1000, 1000.5, K, device=dev).half()   # a zero point beyond the packed step's range
    return a, b


def _same(got, want):   # NaNs equal to NaNs
    return torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got.nan_to_num(7, 65500, -65500), want.nan_to_num(7, 65500, -65500))


@pytest.mark.parametrize("n,M,N,K", [(2, 2, 3, 64), (3, 65, 130, 128), (1, 200, 257, 192), (2, 64, 256, 256), (5, 63, 255, 64), (1, 129, 520, 128),
                                     (2, 31, 1000, 256)])
@pytest.mark.parametrize("special", [False, True])
def test_against_the_oracle(dev, n, M, N, K, special):
    from duqlinear4bitcuda_amd.nn import AsymQuantMatMul, SymQuantMatMul
    print("product tiles", n, M, N, K, special, flush=True)
    a, b = _inputs(n, M, N, K, dev, special)
    got_s, got_a = SymQuantMatMul()(a, b), AsymQuantMatMul()(a, b)
    for i in range(n):
        x, w = a[i].cpu().numpy(), b[i].cpu().numpy()
        with np.errstate(all="ignore"):
            sa, sb = orc.sym_scales(x), orc.sym_scales(w)
            want = orc.sym_dequant(orc.matmul_s4(orc.sym_quant(x, sa), orc.sym_quant(w, sb)), sa, sb)
            assert _same(got_s[i].cpu(), torch.from_numpy(np.asarray(want))), i
            (sa, za), (sb, zb) = orc.asym_scales_zeros(x), orc.asym_scales_zeros(w)
            want = orc.asym_dequant(orc.matmul_s4(orc.asym_quant(x, sa, za), orc.asym_quant(w, sb, zb)), sa, za, sb, zb)
            assert _same(got_a[i].cpu(), torch.from_numpy(np.asarray(want))), i


# one tile to many for a workgroup, runs of unequal length, outputs stored in all three ways
@pytest.mark.parametrize("n,M,N,K", [(32, 2048, 2048, 128), (1, 4090, 4090, 64), (12, 1111, 1111, 128), (40, 300, 1990, 192), (8, 2000, 2008, 256),
                                     (3, 5000, 301, 128), (1, 40, 70000, 64), (700, 70, 66, 64), (2, 1000, 2016, 192)])
def test_against_separate_launches(dev, n, M, N, K):
    from duqlinear4bitcuda_amd import _HIP as hip
    from duqlinear4bitcuda_amd.nn import AsymQuantMatMul, SymQuantizer, SymQuantMatMul
    print("product tiles", n, M, N, K, flush=True)
    a, b = _inputs(n, M, N, K, dev, False)
    (qa, sa, za), (qb, sb, zb) = (hip.quantize_rows_asym(x) for x in (a, b))
    assert torch.equal(AsymQuantMatMul()(a, b), hip.batch_linear4bit_forward(hip.EPI_ASYM, qa, sa, za, qb, sb, zb))
    m = SymQuantMatMul()
    m.quantizer_A, m.quantizer_B = SymQuantizer(0.875), SymQuantizer(0.9, qmax=7)
    (qa, sa), (qb, sb) = hip.quantize_rows_sym(a, 0.875, 6), hip.quantize_rows_sym(b, 0.9, 7)
    assert torch.equal(m(a, b), hip.batch_linear4bit_forward(hip.EPI_SYM, qa, sa, None, qb, sb))


@pytest.mark.parametrize("n,M,N,K", [(12, 1100, 2016, 256), (8, 999, 1500, 256)])
def test_many_rows_of_256(dev, n, M, N, K):
    test_against_separate_launches(dev, n, M, N, K)


# one tile and a few, which a recording runs as two launches, and more
@pytest.mark.parametrize("n,M,N,K", [(1, 64, 64, 256), (1, 50, 200, 128), (11, 60, 64, 192), (15, 64, 64, 256), (31, 60, 64, 256), (32, 64, 64, 256), (1, 16, 4096, 128), (8, 300, 300, 128)])
def test_in_a_recording(dev, n, M, N, K):
    from duqlinear4bitcuda_amd.nn import AsymQuantMatMul
    print("product tiles, recorded", n, M, N, K, flush=True)
    f = AsymQuantMatMul()
    a, b = _inputs(n, M, N, K, dev, False)
    f(a, b)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = f(a, b)
    for k in range(4):
        a.mul_(1.25), b.sub_(0.5)
        want = f(a, b)
        graph.replay()
        assert torch.equal(y, want), k
        torch.cuda.synchronize()
