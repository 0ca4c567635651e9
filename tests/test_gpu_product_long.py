"""Products of long rows with few columns (csrc/duq_product_long.hip): every length of row that a lane's share changes at, rows and columns
that end anywhere in a tile, clips and code ranges of either operand, rows of zeros, infinities and NaN; against the oracle, and all of it
against quantizers and product as launches of their own."""
import numpy as np
import pytest
import torch

from oracle import duq_oracle as orc

pytestmark = pytest.mark.gpu


def _inputs(n, M, N, K, dev, special=False):
    g = torch.Generator(device=dev).manual_seed(n + M + N + K)
    a = torch.softmax(2 * torch.randn(n, M, K, device=dev, generator=g), -1).half()
    b = torch.randn(n, N, K, device=dev, generator=g).half()
    if special:
        for x in (a, b):
            x[0, 0] = 0
            x[0, -1] = 1.5
            x[-1, x.shape[1] // 2, K - 1] = float("inf")
            x[-1, x.shape[1] // 3, 0] = float("nan")
            x[1, x.shape[1] // 2] = 65504
            x[1, x.shape[1] // 2, ::2] = -65504
            x[1, x.shape[1] // 3] = torch.linspace(1000, 1000.5, K, device=dev).half()   # a zero point beyond the packed step's range
    return a, b


def _same(got, want):   # NaNs equal to NaNs
    return torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got.nan_to_num(7, 65500, -65500), want.nan_to_num(7, 65500, -65500))


def _separate(a, b, sym):
    from duqlinear4bitcuda_amd import _HIP as hip
    if sym:
        (qa, sa), (qb, sb) = hip.quantize_rows_sym(a, 0.875, 6), hip.quantize_rows_sym(b, 0.9, 7)
        return hip.batch_linear4bit_forward(hip.EPI_SYM, qa, sa, None, qb, sb)
    (qa, sa, za), (qb, sb, zb) = (hip.quantize_rows_asym(x) for x in (a, b))
    return hip.batch_linear4bit_forward(hip.EPI_ASYM, qa, sa, za, qb, sb, zb)


@pytest.mark.parametrize("n,M,N,K", [(32, 33, 1, 320), (33, 50, 31, 512), (32, 64, 33, 576), (22, 95, 64, 1024), (17, 127, 65, 1088), (16, 129, 128, 1536),
                                     (16, 513, 129, 1600), (8, 1030, 255, 2048), (33, 1000, 200, 2112), (64, 64, 32, 3072), (64, 80, 40, 3136), (32, 150, 72, 4096)])
@pytest.mark.parametrize("special", [False, True])
def test_against_the_oracle_and_separate_launches(dev, n, M, N, K, special):
    from duqlinear4bitcuda_amd.nn import AsymQuantMatMul, SymQuantizer, SymQuantMatMul
    print("long product", n, M, N, K, special, flush=True)
    a, b = _inputs(n, M, N, K, dev, special)
    m = SymQuantMatMul()
    m.quantizer_A, m.quantizer_B = SymQuantizer(0.875), SymQuantizer(0.9, qmax=7)
    got_a, got_s, default = AsymQuantMatMul()(a, b), m(a, b), SymQuantMatMul()(a, b)
    assert _same(got_a, _separate(a, b, False))
    assert _same(got_s, _separate(a, b, True))
    for i in (0, 1, n - 1):
        x, w = a[i].cpu().numpy(), b[i].cpu().numpy()
        with np.errstate(all="ignore"):
            sa, sb = orc.sym_scales(x), orc.sym_scales(w)
            want = orc.sym_dequant(orc.matmul_s4(orc.sym_quant(x, sa), orc.sym_quant(w, sb)), sa, sb)
            assert _same(default[i].cpu(), torch.from_numpy(np.asarray(want))), i
            (sa, za), (sb, zb) = orc.asym_scales_zeros(x), orc.asym_scales_zeros(w)
            want = orc.asym_dequant(orc.matmul_s4(orc.asym_quant(x, sa, za), orc.asym_quant(w, sb, zb)), sa, za, sb, zb)
            assert _same(got_a[i].cpu(), torch.from_numpy(np.asarray(want))), i


# large ones, and what lies on either side of the rule
@pytest.mark.parametrize("n,M,N,K", [(32, 2039, 128, 2048), (40, 1021, 64, 1024), (8, 4096, 256, 4096), (8, 4090, 256, 2176), (1, 4090, 64, 4096),
                                     (2, 992, 64, 512), (8, 255, 256, 2048), (8, 256, 257, 512), (4, 1000, 128, 4160), (63, 32, 16, 448), (700, 32, 7, 320)])
def test_against_separate_launches(dev, n, M, N, K):
    from duqlinear4bitcuda_amd.nn import AsymQuantMatMul
    print("long product", n, M, N, K, flush=True)
    a, b = _inputs(n, M, N, K, dev)
    assert torch.equal(AsymQuantMatMul()(a, b), _separate(a, b, False))


def test_in_a_recording(dev):
    from duqlinear4bitcuda_amd.nn import AsymQuantMatMul
    print("long product, recorded", flush=True)
    f = AsymQuantMatMul()
    a, b = _inputs(8, 300, 80, 704, dev)
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
