"""The row quantizers on short rows (several rows per wavefront up to 512 elements): lane-group and pass remainders,
rows that need the element-wise path beside ordinary ones in one wavefront."""
import numpy as np
import pytest
import torch

from oracle import duq_oracle as orc
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K", [(1, 32), (63, 64), (130, 96), (33, 128), (67, 160), (17, 256), (21, 288), (9, 480), (300, 512), (5, 544),
                                 (131100, 64), (65700, 96), (33001, 256), (16389, 512)])
def test_quantize_short_rows(dev, M, K):
    from duqlinear4bitcuda_amd import _HIP as hip
    print("short rows", M, K, flush=True)
    x = cases.acts_normal(M, K, seed=M + K)
    if M > 8:
        x[1] = 0
        x[2, 5] = np.nan
        x[3, 7] = np.inf
        x[4] = np.float16(1.5)
        x[5] = x[5] * 0.01 + np.float16(900.0)
        x[M - 1, 0] = np.float16(-60000)
    X = cases.t(x, dev)
    with np.errstate(invalid="ignore", over="ignore", divide="ignore"):
        for qmax, clip in ((6, 1.0), (7, 0.6)):
            s_want = orc.sym_scales(x, clip)
            q, s = hip.quantize_rows_sym(X, clip=clip, qmax=qmax)
            assert cases.bits_equal(s.cpu().numpy(), s_want) and np.array_equal(q.cpu().numpy(), orc.sym_quant(x, s_want, qmax))
        s_want, z_want = orc.asym_scales_zeros(x)
        q, s, z = hip.quantize_rows_asym(X)
        assert cases.bits_equal(s.cpu().numpy(), s_want) and cases.bits_equal(z.cpu().numpy(), z_want)
        assert np.array_equal(q.cpu().numpy(), orc.asym_quant(x, s_want, z_want))
        want = orc.asym_quant_shifted(x)
        got = [t.cpu().numpy() for t in hip.quantize_rows_asym_shifted(X)]
        assert np.array_equal(got[0], want[0]) and cases.bits_equal(got[1], want[1]) and cases.bits_equal(got[2], want[2])
        assert np.array_equal(got[3].reshape(-1), want[3].reshape(-1))


@pytest.mark.parametrize("K", [64, 128, 192, 256])
def test_products_of_extreme_codes(dev, K):
    """Short rows, whose accumulators start at a float's bits: sums at both ends of their range (every code -8, and -8 against
    7) and around zero, through the four epilogues that read them so, against the stand-alone ones on int32."""
    from duqlinear4bitcuda_amd import _HIP as hip
    M, N = 70, 300
    a = torch.randint(0, 256, (M, K // 2), dtype=torch.uint8, device=dev)
    b = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, device=dev)
    a[:20], a[20:40], b[:99], b[99:180] = 0x88, 0x77, 0x88, 0x77
    acc = hip.matmul(a, b)
    assert int(acc.max()) == 64 * K and int(acc.min()) == -56 * K
    h = lambda n: (torch.rand(n, device=dev) * 4 - 2).half()
    sr, zr, s1, z1, s2, z2, bias = h(M), h(M).round(), h(N), h(N).round(), h(N), h(N).round(), h(N)
    steps = ((hip.EPI_SYM, (sr, None), (s1, None, None, None), hip.sym_dequant(acc, sr, s1)),
             (hip.EPI_ASYM, (sr, zr), (s1, z1, None, None), hip.asym_dequant(acc, sr, zr, s1, z1)),
             (hip.EPI_SYM_DUAL, (sr, None), (s1, None, s2, None), hip.sym_dual_dequant(acc, sr, s1, s2)),
             (hip.EPI_ASYM_DUAL, (sr, zr), (s1, z1, s2, z2), hip.asym_dual_dequant(acc, sr, zr, s1, z1, s2, z2)))
    for mode, r, c, y in steps:
        for add in (None, bias):
            got = hip.batch_linear4bit_forward(mode, a[None], *(t if t is None else t[None] for t in r), b[None],
                                               *(t if t is None else t[None] for t in c), bias=None if add is None else add[None])
            want = y if add is None else y + add
            assert torch.equal(got[0].view(torch.int16), want.view(torch.int16)), (mode, add is None)
