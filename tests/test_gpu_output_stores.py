"""Output rows that are not whole cache lines: larger outputs than the L2s hold are stored another way.  The same rows of a call on
either side of that line, and of the two kinds of width, agree."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# N: whole lines, 16-byte rows, others; M: 16 Mi outputs at most, and more (integer path: short rows, the stream kernel and, whole
# lines only, 256 x 256 tiles; 6-bit floats: 128 x 256 and 256 x 256)
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


# more than 16 Mi outputs of 16-byte rows that are no whole lines in every kind of the prefill kernel's tiles; `part` rows, which are
# compared with them, run smaller ones
@pytest.mark.parametrize("M,N,plan", [(16390, 1032, (128, 128, 0, 0, 0)), (772, 25656, (128, 256, 0, 0, 0)), (1062, 22008, (256, 256, 0, 0, 0)),
                                      (798, 21272, (128, 256, 18688, 128, 128)), (810, 21016, (128, 256, 18688, 64, 128)),
                                      (1323, 16400, (256, 256, 10752, 128, 256)), (1825, 11000, (256, 256, 8192, 192, 128)),
                                      (3027, 6152, (256, 256, 5376, 128, 128)), (11993, 1400, (256, 256, 1280, 64, 128)),
                                      (8200, 16408, (256, 256, 15872, 192, 128))])   # (more than 128 Mi)
def test_prefill_tiles_past_the_line(dev, M, N, plan):
    from duqlinear4bitcuda_amd import _HIP as hip
    K, part = 2112, 130
    print("output stores, prefill tiles", M, N, plan, flush=True)
    assert hip.gemm_plan_for(M, N, K) == plan and M * N > 16 << 20 and hip.gemm_plan_for(part, N, K) != plan
    g = torch.Generator(device=dev).manual_seed(N)
    codes = lambda *shape: torch.randint(0, 256, shape, generator=g, device=dev, dtype=torch.uint8)
    q, w = codes(M, K // 2), codes(N, K // 2)
    sx, sw = (torch.rand(r, generator=g, device=dev).half() / 64 for r in (M, N))
    zx, zw = (torch.randint(0, 15, (r,), generator=g, device=dev).half() for r in (M, N))
    got = hip.linear4bit_forward(hip.EPI_ASYM, q, sx, zx, w, sw, zw)
    for lo in (*range(0, M - part, 4 * part), M - part):
        rows = slice(lo, lo + part)
        want = hip.linear4bit_forward(hip.EPI_ASYM, q[rows], sx[rows], zx[rows], w, sw, zw)
        assert torch.equal(got[rows].view(torch.int16), want.view(torch.int16)), lo


# the same of the 6-bit float path: up to and above 100 Mi outputs, rows that begin at half lines
@pytest.mark.parametrize("M,N", [(2000, 10576), (5300, 20016), (2000, 10592), (900, 20000)])
def test_fp6_past_the_line(dev, M, N):
    from duqlinear4bitcuda_amd import _HIP as hip
    K, part = 640, 130
    print("output stores, 6-bit floats", M, N, flush=True)
    g = torch.Generator(device=dev).manual_seed(N)
    codes = lambda *shape: torch.randint(0, 256, shape, generator=g, device=dev, dtype=torch.uint8)
    q, w = hip.activation_shadow_bf6(codes(M, K // 2)), hip.weight_shadow_bf6(codes(N, K // 2))
    sx, sw = (torch.rand(r, generator=g, device=dev).half() / 64 for r in (M, N))
    got = hip.linear4bit_forward_bf6(hip.EPI_SYM, q, sx, None, w, sw)
    for lo in (*range(0, M - part, 4 * part), M - part):
        rows = slice(lo, lo + part)
        want = hip.linear4bit_forward_bf6(hip.EPI_SYM, q[rows], sx[rows], None, w, sw)
        assert torch.equal(got[rows].view(torch.int16), want.view(torch.int16)), lo


# every kernel that takes batches (rows of up to 256 elements in tiles of 64 and 32 rows, of 640: 64 x 128, of 2048: prefill tiles), rows of
# whole and half lines, of 16-byte pieces and others, on either side of 16 Mi and of 64 Mi outputs in all problems together
@pytest.mark.parametrize("b,M", [(9, 1000), (7, 1000), (300, 30), (35, 1000)])
@pytest.mark.parametrize("N", [2048, 2016, 2008, 1998])
@pytest.mark.parametrize("K", [128, 192, 256, 640, 2048])
def test_batches(dev, b, M, N, K):
    from duqlinear4bitcuda_amd import _HIP as hip
    print("output stores of a batch", b, M, N, K, flush=True)
    g = torch.Generator(device=dev).manual_seed(N + K)
    codes = lambda *shape: torch.randint(0, 256, shape, generator=g, device=dev, dtype=torch.uint8)
    q, w = codes(b, M, K // 2), codes(b, N, K // 2)
    sx, sw = (torch.rand(b, r, generator=g, device=dev).half() / 64 for r in (M, N))
    zx, zw = (torch.randint(0, 15, (b, r), generator=g, device=dev).half() for r in (M, N))
    for mode, z in ((hip.EPI_SYM, (None, None)), (hip.EPI_ASYM, (zx, zw))):
        got = hip.batch_linear4bit_forward(mode, q, sx, z[0], w, sw, z[1])
        for i in sorted({0, 1, b // 2, b - 1}):
            zi = [None if t is None else t[i] for t in z]
            want = hip.linear4bit_forward(mode, q[i], sx[i], zi[0], w[i], sw[i], zi[1])
            assert torch.equal(got[i].view(torch.int16), want.view(torch.int16)), (mode, i)


# one problem of short rows: either side of 16 Mi and of 128 Mi outputs, of 128 and 192 elements
@pytest.mark.parametrize("N,K,M", [(2016, 128, 9000), (2016, 192, 9000), (2008, 192, 9000), (2008, 256, 9000), (2008, 256, 8000), (8200, 256, 16400), (8200, 192, 16400)])
def test_short_rows(dev, N, K, M):
    from duqlinear4bitcuda_amd import _HIP as hip
    print("output stores, short rows", M, N, K, flush=True)
    g = torch.Generator(device=dev).manual_seed(N + K)
    codes = lambda *shape: torch.randint(0, 256, shape, generator=g, device=dev, dtype=torch.uint8)
    q, w = codes(M, K // 2), codes(N, K // 2)
    sx, sw = (torch.rand(r, generator=g, device=dev).half() / 64 for r in (M, N))
    got = hip.linear4bit_forward(hip.EPI_SYM, q, sx, None, w, sw)
    for lo in (0, M // 2 - 65, M - 130):   # (as many rows: outputs that are always streamed)
        part = slice(lo, lo + 130)
        want = hip.linear4bit_forward(hip.EPI_SYM, q[part], sx[part], None, w, sw)
        assert torch.equal(got[part].view(torch.int16), want.view(torch.int16)), lo
