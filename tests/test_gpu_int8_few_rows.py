"""The 8-bit layer on up to eight rows (quantizer inside the GEMM's launch) and its row quantizer: rows of every kind, lengths
that end inside a wavefront's share, both weight layouts."""
import numpy as np
import pytest
import torch

from oracle import duq_oracle as orc
from tests import cases

pytestmark = pytest.mark.gpu


def _rows(M, K, seed):
    """Ordinary rows, and in the first places of larger sets those that leave the quick path: zeros, a constant, a NaN, an
    infinity, a row far off zero for its spread, tiny and huge values."""
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal((M, K)) * rng.uniform(0.1, 30, (M, 1))).astype(np.float32)
    with np.errstate(over="ignore"):
        odd = (x[0] * 0, x[0] * 0 + 3.25, np.where(np.arange(K) == K - 1, np.nan, x[0]), np.where(np.arange(K) == K // 2, np.inf, x[0]),
               x[0] + np.float32(1e5), x[0] * np.float32(1e-38), x[0] * np.float32(1e36),
               (np.arange(K) % 128 / 2 - 31.75).astype(np.float32))   # quotients half way between integers
    for i in range(min(M - 1, len(odd))):
        x[i + 1] = odd[(i + seed) % len(odd)]
    return x.astype(np.float32)


@pytest.mark.parametrize("M,K", [(9, 4), (9, 252), (9, 260), (12, 1024), (12, 1028), (9, 4096), (9, 11008), (9, 16384), (9, 16388), (9, 32768),
                                 (9, 32772)])
def test_row_quantizer(dev, M, K):
    from duqlinear4bitcuda_amd import _HIP as hip
    print("8-bit rows", M, K, flush=True)
    x = _rows(M, K, 1)
    with np.errstate(all="ignore"):
        s_want, z_want = orc.asym8_scales_zeros(x, device_division=True)
        q_want = orc.asym_quant_8bit(x, s_want, z_want)
    q, s, z = hip.quantize_rows_asym_8bit(torch.from_numpy(x).to(dev))
    assert np.array_equal(s.cpu().numpy().reshape(-1), s_want.reshape(-1), equal_nan=True)
    assert np.array_equal(z.cpu().numpy().reshape(-1), z_want.reshape(-1), equal_nan=True)
    assert np.array_equal(q.cpu().numpy(), q_want)


@pytest.mark.parametrize("M,N,K", [(1, 1, 32), (1, 40, 4096), (2, 17, 64), (2, 4100, 2048), (3, 33, 2080), (4, 300, 1056), (5, 16, 96),
                                   (7, 4113, 4064), (8, 4096, 4096), (8, 129, 2048), (8, 70, 32), (6, 9000, 512)])
def test_quantizer_inside_the_gemm(dev, M, N, K):
    """The same bits as the two launches, whose kernels the oracle tests cover."""
    from duqlinear4bitcuda_amd import _HIP as hip
    print("8-bit few rows", M, N, K, flush=True)
    gen = torch.Generator(device=dev).manual_seed(M * 31 + K)
    w = torch.randint(0, 128, (N, K), generator=gen, device=dev, dtype=torch.int8)
    sw = torch.rand(N, generator=gen, device=dev) * 0.01
    zw = torch.randint(0, 127, (N,), generator=gen, device=dev).float()
    bias = torch.randn(N, generator=gen, device=dev)
    tiled = hip.weight_tile_8bit(w)
    for seed in (0, 3, 6):
        x = torch.from_numpy(_rows(M, K, seed)).to(dev)
        q, s, z = hip.quantize_rows_asym_8bit(x)
        for b in (None, bias):
            want = hip.linear8bit_forward(q, s, z, w, sw, zw, b)
            for t in (None, tiled):
                got = hip.quantize_linear8bit_forward(x, w, t, sw, zw, b)
                assert torch.equal(got.view(torch.int32), want.view(torch.int32)), (seed, b is None, t is None)


@pytest.mark.parametrize("M", [1, 3, 4])
def test_a_misaligned_copy_is_not_read(dev, M):
    """Up to four rows with both weights take the weight as stored where the tiled copy is not 16-byte aligned (a buffer of
    zeros here, which would show); more rows, which have to read the copy, are refused."""
    from duqlinear4bitcuda_amd import _HIP as hip
    from duqlinear4bitcuda_amd import _lib
    print("8-bit misaligned copy", M, flush=True)
    lib, (N, K) = _lib.load(), (96, 256)
    gen = torch.Generator(device=dev).manual_seed(M)
    w = torch.randint(1, 128, (N, K), generator=gen, device=dev, dtype=torch.int8)
    sw, zw = torch.rand(N, generator=gen, device=dev), torch.randint(0, 127, (N,), generator=gen, device=dev).float()
    x = torch.randn(8, K, generator=gen, device=dev)
    y = torch.empty(8, N, device=dev)
    copy = torch.zeros(N * K + 16, device=dev, dtype=torch.int8)[4:]
    ws = torch.empty(lib.duq_quantize_linear8bit_workspace_bytes(8, K), device=dev, dtype=torch.uint8)
    call = lambda m, copy: lib.duq_quantize_linear8bit_forward(
        x.data_ptr(), w.data_ptr(), copy.data_ptr(), sw.data_ptr(), zw.data_ptr(), None, m, N, K, y.data_ptr(), ws.data_ptr(),
        ws.numel(), torch.cuda.current_stream().cuda_stream)
    assert call(M, copy) == 0
    want = hip.quantize_linear8bit_forward(x[:M], w, None, sw, zw)
    assert torch.equal(y[:M].view(torch.int32), want.view(torch.int32))
    assert call(8, copy) == -5


@pytest.mark.parametrize("M,N,K", [(129, 2561, 64), (257, 2303, 96), (130, 5122, 64), (65, 4095, 1536), (70, 131, 1536), (640, 515, 64),
                                   (8200, 2050, 32)])
def test_ragged_columns_of_the_tiles(dev, M, N, K):
    """Prefill-sized tiles whose rows end inside a group of four columns: every output against torch, none past the end."""
    from duqlinear4bitcuda_amd import _HIP as hip
    print("8-bit ragged", M, N, K, flush=True)
    gen = torch.Generator(device=dev).manual_seed(N)
    a = torch.randint(-128, 128, (M, K), generator=gen, device=dev, dtype=torch.int8)
    w = torch.randint(-128, 128, (N, K), generator=gen, device=dev, dtype=torch.int8)
    want = (a.double() @ w.double().T).to(torch.int32)   # (exact: |sum| < 2^53)
    acc = hip.matmul_8bit(a, w)
    assert torch.equal(acc, want)
    sx, zx = torch.rand(M, generator=gen, device=dev), torch.randint(0, 127, (M,), generator=gen, device=dev).float()
    sw, zw = torch.rand(N, generator=gen, device=dev), torch.randint(0, 127, (N,), generator=gen, device=dev).float()
    bias = torch.randn(N, generator=gen, device=dev)
    for b in (None, bias):
        y = (sx[:, None] * sw) * (want.float() - (zx[:, None] + zw))
        y = y if b is None else y + b
        for t, wt in ((None, w), (N, hip.weight_tile_8bit(w))):
            got = hip.linear8bit_forward(a, sx, zx, wt, sw, zw, b, tiled_rows=t)
            assert torch.equal(got.view(torch.int32), y.view(torch.int32)), (b is None, t)


@pytest.mark.parametrize("M,N,K", [(2048, 11008, 2048), (1999, 11007, 2080),    # 96 x 256 tiles behind whole rounds
                                   (2040, 6100, 4096),                          # 96 x 256 tiles alone
                                   (1024, 10500, 4096), (1950, 5005, 4096), (2048, 8300, 2112)])  # 64 x 256, 64 x 128 behind
def test_uneven_rounds_of_the_tiles(dev, M, N, K):
    test_ragged_columns_of_the_tiles(dev, M, N, K)


@pytest.mark.parametrize("M,N,K", [(9, 1, 32), (16, 4100, 1056), (31, 1031, 4128), (40, 2400, 96), (60, 1600, 2080), (64, 8190, 544),
                                   (129, 1040, 1088), (190, 1025, 2080), (250, 1500, 160), (129, 2600, 992), (96, 4000, 1024),
                                   (4081, 16, 64), (12810, 10, 64), (3, 50, 8224), (12, 9000, 4192),
                                   # and on both weight layouts: one column tile a workgroup and two, one to four row tiles
                                   (16, 4090, 992), (31, 4090, 2112), (40, 4090, 2112), (16, 4100, 992), (31, 8190, 4128),
                                   (48, 8190, 2144), (64, 8190, 2112), (64, 4090, 544), (190, 1353, 992), (64, 8190, 480), (16, 8200, 480)])
def test_rows_through_lds(dev, M, N, K):
    """Every tile of the LDS kernel, groups of rows, ends inside a tile and a stage, up to the most groups there can be."""
    from duqlinear4bitcuda_amd import _lib
    assert _lib.load().duq_gemm8_kernel_for(M, N, K, 0) == 3
    test_ragged_columns_of_the_tiles(dev, M, N, K)
