"""Prefill problems whose rounds of tiles do not come out even: whole rounds of 256 x 256 or 128 x 256 tiles and the columns that
are left in smaller ones, and 192 x 128 tiles alone; rows and columns that end inside either kind of tile."""
import pytest

from tests.test_gpu_prefill_tiles import test_prefill_tiles as check

pytestmark = pytest.mark.gpu

# rows and columns of the first tiles, the column up to which they reach, rows and columns of the tiles behind it
SHAPES = [(1999, 11007, 4160, (256, 256, 8192, 192, 128)), (1985, 11000, 4096, (256, 256, 8192, 192, 128)),
          (4000, 8200, 4160, (256, 256, 8192, 64, 128)), (1999, 9001, 2112, (256, 256, 8192, 64, 128)),
          (935, 20001, 2112, (256, 256, 16384, 128, 128)), (1203, 15441, 2176, (256, 256, 13056, 128, 128)),
          (1801, 12518, 2112, (256, 256, 8192, 128, 256)),
          (2048, 6144, 4096, (128, 256, 4096, 128, 128)), (2000, 6100, 2112, (128, 256, 4096, 128, 128)),
          (690, 13001, 2112, (128, 256, 10752, 64, 128)), (1999, 5003, 2112, (128, 256, 4096, 64, 128)),
          (520, 21912, 2560, (128, 256, 13056, 192, 128)),
          # (int32 outputs on the stream kernel; on 128 x 128 tiles)
          (2355, 3344, 2496, (128, 256, 3328, 64, 128)), (4160, 3924, 5888, (256, 256, 3840, 64, 128))]


@pytest.mark.parametrize("M,N,K,plan", SHAPES)
def test_mixed(dev, M, N, K, plan):
    from duqlinear4bitcuda_amd import _HIP as hip
    print("mixed", M, N, K, flush=True)
    assert hip.gemm_plan_for(M, N, K) == plan
    assert hip.gemm_stream_tile_for(M, N, K) == 128256   # (names one tile for all of them)
    check(dev, M, N, K, 1)


@pytest.mark.parametrize("M,N,K,n", [(1536, 4096, 2048, 1), (1501, 4001, 4160, 1), (700, 8190, 2112, 1), (190, 1000, 4096, 17)])
def test_192_row_tiles(dev, M, N, K, n):
    from duqlinear4bitcuda_amd import _HIP as hip
    print("192 x 128", M, N, K, n, flush=True)
    if n == 1:
        assert hip.gemm_stream_tile_for(M, N, K) == 192128
    check(dev, M, N, K, n)
