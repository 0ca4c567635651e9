"""Prefill problems whose rounds of tiles do not come out even: whole rounds of 128 x 256 tiles and the columns that are left in
192 x 128, 128 x 128 or 64 x 128 ones, and 192 x 128 tiles alone; rows and columns that end inside either kind of tile."""
import pytest

from tests.test_gpu_prefill_tiles import test_prefill_tiles as check

pytestmark = pytest.mark.gpu

SHAPES = [(1999, 11007, 4160), (1985, 11000, 4096),      # 192 x 128 behind two rounds
          (2048, 6144, 4096), (2000, 6100, 2112),        # 128 x 128 behind one
          (4000, 8200, 4160), (1999, 9001, 2112)]        # 64 x 128 behind four and two


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_mixed(dev, M, N, K):
    from duqlinear4bitcuda_amd import _HIP as hip
    print("mixed", M, N, K, flush=True)
    assert hip.gemm_stream_tile_for(M, N, K) == 128256
    check(dev, M, N, K, 1)


# (the query names one tile for both kinds of first part)
@pytest.mark.parametrize("M,N,K", [(690, 13001, 2112), (1999, 5003, 2112),    # 64 x 128 behind one round of 128 x 256
                                   (520, 21912, 2560),                       # 192 x 128 behind 1
                                   (935, 20001, 2112), (1203, 15441, 2176),    # 128 x 128 behind one round of 256 x 256
                                   (1801, 12518, 2112),                       # 128 x 256 behind one
                                   (2355, 3344, 2496), (4160, 3924, 5888)])   # int32 outputs: stream kernel, 128 x 128
def test_mixed_of_either_kind(dev, M, N, K):
    from duqlinear4bitcuda_amd import _HIP as hip
    print("mixed", M, N, K, flush=True)
    assert hip.gemm_stream_tile_for(M, N, K) == 128256
    check(dev, M, N, K, 1)


@pytest.mark.parametrize("M,N,K,n", [(1536, 4096, 2048, 1), (1501, 4001, 4160, 1), (700, 8190, 2112, 1), (190, 1000, 4096, 17)])
def test_192_row_tiles(dev, M, N, K, n):
    from duqlinear4bitcuda_amd import _HIP as hip
    print("192 x 128", M, N, K, n, flush=True)
    if n == 1:
        assert hip.gemm_stream_tile_for(M, N, K) == 192128
    check(dev, M, N, K, n)
