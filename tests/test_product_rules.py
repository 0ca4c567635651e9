"""Rules of the products of activations (csrc/duq_product.hip, csrc/duq_product_long.hip), asked without a GPU."""
import pytest

ROW, TILES, LONG, TWO = 1, 2, 3, 4


def _path(mode, n, M, N, K, recorded=0):
    from duqlinear4bitcuda_amd import _lib
    return _lib.load().duq_product_path_for(mode, n, M, N, K, recorded)


def _parametrised(name, module):
    """The shapes of a parametrised test."""
    import importlib
    mark, = (m for m in getattr(importlib.import_module(module), name).pytestmark if m.name == "parametrize" and m.args[0] == "n,M,N,K")
    return mark.args[1]


def test_shapes_of_the_short_row_tests_reach_that_kernel():
    of = lambda name: _parametrised(name, "tests.test_gpu_product_tiles")
    for shape in of("test_against_the_oracle") + of("test_against_separate_launches"):
        want = TWO if shape == (8, 2000, 2008, 256) else TILES   # (rows of 256, large outputs whose rows begin anywhere: not that kernel's)
        assert _path(0, *shape) == _path(1, *shape) == want, shape
    for shape in of("test_many_rows_of_256"):
        assert _path(0, *shape) == _path(1, *shape) == TILES, shape
    for shape in of("test_in_a_recording"):
        assert _path(1, *shape) == TILES, shape
    # a recording keeps two launches for a few tiles: both sides of that are there
    assert [_path(1, *shape, 1) for shape in of("test_in_a_recording")] == [TWO, TWO, TWO, TWO, TWO, TILES, TWO, TILES]


def test_shapes_of_the_long_row_tests_reach_that_kernel():
    of = lambda name: _parametrised(name, "tests.test_gpu_product_long")
    for shape in of("test_against_the_oracle_and_separate_launches"):
        assert _path(0, *shape) == _path(1, *shape) == _path(1, *shape, 1) == LONG, shape
    assert [_path(1, *shape) for shape in of("test_against_separate_launches")] == [LONG] * 4 + [TWO] * 6 + [LONG]
    assert _path(1, 8, 300, 80, 704) == LONG


@pytest.mark.parametrize("there,beside", [
    # short rows: their length, one row of a, width, rows of 256 where a and the blocks of columns are few (asymmetric), large unaligned outputs
    ((8, 500, 500, 256), (8, 500, 500, 320)), ((8, 2, 500, 128), (8, 1, 500, 128)), ((1, 100, 1 << 24, 64), (1, 100, (1 << 24) + 1, 64)),
    ((8, 1024, 1216, 256), (8, 1025, 1216, 256)), ((41, 1025, 256, 256), (40, 1025, 256, 256)), ((8, 1024, 2047, 256), (9, 1024, 2047, 256)),
    # long rows: their length, columns, problems, rows of a, tiles
    ((32, 300, 64, 320), (32, 300, 64, 256)), ((32, 300, 64, 4096), (32, 300, 64, 4160)), ((32, 300, 256, 1024), (32, 300, 257, 1024)),
    ((2, 2048, 64, 1024), (1, 4096, 64, 1024)), ((64, 32, 32, 1024), (64, 31, 31, 1024)), ((8, 256, 256, 1536), (8, 255, 256, 1536)),
    ((64, 256, 128, 2048), (64, 255, 128, 2048)), ((64, 32, 16, 2048), (63, 32, 16, 2048)), ((128, 32, 16, 2112), (127, 32, 16, 2112)),
    ((8, 1024, 256, 2048), (8, 992, 256, 2048)), ((8, 4096, 256, 2112), (8, 4064, 256, 2112))])
def test_either_side_of_the_thresholds(there, beside):
    short = there[3] <= 256
    assert _path(1, *there) == (TILES if short else LONG) and _path(1, *beside) in (ROW, TILES, TWO) and _path(1, *there) != _path(1, *beside)


# single problems: runs of three to five tiles for most of the CUs but not for all, runs of one in a second round, rows of 256 (asymmetric),
# outputs past what the last-level cache holds
@pytest.mark.parametrize("mode,there,beside", [
    (1, (3453, 3456, 128), (3067, 3072, 128)), (1, (2813, 2816, 128), (2941, 2944, 128)), (1, (3581, 3584, 128), (3197, 3200, 128)),
    (1, (2047, 4096, 128), (2049, 4096, 128)), (1, (4605, 1792, 128), (4605, 2048, 128)), (1, (3069, 3072, 64), (3069, 3072, 128)),
    (1, (2397, 3200, 128), (2493, 3328, 128)), (1, (4093, 4096, 192), (3581, 3584, 192)), (1, (4605, 4608, 192), (4029, 4352, 192)),
    (0, (4093, 4096, 256), (3709, 3712, 256)), (0, (4029, 4352, 192), (4029, 4352, 256)), (1, (1024, 20480, 256), (1025, 20480, 256)),
    (0, (8192, 19200, 128), (8192, 19201, 128))])
def test_single_problems(mode, there, beside):
    assert (_path(mode, 1, *there), _path(mode, 1, *beside)) == (TILES, TWO)
    assert _path(mode, 2, *beside) == (TWO if mode and beside[2] > 192 and beside[1] > 6144 else TILES)


# several problems of rows of 256 (asymmetric): how much of a round of runs of five tiles or more is empty, by the number of problems
@pytest.mark.parametrize("there,beside", [((6, 1725, 1728, 256), (6, 1597, 1600, 256)), ((8, 1405, 1408, 256), (8, 1400, 1400, 256)),
                                          ((12, 1126, 1144, 256), (12, 1085, 1088, 256)), ((13, 1085, 1088, 256), (12, 1085, 1088, 256)),
                                          ((48, 1100, 256, 256), (12, 1059, 1064, 256)), ((10, 1085, 1088, 256), (10, 1289, 1312, 256))])
def test_several_problems(there, beside):
    assert (_path(1, *there), _path(1, *beside)) == (TILES, TWO)
    assert _path(0, *beside) == _path(1, *beside[:3], 192) == TILES


def test_no_path_for_what_is_refused():
    assert [_path(m, *s) for m, s in ((2, (8, 64, 64, 64)), (1, (0, 64, 64, 64)), (1, (8, 0, 64, 64)), (1, (8, 64, 0, 64)),
                                      (1, (8, 64, 64, 0)), (1, (8, 64, 64, 96)))] == [0] * 6


def test_long_rows_read_their_own_codes_only():
    """A workgroup of the launch for long rows has wavefronts for one, two, four or eight tiles of 32 columns, and of three, five,
    six or seven the rest reads nothing: what lies behind a problem's codes need not be there."""
    from duqlinear4bitcuda_amd import _lib

    reads = _lib.load().duq_product_long_reads_for
    for N in range(1, 257):
        for K in range(64, 4097, 64):
            assert reads(N, K) == (N + 31) // 32 * 32 * (K // 2), (N, K)
    assert reads(0, 512) == reads(257, 512) == reads(64, 0) == reads(64, 4160) == reads(64, 100) == 0
