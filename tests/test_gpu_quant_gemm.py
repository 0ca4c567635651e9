"""The kernel that quantizes its rows, multiplies and dequantizes (``csrc/duq_quant_gemm.hip``): the oracle's bits at the edges of
its tiles, what it hands out of its quantizer, and the rule that picks its tile."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import duq_oracle as orc
from tests import cases
from tests.test_gpu_random_shapes import hip, test_random_shapes_fp16_input as _against_the_oracle  # noqa: F401 (fixture)


def _tile(M, N, K):
    from duqlinear4bitcuda_amd import _lib

    t = _lib.load().duq_quant_gemm_tile_for(M, N, K)
    return t & 255, t >> 8 & 255, t >> 16 & 255


# tile (rows, column tiles, chunks), then shapes at its edges: one row in the last group, one column in the last tile, short rows,
# rows that end inside a slice, the longest rows
EDGES = {
    (8, 1, 1): [(3, 1, 64), (8, 4096, 4096), (9, 17, 2112), (17, 1024, 3136), (5, 4096, 8192), (6, 33, 4160), (250, 100, 4032)],
    (8, 2, 1): [(8, 8190, 3072), (65, 700, 4096), (120, 500, 2560)],
    (8, 3, 1): [(8, 12288, 4096), (3, 9000, 2112), (24, 4000, 3072)],
    (16, 1, 1): [(500, 100, 64), (513, 110, 1088), (1000, 50, 1984)],
    (16, 2, 1): [(16, 8192, 64), (130, 777, 960), (33, 2700, 2048)],
    (16, 3, 1): [(40, 4000, 2048), (33, 4000, 1984)],
    (16, 8, 1): [(16, 30000, 2048), (64, 8100, 2048), (100, 4200, 1984)],
    (32, 4, 1): [(512, 1024, 512), (500, 1023, 576), (60, 8190, 512), (2000, 17, 576)],
    (32, 4, 2): [(500, 2001, 960), (1000, 1000, 1024), (40, 16001, 64)],
    (32, 4, 3): [(200, 6002, 512)],
    (32, 4, 4): [(64, 30003, 512)],
}
LONG = {  # two sets of registers one after the other
    (16, 2, 1): [(32, 4000, 4032), (513, 1, 2112), (1024, 64, 4096)],   # (the last two: as many groups of rows as there may be)
    (16, 3, 1): [(13, 12287, 3072)],
    (16, 1, 4): [(9, 16383, 4096)],
}
SHAPES = [(t, s) for edges in (EDGES, LONG) for t, shapes in edges.items() for s in shapes]


@pytest.mark.parametrize("tile,shape", SHAPES)
def test_shapes_reach_their_tile(tile, shape):
    assert _tile(*shape) == tile


def test_the_rule_gives_no_other_tile():
    """The tiles above are the ones there are kernels for (several chunks of columns are one kernel, whatever their number)."""
    kind = lambda rows, cols, chunks, K: (rows, cols, chunks > 1, rows == 16 and K > 2048)
    there = {kind(*t, s[2]) for t, s in SHAPES}
    rows = [*range(3, 34), 40, 64, 65, 100, 128, 129, 200, 256, 257, 500, 512, 513, 700, 1000, 1024, 1025, 2000, 2048]
    for M in rows:
        for N in (1, 16, 17, 48, 64, 65, 128, 200, 300, 512, 1000, 2048, 4096, 8192, 16384, 28672, 65536):
            for K in (64, 512, 576, 1024, 1088, 2048, 2112, 3072, 4096, 4160, 8192):
                tile = _tile(M, N, K)
                assert tile[0] == 0 or kind(*tile, K) in there, (M, N, K, tile)


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(SHAPES)))
def test_tiles_against_the_oracle(hip, dev, i):  # noqa: F811
    M, N, K = SHAPES[i][1]
    for mode in (i % 6, (i + 3) % 6):   # a symmetric and an asymmetric epilogue
        _against_the_oracle(hip, dev, M, N, K, mode)


# three and four rows, which go to one kernel or the other by their length, the columns and the quantizer
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(3, 1030, 2112), (4, 1001, 4096), (3, 2048, 4160), (4, 2050, 4160), (4, 2048, 6208), (3, 4096, 8192), (4, 16390, 3008)])
def test_few_long_rows(hip, dev, M, N, K):  # noqa: F811
    for mode in range(6):
        _against_the_oracle(hip, dev, M, N, K, mode)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(3, 4097, 3392), (4, 1000, 4096), (3, 13001, 2560), (4, 12289, 4032), (3, 333, 5696), (4, 2049, 6208), (4, 400, 7168)])
def test_more_long_rows(hip, dev, M, N, K):  # noqa: F811
    test_few_long_rows(hip, dev, M, N, K)


# rows that the rows kernel takes out of LDS in two halves (K > 12288), the last one a piece, a part and the whole of its range
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(3, 37, 12352), (4, 1001, 12352), (4, 300, 14336), (3, 515, 14400), (4, 33, 16320), (4, 1030, 16384)])
def test_rows_in_two_halves(hip, dev, M, N, K):  # noqa: F811
    test_few_long_rows(hip, dev, M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(20, 40, 2112), (33, 2700, 2048), (500, 2001, 960), (40, 4000, 4096)])
def test_rows_that_are_not_finite_beside_rows_that_are(hip, dev, M, N, K):  # noqa: F811
    """A wavefront holds several rows: a zero row, an infinity and a NaN among them, and a scale that underflows."""
    x = cases.acts_outliers(M, K, seed=M)
    x[1], x[4, 3], x[6, K - 1], x[9] = 0, np.inf, np.nan, np.float16(6e-8)
    x[11] = -x[11]
    wq, sw = cases.weights_random_nibbles(N, K, seed=3)
    with np.errstate(all="ignore"):
        want = orc.linear4bit_sq_forward(x, wq, sw)[0]
    got = hip.quantize_linear4bit_forward(cases.t(x, dev), cases.t(wq, dev), cases.t(sw, dev))
    assert cases.bits_equal(got.cpu().numpy(), want)
    u = cases.acts_uniform(M, K, seed=M + 1)
    u[1], u[4, 3], u[6, K - 1], u[9], u[11] = 0, np.inf, np.nan, 3, -u[11]
    w = (np.random.default_rng(M).standard_normal((N, K)) * 0.02).astype(np.float16)
    wq, sw, zw, adj = orc.weight_asym_shifted_from_linear(w)
    with np.errstate(all="ignore"):
        want = orc.linear4bit_asq_rowsum_forward(u, wq, sw, zw, adj)[0]
    got = hip.quantize_linear4bit_forward_asym(hip.EPI_ASYM_ROWSUM, cases.t(u, dev), cases.t(wq, dev), cases.t(sw, dev),
                                               cases.t(zw, dev), None, None, cases.t(adj, dev))
    assert cases.bits_equal(got.cpu().numpy(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(13, 3000, 2048), (37, 500, 960), (100, 5000, 768), (9, 16384, 2560), (21, 600, 4096), (7, 4096, 6208)])
def test_codes_and_parameters_of_the_rows(hip, dev, M, N, K):  # noqa: F811
    """What the caller may ask for of the quantizer: the stand-alone quantizer's bits, whatever the launch."""
    T = lambda v: cases.t(v, dev)
    wq, sw = cases.weights_random_nibbles(N, K, seed=5)
    x = T(cases.acts_outliers(M, K, seed=M))
    y, q, s = hip.quantize_linear4bit_forward(x, T(wq), T(sw), return_quantized=True)
    q0, s0 = hip.quantize_rows_sym(x)[:2]
    assert torch.equal(q, q0) and torch.equal(s, s0)
    assert torch.equal(y, hip.linear4bit_forward(hip.EPI_SYM, q0, s0, None, T(wq), T(sw)))
    x, adj = T(cases.acts_uniform(M, K, seed=M)), torch.zeros(N, dtype=torch.int32, device=dev)
    y, q, s, z, r = hip.quantize_linear4bit_forward_asym(hip.EPI_ASYM_ROWSUM, x, T(wq), T(sw), T(sw), None, None, adj, return_quantized=True)
    for got, want in zip((q, s, z, r), hip.quantize_rows_asym_shifted(x)):
        assert torch.equal(got.flatten(), want.flatten())


def test_every_shape_without_room_for_codes_has_its_kernel():
    """Callers bring no workspace for these, so there are no two launches to fall back to: up to eight rows of up to 4096
    elements the rows kernel, everything else a tile of this one."""
    from duqlinear4bitcuda_amd import _lib

    lib = _lib.load()
    rng = np.random.default_rng(8)
    seen = 0
    for M in range(3, 17):
        for K in [64, 1024, 1088, 2048, 2112, 2496, 2560, 3072, 3136, 3584, 4096, 4160, 8192] + list(64 * rng.integers(1, 129, 12)):
            for N in [1, 16, 4096, 4097, 8192, 12288, 12289, 16384, 16385] + list(rng.integers(1, 40000, 12)):
                M, N, K = int(M), int(N), int(K)
                if lib.duq_quantize_linear4bit_workspace_bytes(M, N, K) or (M <= 4 or (M <= 8 and K <= 4096)):
                    continue
                seen += 1
                assert _tile(M, N, K)[0], (M, N, K)
    assert seen > 500


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,launches", [(32, 4000, 4032, 2), (40, 600, 3008, 1), (36, 604, 7680, 2), (48, 1024, 1024, 1)])
def test_recorded_calls(hip, dev, M, N, K, launches):  # noqa: F811
    """Replays of a recording, where a launch less counts for less, give the eager call's bits."""
    from duqlinear4bitcuda_amd import _lib

    assert 1 + (_lib.load().duq_quant_gemm_tile_for(M, N, K) >> 24) == launches
    T = lambda v: cases.t(v, dev)
    wq, sw = cases.weights_random_nibbles(N, K, seed=7)
    wq, sw = T(wq), T(sw)
    x = T(cases.acts_outliers(M, K, seed=M))
    want = hip.quantize_linear4bit_forward(x, wq, sw)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = hip.quantize_linear4bit_forward(x, wq, sw)
    for _ in range(3):
        got.fill_(0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("mode,one,two", [
    (1, (12, 16000, 2112), (62, 3467, 2368)), (5, (9, 16383, 3584), (9, 16383, 4096)),                                  # sixteen long rows
    (0, (974, 1824, 256), (974, 1824, 640)), (2, (64, 30000, 640), (378, 4757, 640)), (1, (143, 12886, 960), (363, 5035, 576)),   # four chunks
    (4, (391, 3470, 640), (463, 3469, 640)),                                                                            # three, four
    (5, (604, 2231, 448), (498, 2093, 832)), (5, (986, 1934, 448), (313, 4875, 640)), (5, (201, 4000, 960), (201, 6802, 960))])
def test_several_chunks_or_two_launches(mode, one, two):
    from duqlinear4bitcuda_amd import _lib

    path = _lib.load().duq_quantize_linear4bit_path_for
    assert _tile(*one)[0] and _tile(*two)[2] > 1
    assert (path(mode, *one, 0), path(mode, *two, 0)) == (2, 3)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(62, 3467, 2368), (276, 6397, 640), (143, 12886, 960), (498, 2093, 832), (9, 16383, 4096)])
def test_on_either_side_of_several_chunks(hip, dev, M, N, K):  # noqa: F811
    for mode in (1, 4, 5):
        _against_the_oracle(hip, dev, M, N, K, mode)


def test_the_query_says_what_runs():
    """Over every mode, eager and recorded: two launches only where the caller is asked for room, a tile that is given up in a recording only
    there, and the rows kernel where three and four long rows are ahead on it."""
    from duqlinear4bitcuda_amd import _lib

    lib = _lib.load()
    path = lib.duq_quantize_linear4bit_path_for
    for M in [1, 2, 3, 4, 5, 8, 9, 13, 16, 17, 32, 64, 200, 1000, 2048, 2049]:
        for N in (1, 1000, 2048, 2049, 4096, 4097, 12288, 12289, 16384, 16385, 28672):
            for K in (64, 1024, 2048, 2112, 4096, 4160, 6144, 6208, 8192, 8256, 11008):
                tile = lib.duq_quant_gemm_tile_for(M, N, K)
                for mode in range(6):
                    room = lib.duq_quantize_linear4bit_workspace_bytes(M, N, K) if mode in (0, 2) else \
                        lib.duq_quantize_linear4bit_asym_workspace_bytes(mode, M, N, K)
                    eager, recorded = path(mode, M, N, K, 0), path(mode, M, N, K, 1)
                    assert (eager, recorded) in ((1, 1), (2, 2), (2, 3), (3, 3)) and (room or 3 not in (eager, recorded)), (mode, M, N, K)
                    assert (recorded != eager) == bool(tile >> 24) or eager != 2, (mode, M, N, K)
                    given_up = (M in (3, 4) and K > 2048 and eager == 1) or ((tile >> 16 & 255) > 1 and M > 8 and eager == 3)
                    assert (eager == 2) == bool(tile) or given_up, (mode, M, N, K)
    assert [path(m, 3, 4096, 4096, 0) for m in range(6)] == [1, 1, 1, 1, 2, 1] and path(0, 3, 4096, 2048, 0) == path(1, 4, 4096, 5120, 0) == 2
    assert path(4, 3, 12289, 4032, 1) == path(5, 4, 12289, 2112, 1) == 2   # (no room: no two launches)
    for mode, there, beside in ((0, (4, 4096, 5632), (4, 4096, 5696)), (1, (4, 4096, 4160), (3, 4096, 4160)), (2, (4, 300, 4160), (4, 300, 4096)),
                                (4, (3, 12288, 3072), (3, 12289, 3072)), (4, (3, 1000, 5120), (3, 1000, 5184)), (4, (4, 2049, 6208), (4, 2048, 6208)),
                                (4, (4, 1000, 6144), (4, 1000, 6208)), (4, (4, 13000, 3904), (4, 13000, 3840)), (4, (4, 13000, 4032), (4, 13000, 4096)),
                                (5, (4, 4097, 4096), (4, 4096, 4096)), (5, (3, 1000, 3264), (3, 1000, 3328)), (5, (4, 1000, 6208), (3, 1000, 6208)),
                                (5, (3, 2049, 8192), (3, 2048, 8192))):
        assert (path(mode, *there, 0), path(mode, *beside, 0)) == (2, 1), (mode, there, beside)
    assert path(6, 3, 64, 64, 0) == path(0, 0, 64, 64, 0) == path(0, 3, 64, 96, 0) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(20, 1000, 1024), (100, 300, 4096), (300, 700, 512), (60, 12001, 512)])
@pytest.mark.parametrize("mode", range(6))
def test_a_layers_workspace_is_left_alone_by_the_one_kernel(hip, dev, M, N, K, mode):  # noqa: F811
    """The workspace of duq_quantize_linear4bit_forward_layer, where nobody looks for codes, is asked for as where two launches run."""
    from duqlinear4bitcuda_amd import _lib

    lib = _lib.load()
    assert _tile(M, N, K)[0]
    T = lambda v: cases.t(v, dev)
    x = T(cases.acts_outliers(M, K, seed=M) if mode in (0, 2) else cases.acts_uniform(M, K, seed=M))
    wq, sw = (T(v) for v in cases.weights_random_nibbles(N, K, seed=5))
    adj, s2 = torch.arange(N, dtype=torch.int32, device=dev), (sw * 2).contiguous()
    p = lambda t, used: t.data_ptr() if used else None
    layer = _lib.FusedLayer(mode, 1.0, 6, N, K, wq.data_ptr(), sw.data_ptr(), p(s2, mode in (1, 3, 4, 5)), p(s2, mode in (2, 3, 5)),
                            p(sw, mode in (3, 5)), p(adj, mode >= 4), p(adj, mode == 5), None)
    need = lib.duq_quantize_linear4bit_workspace_bytes(M, N, K) if mode in (0, 2) else \
        lib.duq_quantize_linear4bit_asym_workspace_bytes(mode, M, N, K)
    room = torch.full((need,), 0xA5, dtype=torch.uint8, device=dev)
    y = torch.empty(M, N, dtype=torch.float16, device=dev)
    stream = torch.cuda.current_stream().cuda_stream
    call = lambda n: lib.duq_quantize_linear4bit_forward_layer(ctypes.addressof(layer), x.data_ptr(), M, y.data_ptr(), room.data_ptr(), n, stream)
    assert call(need - 1) == -2 and call(need) == 0
    torch.cuda.synchronize()
    assert bool((room == 0xA5).all())
    if mode in (0, 2):
        q, s = hip.quantize_rows_sym(x)[:2]
        want = hip.linear4bit_forward(mode, q, s, None, wq, sw, None, s2 if mode == 2 else None)
    elif mode in (1, 3):
        q, s, z = hip.quantize_rows_asym(x)
        want = hip.linear4bit_forward(mode, q, s, z, wq, sw, s2, s2 if mode == 3 else None, sw if mode == 3 else None)
    else:
        q, s, z, r = hip.quantize_rows_asym_shifted(x)
        want = hip.linear4bit_forward_rowsum(q, s, z, r, wq, sw, s2, adj) if mode == 4 else \
            hip.linear4bit_forward_dual_rowsum(q, s, z, r, wq, sw, s2, s2, sw, adj, adj)
    assert cases.bits_equal(y.cpu().numpy(), want.cpu().numpy())
