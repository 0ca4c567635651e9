"""The 8-bit kernel that quantizes its rows, multiplies and dequantizes (``csrc/duq_quant_gemm8.hip``): the oracle's bits at the
edges of its tiles, on the weight as stored and on the tiled copy, and the rule that picks its tile."""
import numpy as np
import pytest
import torch

from oracle import duq_oracle as orc
from tests import cases
from tests.test_gpu_random_shapes import hip  # noqa: F401 (fixture)


def _tile(M, N, K):
    from duqlinear4bitcuda_amd import _lib

    t = _lib.load().duq_quant_gemm8_tile_for(M, N, K)
    return t & 255, t >> 8 & 255, t >> 16


# tile (rows, column tiles, chunks), then shapes at its edges: one row in the last group, one column in the last tile, short rows,
# rows that end inside a slice, the longest rows
EDGES = {
    (8, 1, 1): [(3, 4096, 2080), (8, 4096, 4096), (9, 33, 2080), (250, 120, 4064), (17, 1300, 3296)],
    (8, 2, 1): [(8, 8190, 2048), (33, 1000, 2048), (57, 580, 1952)],
    (8, 3, 1): [(8, 12288, 2016)],
    (16, 1, 1): [(3, 1, 32), (500, 100, 32), (33, 1300, 544), (65, 770, 1024)],
    (16, 2, 1): [(16, 8177, 1024), (130, 777, 992), (33, 2700, 2048)],
    (16, 3, 1): [(16, 12001, 1024), (40, 4000, 1984)],
    (16, 8, 1): [(16, 30000, 1024), (10, 20001, 928)],
    (32, 4, 1): [(512, 1024, 512), (500, 1023, 576), (64, 8190, 1024), (97, 3900, 992)],
    (32, 4, 2): [(1000, 1000, 512), (60, 12001, 480)],
}
SHAPES = [(t, s) for t, shapes in EDGES.items() for s in shapes]


@pytest.mark.parametrize("tile,shape", SHAPES)
def test_shapes_reach_their_tile(tile, shape):
    assert _tile(*shape) == tile


def _want(x, w, sw, zw, bias):
    with np.errstate(all="ignore"):
        s, z = orc.asym8_scales_zeros(x)
        acc = orc.matmul_s8(orc.asym_quant_8bit(x, s, z), w).astype(np.int32)
        y = orc.asym_dequant_hprec(acc, s, z, sw, zw)
        return y if bias is None else (y + bias[None, :]).astype(np.float32)


def _same(got, want):
    nan = np.isnan(got) & np.isnan(want)
    return bool(np.all((got.view(np.uint32) == want.view(np.uint32)) | nan))


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(SHAPES)))
def test_tiles_against_the_oracle(hip, dev, i):  # noqa: F811
    M, N, K = SHAPES[i][1]
    rng = np.random.default_rng(i)
    x = rng.normal(0.3, 1.0, (M, K)).astype(np.float32)
    if i % 2:   # rows that are not finite, without spread or far off zero for theirs, beside rows that are
        x[M - 1] = 0
        x[0, K - 1], x[M // 2, 0] = np.inf, np.nan
        x[1] = 1000 + x[1] * np.float32(1e-3)
    w = rng.integers(0, 128, (N, K)).astype(np.int8)
    sw = rng.uniform(0.0001, 0.01, (N, 1)).astype(np.float32)
    zw = np.rint(rng.uniform(-60, 10, (N, 1))).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32) if i % 3 else None
    T = lambda v: None if v is None else cases.t(v, dev)
    want = _want(x, w, sw, zw, bias)
    for copy in (None, hip.weight_tile_8bit(T(w))):
        got = hip.quantize_linear8bit_forward(T(x), T(w), copy, T(sw), T(zw), T(bias))
        assert _same(got.cpu().numpy(), want), copy is None


@pytest.mark.gpu
def test_layer_replayed_as_a_graph(dev):
    from duqlinear4bitcuda_amd import nn as qnn

    lin = torch.nn.Linear(1024, 1000, dtype=torch.float32, device=dev)
    layer = qnn.LinearQuant8bitASQ.from_linear(lin).to(dev)
    x = torch.randn(50, 1024, device=dev)
    want = layer(x)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph), torch.no_grad():
        got = layer(x)
    for _ in range(3):
        got.fill_(0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


def test_every_tile_that_the_rule_gives_has_its_kernel():
    """A tile without one would end the call in an error.  (Eight pieces of four elements or sixteen for a lane, one chunk of columns or
    several: what there are kernels for, and what the shapes above run.)"""
    import os
    import re

    path = os.path.join(os.path.dirname(__file__), "..", "duqlinear4bitcuda_amd", "csrc", "duq_quant_gemm8.hip")
    there = {(int(r), int(u), int(c), b == "2") for r, u, c, b in re.findall(r"^    DUQ_Q8\((\d+), (\d+), (\d+), (\d+)\)$", open(path).read(), re.M)}
    kind = lambda rows, cols, chunks, K: (rows, 8 if rows * K <= 16384 else 16, cols, chunks > 1)
    assert {kind(*t, s[2]) for t, s in SHAPES + MORE} == there and len(there) == 14
    seen = set()
    for M in [*range(3, 34), 40, 63, 64, 65, 100, 128, 129, 200, 256, 257, 500, 512, 513, 700, 1000, 1024, 1025, 1536, 2000, 2047, 2048, 2049]:
        for N in (1, 16, 17, 33, 48, 64, 65, 128, 200, 300, 512, 1000, 2048, 2053, 4096, 4097, 8192, 8193, 12288, 16384, 28672, 65536, 65537):
            for K in range(32, 4129, 32):
                tile = _tile(M, N, K)
                if tile[0]:
                    seen.add(kind(*tile, K))
                else:
                    assert tile == (0, 0, 0)
    assert seen == there


# the rest of the tiles: eight rows of at most 2048 elements, sixteen of more than 1024
MORE = [((8, 1, 1), (8, 4001, 1024)), ((8, 1, 1), (5, 436, 1600)), ((8, 1, 1), (7, 130, 2048)), ((16, 1, 1), (9, 2053, 1056)), ((16, 1, 1), (33, 1297, 1504))]


@pytest.mark.parametrize("tile,shape", MORE)
def test_more_shapes_reach_their_tile(tile, shape):
    assert _tile(*shape) == tile


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(len(MORE)))
def test_more_tiles_against_the_oracle(hip, dev, monkeypatch, i):  # noqa: F811
    monkeypatch.setitem(globals(), "SHAPES", MORE)
    test_tiles_against_the_oracle(hip, dev, i)
