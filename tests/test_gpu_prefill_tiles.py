"""The prefill kernel (csrc/duq_prefill.hip) on every tile it has: rows, columns and k that end inside a tile, a stage and a
16-byte piece, widths that leave output rows at any alignment; accumulators against an exact float32 product on the GPU,
every epilogue against the stand-alone one."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (M, N, K, batch): 64 x 64, 96 x 64, 64 x 128, 192 x 128, 128 x 128, 128 x 256 and 256 x 256 tiles, the stream kernel's 64 x 128 and
# the short-row kernel
SHAPES = [(65, 8193, 2624, 1), (70, 8200, 4160, 1), (33, 8193, 12352, 1), (1, 16387, 30784, 1), (1000, 4101, 2112, 1), (897, 4096, 8256, 1),
          (1999, 4093, 4160, 1), (2048, 4096, 4096, 1), (4090, 4081, 2112, 1), (4096, 4104, 4096, 1),
          (300, 2001, 576, 1), (33, 257, 320, 5), (50, 131, 192, 6), (7, 515, 64, 3), (513, 129, 2368, 4), (2, 5, 4096, 2)]


@pytest.mark.parametrize("M,N,K,n", SHAPES)
def test_prefill_tiles(dev, M, N, K, n):
    from duqlinear4bitcuda_amd import _HIP as hip
    print("prefill tiles", M, N, K, n, flush=True)
    assert n > 1 or hip.gemm_kernel_for(M, N, K) in (6, 7)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    rnd = lambda *s: torch.randint(0, 256, s, dtype=torch.uint8, device=dev, generator=g)

    def signed(p):  # [..., K/2] -> float32 [..., K]
        lo, hi = (p & 15).to(torch.int8), (p >> 4).to(torch.int8)
        v = torch.stack((lo, hi), -1).flatten(-2)
        return torch.where(v > 7, v - 16, v).float()

    a, b = rnd(n, M, K // 2), rnd(n, N, K // 2)
    want = torch.stack([signed(a[i]) @ signed(b[i]).T for i in range(n)]).int()   # exact: |sums| < 2^24
    acc = hip.matmul(a[0], b[0])[None] if n == 1 else hip.batched_matmul(a, b)
    assert torch.equal(acc, want)
    h = lambda *s: (torch.rand(*s, device=dev, generator=g) * 4 - 1).half()
    i = lambda *s: torch.randint(-5000, 5000, s, device=dev, generator=g).int()
    sr, zr, rr = h(n, M), h(n, M).round(), i(n, M)
    s1, z1, s2, z2, bias, r1 = h(n, N), h(n, N).round(), h(n, N), h(n, N), h(n, N), i(n, N)
    flat = lambda f, *t: torch.stack([f(*(x[k] for x in t)) for k in range(n)])
    steps = ((hip.EPI_SYM, (sr, None, s1, None, None, None), flat(hip.sym_dequant, acc, sr, s1)),
             (hip.EPI_ASYM, (sr, zr, s1, z1, None, None), flat(hip.asym_dequant, acc, sr, zr, s1, z1)),
             (hip.EPI_SYM_DUAL, (sr, None, s1, None, s2, None), flat(hip.sym_dual_dequant, acc, sr, s1, s2)),
             (hip.EPI_ASYM_DUAL, (sr, zr, s1, z1, s2, z2), flat(hip.asym_dual_dequant, acc, sr, zr, s1, z1, s2, z2)))
    for mode, (r, z, c1, y1, c2, y2), y in steps:
        for off in (0, 1):   # parameter arrays at an odd address: no 64-bit loads
            place = lambda t: t if t is None or not off else torch.cat([t.flatten()[:1], t.flatten()])[1:]
            got = hip.batch_linear4bit_forward(mode, a, r, z, b, *(place(t) for t in (c1, y1, c2, y2)), bias=place(bias))
            assert torch.equal(got.view(torch.int16), (y + bias[:, None]).view(torch.int16)), (mode, off)
    if n == 1:
        got = hip.linear4bit_forward_rowsum(a[0], sr, zr, rr, b[0], s1, z1, r1)
        assert torch.equal(got.view(torch.int16), hip.asym_rowsum_dequant(acc[0], sr, zr, rr, s1, z1, r1).view(torch.int16))
        # the dual-uniform row-sum epilogue, inside the GEMM where its kernel applies it
        got = hip.linear4bit_forward_dual_rowsum(a[0], sr[0], zr[0], rr[0], b[0], s1[0], z1[0], s2[0], z1[0], r1[0], r1[0], bias[0])
        want = hip.asym_dual_rowsum_dequant(acc[0], a[0], sr[0], zr[0], rr[0], b[0], s1[0], z1[0], s2[0], z1[0], r1[0], r1[0], bias[0])
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


# tiles whose eight wavefronts split every stage: odd and even numbers of stages, a k that ends inside a piece, few rows, columns
# that end anywhere (tile 0: a shape the query names no tile for)
SPLIT = [(65, 4100, 2112, 64064), (200, 2101, 4160, 64064), (17, 8201, 16448, 0), (6, 8193, 20032, 0), (64, 11008, 4096, 64064),
         (250, 2049, 8256, 64064), (64, 11007, 4160, 64064),
         (256, 4096, 4096, 64064), (96, 8193, 4160, 96064), (77, 13824, 5120, 96064), (65, 12001, 16448, 96064)]


@pytest.mark.parametrize("M,N,K,tile", SPLIT)
def test_tiles_split_over_k(dev, M, N, K, tile):
    from duqlinear4bitcuda_amd import _HIP as hip
    assert hip.gemm_stream_tile_for(M, N, K) == tile
    test_prefill_tiles(dev, M, N, K, 1)


@pytest.mark.parametrize("M,N,K,n", [(1, 130, 4160, 5), (63, 64, 2112, 7)])
def test_tiles_split_over_k_batched(dev, M, N, K, n):
    test_prefill_tiles(dev, M, N, K, n)
