"""The 8-bit GEMM on tiles whose eight wavefronts split K (csrc/duq_int8.hip, split kernel): rows, columns and k that end
inside a tile, a 256-k chunk and a pair of chunks; int32 against an exact product, the fused result against the stand-alone
dequant, with weights in both layouts."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(65, 4096, 4096), (33, 515, 4192), (49, 1001, 2080), (100, 1030, 1568), (200, 2048, 8192), (17, 8200, 4128),
                                   (64, 33, 4096), (128, 95, 11008), (1000, 40, 1536), (50, 16384, 4128), (256, 4095, 1824)])
def test_split_tiles(dev, M, N, K):
    from duqlinear4bitcuda_amd import _HIP as hip
    print("8-bit split tiles", M, N, K, flush=True)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    a = torch.randint(-128, 128, (M, K), dtype=torch.int8, device=dev, generator=g)
    w = torch.randint(-128, 128, (N, K), dtype=torch.int8, device=dev, generator=g)
    acc = hip.matmul_8bit(a, w)
    assert torch.equal(acc, (a.double() @ w.double().T).int())   # exact: |sums| < 2^53
    r = lambda n: torch.rand(n, device=dev, generator=g) * 3 - 1
    sx, zx, sw, zw, bias = r(M), r(M), r(N), r(N), r(N)
    for b in (None, bias):
        want = (sx[:, None] * sw) * (acc.float() - (zx[:, None] + zw))   # one rounding per operator, as the layer states it
        want = want if b is None else want + b
        assert torch.equal(hip.linear8bit_forward(a, sx, zx, w, sw, zw, b), want)
        assert torch.equal(hip.linear8bit_forward(a, sx, zx, hip.weight_tile_8bit(w), sw, zw, b, tiled_rows=N), want)
