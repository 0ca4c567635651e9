"""The 8-bit layer's row quantizer: rows of every kind, lengths that end inside a wavefront's share."""
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
