"""The LDS and wide kernels of the decode family (any length, narrow problems, and many columns) at the edges of its tiles, stages and rule, against the
oracle, through the C ABI and the dual-uniform row-sum layer, whose epilogue it applies itself."""
import numpy as np
import pytest

from oracle import duq_oracle as orc
from tests import cases
from tests.test_gpu_decode import hip, test_decode_kernels_against_the_oracle as _against_the_oracle  # noqa: F401 (fixture)
from tests.test_gpu_module_decode import library_calls, test_dual_uniform_rowsum_layer_decode as _dual_rowsum  # noqa: F401

pytestmark = pytest.mark.gpu

# 16 columns a workgroup (stages of one kilobyte a row: 2048 elements): one row tile to four, columns and rows that end inside
# one, less than a stage, stage boundaries, the longest rows; up to four rows beyond the rows kernel's.  32 columns (stages of
# 1024 elements): the same, from 4097 columns on.
SHAPES = [(5, 1, 64), (16, 17, 2048), (17, 15, 2112), (33, 4096, 960), (49, 31, 16448), (64, 48, 1984), (63, 2049, 4160),
          (8, 16, 65536), (1, 20, 16448), (1, 20, 30784), (1, 2050, 16448), (4, 33, 20480),
          (5, 4097, 4160), (20, 4100, 1088), (40, 4127, 64), (64, 8192, 1024), (16, 8180, 5184), (3, 4100, 18496), (2, 4112, 30784),
          (32, 8200, 8256), (16, 8193, 12352),
          # groups of rows in workgroups of their own: every tile, the most groups there can be, a last group with one row
          (65, 256, 512), (129, 1040, 1088), (190, 1025, 2112), (250, 1500, 1024), (129, 2600, 960), (193, 1030, 4160), (96, 4000, 1024),
          (128, 4090, 1088), (4081, 16, 576), (1000, 130, 640),
          (70, 1600, 1088), (60, 1600, 2112), (12810, 10, 512),
          # the wide kernel: every form, one to several column tiles per workgroup, a last workgroup with fewer
          (5, 8193, 6208), (16, 16400, 5184), (17, 8200, 64), (32, 12300, 2112), (24, 16390, 8192), (40, 8250, 2048), (49, 16387, 1088)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_lds_kernel_against_the_oracle(hip, dev, M, N, K):  # noqa: F811
    _against_the_oracle(hip, dev, M, N, K)


@pytest.mark.parametrize("M,N,K", [(1, 40, 16448), (7, 37, 16448), (33, 130, 2112), (24, 4110, 1088), (3, 50, 16448), (20, 8210, 2112), (130, 1000, 1088)])
def test_lds_kernel_rowsum_epilogues(hip, dev, library_calls, M, N, K):  # noqa: F811
    x = cases.acts_uniform(M, K, seed=31 + M)
    w = (np.random.default_rng(M).standard_normal((N, K)) * 0.02).astype(np.float16)
    wq, sw, zw, adj = orc.weight_asym_shifted_from_linear(w)
    want, *_ = orc.linear4bit_asq_rowsum_forward(x, wq, sw, zw, adj)
    q, s, z, r = hip.quantize_rows_asym_shifted(cases.t(x, dev))
    y = hip.linear4bit_forward_rowsum(q, s, z, r, cases.t(wq, dev), cases.t(sw, dev), cases.t(zw, dev), cases.t(adj, dev))
    assert cases.bits_equal(y.cpu().numpy(), want)
    _dual_rowsum(dev, library_calls, M, N, K)
