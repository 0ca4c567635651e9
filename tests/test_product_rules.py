"""Rules of the products of activations (csrc/duq_product.hip, csrc/duq_product_long.hip), asked without a GPU."""


def test_long_rows_read_their_own_codes_only():
    """A workgroup of the launch for long rows has wavefronts for one, two, four or eight tiles of 32 columns, and of three, five,
    six or seven the rest reads nothing: what lies behind a problem's codes need not be there."""
    from duqlinear4bitcuda_amd import _lib

    reads = _lib.load().duq_product_long_reads_for
    for N in range(1, 257):
        for K in range(64, 4097, 64):
            assert reads(N, K) == (N + 31) // 32 * 32 * (K // 2), (N, K)
    assert reads(0, 512) == reads(257, 512) == reads(64, 0) == reads(64, 4160) == reads(64, 100) == 0
