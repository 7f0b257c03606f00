"""CPU checks of the choice between the mid-tile and the large-tile kernels."""
import pytest


@pytest.mark.parametrize("G,N,K,M,rows", [
    (32, 5760, 2880, 131072, 256), (4, 2880, 2880, 16384, 256), (7, 2048, 1424, 20000, 192),   # rows enough
    (32, 5760, 2880, 256, 64), (32, 5760, 2880, 3072, 128), (7, 2048, 1424, 5003, 128), (1, 16, 16, 1, 64),
    (257, 2048, 1424, 300, 192),                             # more groups than it holds
    (1, 16, 16, 0, 192), (1, 16, 16, 2 ** 31 - 257, 192),    # no rows; more tiles than one launch
])
def test_gemm_tile_rows(pkg, G, N, K, M, rows):
    assert pkg.persistent.tile_rows(G, N, K, K, K, N, M) == rows


def test_gemm_rows_of_c_within_32_bits(pkg):
    assert pkg.persistent.tile_rows(4, 2048, 1424, 1424, 1424, 2 ** 24 - 512 - 8, 100) == 64
    assert pkg.persistent.tile_rows(4, 2048, 1424, 1424, 1424, 2 ** 24, 100) == 192
