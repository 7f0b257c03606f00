"""CPU checks of the choice between the mid-tile and the large-tile kernels."""
import random

import pytest


@pytest.mark.parametrize("G,N,K,M,rows", [
    (32, 5760, 2880, 131072, 256), (4, 2880, 2880, 16384, 256), (7, 2048, 1424, 20000, 192),   # rows enough
    (32, 5760, 2880, 256, 64), (32, 5760, 2880, 3072, 128), (7, 2048, 1424, 5003, 192), (7, 2048, 1424, 3000, 128), (1, 16, 16, 1, 64),
    (257, 2048, 1424, 300, 192),                             # more groups than it holds
    (1, 16, 16, 0, 192), (1, 16, 16, 2 ** 31 - 257, 192),    # no rows; more tiles than one launch
])
def test_gemm_tile_rows(pkg, G, N, K, M, rows):
    assert pkg.persistent.tile_rows(G, N, K, K, K, N, M) == rows


def test_gemm_rows_of_c_within_32_bits(pkg):
    assert pkg.persistent.tile_rows(4, 2048, 1424, 1424, 1424, 2 ** 24 - 512 - 8, 100) == 64
    assert pkg.persistent.tile_rows(4, 2048, 1424, 1424, 1424, 2 ** 24, 100) == 192


@pytest.mark.parametrize("G,m,n,M,mode,rows", [
    (32, 2880, 5760, 131072, 0, 320), (4, 2880, 2880, 16384, 2, 320), (12, 1600, 1600, 100000, 0, 320),
    (1, 16, 16, 0, 0, 128), (4, 64, 128, 512, 0, 128), (4, 2880, 2880, 1024, 0, 320), (4, 2880, 2880, 1024, 2, 128), (8, 512, 1024, 100000, 0, 128),
    (12, 1600, 1600, 1000, 2, 128), (257, 64, 128, 512, 0, 192),
    (4, 64, 128, 2 ** 31, 0, 192),                           # no 32-bit token count
    (256, 65536, 65536, 256, 0, 192),                        # more tiles than one launch
])
def test_wgrad_tile_rows(pkg, G, m, n, M, mode, rows):
    assert pkg.load_library().ggemm_vark_tile_rows(G, m, n, n, mode, M, 256) == rows


def test_wgrad_fp32_modes_take_the_same_kernel(pkg):
    """Accumulating adds what the fp32 mode writes, bit for bit, only if one kernel computes both."""
    rows = pkg.load_library().ggemm_vark_tile_rows
    for G in (1, 4, 32):
        for m, n in ((64, 128), (1600, 1600), (2880, 2880), (2880, 5760), (2048, 528)):
            for M in (16, 1000, 4096, 16384, 131072):
                assert rows(G, m, n, n, 1, M, 256) == rows(G, m, n, n, 2, M, 256)


def test_wgrad_unaligned_rows_of_c_keep_the_192_row_kernel(pkg):
    rows = pkg.load_library().ggemm_vark_tile_rows
    assert rows(4, 64, 128, 136, 0, 512, 256) == 128 and rows(4, 64, 128, 132, 0, 512, 256) == 192
    assert rows(4, 64, 128, 132, 1, 512, 256) == 128


def test_gemm_workgroups_cover_the_rows_of_any_offsets():
    """Model of the mid-tile GEMM's rows (load_groups) and grid (capi): every row that a group holds is taken
    once, by the first group that holds it, and the tiles are no more than the workgroups, also where offsets
    decrease and rise again (from the first on, which is zero)."""
    rng = random.Random(0)
    for rows in (64, 128):
        for _ in range(300):
            G, M, n_tn = rng.randint(1, 256), rng.randint(1, 3000), rng.randint(1, 9)
            offs = [0] + [rng.randint(0, M) for _ in range(G)]
            if rng.random() < 0.5:
                offs.sort()
            grid = -(-(M // rows + min(G, M)) * n_tn // 256) * 256
            held, taken, tiles, past = set(), [], 0, 0
            for a, b in zip(offs, offs[1:]):
                held |= set(range(a, b))
                start = max(a, past)
                taken += range(start, b)
                assert offs != sorted(offs) or start == a
                tiles += -(-max(b - start, 0) // rows) * n_tn
                past = max(past, b)
            assert len(taken) == len(set(taken)) and set(taken) == held and tiles <= grid
            order = [b - b % 256 + b % 8 * 32 + b % 256 // 8 for b in range(grid)]
            assert sorted(order) == list(range(grid))


@pytest.mark.parametrize("G,m,n,M,mode,rows", [
    (1, 2880, 2880, 100930, 0, 320), (1, 2880, 2880, 100930, 2, 320), (2, 2880, 3312, 106369, 0, 192),
    (5, 2544, 1744, 17692, 0, 192), (1, 1984, 5760, 114333, 0, 256),
    (14, 2880, 144, 80476, 2, 128), (8, 512, 1024, 1000, 0, 128), (2, 1024, 2048, 8000, 0, 128), (12, 1600, 1600, 1000, 1, 128),   # still mid
])
def test_wgrad_of_whole_rounds(pkg, G, m, n, M, mode, rows):
    """Launches on which the mid tiles measured slower than the large ones, next to some they serve."""
    assert pkg.load_library().ggemm_vark_tile_rows(G, m, n, n, mode, M, 256) == rows


@pytest.mark.parametrize("G,N,K,M,rows", [
    (13, 2880, 2880, 5788, 256), (15, 2560, 5760, 7007, 256), (2, 2320, 2880, 3715, 128),
    (4, 2880, 2880, 8192, 128), (8, 512, 1024, 100000, 128), (32, 5760, 2880, 3072, 128), (32, 5760, 2880, 256, 64),
])
def test_gemm_of_whole_rounds(pkg, G, N, K, M, rows):
    assert pkg.persistent.tile_rows(G, N, K, K, K, N, M) == rows
