"""The mid-tile kernels, which the library runs for launches of few rows or small tiles' worth of
output, against the 512-thread kernels: the same K partition and MFMA, so the same bits."""
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu


def _fp8_bytes(shape, gen, pad, cuda):
    """Random fp8 bytes without NaN and infinity codes, rows `pad` bytes longer than the view."""
    t = torch.randint(0, 256, shape[:-1] + (shape[-1] + pad,), generator=gen, dtype=torch.int32)
    return (t.to(torch.uint8) & 0xbb).to(cuda)[..., :shape[-1]]


GEMM = [  # rows of each group, N, K, tile rows
    ([5], 16, 16, 64),
    ([0, 1, 63, 64, 65, 0, 129, 200], 208, 272, 64),
    ([3] * 256, 144, 128, 64),                       # the most groups it takes
    ([300, 0, 5, 4000], 640, 2880, 64),
    ([700, 715, 0, 1200, 127, 128, 2133], 2048, 1424, 128),
]


@pytest.mark.parametrize("lens,N,K,rows", GEMM, ids=[f"{r[3]}rows{i}" for i, r in enumerate(GEMM)])
def test_gemm_equals_512_thread_kernel(pkg, cuda, lens, N, K, rows):
    gen = torch.Generator().manual_seed(N + K)
    G, M = len(lens), sum(lens)
    offs = torch.tensor([0] + lens, device=cuda).cumsum(0)
    s = torch.tensor(0.01, device=cuda)
    for dt, pad in itertools.product((torch.float8_e4m3fn, torch.float8_e5m2), (0, 48)):
        # a few rows past the last group, and rows, weights and results that are longer than their views
        a = _fp8_bytes((M + 3, K), gen, pad, cuda).view(dt)
        b = _fp8_bytes((G, N, K), gen, pad, cuda).view(torch.float8_e4m3fn)
        assert pkg.persistent.tile_rows(G, N, K, K + pad, K + pad, N + pad, M + 3) == rows
        outs = []
        for kernel in ("auto", "512"):
            buf = torch.full((M + 3, N + pad), 7.0, dtype=torch.bfloat16, device=cuda)
            print(f"[gpu-case] mid gemm {dt} {lens[:8]} N={N} K={K} pad={pad} {kernel}", flush=True)
            pkg.grouped_gemm_fp8_tensorwise(a, b, s, s, offs, out=buf[:, :N], kernel=kernel)
            torch.cuda.synchronize()
            assert bool((buf[M:] == 7).all()) and bool((buf[:, N:] == 7).all())   # nothing outside is written
            outs.append(buf[:M, :N].contiguous().view(torch.int16))
        assert torch.equal(*outs)
