"""The mid-tile kernels, which the library runs for launches of few rows or small tiles' worth of
output, against the 512-thread kernels: the same K partition and MFMA, so the same bits."""
import itertools

import pytest
import torch

from oracle import vark_oracle
from test_vark_backward_walk_host import walks_backwards

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
    ([400, 415, 0, 900, 127, 128, 1030], 2048, 1424, 128),
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


# rows of each group, OUT_M, OUT_N: ragged stages, tiles' edges, the ranked and the unranked deal
WGRAD = [
    ([5], 16, 16), ([0, 1, 127, 128, 129, 0, 300, 200], 208, 272), ([300, 0, 7], 640, 1152),
    ([3, 1] * 32, 128, 144), ([2, 0, 1] * 85 + [140], 144, 128),
]


@pytest.mark.parametrize("lens,m,n", WGRAD, ids=[f"{len(r[0])}groups{r[1]}x{r[2]}" for r in WGRAD])
def test_wgrad_equals_192_row_kernel(pkg, cuda, lens, m, n):
    """The bf16 result equals the drop-in code object's (the 192-row kernel), the transposed formats'
    result is the transpose's, and the fp32 modes agree with both, through padded and offset rows."""
    from ggemm_asm_amd import harness
    from ggemm_asm_amd.vark import weight_grad_fp8
    gen = torch.Generator().manual_seed(m + n)
    G, M = len(lens), sum(lens)
    offs = torch.tensor([0] + lens, device=cuda).cumsum(0)
    s = torch.tensor(0.01, device=cuda)
    run = pkg.grouped_gemm_fp8_tensorwise_variable_k
    module, func, _ = harness.load_kernel(pkg.CODE_OBJECT_PATH)
    try:
        for pad in (0, 48):
            assert pkg.load_library().ggemm_vark_tile_rows(G, m, n, n + pad, 0, M + 3, 256) == 128
            assert pkg.load_library().ggemm_vark_tile_rows(G, m, n, n + pad, 1, M + 3, 256) == 128
            lhs, rhs = (_fp8_bytes((M + 3, w), gen, pad, cuda) for w in (m, n))
            print(f"[gpu-case] mid wgrad {lens[:8]} {m}x{n} pad={pad}", flush=True)
            buf = torch.full((G, m, n + pad), 7.0, dtype=torch.bfloat16, device=cuda)
            run(lhs, rhs, s, s, offs, out=buf[..., :n])
            torch.cuda.synchronize()
            assert bool((buf[..., n:] == 7).all())
            got = buf[..., :n].contiguous()
            cl, cr = lhs.contiguous(), rhs.contiguous()
            ref = torch.full_like(got, 7.0)
            torch.cuda.synchronize()
            harness.launch_variable_k_kernel(func, cl, cr, ref, s, s, offs, G, m, n, harness.get_num_cus(0))
            torch.cuda.synchronize()
            assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
            f32 = run(lhs, rhs, s, s, offs, out_dtype=torch.float32)
            assert torch.equal(f32.bfloat16().view(torch.int16), got.view(torch.int16))
            wide = torch.randn((G, m, n + 12), device=cuda)
            acc = wide.clone()
            run(lhs, rhs, s, s, offs, out=acc[..., :n], accumulate=True)
            assert torch.equal(acc[..., :n], wide[..., :n] + f32) and torch.equal(acc[..., n:], wide[..., n:])
            e4m3, e5m2 = lhs.view(torch.float8_e4m3fn), rhs.view(torch.float8_e5m2)
            dw = weight_grad_fp8(e5m2, e4m3, s, s, offs)     # [G, n, m]
            err = (dw.transpose(1, 2).float() - f32).abs()
            # both round the same fp32 sums (of up to 3 more orders of additions) to bf16
            assert bool((err <= 2.0 ** -8 * f32.abs() + 1e-5 * float(f32.abs().max())).all())
    finally:
        harness.unload_kernel(module)


# m, n, lengths, tile rows, tiles of a group, stage, and for the fp32 and the accumulating mode (epilogue weight,
# stages that a tile's C is worth) as the kernels give them to make_sched
WALKS = [
    (1600, 1600, [900, 200, 31, 200, 200, 200, 4524, 4389, 200, 64, 900, 4443, 1, 1, 1, 1, 31, 900, 200, 0, 31, 900,
                  0, 1], 320, 25, 64, ((3, 16), (3, 32))),
    (2112, 1904, [5000, 3000, 0, 7, 64, 1, 31, 900] * 4, 192, 55, 128, ((2, 8), (4, 16))),
]


@pytest.mark.parametrize("m,n,lens,tile,tpg,stage,modes", WALKS, ids=["wide", "192row"])
def test_fp32_backward_walk_of_light_tiles(pkg, cuda, m, n, lens, tile, tpg, stage, modes):
    """Skewed lengths whose many small groups make the odd XCDs walk their tiles backwards, on the
    wide and the 192-row kernel, several rounds of them: the fp32 result rounds to the bf16 one (whose walk
    is forward), lies within the exact result's bound, and accumulating adds it exactly."""
    assert all(walks_backwards(lens, tpg, stage, *mode) for mode in modes)
    gen = torch.Generator().manual_seed(m)
    offs = torch.tensor([0] + lens, device=cuda).cumsum(0)
    rows = pkg.load_library().ggemm_vark_tile_rows
    assert [rows(len(lens), m, n, n, mode, sum(lens), 256) for mode in (0, 1, 2)] == [tile] * 3
    lhs, rhs = (_fp8_bytes((sum(lens), w), gen, 0, cuda) for w in (m, n))
    s = torch.tensor(0.01, device=cuda)
    run = pkg.grouped_gemm_fp8_tensorwise_variable_k
    bf16 = run(lhs, rhs, s, s, offs)
    f32 = run(lhs, rhs, s, s, offs, out=torch.full((len(lens), m, n), float("nan"), device=cuda),
              out_dtype=torch.float32)
    assert torch.equal(f32.bfloat16().view(torch.int16), bf16.view(torch.int16))
    for g in (lens.index(max(lens)), lens.index(900), lens.index(31), lens.index(0)):
        lo, hi = int(offs[g]), int(offs[g + 1])
        l, r = lhs[lo:hi, :192].cpu().numpy(), rhs[lo:hi, n - 208:].cpu().numpy()
        got = f32[g:g + 1, :192, n - 208:].double().cpu().numpy()
        bad, _ = vark_oracle.mfma_bound_violations(got, l, r, [0, hi - lo], 0.01, 0.01, out_rounding=0.0)
        assert not bad.any()
    c0 = torch.randn_like(f32)
    acc = c0.clone()
    run(lhs, rhs, s, s, offs, out=acc, accumulate=True)
    assert torch.equal(acc, c0 + f32)


@pytest.mark.parametrize("lens,N,K,kernel", [([0, 0], 208, 272, "auto"), ([70, 0, 5], 2048, 528, "auto"),
                                             ([300, 300], 208, 272, "512"), ([300, 1], 640, 128, "wide")])
def test_zero_tail_in_the_same_launch(pkg, cuda, lens, N, K, kernel):
    """Rows past the last group become zero, and only those, on every kernel; all rows when no group
    has one."""
    gen = torch.Generator().manual_seed(N)
    M, G, s = sum(lens) + 300, len(lens), torch.tensor(0.01, device=cuda)
    offs = torch.tensor([0] + lens, device=cuda).cumsum(0)
    a = _fp8_bytes((M, K), gen, 0, cuda).view(torch.float8_e4m3fn)
    b = _fp8_bytes((G, N, K), gen, 0, cuda).view(torch.float8_e4m3fn)
    buf = torch.full((2, M + 64, N + 16), 7.0, dtype=torch.bfloat16, device=cuda)
    for z in (0, 1):
        pkg.grouped_gemm_fp8_tensorwise(a, b, s, s, offs, out=buf[z, :M, :N], kernel=kernel, zero_tail=bool(z))
    torch.cuda.synchronize()
    rows = sum(lens)
    assert torch.equal(buf[0, :rows].view(torch.int16), buf[1, :rows].view(torch.int16))
    assert bool((buf[0, rows:] == 7).all()) and bool((buf[1, rows:M, :N] == 0).all())
    assert bool((buf[1, M:] == 7).all()) and bool((buf[1, :, N:] == 7).all())


@pytest.mark.parametrize("lens", [[5], [0, 3], [1, 0, 0]], ids=str)
def test_launches_of_one_to_three_tiles_on_the_192_row_kernel(pkg, cuda, lens):
    """The schedule's smallest launches: fewer units of work than slices, on the tensorwise (K=32) and
    the MXFP8 kernel, after a launch that leaves its schedule and stages in the LDS."""
    gen = torch.Generator().manual_seed(len(lens))
    G, M, m, n = len(lens), sum(lens), 64, 128
    offs = torch.tensor([0] + lens, device=cuda).cumsum(0)
    s = torch.tensor(0.01, device=cuda)
    run = pkg.grouped_gemm_fp8_tensorwise_variable_k
    full = torch.tensor([0, 600], device=cuda)
    large = [_fp8_bytes((600, w), gen, 0, cuda) for w in (1920, 5760)]
    x, dy = (torch.randn((M, w), generator=gen).to(cuda) for w in (m, n))
    e4m3, e5m2 = x.to(torch.float8_e4m3fn), dy.to(torch.float8_e5m2)
    ql, sl, padded = pkg.quantize_mxfp8_grouped(x, offs, "e4m3")
    qr, sr, _ = pkg.quantize_mxfp8_grouped(dy, offs, "e5m2")
    run(*large, s, s, full, mfma="k32")
    k32 = run(e4m3, e5m2, s, s, offs, mfma="k32")
    run(*large, s, s, full, mfma="k32")
    mx = pkg.grouped_gemm_mxfp8_variable_k(ql, qr, sl, sr, padded)
    # the fp8 MFMA drops bits some 11 places below a block's largest product, up to 2^-9 of it per block:
    # the rigorous bound on the same bytes, and one rounding to bf16
    for got, l, r, o, kw in ((k32, e4m3, e5m2, offs, {}), (mx, ql, qr, padded, {"lhs_sc": sl, "rhs_sc": sr})):
        bytes_l, bytes_r = (t.view(torch.uint8).cpu().numpy() for t in (l, r))
        scale = 1.0 if kw else float(s)
        bad, _ = vark_oracle.mfma_bound_violations(got.double().cpu().numpy(), bytes_l, bytes_r, o.cpu().numpy(),
                                                   scale, scale, **{k: v.cpu().numpy() for k, v in kw.items()})
        assert not bad.any()


@pytest.mark.parametrize("mode", ["bf16", "f32", "accumulate"])
def test_wgrad_empty_groups_do_not_see_the_scales(pkg, cuda, mode):
    """A group without tokens gives zeros and leaves an accumulated C as it is, -0 included, also where
    a scale is NaN or infinite (an activation was)."""
    lens, m, n = [0, 5, 0, 200], 64, 144
    gen = torch.Generator().manual_seed(3)
    offs = torch.tensor([0] + lens, device=cuda).cumsum(0)
    assert pkg.load_library().ggemm_vark_tile_rows(len(lens), m, n, n, int(mode != "bf16"), sum(lens), 256) == 128
    lhs, rhs = (_fp8_bytes((sum(lens), w), gen, 0, cuda) for w in (m, n))
    one = torch.ones((), device=cuda)
    for bad in (float("nan"), float("inf")):
        c0 = torch.full((len(lens), m, n), -0.0 if mode == "accumulate" else 7.0,
                        dtype=torch.bfloat16 if mode == "bf16" else torch.float32, device=cuda)
        c = pkg.grouped_gemm_fp8_tensorwise_variable_k(lhs, rhs, one * bad, one, offs, out=c0.clone(),
                                                       out_dtype=c0.dtype, accumulate=mode == "accumulate")
        for g in (0, 2):
            assert bool((c[g] == 0).all()) and bool(torch.signbit(c[g]).all()) == (mode == "accumulate")
        assert not bool(torch.isfinite(c[1]).any()) and not bool(torch.isfinite(c[3]).any())


@pytest.mark.parametrize("offs", [[0, 100, 300], [0, 0], [0, 700], [0, 100, 2000], [0, 90, -5]], ids=str)
def test_clear_tail_entry_equals_zero_tail(pkg, cuda, offs):
    """ggemm_persistent_clear_tail, for C callers with a GEMM launch of their own: the rows that zero_tail
    clears, of rows longer than N in a buffer with more rows, and no others."""
    N, K, M, G = 208, 272, 700, len(offs) - 1
    gen = torch.Generator().manual_seed(2)
    s, at = torch.tensor(0.01, device=cuda), torch.tensor(offs, device=cuda)
    a = _fp8_bytes((M, K), gen, 0, cuda).view(torch.float8_e4m3fn)
    b = _fp8_bytes((G, N, K), gen, 0, cuda).view(torch.float8_e4m3fn)
    buf = torch.full((2, M + 64, N + 16), 7.0, dtype=torch.bfloat16, device=cuda)
    for z in (0, 1):
        pkg.grouped_gemm_fp8_tensorwise(a, b, s, s, at, out=buf[z, :M, :N], zero_tail=bool(z))
    assert pkg.load_library().ggemm_persistent_clear_tail(
        buf[0].data_ptr(), N, N + 16, at.data_ptr(), G, M, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(buf[0].view(torch.int16), buf[1].view(torch.int16))
    rows = min(max(offs[-1], 0), M)
    assert bool((buf[0, rows:M, :N] == 0).all()) and bool((buf[0, M:] == 7).all()) and bool((buf[0, :, N:] == 7).all())


@pytest.mark.parametrize("N,K,kernel", [(208, 272, "auto"), (2048, 528, "auto"), (208, 272, "512"), (640, 128, "wide")])
@pytest.mark.parametrize("offs", [[0, 300, 200], [0, 700, 650, 10], [0, 90, -5], [0, 100, 2000]], ids=str)
def test_zero_tail_past_offsets_that_decrease(pkg, cuda, offs, N, K, kernel):
    """Rows from the last offset on become zero also where an earlier group ends past it (its tiles write
    none of them), the rows before it are the GEMM's; all rows for a negative last offset, none for one
    past the rows."""
    gen = torch.Generator().manual_seed(N)
    M, G, s = 700, len(offs) - 1, torch.tensor(0.01, device=cuda)
    a = _fp8_bytes((M, K), gen, 0, cuda).view(torch.float8_e4m3fn)
    b = _fp8_bytes((G, N, K), gen, 0, cuda).view(torch.float8_e4m3fn)
    at = torch.tensor(offs, device=cuda)
    buf = torch.full((2, M + 64, N + 16), 7.0, dtype=torch.bfloat16, device=cuda)
    for z in (0, 1):
        pkg.grouped_gemm_fp8_tensorwise(a, b, s, s, at, out=buf[z, :M, :N], kernel=kernel, zero_tail=bool(z))
    torch.cuda.synchronize()
    rows = min(max(offs[-1], 0), M)
    assert torch.equal(buf[0, :rows].view(torch.int16), buf[1, :rows].view(torch.int16))
    assert bool((buf[1, rows:M, :N] == 0).all())
    assert bool((buf[1, M:] == 7).all()) and bool((buf[1, :, N:] == 7).all())


def test_gemm_rows_of_several_groups(pkg, cuda):
    """Offsets that fall and rise again: rows of several groups have more tiles than the launch has
    workgroups, and the rows that only the last of them holds are computed too. One weight for all
    groups, so that every row has one result."""
    N, K, M = 128, 272, 512
    gen = torch.Generator().manual_seed(1)
    offs = torch.tensor([0, 400] * 127 + [0, 512], device=cuda)
    G, s = offs.numel() - 1, torch.tensor(0.01, device=cuda)
    assert pkg.persistent.tile_rows(G, N, K, K, K, N, M) == 64
    a = _fp8_bytes((M, K), gen, 0, cuda).view(torch.float8_e4m3fn)
    b = _fp8_bytes((1, N, K), gen, 0, cuda).view(torch.float8_e4m3fn)
    out = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=cuda)
    pkg.grouped_gemm_fp8_tensorwise(a, b.expand(G, N, K).contiguous(), s, s, offs, out=out)
    one = pkg.grouped_gemm_fp8_tensorwise(a, b, s, s, torch.tensor([0, M], device=cuda), kernel="512")
    assert torch.equal(out.view(torch.int16), one.view(torch.int16))
