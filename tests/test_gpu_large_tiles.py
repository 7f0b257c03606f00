"""The 192-row wgrad kernel behind the automatic choice, on shapes small enough for the oracle: groups
without tokens past 256 keep the mid tiles out, so that the tensorwise kernel runs at every output mode, on
both tile widths."""
import pytest
import torch

import test_gpu_parity as parity

pytestmark = pytest.mark.gpu
SPARE = [0] * 257


def _on_192_rows(pkg, lens, om, on, modes=(0, 1, 2)):
    for mode in modes:
        assert pkg.load_library().ggemm_vark_tile_rows(len(lens), om, on, on, mode, sum(lens), 256) == 192


@pytest.mark.parametrize("lens,om,on", [([127, 128, 129, 0, 256, 257], 208, 336), ([1, 2, 3, 5, 8, 13], 16, 16),
                                        ([300, 0, 645], 64, 1152), ([255, 0, 129, 640], 208, 1728),
                                        ([4096 + 77, 31], 384, 320)], ids=["c320", "tiny", "c384", "half384", "long"])
def test_ragged_groups_vs_oracle(pkg, orc, cuda, lens, om, on):
    _on_192_rows(pkg, lens + SPARE, om, on, (0,))
    parity.test_ragged_groups_vs_oracle(pkg, orc, cuda, lens + SPARE, om, on, "k128")


@pytest.mark.parametrize("lens,om,on", [([127, 128, 0, 255, 256, 257], 208, 336), ([300, 0, 645], 208, 768),
                                        ([300, 0, 129], 16, 1728), ([31] * 4 + [0] * 2, 16, 384)],
                         ids=["c320", "c384", "half384", "tiny"])
def test_fp32_output_and_accumulate(pkg, orc, cuda, lens, om, on):
    _on_192_rows(pkg, lens + SPARE, om, on)
    parity.test_fp32_output_and_accumulate(pkg, orc, cuda, lens + SPARE, om, on)


@pytest.mark.parametrize("kind", ["bf16", "f32", "f32_acc"])
@pytest.mark.parametrize("on", [320, 384])
def test_offsets_past_token_count_are_clamped(pkg, orc, cuda, kind, on):
    """As on the mid tiles: rows past M hold bytes that would change the result; offsets before 0 and past M
    are clamped, a group past M is empty."""
    M, om = 457, 208
    offs = torch.tensor([-64, 100, 100, 400, 600] + [800] * 258, dtype=torch.int64)
    clamped, G = offs.clamp(min=0, max=M), offs.numel() - 1
    lens = torch.diff(clamped).tolist()
    _on_192_rows(pkg, lens, om, on)
    lhs, rhs, _, _, (sl, sr) = parity._rand_bytes_problem(lens, om, on, seed=43)
    dl, dr = (torch.cat([t, torch.full((512, t.shape[1]), 0x38, dtype=torch.uint8)]).to(cuda)[:M] for t in (lhs, rhs))
    s1, s2 = (torch.tensor(v, dtype=torch.float32, device=cuda) for v in (sl, sr))
    fp32 = kind != "bf16"
    out = torch.zeros((G, om, on), dtype=torch.float32 if fp32 else torch.bfloat16, device=cuda)
    pkg.grouped_gemm_fp8_tensorwise_variable_k(dl, dr, s1, s2, offs.to(cuda), out=out, out_dtype=out.dtype,
                                               accumulate=kind == "f32_acc")
    torch.cuda.synchronize()
    if fp32:
        ref = orc.vark_wgrad_tensorwise_f32(lhs.numpy(), rhs.numpy(), sl, sr, clamped.numpy())
        parity._f32_parity(orc, out.cpu().numpy(), ref, f"192-row clamp/{kind}")
    else:
        ref = orc.vark_wgrad_tensorwise(lhs.numpy(), rhs.numpy(), sl, sr, clamped.numpy())
        parity._assert_parity(orc, pkg.as_bf16_bits(out), ref, clamped.numpy(), "192-row clamp/bf16")
    assert bool((out[1] == 0).all()) and bool((out[4:] == 0).all())


def test_gemm_of_spread_starts(pkg, cuda):
    """Three tiles a workgroup, C rows off the 128-byte lines: the workgroups start one after the other. The
    same rows with C on the lines, where they start as one, have the same bits."""
    G, N, K, s = 3, 16, 512, torch.tensor(0.01, device=cuda)
    M = 768 * 192 + 5
    gen = torch.Generator().manual_seed(4)
    a = torch.randn((M, K), generator=gen).to(torch.float8_e4m3fn).to(cuda)
    b = torch.randn((G, N, K), generator=gen).to(torch.float8_e4m3fn).to(cuda)
    offs = torch.tensor([0, 700, 701, M], device=cuda)
    outs = [torch.full((M, stride), 7.0, dtype=torch.bfloat16, device=cuda)[:, :N] for stride in (24, 64)]
    for out in outs:
        pkg.grouped_gemm_fp8_tensorwise(a, b, s, s, offs, out=out, kernel="512")
    assert torch.equal(*(o.contiguous().view(torch.int16) for o in outs))


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_wgrad_of_spread_starts(pkg, orc, cuda, mode):
    """Three 320 x 320 tiles a workgroup and one to four stages each, the workgroups started one after the
    other: two groups against the exact result's bound."""
    lens, m, n = [300, 1, 0, 517] * 12, 1280, 1280
    assert pkg.load_library().ggemm_vark_tile_rows(len(lens), m, n, n, mode, sum(lens), 256) == 320
    assert len(lens) * 16 >= 3 * 256 and 1 <= sum(-(-v // 64) for v in lens) / len(lens) / 2 <= 4
    gen = torch.Generator().manual_seed(mode)
    lhs, rhs = ((torch.randint(0, 256, (sum(lens), w), generator=gen).to(torch.uint8) & 0xbb) for w in (m, n))
    offs, s = torch.tensor([0] + lens).cumsum(0), torch.tensor(0.01, device=cuda)
    dt = torch.float32 if mode else torch.bfloat16
    c0 = torch.zeros((len(lens), m, n), dtype=dt, device=cuda) if mode == 2 else None
    c = pkg.grouped_gemm_fp8_tensorwise_variable_k(lhs.to(cuda), rhs.to(cuda), s, s, offs.to(cuda), out=c0,
                                                   out_dtype=dt, accumulate=mode == 2)
    for g in (1, 47):
        lo, hi = int(offs[g]), int(offs[g + 1])
        bad, _ = orc.mfma_bound_violations(c[g:g + 1, -160:, :176].double().cpu().numpy(), lhs[lo:hi, m - 160:].numpy(),
                                           rhs[lo:hi, :176].numpy(), [0, hi - lo], 0.01, 0.01,
                                           out_rounding=0.0 if mode else 2.0 ** -8)
        assert not bad.any()
    assert bool((c[2::4] == 0).all())
