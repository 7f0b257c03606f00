"""The weight gradient in the weight's own orientation (e5m2 LHS, e4m3 RHS) against the oracle."""
import pytest
import torch

from oracle import vark_oracle as orc

pytestmark = pytest.mark.gpu


# N, K, groups without tokens after the others (more than 256 groups keep the mid tiles out), tile rows: the mid
# tiles, both wide tiles (320 x 320, 256 x 384 with a partial M-tile), the 192-row kernel on both of its tile
# widths and at its smallest shape; groups empty, of one token, around a stage and ragged
@pytest.mark.parametrize("N,K,spare,rows", [(16, 16, 0, 128), (1280, 640, 0, 128), (1920, 960, 0, 320),
                                            (1040, 1920, 0, 256), (192, 320, 257, 192), (208, 1728, 257, 192),
                                            (16, 16, 257, 192)])
def test_weight_grad_fp8(pkg, N, K, spare, rows):
    lens = [0, 1, 63, 64, 65, 200, 0, 131] + [0] * spare
    M = sum(lens) + 5                                     # rows past the last group are not read
    assert pkg.load_library().ggemm_vark_tile_rows(len(lens), N, K, K, 0, M, 256) == rows
    gen = torch.Generator().manual_seed(N + K)
    dy = (torch.randn(M, N, generator=gen) * 8).to(torch.float8_e5m2)
    x = (torch.randn(M, K, generator=gen) * 8).to(torch.float8_e4m3fn)
    offs = torch.tensor([0] + lens).cumsum(0)
    sdy, sx = 0.25, 0.037
    ref = orc.vark_wgrad_tensorwise(x.view(torch.uint8).numpy(), dy.view(torch.uint8).numpy(), sx, sdy, offs.numpy())
    from ggemm_asm_amd.vark import weight_grad_fp8
    dev = torch.device("cuda")
    dw = weight_grad_fp8(dy.to(dev), x.to(dev), torch.tensor(sdy, device=dev), torch.tensor(sx, device=dev), offs.to(dev))
    assert dw.is_contiguous() and tuple(dw.shape) == (len(lens), N, K)
    m = orc.compare(pkg.as_bf16_bits(dw.transpose(1, 2)), ref, offs.numpy())
    assert orc.parity_ok(m), m
