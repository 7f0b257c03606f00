"""The quantizers' two ways to load x, on both sides of the sizes where the choice changes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,mb", [(torch.bfloat16, 1), (torch.bfloat16, 299), (torch.bfloat16, 301),
                                      (torch.bfloat16, 1099), (torch.bfloat16, 1101), (torch.float32, 499),
                                      (torch.float32, 501)], ids=str)
def test_amax_on_both_sides_of_the_size_rule(pkg, cuda, dtype, mb):
    """The largest element found in the last row and the first, alone and before each quantizing pass."""
    cols = 2880
    rows = mb * 1000 * 1000 // (cols * dtype.itemsize) // 16 * 16
    x = torch.empty((rows, cols), dtype=dtype, device=cuda).normal_()
    for at, v in (((rows - 1, cols - 1), 100.0), ((0, 0), -200.0)):
        x[at] = v
        q, scale, am = pkg.quantize_fp8_tensorwise(x)
        _, q_t, scale_t, am_t = pkg.quantize_fp8_tensorwise_transpose(x, keep=False)
        assert float(am) == float(am_t) == float(pkg.amax(x)) == abs(v)
        assert float(scale) == float(scale_t) == float(torch.tensor(abs(v)) / 448)
        assert torch.equal(q.view(torch.uint8).t(), q_t.view(torch.uint8))
        assert float(q[at].float()) == (448.0 if v > 0 else -448.0)


@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
@pytest.mark.parametrize("rows,align", [(5744, None), (5760, None), (5744, 128)])
@pytest.mark.parametrize("mb", [274, 276])
def test_transposing_pass_on_both_sides_of_its_load_rule(pkg, cuda, mb, rows, align, fmt):
    """q^T rows off 128-byte lines, on them and padded to them, just below 275 MB of bf16 and just above: the
    same bytes as the streaming pass writes, which has one way to load."""
    batch = 16
    cols = mb * 1000 * 1000 // (2 * batch * rows) // 16 * 16 + (16 if mb > 275 else 0)
    x = torch.empty((batch, rows, cols), dtype=torch.bfloat16, device=cuda).normal_()
    x[-1, -1, -1], x[0, 0, 0] = 100.0, -200.0
    assert (x.nbytes > 275e6) == (mb > 275)
    q, scale, am = pkg.quantize_fp8_tensorwise(x.view(batch * rows, cols), fmt=fmt)
    q2, q_t, scale_t, am_t = pkg.quantize_fp8_tensorwise_transpose(x, fmt=fmt, row_align=align)
    assert q_t.stride(-2) == (rows if align is None else -(-rows // align) * align)
    assert float(am) == float(am_t) == 200.0 and float(scale) == float(scale_t)
    u = q.view(torch.uint8).view(batch, rows, cols)
    assert torch.equal(u, q2.view(torch.uint8))
    assert torch.equal(u.transpose(1, 2), q_t.view(torch.uint8))
