"""The amax pass's two ways to load x, on both sides of the sizes where the choice changes."""
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
