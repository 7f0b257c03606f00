"""The quantizers with and without a workspace: the same bytes, scale and amax."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,cols", [(0, 16), (1, 16), (3, 64), (1024, 128), (70001, 48)])
def test_workspace_equals_atomic_amax(pkg, cuda, rows, cols, dtype):
    lib = pkg.load_library()
    x = torch.randn((max(rows, 1), cols), generator=torch.Generator().manual_seed(rows)).to(dtype).to(cuda)
    stream = torch.cuda.current_stream().cuda_stream
    f32 = int(dtype == torch.float32)
    got = []
    for ws in (torch.full((2048,), -1, dtype=torch.int32, device=cuda), None):   # any content before the call
        q = torch.zeros((max(rows, 1), cols), dtype=torch.uint8, device=cuda)
        qt = torch.zeros((cols, 16 * max(rows // 16, 1)), dtype=torch.uint8, device=cuda)
        scale, amax = torch.full((2, 2), 7.0, device=cuda)
        name, tail = ("_ws", (ws.data_ptr(), stream)) if ws is not None else ("", (stream,))
        rc = getattr(lib, "ggemm_quant_fp8_tensorwise" + name)(
            x.data_ptr(), f32, rows, cols, cols, 0, q.data_ptr(), cols, scale.data_ptr(), amax.data_ptr(), *tail)
        assert rc == 0
        if rows >= 16:
            rc = getattr(lib, "ggemm_quant_fp8_tensorwise_transpose" + name)(
                x.data_ptr(), f32, 1, rows // 16 * 16, cols, 1, None, cols, qt.data_ptr(), qt.stride(0),
                scale[1:].data_ptr(), amax[1:].data_ptr(), *tail)
            assert rc == 0
        torch.cuda.synchronize()
        got.append((q, qt, scale, amax))
    assert all(torch.equal(a, b) for a, b in zip(*got))
    assert float(got[0][3][0]) == (float(x.float().abs().max()) if rows else 0.0)
