"""CPU checks of what the torch ops refuse before anything is launched."""
import pytest
import torch

from __graft_entry__ import load_package

load_package()
from ggemm_asm_amd import _lib, quant, vark  # noqa: E402


@pytest.fixture
def launches(monkeypatch):
    """Calls that get past the checks, of tensors that stand for the GPU's."""
    calls = []
    monkeypatch.setattr(_lib, "launch", lambda name, *a: calls.append(name))
    monkeypatch.setattr(vark, "_check_inputs", lambda *a, **k: None)
    return calls


@pytest.mark.parametrize("bad", [torch.ones((), dtype=torch.float64), torch.ones(2), torch.ones((), device="meta")],
                         ids=["dtype", "elements", "device"])
def test_weight_grad_scales_are_checked(launches, bad):
    """The kernel reads a scale as one fp32 on its own device: anything else is another number or an
    address that is not the GPU's."""
    dy, x = torch.zeros((8, 32), dtype=torch.float8_e5m2), torch.zeros((8, 16), dtype=torch.float8_e4m3fn)
    one, offs = torch.ones(()), torch.tensor([0, 8])
    vark.weight_grad_fp8(dy, x, one, one, offs)
    assert launches == ["ggemm_vark_wgrad_fp8_swapped"]
    for scales in ((one, bad), (bad, one)):
        with pytest.raises(ValueError, match="scales"):
            vark.weight_grad_fp8(dy, x, *scales, offs)
    assert len(launches) == 1


@pytest.mark.parametrize("op", ["quantize_fp8_tensorwise_delayed", "quantize_fp8_tensorwise_transpose_delayed"])
@pytest.mark.parametrize("slot", [3, 2 ** 32 + 3, torch.zeros(1, dtype=torch.int32, device="meta")], ids=str)
def test_history_lengths_past_32_bits_are_refused(monkeypatch, op, slot):
    """A history of 2^32 + 16 entries is no history of 16, nor its slot 2^32 + 3 the slot 3."""
    monkeypatch.setattr(quant, "_check", lambda x, fmt: None)
    x = torch.empty((32, 64), dtype=torch.bfloat16, device="meta")
    with pytest.raises(OverflowError):
        getattr(quant, op)(x, torch.empty(2 ** 32 + 16, device="meta"), slot)
