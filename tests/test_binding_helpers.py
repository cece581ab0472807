"""The native binding's allocation helpers behave as torch.empty does: torch's own errors."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from mxfp4_int8_m5_amd import _lib


def test_an_error_keeps_its_type():
    class Refuse(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            raise KeyError("refused")

    like = torch.zeros(1)
    with Refuse(), pytest.raises(KeyError, match="refused"):
        _lib.native().empty_i8(like, 4)
    with pytest.raises(TypeError):
        _lib.native().empty_i8(like)
    with pytest.raises(RuntimeError):
        _lib.native().empty_i8(like, -4)


@pytest.mark.gpu
def test_out_of_memory_is_torchs():
    like = torch.zeros(1, device="cuda")
    torch.cuda.set_per_process_memory_fraction(0.25)   # the allocator refuses by itself beyond it
    try:
        with pytest.raises(torch.cuda.OutOfMemoryError):
            _lib.native().empty_u8(like, torch.cuda.get_device_properties(0).total_memory // 2)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
