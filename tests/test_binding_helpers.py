"""The native binding's allocation helpers behave as torch.empty does: torch's own errors, other threads running meanwhile."""
import sys
import threading
import time

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


def test_other_threads_run_during_an_allocation():
    """A first allocation of a size asks the driver, and one that finds no memory waits for the GPU: neither holds the GIL.
    Here deterministic mode's filling of a large tensor takes the time."""
    count, done = [0], threading.Event()

    def spin():
        while not done.is_set():
            count[0] += 1

    like, was, interval = torch.zeros(1), torch.are_deterministic_algorithms_enabled(), sys.getswitchinterval()
    worker = threading.Thread(target=spin)
    try:
        torch.use_deterministic_algorithms(True)
        sys.setswitchinterval(1e-4)
        worker.start()
        rates = []
        for work in (lambda: time.sleep(0.1), *[lambda: _lib.native().empty_u8(like, 1 << 30)] * 3):
            t0, c0 = time.perf_counter(), count[0]
            t = work()
            rates.append((count[0] - c0) / (time.perf_counter() - t0))
    finally:
        done.set()
        worker.join()
        sys.setswitchinterval(interval)
        torch.use_deterministic_algorithms(was)
    assert bool((t[::1 << 20] == 255).all())   # the fill took place
    # held, the count stops but for a turn or two of the interpreter: 0.2 % of a fill of 0.1 s
    assert min(rates[1:]) > 0.05 * rates[0], rates
