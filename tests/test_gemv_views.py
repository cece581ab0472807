"""Which layouts of several rows the decode GEMV's wrapper takes: what it hands to the library, without a GPU."""
import pytest
import torch

from mxfp4_int8_m5_amd import _lib, sc_decode


class Recorder:
    """Stands in for the native binding: keeps the operands of the launch."""
    def __getattr__(self, name):
        return getattr(self.real, name)

    def __init__(self, real):
        self.real = real

    def scmx_gemv_rows_workspace(self, *_):
        return 0

    def scmx_gemv_rows(self, fmt, xq, xscale, codes, bcodes, wscale, res, *_):
        self.operands = xq, xscale, res


@pytest.mark.parametrize("rows", [3, 5, 6, 7])
def test_rows_between_the_kernel_sizes_may_be_views(rows, monkeypatch):
    nat = Recorder(_lib.native())
    monkeypatch.setattr(_lib, "native", lambda: nat)
    x = torch.arange(rows * 512, dtype=torch.int32).to(torch.int8).view(rows, 512)[:, 256:]
    xs, res = torch.rand(rows, 2)[:, 0], torch.rand(rows, 128).to(torch.bfloat16)[:, :64]
    sc_decode.gemv(x, None, None, xs, None, 64, 2, res=res)
    for got, want in zip(nat.operands, (x, xs, res)):
        assert got.is_contiguous() and torch.equal(got, want)
    sc_decode.gemv(x.to(torch.bfloat16), None, None, None, None, 64, 1, pro=1)
    assert nat.operands[0].is_contiguous() and nat.operands[1] is nat.operands[2] is None
