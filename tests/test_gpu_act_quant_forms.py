"""The activation quantizer in both layouts against the oracle, bit for bit, through each of its forms: a workgroup per row (few
rows, long rows), a wave per row with whole and with partial register pieces (codes of long blocked rows leaving in two turns),
and the forms that read a row twice."""
import numpy as np
import pytest

from oracle import bf16, linear
from tests.util import blocked_layout, dev, host, llm_acts

pytestmark = pytest.mark.gpu

# (rows, rows with padding, row length)
WORKGROUP = [(3, 3, 2080), (5, 8, 4096), (1, 1, 4128), (7, 7, 8192), (256, 256, 2560), (3, 4, 8224), (300, 301, 12288), (2, 2, 16384)]
WAVE = [(5, 6, k) for k in (32, 512, 544, 1024, 1056, 1536, 1568, 2048)] + \
       [(258, 259, k) for k in (2080, 2560, 3072, 3584, 4096, 4128, 5120, 5632, 6144, 6176, 7680, 8192)]
TWICE = [(5, 7, 1000), (3, 3, 16416), (260, 260, 8), (258, 258, 20480)]
BLOCKED = [(1, 32, 544), (20, 32, 1024), (70, 96, 1056), (128, 128, 2048),                      # a workgroup per row
           (250, 256, 4096), (33, 64, 4128), (40, 64, 8192), (3, 32, 8224), (32, 32, 12288), (9, 32, 16384), (289, 320, 12320),
           (32, 32, 32), (7, 32, 512), (130, 160, 544), (130, 160, 1024), (160, 160, 1536), (129, 160, 1568), (130, 160, 2048),
           (260, 288, 2080), (288, 288, 3072), (257, 288, 3584), (260, 288, 4096), (257, 288, 5120), (260, 288, 6144),
           (257, 288, 6176), (260, 288, 8192), (257, 288, 8224), (288, 288, 11808), (257, 288, 12288),   # a wave per row
           (5, 32, 16416), (260, 288, 20480)]                                                     # read twice


def acts(m, k):
    rng = np.random.default_rng(m * k)
    bits, x = llm_acts(rng, m, k)
    if m > 2:   # a row of zeros, and one whose largest value is its last
        x = x.copy()
        x[1] = 0.0
        x[2, -1] = -4.0 * np.abs(x[2]).max()
        bits = bf16.to_bits(x)
        x = bf16.from_bits(bits)
    return bits, x


@pytest.mark.parametrize("m,mp,k", WORKGROUP + WAVE + TWICE)
def test_rows(m, mp, k):
    from mxfp4_int8_m5_amd import sc_kernels as S
    bits, x = acts(m, k)
    xq, xs = S.act_quant(dev(bits), mp)
    rq, rs = linear.act_quant(x, mp)
    assert np.array_equal(host(xs), rs) and np.array_equal(host(xq), rq)


@pytest.mark.parametrize("m,mp,k", BLOCKED)
def test_blocked(m, mp, k):
    from mxfp4_int8_m5_amd import sc_kernels as S
    bits, x = acts(m, k)
    bx, xs = S.act_quant_blocked(dev(bits), mp)
    rq, rs = linear.act_quant(x, mp)
    assert np.array_equal(host(xs), rs) and np.array_equal(host(bx.data), blocked_layout(rq))


@pytest.mark.parametrize("m,k", [(3, 4096), (2, 12288)])
def test_rows_into_unaligned_codes(m, k):
    """Codes 8 bytes past an aligned address: the forms with 16-byte stores stand back."""
    import torch

    from mxfp4_int8_m5_amd import _lib
    bits, x = acts(m, k)
    xq, xs = torch.empty(m * k + 8, dtype=torch.int8, device="cuda")[8:], torch.empty(m, dtype=torch.float32, device="cuda")
    _lib.native().scmx_act_quant(dev(bits), xq, xs, m, m, k)
    rq, rs = linear.act_quant(x, m)
    assert np.array_equal(host(xs), rs) and np.array_equal(host(xq).reshape(m, k), rq)
