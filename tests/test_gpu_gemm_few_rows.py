"""The few-row GEMM (blocked activations, up to 128 rows) against the tiled one on row-layout activations, whose results other
tests hold against the oracle: the same bits at the edges of its row tiles, with ragged column groups, with fewer K steps
than waves and with more than its loads in flight, for every weight format and epilogue; and just past its range."""
import numpy as np
import pytest
import torch

from oracle import bf16, layout
from tests.test_gpu_gemv_rows import FORMATS, packed
from tests.util import dev, host, llm_acts, product_format, random_packed

pytestmark = pytest.mark.gpu
GENERIC = layout.Format(block=32, code_mag=(0, 1, 2, 3, 4, 5, 6, 7), mult=(1, 3, 9, 15))


@pytest.mark.parametrize("name", [*FORMATS, "generic"])
@pytest.mark.parametrize("n,k", [(2048, 2048), (64, 128), (24, 384), (16, 896), (904, 4864), (40, 6144), (64, 12288), (64, 16640), (7512, 256)])
@pytest.mark.parametrize("m", [1, 15, 17, 32, 49, 64, 65, 96, 97, 128, 129, 290])
def test_equals_the_tiled_kernel(m, n, k, name):
    from mxfp4_int8_m5_amd import sc_kernels as S
    rng = np.random.default_rng(m * n + k)
    if name == "generic":
        c, b, w, _ = random_packed(rng, n, k, GENERIC)
        codes, bc, ws, fmt = dev(c), dev(b), dev(w), product_format(GENERIC)
    else:
        codes, bc, ws, fmt = packed(rng, n, k, name)
    x = dev(llm_acts(rng, m, k)[0])
    res = dev(bf16.to_bits(rng.standard_normal((m, n)).astype(np.float32)))
    wq = S.PackedWq(codes, bc, n, k, fmt, ws)
    xr, xs = S.act_quant(x, m)
    xb, xsb = S.act_quant_blocked(x, -(-m // 32) * 32)
    xb = S.BlockedXq(xb.data, m, k)
    assert np.array_equal(host(S.mm_i8_i32(xb, wq)), host(S.mm_i8_i32(xr, wq)))
    for epi in (1, 2, 3):
        kw = {"res": res} if epi == 2 else {}
        assert np.array_equal(host(S.mm_epi(xb, wq, xsb, ws, epi, **kw)), host(S.mm_epi(xr, wq, xs, ws, epi, **kw))), epi
    y = S.linear_w4a8(x, codes, bc, ws, n, 1, fmt=fmt)
    assert np.array_equal(host(y), host(S.mm_epi(xr, wq, xs, ws, 1)))


@pytest.mark.parametrize("name", [*FORMATS, "generic"])
@pytest.mark.parametrize("m,n,k", [(97, 1376, 2176), (112, 1544, 4224), (128, 2048, 4096)])
def test_two_groups_of_four_row_tiles(m, n, k, name):
    test_equals_the_tiled_kernel(m, n, k, name)
