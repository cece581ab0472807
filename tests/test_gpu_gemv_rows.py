"""Several activation rows against one pass over the weights, at the row counts between the kernels' sizes and for every
format that has a half-precision MFMA form: wide and narrow layers, one piece of K and several, ragged row groups (which
leave for the general kernels).  Each row must be the bits of a one-row call, which other tests hold against the oracle."""
import numpy as np
import pytest
import torch

from oracle import bf16, layout
from tests.util import dev, host, llm_acts, product_format

pytestmark = pytest.mark.gpu
F32 = np.float32
FORMATS = {"published": layout.Format(), "sixteen": layout.Format(block=16),
           "range": layout.Format(block=16, mult=tuple(range(1, 11)), bc_bits=4),
           "high_range": layout.Format(block=16, mult=tuple(range(3, 11)), bc_bits=4), "mxfp4": None}


def packed(rng, n, k, name):
    from mxfp4_int8_m5_amd import sc_format as F
    codes = dev(rng.integers(0, 2 ** 32, n * k // 8, dtype=np.uint64).astype(np.uint32))
    ws = np.exp2(rng.integers(-12, -6, n)).astype(F32)
    fmt = FORMATS[name]
    if fmt is None:
        e8 = (rng.integers(0, 4, (n, k // 32)) + rng.integers(100, 120, (n, 1))).astype(np.uint8)
        return codes, dev(e8), F.mxfp4_row_scales(dev(e8)), F.MXFP4
    bc = rng.integers(0, len(fmt.mult), (n, k // fmt.block)).astype(np.uint8)
    per = 8 // fmt.bc_bits
    b = (bc.reshape(n, -1, per) << (np.arange(per, dtype=np.uint8) * fmt.bc_bits)).sum(-1).astype(np.uint8)
    return codes, dev(b), dev(ws), product_format(fmt)


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("n,k", [(32768, 2048), (32784, 1536), (32768, 512), (2048, 2048), (48, 512), (16, 6144), (64, 8192),
                                 (20, 1024), (1022, 512), (64, 896)])
@pytest.mark.parametrize("rows", [2, 3, 5, 8])
def test_rows_equal_single_rows(rows, n, k, name):
    from mxfp4_int8_m5_amd import sc_decode as G
    rng = np.random.default_rng(rows * n + k)
    codes, bc, ws, fmt = packed(rng, n, k, name)
    x = dev(llm_acts(rng, rows, k)[0])
    nw = dev(llm_acts(rng, 1, k)[0][0])
    xq = torch.from_numpy(rng.integers(-127, 128, (rows, k)).astype(np.int8)).cuda()
    xs = torch.from_numpy(rng.uniform(1e-3, 1e-2, rows).astype(F32)).cuda()
    res = dev(bf16.to_bits(rng.standard_normal((rows, n)).astype(F32)))
    for pro, epi in ((0, 1), (1, 2), (2, 3)):
        if epi == 3 and n % 4:
            continue
        kw = {"pro": pro, "fmt": fmt}
        if pro == 2:
            kw.update(nw=nw, eps=1e-6)
        a, s = (xq, xs) if pro == 0 else (x, None)
        y = host(G.gemv(a, codes, bc, s, ws, n, epi, res=res if epi == 2 else None, **kw))
        for b in range(rows):
            one = host(G.gemv(a[b], codes, bc, None if s is None else s[b:b + 1], ws, n, epi,
                              res=res[b] if epi == 2 else None, **kw))
            assert np.array_equal(y[b], one), (pro, epi, b)
