"""Several activation rows against one pass over the weights, at the row counts between the kernels' sizes and for every
format that has a half-precision MFMA form: wide and narrow layers, one piece of K and several, ragged row groups (which
leave for the general kernels).  Each row must be the bits of a one-row call, which other tests hold against the oracle."""
import numpy as np
import pytest
import torch

from oracle import bf16, layout, linear
from tests.util import dev, host, llm_acts, product_format, random_packed

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


@pytest.mark.parametrize("rows", [3, 5, 6, 7, 11])
def test_views_of_rows(rows):
    """Row counts between the kernels' sizes have always been taken from any layout: columns of a wider matrix, every other row."""
    from mxfp4_int8_m5_amd import sc_decode as G
    rng = np.random.default_rng(rows)
    n, k = 256, 512
    codes, bc, ws, fmt = packed(rng, n, k, "published")
    x = dev(llm_acts(rng, rows, 2 * k)[0])
    xs = torch.from_numpy(rng.uniform(1e-3, 1e-2, 2 * rows).astype(F32)).cuda()
    xq = torch.from_numpy(rng.integers(-127, 128, (rows, 2 * k)).astype(np.int8)).cuda()
    res = dev(bf16.to_bits(rng.standard_normal((rows, 2 * n)).astype(F32)))
    if rows > 8:   # eight rows and a rest of three: the first eight have to be contiguous
        x, xq, xs, res = x[:, :k].contiguous(), xq[:, :k].contiguous(), xs[:rows], res[:, :n].contiguous()
    else:
        x, xq, xs, res = x[:, k:], xq[:, k:], xs[::2], res[:, n:]
        assert not any(t.is_contiguous() for t in (x, xq, xs, res))
    c = lambda t: t.contiguous()   # noqa: E731
    for epi in (1, 2):
        r = {"res": res} if epi == 2 else {}
        rc = {"res": c(res)} if epi == 2 else {}
        assert torch.equal(G.gemv(xq, codes, bc, xs, ws, n, epi, fmt=fmt, **r), G.gemv(c(xq), codes, bc, c(xs), ws, n, epi, fmt=fmt, **rc))
        assert torch.equal(G.gemv(x, codes, bc, None, ws, n, epi, pro=1, fmt=fmt, **r),
                           G.gemv(c(x), codes, bc, None, ws, n, epi, pro=1, fmt=fmt, **rc))


@pytest.mark.parametrize("rows", [1, 2, 3, 8])
@pytest.mark.parametrize("k", [128, 896, 2176])
@pytest.mark.parametrize("fmt", [layout.Format(block=16, mult=tuple(range(1, 11)), bc_bits=4), layout.Format(block=16),
                                 layout.Format(code_mag=(0, 1, 2, 3, 4, 5, 6, 7), mult=(1, 3, 9, 15)),
                                 layout.Format(block=8, code_mag=(0, 1, 2, 3, 4, 5, 6, 7), mult=(1, 3, 9, 15), bc_bits=8)])
def test_block_codes_at_the_end_of_their_memory(fmt, k, rows):
    """Rows that do not fill the lanes of a step: the lanes past the end read no block codes past the last row.  The block codes
    are the last bytes of an allocation that is whole pages of its own (20 MiB)."""
    from mxfp4_int8_m5_amd import sc_decode as G
    rng = np.random.default_rng(k + rows)
    n, pf = 1152, product_format(fmt)
    c, b, w, q = random_packed(rng, n, k, fmt)
    whole = torch.empty(20 << 20, dtype=torch.uint8, device="cuda")
    bc = whole[-b.size:].view(b.shape)
    bc.copy_(dev(b))
    xq = rng.integers(-127, 128, (rows, k)).astype(np.int8)
    xs = rng.uniform(1e-3, 1e-2, rows).astype(F32)
    y = host(G.gemv(dev(xq), dev(c), bc, dev(xs), dev(w), n, 1, fmt=pf)).reshape(rows, n)
    assert np.array_equal(y, linear.gemv(xq, xs, q, w, 1).reshape(rows, n))
