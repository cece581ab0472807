"""The device quantizers where a thread owns a block and a workgroup several rows: row lengths that leave part of the last
workgroup empty, rows longer than a workgroup has threads, pointers without 16-byte alignment, and weights built so that
float32 sums cannot decide between exponents.  Against the numpy oracle, bit for bit."""
import numpy as np
import pytest
import torch

from oracle import bf16, family, layout
from tests.util import host, llm_weights, product_format

pytestmark = pytest.mark.gpu
F32 = np.float32


def _device(w, as_bf16, shift):
    """w on the GPU, `shift` elements past an aligned address."""
    t = torch.from_numpy(w).cuda()
    t = t.to(torch.bfloat16) if as_bf16 else t
    if not shift:
        return t
    buf = torch.zeros(w.size + shift, dtype=t.dtype, device="cuda")
    buf[shift:] = t.reshape(-1)
    return buf[shift:].view(w.shape)


@pytest.mark.parametrize("block", [16, 32])
@pytest.mark.parametrize("n,k,as_bf16,shift", [(1, 128, False, 0), (67, 128, True, 0), (19, 896, True, 0), (3, 4864, True, 3),
                                               (5, 6144, False, 1), (2, 8192, True, 0), (3, 12288, False, 0), (130, 384, True, 0)])
def test_published_format(n, k, as_bf16, shift, block):
    from mxfp4_int8_m5_amd import sc_format as SF
    rng = np.random.default_rng(n * k + block)
    w = llm_weights(rng, n, k).astype(F32)
    # blocks whose candidates tie or nearly tie: whole levels (zero error at two exponents), one value far below the rest
    lv = np.array([0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0])
    w[0, :64] = rng.choice(lv, 64) * 2.0 ** -4
    w[0, 64:96] = 3.0
    w[0, 64] = 2.0 ** -60
    w[-1, :32] = 1.25 * np.where(np.arange(32) % 2, 1, -1)
    if as_bf16:
        w = bf16.from_bits(bf16.to_bits(w))
    fmt = layout.Format(block=block)
    codes, bc, ws, q = layout.quantize(w.astype(np.float64), fmt)
    dc, db, dw, dq = SF.quantize(_device(w, as_bf16, shift), product_format(fmt))
    assert np.array_equal(host(dc).view(np.uint32), codes)
    assert np.array_equal(host(db), bc) and np.array_equal(host(dw), ws) and np.array_equal(host(dq), q)


@pytest.mark.parametrize("name", ["e2m1/B16/M1..10", "e2m1/B32/M1..8", "int4/B16/M1..16"])
@pytest.mark.parametrize("n,k,as_bf16,shift", [(1, 128, False, 0), (9, 256, True, 0), (6, 896, True, 1), (3, 4864, False, 0),
                                               (2, 12288, True, 0), (5, 2048, False, 1)])
def test_family(n, k, as_bf16, shift, name):
    from mxfp4_int8_m5_amd import pack_format as P
    fam = family.member(name)
    sf = fam.storage()
    rng = np.random.default_rng(n * k)
    w = llm_weights(rng, n, k).astype(F32)
    w[0, :128] = rng.integers(-24, 25, 128) * F32(np.abs(w[0]).max() / 24)   # quotients on and next to the midpoints
    if as_bf16:
        w = bf16.from_bits(bf16.to_bits(w))
    _, qi, base, scales = family.quantize(w, fam)
    codes, bc, ws = family.pack_parts(qi, base, scales, sf)
    dc, db, dw, _ = P.pack_matrix(_device(w, as_bf16, shift), name)
    assert np.array_equal(host(dw), ws) and np.array_equal(host(db), bc)
    assert np.array_equal(host(dc).view(np.uint32), codes)


@pytest.mark.parametrize("name", ["e2m1/B16/M1..10", "int4/B16/M1..16"])
def test_family_many_blocks(name):
    """Enough blocks for a thread to take all bases of one (70400 and 35200; the shapes above spread a block's bases over threads)."""
    test_family(1100, 512, True, 0, name)
    test_family(1100, 1024, True, 0, name)


@pytest.mark.parametrize("block", [16, 32])
@pytest.mark.parametrize("as_bf16", [False, True])
@pytest.mark.parametrize("share", [0.002, 0.1, 1.0])
def test_published_format_ties(share, as_bf16, block):
    """Blocks of whole levels, whose sums tie or vanish at two exponents, among blocks that do not: none or a few of a wave's
    lanes have one (the wave sums it), many or all (each lane its own)."""
    from mxfp4_int8_m5_amd import sc_format as SF
    rng = np.random.default_rng(int(1000 * share) + block)
    n, k = 70, 1024
    w = llm_weights(rng, n, k).astype(F32)
    tied = np.repeat(rng.random((n, k // block)) < share, block, axis=1)
    w[tied] = (rng.choice([0.0, 1.0, 2.0, 3.0, 4.0, 6.0], tied.sum()) * rng.choice([-1, 1], tied.sum()) * 2.0 ** -4).astype(F32)
    if as_bf16:
        w = bf16.from_bits(bf16.to_bits(w))
    fmt = layout.Format(block=block)
    codes, bc, ws, q = layout.quantize(w.astype(np.float64), fmt)
    dc, db, dw, dq = SF.quantize(_device(w, as_bf16, 0), product_format(fmt))
    assert np.array_equal(host(dc).view(np.uint32), codes)
    assert np.array_equal(host(db), bc) and np.array_equal(host(dw), ws) and np.array_equal(host(dq), q)


@pytest.mark.parametrize("block", [16, 32])
@pytest.mark.parametrize("as_bf16", [False, True])
def test_family_codebook_without_a_zero(monkeypatch, as_bf16, block):
    """Smallest magnitude 1: a zero weight has no sign, costs nothing whatever the scale, and is stored as code 0."""
    from mxfp4_int8_m5_amd import pack_format as P
    monkeypatch.setitem(family.CODEBOOKS, "one", (1, 2, 3, 4, 5, 6, 7, 8))
    fam = family.Family("one", block, tuple(range(1, 11)))
    sf = fam.storage()
    rng = np.random.default_rng(block)
    w = llm_weights(rng, 24, 512).astype(F32)
    w[rng.random(w.shape) < 0.4] = 0.0
    w[0] = 0.0
    if as_bf16:
        w = bf16.from_bits(bf16.to_bits(w))
    _, qi, base, scales = family.quantize(w, fam)
    m = np.rint(scales / base[:, None]).astype(np.int64)
    idx = np.searchsorted(sf.code_mag, np.abs(qi) // np.repeat(m, block, axis=1))
    codes, bc, ws = layout.pack_rows((idx | (qi < 0) << 3).astype(np.uint8), np.searchsorted(sf.mult, m).astype(np.uint8), base, sf)
    dc, db, dw, _ = P.pack_matrix(_device(w, as_bf16, 0), "one", product_format(sf))
    assert np.array_equal(host(dw), ws) and np.array_equal(host(db), bc)
    assert np.array_equal(host(dc).view(np.uint32), codes)
