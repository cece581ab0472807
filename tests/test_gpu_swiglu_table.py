"""The SwiGLU epilogue's table of the sigmoid (entries from |g| = 2^-8 on, both ends held) through the kernels that copy it to LDS and
those that read it from memory, and the two-at-a-time form of it: every bf16 gate, with an up value of either sign, against the oracle."""
import numpy as np
import pytest
import torch

from oracle import bf16, layout, linear
from tests.util import F32, FORMATS, blocked_layout, dev, host, product_format, random_packed

pytestmark = pytest.mark.gpu


# few rows; tiles from blocked activations and by rows; expert slots of 64 (the packed tiles, which copy the table behind their K loop:
# eight waves up to K = 512, four beyond), 128 and 256 rows
@pytest.mark.parametrize("path,m,k", [("blocked", 5, 256), ("blocked", 300, 256), ("rows", 300, 256), (64, 70, 256), (64, 70, 768), (64, 20, 768),
                                      (128, 70, 256), (256, 70, 256)])
def test_every_gate(path, m, k):
    from mxfp4_int8_m5_amd import sc_kernels as S
    from mxfp4_int8_m5_amd import sc_moe as M
    n = 4 * 32768
    gate = bf16.from_bits(np.arange(65536, dtype=np.uint32).astype(np.uint16))
    ws = np.empty((n // 4, 4), F32)
    ws[:, 0], ws[:, 1], ws[:, 2], ws[:, 3] = gate[0::2], gate[1::2], F32(1.0), F32(-0.3984375)
    ws = ws.reshape(-1)
    code4 = np.zeros((n, k), np.uint8)
    code4[:, 0] = 1                                               # weight rows (1, 0, 0, ...): acc = xq[:, 0]
    codes, bc, _ = layout.pack_rows(code4, np.zeros((n, k // 32), np.uint8), ws)
    xq = np.zeros((-(-m // 32) * 32, k), np.int8)
    xq[:, 0] = np.where(np.arange(len(xq)) % 2, -1, 1)
    xs = np.ones(len(xq), F32)
    dc, db, dw, fmt = dev(codes), dev(bc), dev(ws), product_format(layout.DEFAULT)
    if isinstance(path, str):
        x = S.BlockedXq(dev(blocked_layout(xq)), m, k) if path == "blocked" else dev(xq[:m])
        got = S.mm_epi(x, S.PackedWq(dc, db, n, k, fmt, dw), dev(xs[:m]), dw, 3)[:m]
    else:
        off, ts, mt = M.segments(torch.zeros(m, dtype=torch.int32, device="cuda"), 1, path)
        got = M.moe_mm(dev(xq[:m]), m, dc[None], db[None], dw[None], off, ts, mt, n, 3, dev(xs[:m]), tile=(path, 64, 4), fmt=fmt)
    with np.errstate(all="ignore"):
        want = dev(linear.epilogue(np.stack([np.ones(n, np.int32), -np.ones(n, np.int32)]), np.ones(2, F32), ws, 3))
    nan = want.isnan()
    for r in range(2):
        rows = got[r::2]
        assert torch.equal(rows.isnan(), nan[r].expand_as(rows))
        assert torch.equal(rows.view(torch.int16)[:, ~nan[r]], want[r].view(torch.int16)[~nan[r]].expand(len(rows), -1))
    assert host(nan).sum() < 2000


# staged tiles several of which share a CU copy the table behind their K loop as well: expert slots of 64 rows where K is no multiple of
# 256 (one K step, odd and even counts of them), 64x64 by rows
@pytest.mark.parametrize("path,m,k", [(64, 70, 128), (64, 70, 384), (64, 20, 896), ("rows", 50, 128), ("rows", 64, 384)])
def test_every_gate_where_workgroups_share_a_cu(path, m, k):
    test_every_gate(path, m, k)


# 128x64 by rows, with more tiles than CUs and fewer, rows and columns that end inside a tile; 64x64; the tiles of test_gemm_tile_choice.py
SHARED = [(3, 160, 12288, 1152), (3, 131, 11656, 1152), (3, 67, 8288, 128), (4, 300, 6144, 512), (4, 300, 6152, 896)]


@pytest.mark.parametrize("epi", [1, 2, 3])
@pytest.mark.parametrize("tile,m,n,k", SHARED)
def test_epilogues_where_workgroups_share_a_cu(tile, m, n, k, epi):
    """INT8 weights, the published format and table decode, bit for bit against the oracle's epilogue of the exact sums."""
    from mxfp4_int8_m5_amd import sc_kernels as S
    from tests.test_gpu_gemm_tiles import product
    rng = np.random.default_rng(m + n + epi)
    xq = rng.integers(-127, 128, (m, k)).astype(np.int8)
    xs = (2.0 ** -7 * (0.5 + rng.random(m))).astype(F32)
    res = bf16.to_bits(rng.standard_normal((m, n)).astype(F32)) if epi == 2 else None
    for fmt in (FORMATS[0], FORMATS[4]):
        c, b, w, q = random_packed(rng, n, k, fmt)
        want = linear.epilogue(host(product(dev(xq), dev(q))), xs, w, epi, res)
        forms = [S.PackedWq(dev(c), dev(b), n, k, product_format(fmt), dev(w))] + ([dev(q)] if fmt is FORMATS[0] else [])
        for wq in forms:
            got = S.mm_epi(dev(xq), wq, dev(xs), dev(w), epi, res=dev(res) if epi == 2 else None)
            assert np.array_equal(host(got), want)
