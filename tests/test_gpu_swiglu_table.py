"""The SwiGLU epilogue's table of the sigmoid (entries from |g| = 2^-8 on, both ends held) through the kernels that copy it to LDS and
those that read it from memory, and the two-at-a-time form of it: every bf16 gate, with an up value of either sign, against the oracle."""
import numpy as np
import pytest
import torch

from oracle import bf16, layout, linear
from tests.util import F32, blocked_layout, dev, host, product_format

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
