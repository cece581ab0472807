"""The tiles of the blocked dense GEMM and of the grouped GEMM, INT32 against a float64 product of the decoded weights: ragged rows and
columns, step counts that end in every tail of the unrolled K loops, each weight format."""
import numpy as np
import pytest
import torch

from oracle import bf16, layout, linear
from tests.util import FORMATS, blocked_layout, dev, host, product_format, random_packed

pytestmark = pytest.mark.gpu
NAMES = {"published": FORMATS[0], "sixteen": FORMATS[1], "range": FORMATS[5], "table": FORMATS[4], "mxfp4": None}


def weights(rng, n, k, name):
    """(codes, block codes, row scales, product format, decoded INT8 [n, k]) on the device."""
    from mxfp4_int8_m5_amd import sc_format as F
    c, b, w, q = random_packed(rng, n, k, NAMES[name] or layout.DEFAULT)
    if NAMES[name]:
        return dev(c), dev(b), dev(w), product_format(NAMES[name]), dev(q)
    nib, e8 = layout.to_mxfp4(c, b, w, n, k)
    nib, e8 = dev(nib), dev(e8)
    ws = F.mxfp4_row_scales(e8)
    lift = torch.exp2(torch.log2(dev(w)) - torch.log2(ws))   # a row whose smallest shift is not 0 decodes to smaller integers
    return F.mxfp4_codes(nib), e8, ws, F.MXFP4, (dev(q).double() * lift[:, None].double()).to(torch.int8)


def product(xq, q):
    return (xq.double() @ q.double().T).to(torch.int32)


# (tile of the blocked table on 256 CUs, shapes): every tail of each tile's rotating loop (test_gemm_tile_choice.py checks the tiles)
BLOCKED = [(0, [(1154, 10396, 128), (588, 10004, 384), (518, 10076, 640), (1030, 11864, 4224)]),   # 256x128, four waves (or, by format, another)
           (1, [(935, 12296, 1536), (935, 12296, 1664), (772, 11664, 2176), (653, 11248, 4224)]),  # 256x256
           (2, [(400, 9368, 4096), (588, 6584, 4224), (455, 8240, 4352), (454, 8284, 4480), (387, 9476, 4608), (391, 9536, 4736),
                (645, 8376, 640), (392, 12292, 768), (515, 10144, 896), (530, 9812, 1024), (518, 10316, 1280),
                (273, 11488, 4224)]),                                                              # 256x128, eight waves, both MFMA shapes
           (3, [(1581, 11764, 4224)]),                                                             # the same, several waves of tiles
           (4, [(216, 8564, 256), (146, 11004, 384), (148, 11192, 512), (134, 11848, 640), (130, 10900, 768), (137, 11804, 896)]),   # 256x64
           (5, [(278, 180, 128), (319, 136, 256), (235, 136, 384), (154, 224, 512), (165, 340, 640), (133, 3888, 768),
                (4133, 196, 896)]),                                                                # 128x64
           (6, [(142, 7200, 128), (137, 6856, 256), (149, 8264, 384), (142, 8452, 512), (131, 8704, 640), (141, 144, 768),
                (134, 316, 896)])]                                                                 # 64x64


# whichever tile they take
MORE = [(400, 12296, 384), (1030, 12296, 640), (385, 12288, 4224), (1000, 6152, 768), (1500, 4104, 2048), (600, 4104, 2048),
        (1030, 2052, 1280), (515, 8200, 640), (1025, 8192, 384), (4099, 2052, 128), (770, 1032, 1280), (129, 1028, 256), (300, 260, 896)]

# the same for the larger tiles by rows, which multiply with 32x32x32 up to three quarters of a tile per CU
ROWS = [(0, [(706, 12476, 384), (705, 12352, 512), (642, 10944, 640), (661, 10996, 768), (968, 12392, 256), (796, 12556, 384)]),      # 256x256
        (1, [(709, 5456, 512), (387, 8396, 640), (262, 11020, 768), (257, 11732, 896), (268, 10892, 1152), (265, 10984, 1536),
             (326, 12380, 640)]),                                                                                # 256x128
        (2, [(135, 10940, k) for k in (4096, 4224, 4352, 4480, 4608, 4736)] + [(206, 12332, 128), (196, 12416, 512)]),    # 128x128
        (3, [(67, 8288, 128), (68, 8244, 256), (75, 8268, 384), (68, 9200, 512), (69, 8460, 640), (66, 9780, 768),
             (65, 8416, 896), (68, 8296, 1024), (134, 6552, 256)])]                                              # 128x64


@pytest.mark.parametrize("name", list(NAMES))
@pytest.mark.parametrize("m,n,k", [s for _, shapes in ROWS for s in shapes])
def test_row_tiles(m, n, k, name):
    from mxfp4_int8_m5_amd import sc_kernels as S
    rng = np.random.default_rng(m + n + k)
    codes, bc, ws, fmt, q = weights(rng, n, k, name)
    xq = torch.from_numpy(rng.integers(-127, 128, (m, k)).astype(np.int8)).cuda()
    want = product(xq, q)
    assert torch.equal(S.mm_i8_i32(xq, S.PackedWq(codes, bc, n, k, fmt, ws)), want)
    if name == "published":
        assert torch.equal(S.mm_i8_i32(xq, q), want)


@pytest.mark.parametrize("name", list(NAMES))
@pytest.mark.parametrize("m,n,k", [s for _, shapes in BLOCKED for s in shapes] + MORE)
def test_blocked_tiles(m, n, k, name):
    from mxfp4_int8_m5_amd import sc_kernels as S
    rng = np.random.default_rng(m + n + k)
    codes, bc, ws, fmt, q = weights(rng, n, k, name)
    xq = rng.integers(-127, 128, (-(-m // 32) * 32, k)).astype(np.int8)
    xb = S.BlockedXq(dev(blocked_layout(xq)), m, k)
    assert torch.equal(S.mm_i8_i32(xb, S.PackedWq(codes, bc, n, k, fmt, ws))[:m], product(dev(xq)[:m], q))


# a shape per tile that multiplies with 32x32x32, by layout
@pytest.mark.parametrize("epi", [1, 2, 3])
@pytest.mark.parametrize("m,n,k,blocked", [(935, 12296, 1536, True), (400, 9368, 4096, True), (706, 12480, 384, False), (709, 5456, 512, False),
                                           (135, 10944, 4096, False), (67, 8288, 128, False)])
def test_epilogues_of_launches_that_leave_cus_idle(m, n, k, blocked, epi):
    """Bit for bit against the oracle's epilogue of the exact sums, output rows that are whole 16-byte pieces and not."""
    from mxfp4_int8_m5_amd import sc_kernels as S
    rng = np.random.default_rng(m + n + epi)
    c, b, w, q = random_packed(rng, n, k, FORMATS[0])
    xq = rng.integers(-127, 128, (-(-m // 32) * 32, k)).astype(np.int8)
    xs = (2.0 ** -7 * (0.5 + rng.random(m))).astype(np.float32)
    res = bf16.to_bits(rng.standard_normal((m, n)).astype(np.float32)) if epi == 2 else None
    x = S.BlockedXq(dev(blocked_layout(xq)), m, k) if blocked else dev(xq[:m])
    got = S.mm_epi(x, S.PackedWq(dev(c), dev(b), n, k, product_format(FORMATS[0]), dev(w)), dev(xs), dev(w), epi,
                   res=dev(res) if epi == 2 else None)
    assert np.array_equal(host(got), linear.epilogue(host(product(dev(xq)[:m], dev(q))), xs, w, epi, res))


def grouped(e, n, k, tm, name, counts, rng):
    """The grouped product of expert segments of `counts` gathered rows, INT32, against float64."""
    from mxfp4_int8_m5_amd import sc_moe as M
    ex = np.repeat(np.arange(e), counts).astype(np.int32)
    r = len(ex)
    few = [weights(rng, n, k, name) for _ in range(min(e, 3))]
    pick = [i % len(few) for i in range(e)]
    codes, bc, ws, q = (torch.stack([few[i][f] for i in pick]) for f in (0, 1, 2, 4))
    src = torch.from_numpy(rng.integers(-127, 128, (r + 9, k)).astype(np.int8)).cuda()
    tok = torch.from_numpy(rng.permutation(r + 9)[:r].astype(np.int32)).cuda()
    off, tstart, mt = M.segments(dev(ex), e, tm)
    rows, idx = src[tok.long()], dev(ex).long()
    want = torch.zeros((r, n), dtype=torch.int32, device="cuda")
    for f in range(len(few)):
        sel = (idx % len(few)) == f
        want[sel] = product(rows[sel], few[f][4])
    got = M.moe_mm(src, r, codes, bc, ws, off, tstart, mt, n, 0, tile=(tm, 64, 4), gather=tok, fmt=few[0][3])
    assert torch.equal(got, want)
    if name == "published":
        got = M.moe_mm_i8(rows.contiguous(), r, q.reshape(e * n, k).contiguous(), ws, off, tstart, mt, n, 0, tile=(tm, 64, 4))
        assert torch.equal(got, want)


@pytest.mark.parametrize("name", list(NAMES))
@pytest.mark.parametrize("tm", [64, 128, 256])
@pytest.mark.parametrize("e,n,k", [(3, 1156, 512), (65, 256, 384), (130, 128, 256), (4100, 8, 128)])
def test_grouped_tiles(e, n, k, tm, name):
    """Segments of 0 to a little over 256 rows (a 256-row slot of which 128-row tiles use one or both halves, with and
    without rows past the segment), expert counts either side of one and two levels of the tile's expert search; rows gathered."""
    rng = np.random.default_rng(e + n + k)
    counts = rng.choice([0, 1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 255, 256, 257], e) if e < 1000 else rng.choice([0, 0, 0, 1, 2], e)
    counts[0] += 1
    grouped(e, n, k, tm, name, counts, rng)


# 256 columns a workgroup up to 512 of K, 128 beyond or where the rows of weights do not divide; every tail of six steps
@pytest.mark.parametrize("name", ["published", "sixteen", "range", "mxfp4"])
@pytest.mark.parametrize("n,k", [(256, 256), (512, 512), (128, 512), (384, 256), (128, 768), (256, 1024), (256, 1280), (128, 1792)])
def test_packed_tiles(n, k, name):
    rng = np.random.default_rng(n + k)
    grouped(9, n, k, 64, name, np.array([1, 0, 31, 32, 33, 63, 64, 65, 200]), rng)


# 256-row slots that hold more: whole and cut 256x256 tiles (one that fills the CUs among them), 256x128 ones for narrow
# layers, an expert without rows, K loops of every length up to a trip and two more
@pytest.mark.parametrize("name", list(NAMES))
@pytest.mark.parametrize("counts", [(257, 300, 511), (512, 0, 300)])
@pytest.mark.parametrize("n,k", [(256, 128), (1156, 256), (256, 384), (1156, 512), (256, 640), (22016, 128),
                                 (128, 128), (132, 256), (128, 384), (128, 512), (128, 640), (128, 768), (128, 896)])
def test_tall_segments(n, k, counts, name):
    grouped(3, n, k, 256, name, np.array(counts), np.random.default_rng(n + k))
