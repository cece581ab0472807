"""The grouped GEMM on rows in 256-row slots of blocked activations, and the two kernels that fill the slots: against the row forms and a
float64 product of the decoded weights, with segments that end at every edge of a 16-row block, a wave's turn and a slot."""
import numpy as np
import pytest
import torch

from oracle import bf16, linear
from tests.test_gpu_gemm_tiles import NAMES, product, weights
from tests.util import FORMATS, dev, host

pytestmark = pytest.mark.gpu
EDGES = [0, 1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 192, 255, 256, 257, 300, 511, 512, 513]


def segments(e, counts, rng):
    from mxfp4_int8_m5_amd import sc_moe as M
    ex = np.repeat(np.arange(e), counts).astype(np.int32)
    off, ts, _ = M.segments(dev(ex), e, 256)
    return ex, off, ts


def rows_of_slots(slots, ex, off, ts, k):
    """The sorted rows found in the slots."""
    blocks = host(slots).reshape(-1, k // 32, 2, 32, 16).transpose(0, 3, 1, 2, 4).reshape(-1, k)
    off, ts = host(off), host(ts)
    return blocks[ts[ex] * 256 + np.arange(len(ex)) - off[ex]]


@pytest.mark.parametrize("k", [128, 384, 512, 640, 1024, 2176])
@pytest.mark.parametrize("e", [1, 25, 64, 65, 200])
def test_slots_hold_the_sorted_rows(e, k):
    from mxfp4_int8_m5_amd import sc_kernels as S
    from mxfp4_int8_m5_amd import sc_moe as M
    rng = np.random.default_rng(e + k)
    ex, off, ts = segments(e, rng.choice(EDGES if e < 100 else [0, 1, 8, 9, 40], e) if e > 1 else [77], rng)
    r = len(ex)
    x = dev(bf16.to_bits(rng.standard_normal((r, k)).astype(np.float32)))
    q, s = S.act_quant(x, r)
    slots, xs = M.act_quant_sorted(x, r, off, ts)
    assert torch.equal(xs, s) and np.array_equal(rows_of_slots(slots, ex, off, ts, k), host(q))
    tok = torch.from_numpy(rng.integers(0, r, r + 3).astype(np.int32)).cuda()
    slots, xs = M.gather_blocked(q, s, tok, r, off, ts)
    assert torch.equal(xs, s[tok[:r].long()]) and np.array_equal(rows_of_slots(slots, ex, off, ts, k), host(q[tok[:r].long()]))


@pytest.mark.parametrize("name", ["published", "sixteen", "range", "mxfp4"])
@pytest.mark.parametrize("e,n,k", [(25, 256, 128), (25, 1156, 256), (25, 128, 384), (25, 132, 640), (65, 384, 512), (25, 256, 2176)])
def test_grouped_product_from_slots(e, n, k, name):
    from mxfp4_int8_m5_amd import sc_moe as M
    rng = np.random.default_rng(e + n + k)
    counts = np.concatenate([rng.permutation(EDGES), rng.choice([0, 1, 5], e - 25)])
    ex, off, ts = segments(e, counts, rng)
    r = len(ex)
    few = [weights(rng, n, k, name) for _ in range(3)]
    codes, bc, ws, q = (torch.stack([few[i % 3][f] for i in range(e)]) for f in (0, 1, 2, 4))
    src = torch.from_numpy(rng.integers(-127, 128, (r + 5, k)).astype(np.int8)).cuda()
    tok = torch.from_numpy(rng.permutation(r + 5)[:r].astype(np.int32)).cuda()
    scale = torch.from_numpy((2.0 ** -9 * (0.5 + rng.random(r + 5))).astype(np.float32)).cuda()
    slots, xs = M.gather_blocked(src, scale, tok, r, off, ts)
    rows, idx = src[tok.long()], dev(ex).long() % 3
    want = torch.empty((r, n), dtype=torch.int32, device="cuda")
    for f in range(3):
        want[idx == f] = product(rows[idx == f], few[f][4])
    args = slots, xs, r, k, codes, bc, ws, off, ts, n
    assert torch.equal(M.moe_mm_blocked(*args, 0, few[0][3]), want)
    for epi in (1, 3) if n % 8 == 0 else (1,):   # the row form's epilogue, checked against the oracle elsewhere
        ref = M.moe_mm(src, r, codes, bc, ws, off, ts, 0, n, epi, scale, tile=(256, 64, 4), gather=tok, fmt=few[0][3])
        assert torch.equal(M.moe_mm_blocked(*args, epi, few[0][3]).view(torch.int16), ref.view(torch.int16))


def test_table_formats_are_refused():
    from mxfp4_int8_m5_amd import sc_moe as M
    from tests.util import product_format
    fmt = product_format(FORMATS[4])
    assert not M.takes_slots(1000, 4, 256, 256, fmt) and not M.takes_slots(1000, 4, 256, 128, product_format(FORMATS[0]))
    z = torch.zeros(1 << 20, dtype=torch.int32, device="cuda")
    with pytest.raises(ValueError):
        M.moe_mm_blocked(z.view(torch.int8), z.float(), 10, 256, z, z.view(torch.uint8), z.float().reshape(4, -1), z, z, 8, 1, fmt)


@pytest.mark.parametrize("d,f2,rows", [(512, 2048, 300), (512, 1024, 300), (256, 2048, 90)])   # down from slots, wide and narrow; neither
def test_expert_mlp_is_its_parts(d, f2, rows, e=5):
    from mxfp4_int8_m5_amd import sc_kernels as S
    from mxfp4_int8_m5_amd import sc_moe as M
    rng = np.random.default_rng(d + f2)
    m = rows * e // 2
    gu, dn = ([torch.stack(t) for t in zip(*[weights(rng, n, k, "published")[:3] for _ in range(e)])] for n, k in ((f2, d), (d, f2 // 2)))
    inds = dev(rng.permuted(np.tile(np.arange(e), (m, 1)), axis=1)[:, :2].astype(np.int32))
    tm = M.row_tile(2 * m, e)
    pos, tok, _, off, ts, mt = M.route_sort(inds, e, tm)
    xq, xs = S.act_quant(dev(bf16.to_bits(rng.standard_normal((m, d)).astype(np.float32))), m)
    fmt = weights(rng, 4, 128, "published")[3]
    act = M.moe_mm(xq, 2 * m, *gu, off, ts, mt, f2, 3, xs, tile=(tm, 64, 4), gather=tok, fmt=fmt)
    hq, hs = S.act_quant(act, 2 * m)
    want = M.moe_mm(hq, 2 * m, *dn, off, ts, mt, d, 1, hs, tile=(tm, 64, 4), fmt=fmt)
    assert torch.equal(M.expert_mlp(xq, xs, 2 * m, gu, dn, tok, off, ts, mt, tm, fmt).view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("d,f2,rows,e", [(512, 2048, 150, 40), (1024, 2048, 280, 18)])   # more tiles than CUs; fewer, and many rows
def test_expert_mlp_from_slots_throughout(d, f2, rows, e):
    from mxfp4_int8_m5_amd import sc_moe as M
    assert M.slots_pay(rows * e, e, f2, d, True) and M.slots_pay(rows * e, e, d, f2 // 2, False)
    test_expert_mlp_is_its_parts(d, f2, rows, e)


@pytest.mark.parametrize("k", [4096, 8192, 8320, 8704, 12288])   # beyond 8192: the quantizer's codes pass through LDS in two turns
def test_slots_of_long_rows(k):
    test_slots_hold_the_sorted_rows(25, k)


@pytest.mark.parametrize("k", [4096, 8704, 12288])
def test_grouped_product_of_long_rows(k):
    test_grouped_product_from_slots(25, 132, k, "published")
