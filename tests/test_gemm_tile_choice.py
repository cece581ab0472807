"""The blocked tile that the GEMM's cost table chooses on 256 CUs, recomputed from the table in the source: the shapes of the GPU tile
test reach the tiles that they are listed under, and 32x32x32 and 16x16x64 forms both."""
import os
import re

import pytest

from tests.test_gpu_gemm_tiles import BLOCKED

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mxfp4-int8-m5_amd", "csrc")


def table():
    with open(os.path.join(CSRC, "gemm.hip")) as f:
        body = re.search(r"BLOCKED_TILES\[6\] = \{\n(.*?)\n\};", f.read(), re.S).group(1)
    number = r"[\d.]+f?"
    rows = []
    for line in body.splitlines():
        head = [int(x) for x in re.match(r"\s*\{(\d+), (\d+), (\d+),", line).groups()]
        lists = [[float(x.rstrip("f")) for x in re.findall(number, l)] for l in re.findall(r"\{([^{}]*)\}", line[line.index("{") + 1:])]
        low, mid = (float(x) for x in re.search(r"\}, ([\d.]+)f, ([\d.]+)f\}", line).groups())
        rows.append((*head, *lists, low, mid))
    return rows


def chosen(m, n, k, cus=256):
    times = []
    for bm, bn, occ, f, s, w, low, mid in table():
        full, rest = divmod(-(-m // bm) * -(-n // bn), cus * occ)
        cost = lambda r: max(f[r - 1] + k / 128 * s[r - 1], w[r - 1])
        t = full * cost(occ)
        if rest > cus:
            t += cost(-(-rest // cus))
        elif rest:
            fill = rest / cus
            t += cost(1) * (low if fill <= 0.5 else low + (mid - low) * (fill - 0.5) * 4 if fill <= 0.75 else mid + (1 - mid) * (fill - 0.75) * 4)
        times.append(t)
    return times.index(min(times))


@pytest.mark.parametrize("tile,m,n,k", [(t, *s) for t, shapes in BLOCKED for s in shapes])
def test_the_tile_test_reaches_its_tiles(tile, m, n, k):
    assert chosen(m, n, k) == tile


def test_both_mfma_shapes_are_reached():
    tiles = [-(-m // 256) * -(-n // 128) for m, n, _ in BLOCKED[2][1]]
    assert min(tiles) <= 160 < max(tiles)
