"""The tile that the GEMM's cost tables choose on 256 CUs, recomputed from the tables in the source: the shapes of the GPU tile tests
reach the tiles that they are listed under, and 32x32x32 and 16x16x64 forms both."""
import os
import re

import pytest

from tests.test_gpu_gemm_tiles import BLOCKED, ROWS

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mxfp4-int8-m5_amd", "csrc")


def table(name):
    with open(os.path.join(CSRC, "gemm.hip")) as f:
        body = re.search(name + r"\[\d\] = \{\n(.*?)\n\};", f.read(), re.S).group(1)
    number = r"[\d.]+f?"
    rows = []
    for line in body.splitlines():
        head = [int(x) for x in re.match(r"\s*\{(\d+), (\d+), (\d+),", line).groups()]
        lists = [[float(x.rstrip("f")) for x in re.findall(number, l)] for l in re.findall(r"\{([^{}]*)\}", line[line.index("{") + 1:])]
        low, mid, waves = re.search(r"\}, ([\d.]+)f, ([\d.]+)f(?:, (ONE|SEVERAL))?\}", line).groups()
        rows.append((*head, *lists, float(low), float(mid), waves))
    return rows


def chosen(name, m, n, k, cus=256):
    times = {}
    for i, (bm, bn, occ, f, s, w, low, mid, waves) in enumerate(table(name)):
        if name == "ROW_TILES" and i >= 5 and (-(-m // bm) * -(-n // bn) > cus or k % (256 if i == 5 else 512)):
            continue   # K groups
        if waves and (-(-m // bm) * -(-n // bn) <= cus * occ) != (waves == "ONE"):
            continue
        full, rest = divmod(-(-m // bm) * -(-n // bn), cus * occ)
        cost = lambda r: max(f[r - 1] + k / 128 * s[r - 1], w[r - 1])
        t = full * cost(occ)
        if rest > cus:
            t += cost(-(-rest // cus))
        elif rest:
            fill = rest / cus
            t += cost(1) * (low if fill <= 0.5 else low + (mid - low) * (fill - 0.5) * 4 if fill <= 0.75 else mid + (1 - mid) * (fill - 0.75) * 4)
        times[i] = t
    return min(times, key=times.get)


@pytest.mark.parametrize("name,tile,m,n,k", [(name, t, *s) for name, tiles in (("BLOCKED_TILES", BLOCKED), ("ROW_TILES", ROWS))
                                             for t, shapes in tiles for s in shapes])
def test_the_tile_tests_reach_their_tiles(name, tile, m, n, k):
    assert chosen(name, m, n, k) == tile


def test_both_mfma_shapes_are_reached():
    count = lambda shapes, bm, bn: [-(-m // bm) * -(-n // bn) for m, n, _ in shapes]
    blocked = count(BLOCKED[2][1], 256, 128)
    assert min(blocked) <= 160 < max(blocked)
    for (_, shapes), bm, bn in zip(ROWS, (256, 256, 128, 128), (256, 128, 128, 64)):
        tiles = count(shapes, bm, bn)
        assert min(tiles) <= 192 < max(tiles)
