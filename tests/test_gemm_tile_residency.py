"""What the compiler made of the GEMM tiles, read from the built library: the registers and LDS of each against what the choice of a
tile counts on -- as many workgroups on a CU as the cost tables of gemm.hip and the comments of gemm_grouped.hip say --, and the
place of the sigmoid's table."""
import re
import struct

import msgpack
import pytest

from tests.test_gemm_tile_choice import table

CU_LDS, SIMDS, REGISTERS, MOST_WAVES = 160 * 1024, 4, 512, 8   # gfx950: a CU's LDS; its SIMDs; a SIMD's registers a lane and waves
FIELDS = ("bm", "bn", "bk", "wgm", "wgn", "bmode", "occ", "fd", "skip", "pk", "kg", "adm", "mf")


def code_objects():
    """The GPU's ELF files in the library's offload bundles."""
    import mxfp4_int8_m5_amd as pkg
    with open(pkg._lib.LIB_PATH, "rb") as f:
        lib = f.read()
    at = lib.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        entries, = struct.unpack_from("<Q", lib, at + 24)
        p = at + 32
        for _ in range(entries):
            start, size, n = struct.unpack_from("<QQQ", lib, p)
            if b"gfx950" in lib[p + 24:p + 24 + n]:
                yield lib[at + start:at + start + size]
            p += 24 + n
        at = lib.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


def sections(elf):
    first, = struct.unpack_from("<Q", elf, 40)
    size, count = struct.unpack_from("<HH", elf, 58)
    return [struct.unpack_from("<IIQQQQIIQQ", elf, first + i * size) for i in range(count)]


def descriptors():
    """The metadata of every kernel: the code objects' AMDGPU notes."""
    for elf in code_objects():
        for _, kind, _, _, at, _, _, _, _, _ in sections(elf):
            if kind == 7:   # SHT_NOTE
                name, desc, note = struct.unpack_from("<III", elf, at)
                if note == 32:   # NT_AMDGPU_METADATA
                    yield from msgpack.unpackb(elf[at + 12 + (name + 3 & ~3):][:desc])["amdhsa.kernels"]


@pytest.fixture(scope="module")
def tiles():
    found = []
    for k in descriptors():
        m = re.match(r"_ZN4scmx11gemm_kernelI((?:L[ib]\d+E)+)", k[".name"])
        if m:
            t = dict(zip(FIELDS, map(int, re.findall(r"L[ib](\d+)E", m.group(1)))))
            t["waves"] = t["wgm"] * t["wgn"] * t["kg"]
            per_simd = min(MOST_WAVES, REGISTERS // (-(-k[".vgpr_count"] // 8) * 8))
            t["on_a_cu"] = min(CU_LDS // k[".group_segment_fixed_size"], per_simd * SIMDS // t["waves"])
            t["spilled"] = k[".vgpr_spill_count"]
            found.append(t)
    assert len(found) > 100
    return found


def few(found, n):
    """Of the instances those that share a CU in fewer than n."""
    assert found
    return [t for t in found if t["on_a_cu"] < n]


@pytest.mark.parametrize("name,kind", [("BLOCKED_TILES", 1), ("ROW_TILES", 0)])
def test_workgroups_that_share_a_cu(tiles, name, kind):
    waves = {"BLOCKED_TILES": (4, 8, 8, 8, 8, 4, 4), "ROW_TILES": (8, 8, 8, 8, 4, 8, 8)}[name]
    for (bm, bn, occ, *_), w, groups in zip(table(name), waves, (1, 1, 1, 1, 1, 2, 4) if kind == 0 else (1,) * 7):
        assert few([t for t in tiles if (t["bm"], t["bn"], t["waves"], t["kg"], t["adm"], t["skip"], t["pk"])
                    == (bm, bn, w, groups, kind, 0, 0)], occ) == [], (name, bm, bn)


@pytest.mark.parametrize("shape,n", [((64, 128, 8, 0, 0), 2), ((64, 128, 4, 1, 0), 3), ((64, 256, 8, 1, 0), 2), ((128, 128, 4, 0, 2), 2),
                                     ((256, 128, 4, 0, 1), 2)])
def test_expert_tiles_that_share_a_cu(tiles, shape, n):
    """64 rows with weights staged as INT8 and packed (four waves, eight), 128 gathered rows, 256 rows in slots."""
    assert few([t for t in tiles if (t["bm"], t["bn"], t["waves"], t["pk"], t["adm"]) == shape], n) == []


def test_the_epilogue_tests_reach_their_tiles():
    from tests.test_gemm_tile_choice import chosen
    from tests.test_gpu_swiglu_table import SHARED
    assert [chosen("ROW_TILES", *s) for _, *s in SHARED] == [t for t, *_ in SHARED]


def test_the_sigmoid_table_is_aligned():
    """The tiles copy it in pieces of 16 bytes: the section that holds it has to be placed on one, and its place in there."""
    found = 0
    for elf in code_objects():
        parts = sections(elf)
        for _, kind, _, _, at, size, link, _, _, entry in parts:
            if kind != 11:   # SHT_DYNSYM
                continue
            names = parts[link][4]
            for i in range(at, at + size, entry):
                name, _, _, section, value, _ = struct.unpack_from("<IBBHQQ", elf, i)
                if section and b"g_silu_table" in elf[names + name:elf.index(b"\0", names + name)]:
                    found += 1
                    assert parts[section][8] % 16 == 0 and value % 16 == 0
    assert found == 1
