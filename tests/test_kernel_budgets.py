"""Register budgets of the kernels whose occupancy was set by measurement, read
from the metadata of the built library: a change elsewhere in a kernel must not
take a wave per SIMD from it (a wave has 512 registers of a SIMD to share, in
steps of 8)."""
import re
import struct

import msgpack
import pytest

from unigasfoam_amd import core


def code_objects(blob):
    """The gfx950 ELF images of the offload bundles of a host library."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := blob.find(magic, at)) >= 0:
        n, p = struct.unpack_from("<Q", blob, at + 24)[0], at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, p)
            if b"gfx950" in blob[p + 24:p + 24 + idlen]:
                yield blob[at + off:at + off + size]
            p += 24 + idlen
        at += 24


def kernels(elf):
    """Metadata of an image's kernels (its AMDGPU note)."""
    shoff = struct.unpack_from("<Q", elf, 40)[0]
    entsize, num = struct.unpack_from("<HH", elf, 58)
    for i in range(num):
        kind = struct.unpack_from("<I", elf, shoff + i * entsize + 4)[0]
        off, size = struct.unpack_from("<QQ", elf, shoff + i * entsize + 24)
        p = off
        while kind == 7 and p < off + size:
            nlen, dlen, typ = struct.unpack_from("<III", elf, p)
            d = p + 12 + (nlen + 3) // 4 * 4
            if typ == 32:
                yield from msgpack.unpackb(elf[d:d + dlen])["amdhsa.kernels"]
            p = d + (dlen + 3) // 4 * 4


@pytest.fixture(scope="module")
def table():
    return {k[".name"]: k for image in code_objects(open(core.LIB_PATH, "rb").read()) for k in kernels(image)}


def waves(k):
    return 512 // ((k[".vgpr_count"] + 7) // 8 * 8)


@pytest.mark.parametrize("level, species, least", [(0, 1, 5), (1, 1, 4), (2, 1, 4), (0, 2, 4), (1, 2, 4), (2, 2, 4),
                                                   (0, 8, 4), (1, 8, 3), (2, 8, 3)])
def test_cell_tile(table, level, species, least):
    """Every instance but those whose LDS leaves less room."""
    got = {n: k for n, k in table.items()
           if re.match(rf"_ZN3ugx6k_tileI[fd]Lb0ELi{level}ELi{species}ELi\d+E", n)}
    assert len(got) == 6
    for n, k in got.items():
        if n.startswith("_ZN3ugx6k_tileId") and "ELi256E" in n:
            continue    # 45 KB of LDS: three blocks of a wave per SIMD
        assert waves(k) >= least, (n, k[".vgpr_count"])


@pytest.mark.parametrize("real, least", [("f", 4), ("d", 3)])
def test_move(table, real, least):
    k = next(k for n, k in table.items() if n.startswith(f"_ZN3ugx6k_moveI{real}E"))
    assert waves(k) >= least and k[".private_segment_fixed_size"] == 0


@pytest.mark.parametrize("real", ["f", "d"])
def test_cell_sums_of_eight_species(table, real):
    k = next(k for n, k in table.items() if n.startswith(f"_ZN3ugx11k_cell_sumsI{real}Li0ELi8E"))
    assert waves(k) >= 4 and k[".private_segment_fixed_size"] == 0
