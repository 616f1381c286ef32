"""What the compiler gave the kernels, from the metadata of the built library: registers and scratch.  Needs no GPU."""
import re
import struct

import msgpack
import pytest

from cats_amd.build import KERNEL_LIB


def _code_objects(blob):
    """The gfx950 code objects of the offload bundles in a shared library."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := blob.find(magic, at)) >= 0:
        count = struct.unpack_from("<Q", blob, at + 24)[0]
        o = at + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", blob, o)
            if b"gfx950" in blob[o + 24:o + 24 + n]:
                yield blob[at + off:at + off + size]
            o += 24 + n
        at += 24


def _kernels(elf):
    """amdhsa.kernels of the metadata note (type 32) of a code object."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + i * shentsize)
        end = off + size
        while kind == 7 and off < end:  # SHT_NOTE
            namesz, descsz, ntype = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (namesz + 3) // 4 * 4
            if ntype == 32:
                yield from msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]
            off = desc + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    if not KERNEL_LIB.exists():
        import __graft_entry__

        __graft_entry__.build()
    found = {k[".name"]: k for elf in _code_objects(KERNEL_LIB.read_bytes()) for k in _kernels(elf)}
    assert len(found) > 100
    return found


def _pairs(kernels, pattern):
    """Kernels whose last template argument, a flag, is the only difference: (without, with)."""
    pairs = [(k, kernels[name.replace(m[0], m[1] + "Lb1EE")]) for name, k in kernels.items() if (m := re.search("(" + pattern + ")Lb0EE", name))]
    assert pairs
    return pairs


def test_small_layers_hold_no_registers_for_a_tail(kernels):
    """A plain call of one row has no norm, residual or next norm to hold: fewer registers than a tail's."""
    for plain, tail in _pairs(kernels, r"small_rows_kernelINS_\w+?ELi1ELi\dELb\dE"):
        assert plain[".vgpr_count"] < tail[".vgpr_count"], plain[".name"]
    for plain, tail in _pairs(kernels, r"small_tail_kernelINS_\w+?E"):
        assert plain[".vgpr_count"] < tail[".vgpr_count"], plain[".name"]


def test_nothing_spills(kernels):
    """No kernel has scratch, but for the fp32 wave-per-row passes over rows of x that no workgroup holds in LDS, at eight batch rows."""
    spilled = {n for n, k in kernels.items() if k[".private_segment_fixed_size"] or k[".vgpr_spill_count"]}
    assert {n for n in spilled if not re.search(r"rows_kernelINS_3F32ELi8ELi2ELi8ELb0ELi\dELb0E", n)} == set()


def test_two_register_sets_hold_no_registers_for_a_norm(kernels):
    """The matrix-core gate + up pass over long rows: at least as many registers with a norm as without, in each type."""
    pairs = _pairs(kernels, r"rows_mma_kernelINS_\w+?ELi\dELi2ELb1ELi1E")
    assert len(pairs) == 15
    for plain, norm in pairs:
        assert plain[".vgpr_count"] <= norm[".vgpr_count"], plain[".name"]


def test_wave_per_row_calls_hold_nothing_for_a_norm(kernels):
    """Gate + up of two to four rows with x in LDS: the plain instance has no room for the rows' squares."""
    pairs = _pairs(kernels, r"rows_kernelINS_\w+?ELi[24]ELi2ELi8ELb\dELi1ELb1ELi\dE")
    assert len(pairs) == 12
    for plain, norm in pairs:
        assert plain[".group_segment_fixed_size"] + 512 <= norm[".group_segment_fixed_size"], plain[".name"]
