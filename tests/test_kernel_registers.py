"""Registers of the placement kernels in the library as it was built, from the metadata the compiler leaves in its code
objects: launch_place counts on two workgroups of 1024 lanes per compute unit for launches that only read or only widen."""

import struct

import msgpack
import pytest

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(blob: bytes):
    at = blob.find(BUNDLE)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", blob, at + len(BUNDLE))
        pos = at + len(BUNDLE) + 8
        for _ in range(n):
            offset, size, name_len = struct.unpack_from("<QQQ", blob, pos)
            name = blob[pos + 24: pos + 24 + name_len]
            pos += 24 + name_len
            if b"gfx950" in name and size:
                yield blob[at + offset: at + offset + size]
        at = blob.find(BUNDLE, pos)


def kernels_of(elf: bytes):
    """The entries of ``amdhsa.kernels`` in the code object's AMDGPU metadata note (type 32)."""
    assert elf[:5] == b"\x7fELF\x02"
    phoff, = struct.unpack_from("<Q", elf, 32)
    phentsize, phnum = struct.unpack_from("<HH", elf, 54)
    for k in range(phnum):
        kind, _, offset, _, _, size, _, _ = struct.unpack_from("<IIQQQQQQ", elf, phoff + k * phentsize)
        pos = offset
        while kind == 4 and pos < offset + size:  # PT_NOTE
            name_size, desc_size, note = struct.unpack_from("<III", elf, pos)
            desc = pos + 12 + (name_size + 3) // 4 * 4
            if note == 32 and elf[pos + 12: pos + 18] == b"AMDGPU":
                yield from msgpack.unpackb(elf[desc: desc + desc_size])["amdhsa.kernels"]
            pos = desc + (desc_size + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels(mxp):
    found = {}
    for elf in code_objects(mxp.LIB_PATH.read_bytes()):
        for k in kernels_of(elf):
            found[k[".name"]] = k
    return found


@pytest.mark.parametrize("name, workgroups", [("place_kernel", 2), ("checksum_kernel", 2), ("place_ragged_kernel", 1),
                                              ("place_digest_kernel", 1), ("place_digest_ragged_kernel", 1)])
def test_workgroups_fit_a_compute_unit(kernels, name, workgroups):
    mine = [k for mangled, k in kernels.items() if f"{len(name)}{name}E" in mangled]
    assert len(mine) == 1
    # a SIMD has 512 vector registers a lane; a workgroup of 1024 lanes puts four wavefronts on each of the four SIMDs
    assert mine[0][".vgpr_count"] + mine[0].get(".agpr_count", 0) <= 512 // (4 * workgroups)
    assert mine[0][".vgpr_spill_count"] == 0 and mine[0][".private_segment_fixed_size"] == 0
