"""Register spills of the built row kernels (CPU only: reads the kernel descriptions, the metadata notes of
the code objects inside the library)."""
import os
import re
import struct

import msgpack
import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "particledynamics.jl_amd", "lib",
                   "libpdx.so")


def _code_objects(data):
    """The device ELF images of the offload bundles in a host library."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(magic))
        pos = at + len(magic) + 8
        for _ in range(count):
            offset, size, idlen = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + idlen].decode()
            pos += 24 + idlen
            if "amdgcn" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(magic, at + 1)


def _kernels(elf):
    """The kernel descriptions (amdhsa.kernels) in an ELF image's notes."""
    phoff, = struct.unpack_from("<Q", elf, 32)
    phsize, phnum = struct.unpack_from("<HH", elf, 54)
    for k in range(phnum):
        kind, = struct.unpack_from("<I", elf, phoff + k * phsize)
        if kind != 4:  # PT_NOTE
            continue
        offset, = struct.unpack_from("<Q", elf, phoff + k * phsize + 8)
        size, = struct.unpack_from("<Q", elf, phoff + k * phsize + 32)
        pos = offset
        while pos < offset + size:
            nname, ndesc, _ = struct.unpack_from("<III", elf, pos)
            name = elf[pos + 12:pos + 12 + nname]
            desc = pos + 12 + (nname + 3) // 4 * 4
            if name.startswith(b"AMDGPU"):
                yield from msgpack.unpackb(elf[desc:desc + ndesc], strict_map_key=False).get("amdhsa.kernels", [])
            pos = desc + (ndesc + 3) // 4 * 4


def test_row_kernels_use_no_scratch():
    """No k_pair or k_pair_acc spills its registers: a spill inside the row walk is a memory access per visit."""
    if not os.path.exists(LIB):
        pytest.skip("library not built")
    with open(LIB, "rb") as f:
        data = f.read()
    rows = [k for elf in _code_objects(data) for k in _kernels(elf)
            if re.search(r"k_pair(_acc)?I", k[".name"])]
    assert len(rows) > 400
    spilled = {k[".name"]: (k[".private_segment_fixed_size"], k[".vgpr_spill_count"]) for k in rows
               if k[".private_segment_fixed_size"] or k[".vgpr_spill_count"]}
    assert not spilled, spilled
