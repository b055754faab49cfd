"""Registers of the compiled kernels, from the metadata that the compiler wrote
into the library (no GPU)."""
import os
import struct

import msgpack
import pytest

from conftest import LIB


def _kernels(path):
    """amdhsa.kernels of the gfx950 code objects in the library."""
    data = open(path, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    out = []
    at = data.find(magic)
    while at >= 0:
        n, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(n):
            off, size, ln = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + ln]
            p += 24 + ln
            if b"gfx950" in name and size:
                out += _notes(data[at + off:at + off + size])
        at = data.find(magic, at + 1)
    return out


def _notes(elf):
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    entsize, count = struct.unpack_from("<HH", elf, 0x3A)
    for k in range(count):
        head = struct.unpack_from("<IIQQQQ", elf, shoff + k * entsize)
        if head[1] != 7:                             # SHT_NOTE
            continue
        namesz, descsz, kind = struct.unpack_from("<III", elf, head[4])
        if kind == 32:                               # NT_AMDGPU_METADATA
            q = head[4] + 12 + (namesz + 3) // 4 * 4
            return msgpack.unpackb(elf[q:q + descsz])["amdhsa.kernels"]
    return []


def test_the_assembly_spills_no_registers():
    """k_asm<B, newmark2>, eight instances: no scratch memory, no spilled register."""
    if not os.path.exists(LIB):
        pytest.skip("library not built")
    found = {}
    for k in _kernels(LIB):
        if "5k_asmI" in k[".name"]:
            found[k[".name"]] = (k[".private_segment_fixed_size"], k[".vgpr_spill_count"],
                                 k[".sgpr_spill_count"])
    assert len(found) == 8
    assert set(found.values()) == {(0, 0, 0)}, found
