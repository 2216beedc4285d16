"""What the compiler gave the kernels of the built library, from the metadata of its code objects."""

import os
import struct

import msgpack
import pytest

from dual_mod_public_amd import _build


def _code_objects(data):
    """The gfx code objects of the library's offload bundles."""
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, p)
            if b"gfx" in data[p + 24:p + 24 + length] and size:
                yield data[at + off:at + off + size]
            p += 24 + length
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


def _kernels(elf):
    """The kernel descriptions of a code object: its NT_AMDGPU_METADATA note (type 32)."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    size, num = struct.unpack_from("<HH", elf, 0x3a)
    for i in range(num):
        kind, = struct.unpack_from("<I", elf, shoff + i * size + 4)
        if kind != 7:   # SHT_NOTE
            continue
        p, length = struct.unpack_from("<QQ", elf, shoff + i * size + 0x18)
        end = p + length
        while p < end:
            nsz, dsz, note = struct.unpack_from("<III", elf, p)
            desc = p + 12 + (nsz + 3) // 4 * 4
            if note == 32:
                yield from msgpack.unpackb(elf[desc:desc + dsz], raw=False)["amdhsa.kernels"]
            p = desc + (dsz + 3) // 4 * 4


def test_decode_kernels_hold_their_rows_in_registers():
    """A split's K rows, kept from the scores on, must not go through scratch memory: a spilled form of the
    tape read moved as many bytes there as it read from the tape."""
    if not os.path.exists(_build.LIB):
        pytest.skip("the library is not built")
    with open(_build.LIB, "rb") as f:
        found = [k for elf in _code_objects(f.read()) for k in _kernels(elf) if "k_decode_" in k[".name"]]
    assert len(found) >= 8
    assert [(k[".name"], k[".private_segment_fixed_size"]) for k in found if k[".private_segment_fixed_size"]] == []
