"""No kernel of the library keeps registers in scratch memory, by the metadata of its code objects: a spill or two costs every launch 0.3 us and limits the
waves that a launch may have resident."""
import os
import struct

import pytest

from conftest import PKG

msgpack = pytest.importorskip("msgpack")
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    """The gfx950 code objects of the bundles in the library."""
    at = data.find(BUNDLE)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(BUNDLE))
        p = at + len(BUNDLE) + 8
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", data, p)
            triple = data[p + 24:p + 24 + name]
            p += 24 + name
            if b"gfx950" in triple:
                yield data[at + offset:at + offset + size]
        at = data.find(BUNDLE, at + len(BUNDLE))


def kernels(elf):
    """The kernels' entries in the AMDGPU metadata note (type 32, MessagePack) of a 64-bit little-endian ELF file."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    entsize, count = struct.unpack_from("<HH", elf, 0x3a)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, shoff + i * entsize + 4)
        offset, size = struct.unpack_from("<QQ", elf, shoff + i * entsize + 0x18)
        if kind != 7:                                            # SHT_NOTE
            continue
        name, desc, note = struct.unpack_from("<III", elf, offset)
        if note == 32:
            start = offset + 12 + (name + 3) // 4 * 4
            return msgpack.unpackb(elf[start:start + desc], strict_map_key=False)["amdhsa.kernels"]
    return []


def test_no_kernel_uses_scratch():
    path = os.path.join(PKG, "libsparseops_hip.so")
    if not os.path.exists(path):
        pytest.skip("the library is not built")
    with open(path, "rb") as f:
        found = [k for elf in code_objects(f.read()) for k in kernels(elf)]
    assert len(found) > 300 and any("conv2d_window_kernel" in k[".name"] for k in found)
    assert [(k[".name"], k[".private_segment_fixed_size"]) for k in found if k[".private_segment_fixed_size"] != 0] == []
