"""Where the raster's tile memory begins.  k_tile_raster's dynamic LDS holds
64-bit keys and 16-byte rows, which the compiler reads and writes with
instructions for 16-byte aligned words; it starts where the kernel's own
(static) LDS ends.  The sizes are those of the built library's code object."""
import os
import struct

import msgpack

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(path):
    """The gfx950 ELF images bundled into the library, one per source file."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in target and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + len(MAGIC))


def _kernels(elf):
    """(name, static LDS bytes) of each kernel, from the metadata note."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        kind, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        off, size = struct.unpack_from("<QQ", elf, shoff + i * shentsize + 0x18)
        if kind != 7:   # SHT_NOTE
            continue
        namesz, descsz, _ = struct.unpack_from("<III", elf, off)
        desc = off + 12 + (namesz + 3) // 4 * 4
        for k in msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]:
            yield k[".name"], k[".group_segment_fixed_size"]


def test_raster_tile_memory_is_aligned():
    from sloth_amd import _build

    if not os.path.exists(_build.LIB):
        _build.build()
    sizes = [(name, lds) for elf in _code_objects(_build.LIB) for name, lds in _kernels(elf) if "k_tile_raster" in name]
    assert sizes
    assert [s for s in sizes if s[1] % 16] == []
