"""What the compiler's metadata in the built library says of each kernel (registers, scratch), read on the host."""
import struct

import msgpack

_NOTE, _AMDGPU_METADATA = 7, 32   # section type, note type


def _code_objects(data):
    """The gfx950 ELF images of the library's offload bundles."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        entries, = struct.unpack_from("<Q", data, at + len(magic))
        entry = at + len(magic) + 8
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            if size and b"gfx950" in data[entry + 24:entry + 24 + length]:
                yield data[at + offset:at + offset + size]
            entry += 24 + length
        at = data.find(magic, at + len(magic))


def kernels(path):
    """{mangled name: its metadata}"""
    out = {}
    with open(path, "rb") as f:
        images = list(_code_objects(f.read()))
    for elf in images:
        sections, = struct.unpack_from("<Q", elf, 0x28)
        size, count = struct.unpack_from("<HH", elf, 0x3A)
        for i in range(count):
            _, kind, _, _, at, length = struct.unpack_from("<IIQQQQ", elf, sections + i * size)
            end = at + length if kind == _NOTE else 0
            while at < end:
                name, desc, note = struct.unpack_from("<III", elf, at)
                at += 12 + (name + 3 & ~3)
                if note == _AMDGPU_METADATA:
                    out.update((k[".name"], k) for k in msgpack.unpackb(elf[at:at + desc])["amdhsa.kernels"])
                at += desc + 3 & ~3
    return out
