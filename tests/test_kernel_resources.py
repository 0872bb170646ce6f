"""Scratch memory of the built kernels, from the metadata of the library's code objects."""

import struct

import msgpack

from helpers import load_pkg


def _sections(elf):
    at = struct.unpack_from("<Q", elf, 0x28)[0]
    size, count, names = struct.unpack_from("<HHH", elf, 0x3A)
    head = [struct.unpack_from("<IIQQQQIIQQ", elf, at + i * size) for i in range(count)]
    text = head[names][4]
    for s in head:
        start = text + s[0]
        yield elf[start:elf.index(b"\0", start)], s[1], elf[s[4]:s[4] + s[5]]


def _code_objects(library):
    fat = next(data for name, _, data in _sections(library) if name == b".hip_fatbin")
    at = fat.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        q = at + 32
        for _ in range(struct.unpack_from("<Q", fat, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", fat, q)
            if b"gfx" in fat[q + 24:q + 24 + length] and size:
                yield fat[at + offset:at + offset + size]
            q += 24 + length
        at = fat.find(b"__CLANG_OFFLOAD_BUNDLE__", q)


def _kernels():
    out = {}
    with open(load_pkg().LIB_PATH, "rb") as f:
        library = f.read()
    for elf in _code_objects(library):
        for _, kind, data in _sections(elf):
            q = 0
            while kind == 7 and q < len(data):  # notes
                name, desc, note = struct.unpack_from("<III", data, q)
                q += 12 + (name + 3) // 4 * 4
                if note == 32:
                    out.update({k[".name"]: k for k in msgpack.unpackb(data[q:q + desc])["amdhsa.kernels"]})
                q += (desc + 3) // 4 * 4
    return out


def test_path_kernels_keep_no_parameter_block_in_scratch():
    """The kernels that walk paths may spill some registers, but hold no copy of their parameter block
    (above 700 bytes), which a selection among its members by address makes of it."""
    kernels = {n: k for n, k in _kernels().items() if "pipe_trace" in n or "trace_" in n}
    assert len(kernels) >= 28
    bad = {n: k[".private_segment_fixed_size"] for n, k in kernels.items() if k[".private_segment_fixed_size"] > 256}
    assert not bad, bad
