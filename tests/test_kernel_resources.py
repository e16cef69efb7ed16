"""Registers and scratch memory of the built kernels, from the metadata that the compiler writes into
the library's code objects: the per-cell state lives in registers, so no kernel uses scratch memory."""
import struct

import msgpack
import pytest

from cfd_solvers_amd import build


def _code_objects(data):
    """The gfx950 members of the offload bundles (magic, count, then offset, size and triple each)."""
    at = 0
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        count, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + length]:
                yield data[at + offset:at + offset + size]
            p += 24 + length
        at += 24


def _kernels(elf):
    """The kernels of the code object's metadata note (type 32, msgpack)."""
    table, = struct.unpack_from("<Q", elf, 32)
    entry, count = struct.unpack_from("<HH", elf, 54)
    for k in range(count):
        kind, = struct.unpack_from("<I", elf, table + k * entry)
        offset, = struct.unpack_from("<Q", elf, table + k * entry + 8)
        if kind != 4:  # PT_NOTE
            continue
        name_size, size, note = struct.unpack_from("<III", elf, offset)
        if note == 32:
            start = offset + 12 + (name_size + 3) // 4 * 4
            yield from msgpack.unpackb(elf[start:start + size])["amdhsa.kernels"]


@pytest.fixture(scope="module")
def kernels():
    if not build.LIB.exists():
        build.build()
    return {k[".name"]: k for elf in _code_objects(build.LIB.read_bytes()) for k in _kernels(elf)}


def test_no_kernel_uses_scratch_memory(kernels):
    assert sum("14stream_collideI" in n for n in kernels) == 3 * 5 * 8 and sum("10tiled_stepI" in n for n in kernels) == 48
    used = {n: k[".private_segment_fixed_size"] for n, k in kernels.items() if k[".private_segment_fixed_size"]}
    assert not used, f"{len(used)} kernels, {list(used.items())[:3]}"
