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
    assert sum("14stream_collideI" in n for n in kernels) == 3 * 5 * 8 and any("10tiled_stepI" in n for n in kernels)
    used = {n: k[".private_segment_fixed_size"] for n, k in kernels.items() if k[".private_segment_fixed_size"]}
    assert not used, f"{len(used)} kernels, {list(used.items())[:3]}"


def test_field_kernels_keep_their_waves(kernels):
    """macroscopic and diagnostics_partial run 8 waves a SIMD on periodic lattices (64 of 512 vector
    registers a lane) and at least 7 (72) on bounded ones; the largest are the D3Q27 FP64 ones."""
    for kernel in ("11macroscopicI", "19diagnostics_partialI"):
        for bounded, most in (("Lb0E", 64), ("Lb1E", 72)):
            used = {n: k[".vgpr_count"] for n, k in kernels.items()
                    if kernel in n and n.split(kernel)[1].split("EEvPKv")[0].endswith(bounded)}
            assert len(used) == 3 * 5 * 2
            assert max(used.values()) <= most, max(used.items(), key=lambda i: i[1])
