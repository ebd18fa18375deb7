"""Registers of the built projection and weight-gradient kernels (CPU).

A tile loop that keeps its weights resident has no registers to spare: one
that spills waits for its own loads at each scratch access (element-load forms
that spilled 25 to 187 registers took up to 2.8 times as long as before).
The counts are the compiler's, from the metadata of the code objects that were
built here."""

from __future__ import annotations

import struct

import pytest

from lsso_amd import build

KERNELS = ("linear_kernel", "linear_stream_kernel", "weight_grad_kernel")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data: bytes):
    """The gfx950 ELF images of every offload bundle in a library."""

    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            name = data[entry + 24:entry + 24 + length]
            if name.endswith(build.OFFLOAD_ARCH.encode()) and size:
                yield data[at + offset:at + offset + size]
            entry += 24 + length
        at = data.find(MAGIC, at + len(MAGIC))


def _kernels(image: bytes):
    """amdhsa.kernels of a code object's AMDGPU metadata note."""

    msgpack = pytest.importorskip("msgpack")
    sections, = struct.unpack_from("<Q", image, 40)
    width, count = struct.unpack_from("<HH", image, 58)
    for i in range(count):
        header = struct.unpack_from("<IIQQQQ", image, sections + i * width)
        if header[1] != 7:   # SHT_NOTE
            continue
        at, end = header[4], header[4] + header[5]
        while at < end:
            name_size, size, kind = struct.unpack_from("<III", image, at)
            body = at + 12 + -(-name_size // 4) * 4
            if kind == 32:   # NT_AMDGPU_METADATA
                yield from msgpack.unpackb(image[body:body + size])["amdhsa.kernels"]
            at = body + -(-size // 4) * 4


def test_projection_kernels_do_not_spill() -> None:
    path = build.library_path()
    if not path.is_file():
        import __graft_entry__

        __graft_entry__.build()
    found = {}
    for image in _code_objects(path.read_bytes()):
        for kernel in _kernels(image):
            if any(part in kernel[".name"] for part in KERNELS):
                found[kernel[".name"]] = kernel[".vgpr_spill_count"]
    assert all(any(part in name for name in found) for part in KERNELS)
    assert {name: count for name, count in found.items() if count} == {}
