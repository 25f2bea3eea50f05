"""Registers of the built kernels, as their code objects state them: a GEMM
whose ring or tile spills keeps its results and loses its speed, which no
parity test sees."""

from __future__ import annotations

import os
import re
import struct

import msgpack
import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "local_kimi_amd")


def _code_objects(data: bytes):
    """The gfx950 images of a shared library's offload bundles."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        pos = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, name = struct.unpack_from("<QQQ", data, pos)
            if b"gfx950" in data[pos + 24:pos + 24 + name]:
                yield data[at + offset:at + offset + size]
            pos += 24 + name
        at = data.find(magic, at + 24)


def _kernels(elf: bytes):
    """The kernel descriptions of a code object (its NT_AMDGPU_METADATA note)."""
    table = struct.unpack_from("<Q", elf, 40)[0]
    entry, count = struct.unpack_from("<HH", elf, 58)
    for i in range(count):
        at = table + i * entry
        if struct.unpack_from("<I", elf, at + 4)[0] != 7:  # SHT_NOTE
            continue
        pos, size = struct.unpack_from("<QQ", elf, at + 24)
        end = pos + size
        while pos < end:
            name, desc, kind = struct.unpack_from("<III", elf, pos)
            pos += 12 + (name + 3 & ~3)
            if kind == 32:
                yield from msgpack.unpackb(elf[pos:pos + desc])["amdhsa.kernels"]
            pos += desc + 3 & ~3


@pytest.fixture(scope="module")
def kernels():
    with open(os.path.join(PKG, "liblkamd.so"), "rb") as f:
        found = [k for elf in _code_objects(f.read()) for k in _kernels(elf)]
    assert len(found) > 100
    return found


def _template_args(symbol: str, name: str):
    """The integer template arguments of a mangled kernel name, or None."""
    m = re.search(rf"{name}I((?:L[ib]\d+E)+)E", symbol)
    return None if m is None else tuple(int(v) for v in re.findall(r"L[ib](\d+)E", m.group(1)))


def test_persistent_gemms_hold_their_ring_in_registers(kernels):
    """Two matrices at groups of 32 (format 4) and 64 (5) take four k-steps of
    ring wherever they divide; six, where only they divide, is the one that
    spills."""
    seen = 0
    for k in kernels:
        args = _template_args(k[".name"], "w4a16_persist_kernel")
        if args is None:
            continue
        seen += 1
        fmt, mats, depth = args[:3]
        if (fmt, mats, depth) == (4, 2, 6):
            continue
        assert k[".vgpr_spill_count"] <= 16, (k[".name"], k[".vgpr_spill_count"])
    assert seen > 50


def test_prefill_gemms_use_no_scratch_memory(kernels):
    sizes = {k[".name"]: k[".private_segment_fixed_size"] for k in kernels
             if _template_args(k[".name"], "tile_gemm_kernel") is not None}
    assert len(sizes) >= 18
    assert not {name: size for name, size in sizes.items() if size}
