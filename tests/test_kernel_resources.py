"""Registers and block sizes of the built kernels, read on the CPU from the metadata notes of the library's gfx950
code objects: what a launch needs to be possible, and what a kernel's blocks per CU depend on."""
from __future__ import annotations

import re
import struct

import pytest

msgpack = pytest.importorskip("msgpack")


def _notes(elf):
    """The AMDGPU metadata maps of one code object (ELF64, little-endian): notes of type 32 named AMDGPU."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum = struct.unpack_from("<HH", elf, 58)
    for i in range(shnum):
        _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + i * shentsize)
        if kind != 7:  # SHT_NOTE
            continue
        pos = off
        while pos + 12 <= off + size:
            nlen, dlen, ntype = struct.unpack_from("<III", elf, pos)
            name = elf[pos + 12:pos + 12 + nlen].rstrip(b"\0")
            data = pos + 12 + (nlen + 3) // 4 * 4
            if ntype == 32 and name == b"AMDGPU":
                yield msgpack.unpackb(elf[data:data + dlen])
            pos = data + (dlen + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels_meta():
    from kernels import _capi
    blob = _capi.LIB_PATH.read_bytes()
    found = {}
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", blob):
        count, = struct.unpack_from("<Q", blob, m.end())
        pos = m.end() + 8
        for _ in range(count):
            off, size, idlen = struct.unpack_from("<QQQ", blob, pos)
            target = blob[pos + 24:pos + 24 + idlen]
            pos += 24 + idlen
            if b"gfx950" in target and size:
                for note in _notes(blob[m.start() + off:m.start() + off + size]):
                    found.update({k[".name"]: k for k in note["amdhsa.kernels"]})
    assert len(found) > 100
    return found


def _variants(meta, kernel):
    """{template arguments: metadata} of a kernel template with int and bool arguments."""
    out = {}
    for name, k in meta.items():
        m = re.match(rf"_Z{len(kernel)}{kernel}I((?:L[ib]\d+E)+)E", name)
        if m:
            out[tuple(int(v) for v in re.findall(r"L[ib](\d+)E", m.group(1)))] = k
    assert out, kernel
    return out


def test_row_kernel_leaves_room_for_two_blocks(kernels_meta):
    """k_bwd_gemm<PT, NT, MULTI>: blocks of 512 threads, two to a CU (at most 128 VGPRs) where two of their LDS rings
    fit and the accumulators allow it, and no spills anywhere."""
    for (pt, nt, _), k in _variants(kernels_meta, "k_bwd_gemm").items():
        assert k[".vgpr_spill_count"] == 0, (pt, nt)
        ring = 3 * (2 * 2 * (32 * pt * 32 * nt + 64 * 32 * pt) + 1024)
        if nt <= 2 and 2 * (ring + 256) <= 160 * 1024:
            assert k[".vgpr_count"] <= 128, (pt, nt, k[".vgpr_count"])
