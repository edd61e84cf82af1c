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


def _allocated_vgprs(elf):
    """{kernel: VGPRs a wave is given} from the kernel descriptors (<kernel>.kd, 64 bytes; the low six bits of the
    32-bit word at 48 count eights, less one): what decides the waves per SIMD, also where the compiler rounds the
    allocation up to keep to a limit on them."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum = struct.unpack_from("<HH", elf, 58)
    sec = [struct.unpack_from("<IIQQQQIIQQ", elf, shoff + i * shentsize) for i in range(shnum)]
    for _, kind, _, _, off, size, link, _, _, entsize in sec:
        if kind != 11:  # SHT_DYNSYM
            continue
        names = sec[link][4]
        for p in range(off, off + size, entsize):
            st_name, _, _, shndx, value, _ = struct.unpack_from("<IBBHQQ", elf, p)
            name = elf[names + st_name:elf.index(b"\0", names + st_name)].decode()
            if name.endswith(".kd"):
                at = sec[shndx][4] + value - sec[shndx][3]
                yield name[:-3], ((struct.unpack_from("<I", elf, at + 48)[0] & 63) + 1) * 8


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
                elf = blob[m.start() + off:m.start() + off + size]
                for note in _notes(elf):
                    found.update({k[".name"]: k for k in note["amdhsa.kernels"]})
                for name, n in _allocated_vgprs(elf):
                    found[name]["allocated"] = n
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
            assert k["allocated"] <= 128, (pt, nt, k["allocated"])


def test_walks_and_pair_scan_leave_room_for_two_blocks(kernels_meta):
    """State walks of up to eight waves (2 per SIMD): at most 128 VGPRs, two blocks to a CU. The exact forward scan of
    the halves of wide heads, one wave per SIMD: at most 256 for chunks of 64 and 128 tokens (for 128 with NT = 4 its
    accumulators and S take more)."""
    for (pt, nt, _), k in _variants(kernels_meta, "k_state_fused").items():
        if pt * nt <= 4:
            assert k["allocated"] <= 128, (pt, nt, k["allocated"])
    for (pt, nt, nb, s32), k in _variants(kernels_meta, "k_scan_fwd_chunk").items():
        if s32 and (nb == 1 or nb == 2 and nt < 4):
            assert k["allocated"] <= 256, (pt, nt, nb, k["allocated"])


def test_head_kernel_spills_little(kernels_meta):
    """k_bwd_head<PT, NT, MODE, LATE>: no spills but a few registers with NT = 4, whose dC / dB accumulators and dS
    tiles alone take 128 of the 256 (more only in the variant of the shortest chunks' MODE 3)."""
    for (pt, nt, mode, late), k in _variants(kernels_meta, "k_bwd_head").items():
        if mode != 3 or late or nt < 4:
            assert k[".vgpr_spill_count"] <= (24 if nt == 4 else 0), (pt, nt, mode, k[".vgpr_spill_count"])
