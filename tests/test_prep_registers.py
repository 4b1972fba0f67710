"""Registers of the single-pass prep kernels, from the metadata of the code
objects in the built library: spilled registers are reloaded among the loads of
the next row, and a row then waits for those.  Kernels with either factors or a
perm carry no more than their own gather's values, and R = 4096 rows of four
tiles (13312 to 16384 values) have a whole register file per wave.  CPU only."""
from __future__ import annotations

import re
import struct

import msgpack
import pytest

_KERNEL = re.compile(r"rq_fast_kernelI((?:L[ib]\d+E)+)E")


def _code_objects(blob: bytes):
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := blob.find(magic, at)) >= 0:
        pos = at + len(magic)
        (n,) = struct.unpack_from("<Q", blob, pos)
        pos += 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, pos)
            name = blob[pos + 24 : pos + 24 + idlen]
            pos += 24 + idlen
            if b"amdgcn" in name and size:
                yield blob[at + off : at + off + size]
        at += len(magic)


def _metadata(elf: bytes) -> dict:
    (shoff,) = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        base = shoff + i * shentsize
        (kind,) = struct.unpack_from("<I", elf, base + 4)
        off, size = struct.unpack_from("<QQ", elf, base + 0x18)
        if kind != 7:  # SHT_NOTE
            continue
        nlen, dlen, note = struct.unpack_from("<III", elf, off)
        if note == 32:  # NT_AMDGPU_METADATA
            start = off + 12 + (nlen + 3) // 4 * 4
            return msgpack.unpackb(elf[start : start + dlen], strict_map_key=False)
    return {}


@pytest.fixture(scope="module")
def kernels(rt):
    """(dtype, log4 R, tiles, variant, threads, norm, quant, waves) -> kernel metadata"""
    assert rt.KERNELS_AVAILABLE, rt.LOAD_ERROR
    out = {}
    with open(rt.LIB_PATH, "rb") as f:
        blob = f.read()
    for elf in _code_objects(blob):
        for k in _metadata(elf).get("amdhsa.kernels", []):
            m = _KERNEL.search(k[".name"])
            if m:
                out[tuple(int(v) for v in re.findall(r"L[ib](\d+)E", m.group(1)))] = k
    assert len(out) > 500
    return out


def _spills(kernels, log4r, tiles, variant, threads):
    found = {key: k for key, k in kernels.items() if key[1:5] == (log4r, tiles, variant, threads)}
    assert found
    return found


GENERAL, BOTH = 1, 2  # factors or a perm; both


@pytest.mark.parametrize("log4r", [0, 2, 3, 4, 5])
def test_gather_of_two_narrow_tiles(kernels, log4r):
    for key, k in _spills(kernels, log4r, 2, GENERAL, 192).items():
        assert k[".vgpr_spill_count"] <= 24, key


def test_three_tiles_across_waves(kernels):
    for key, k in _spills(kernels, 6, 3, GENERAL, 256).items():
        if key[0] == 1:  # bf16; f16 keeps another part of its constants in scratch
            assert k[".vgpr_spill_count"] <= 35, key
        assert k[".private_segment_fixed_size"] <= 144, key


@pytest.mark.parametrize("variant", [GENERAL, BOTH])
def test_four_tiles_across_waves(kernels, variant):
    for key, k in _spills(kernels, 6, 4, variant, 256).items():
        assert k[".private_segment_fixed_size"] == 0, key


@pytest.mark.parametrize("threads", [64, 128, 256])
def test_one_narrow_tile_keeps_three_waves(kernels, threads):
    """R = 1024 with factors or a perm: bf16, and f16 behind a norm, hold more than
    128 registers (three waves per SIMD), which many short rows run faster on."""
    for key, k in _spills(kernels, 5, 1, GENERAL, threads).items():
        if key[6] and (key[0] == 1 or key[5]):
            assert k[".vgpr_count"] > 128 and k[".vgpr_spill_count"] == 0, key


def test_one_tile_across_waves_behind_a_norm(kernels):
    for key, k in _spills(kernels, 6, 1, GENERAL, 256).items():
        if key[5]:
            assert k[".vgpr_spill_count"] == 0, key
