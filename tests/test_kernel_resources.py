"""What the compiler made of the kernels whose speed hangs on it, read from the built library's own metadata (no GPU)."""
import os
import struct

import pytest

from flashnn_amd import _lib

msgpack = pytest.importorskip("msgpack")


def _kernels():
    """{kernel name: metadata} of every gfx950 code object in the library: offload bundles, each an ELF file with one note of
    metadata in msgpack."""
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("the library has not been built")
    blob = open(_lib.LIB_PATH, "rb").read()
    magic, found, at = b"__CLANG_OFFLOAD_BUNDLE__", {}, 0
    while (at := blob.find(magic, at)) >= 0:
        count, = struct.unpack_from("<Q", blob, at + 24)
        pos = at + 32
        for _ in range(min(count, 16)):
            offset, size, name_len = struct.unpack_from("<QQQ", blob, pos)
            name = blob[pos + 24:pos + 24 + name_len]
            pos += 24 + name_len
            elf = blob[at + offset:at + offset + size]
            if b"gfx950" not in name or elf[:4] != b"\x7fELF":
                continue
            sections, = struct.unpack_from("<Q", elf, 40)
            step, number = struct.unpack_from("<HH", elf, 58)
            for s in range(number):
                kind, = struct.unpack_from("<I", elf, sections + s * step + 4)
                if kind != 7:                                   # SHT_NOTE
                    continue
                start, _ = struct.unpack_from("<QQ", elf, sections + s * step + 24)
                owner, length, tag = struct.unpack_from("<III", elf, start)
                if tag == 32:                                   # NT_AMDGPU_METADATA
                    body = start + 12 + (owner + 3) // 4 * 4
                    for k in msgpack.unpackb(elf[body:body + length])["amdhsa.kernels"]:
                        found[k[".name"]] = k
        at += len(magic)
    return found


def _ring(kernels, bm, bn, form):
    got = [k for n, k in kernels.items() if f"gemm_a8w8_ring_kernelILi{bm}ELi{bn}E" in n and f"MoeFormE{form}E" in n]
    assert len(got) == 2        # two output types
    return got


def test_moe_tiles_of_whole_blocks_spill_nothing_to_speak_of():
    """The 256x256 tile fills the register file: sharing its code with the search for blocks put together, and the loop
    that goes with it, spilled 16 registers and cost blocks of 256 rows 8 % of their speed."""
    kernels = _kernels()
    assert all(k[".vgpr_spill_count"] <= 2 and k[".sgpr_spill_count"] == 0 for k in _ring(kernels, 256, 256, 1))
    for bm in (64, 128):
        for form in (1, 2):
            assert all(k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0
                       for k in _ring(kernels, bm, 128, form))
