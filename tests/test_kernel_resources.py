"""Registers of built kernels, from the metadata of the library's own code objects (no GPU)."""
import os
import struct

import msgpack
import pytest

import pnfft_amd

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def kernels():
    """{kernel symbol: metadata} of every gfx950 code object in the library."""
    path = os.path.join(os.path.dirname(pnfft_amd.__file__), "libpnfft_amd.so")
    if not os.path.exists(path):
        pytest.skip("library not built")
    data = open(path, "rb").read()
    out = {}
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(count):
            off, size, tlen = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24:pos + 24 + tlen]
            pos += 24 + tlen
            if b"gfx950" in triple:
                out.update(elf_kernels(data[at + off:at + off + size]))
        at = data.find(MAGIC, at + len(MAGIC))
    return out


def elf_kernels(elf):
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    entsize, num = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(num):
        sh = struct.unpack_from("<IIQQQQIIQQ", elf, shoff + i * entsize)
        if sh[1] != 7:  # SHT_NOTE
            continue
        nsz, dsz, kind = struct.unpack_from("<III", elf, sh[4])
        if kind == 32:  # NT_AMDGPU_METADATA
            beg = sh[4] + 12 + (nsz + 3) // 4 * 4
            meta = msgpack.unpackb(elf[beg:beg + dsz], strict_map_key=False)
            return {k[".name"]: k for k in meta["amdhsa.kernels"]}
    return {}


def test_lds_atomic_scatter_holds_two_blocks_per_cu():
    """scatter_tiled_k has a thread for every node of its work item, so its node loop runs once and needs
    registers for one node: FP64 at m = 2 within the 128 of two blocks of eight waves per CU, in both modes, and
    no spills up to m = 5."""
    k = kernels()
    for mode in (1, 2):
        m2 = k[f"_ZN9pnfft_amd12_GLOBAL__N_115scatter_tiled_kIdLi2ELi{mode}EEEvNS_5BArgsIT_EE"]
        assert m2[".vgpr_count"] <= 128
        for m in (2, 3, 4, 5):
            v = k[f"_ZN9pnfft_amd12_GLOBAL__N_115scatter_tiled_kIdLi{m}ELi{mode}EEEvNS_5BArgsIT_EE"]
            assert v[".vgpr_spill_count"] == 0, (m, mode)
