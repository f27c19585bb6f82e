"""Register use of the built kernels, read from the library's own metadata (CPU
only): a kernel that spills vector registers sends every iteration of its loop
through scratch memory."""
import os
import re
import struct

import pytest

from bytes_amd import _lib

msgpack = pytest.importorskip("msgpack")


def _kernels():
    """name -> metadata of every gfx950 kernel in libbytes_amd.so: the ELF notes
    of the code objects in its offload bundles."""
    if not os.path.exists(_lib.LIB_PATH):
        pytest.fail(f"{_lib.LIB_PATH} not built (run python -m bytes_amd.build)")
    d = open(_lib.LIB_PATH, "rb").read()
    magic, out = b"__CLANG_OFFLOAD_BUNDLE__", {}
    at = d.find(magic)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", d, at + 24)
        p = at + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", d, p)
            triple, p = d[p + 24:p + 24 + n], p + 24 + n
            if b"gfx950" in triple and size:
                out.update(_notes(d[at + off:at + off + size]))
        at = d.find(magic, at + 24)
    assert out
    return out


def _notes(elf):
    out = {}
    (shoff,), (width, count) = struct.unpack_from("<Q", elf, 0x28), struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        kind, start, size = (struct.unpack_from("<I", elf, shoff + i * width + 4)
                             + struct.unpack_from("<QQ", elf, shoff + i * width + 24))
        if kind != 7:                                        # SHT_NOTE
            continue
        q = start
        while q < start + size:
            names, descs, _ = struct.unpack_from("<III", elf, q)
            name, q = elf[q + 12:q + 12 + names].rstrip(b"\0"), q + 12 + (names + 3) // 4 * 4
            if name == b"AMDGPU":
                out.update((k[".name"], k) for k in msgpack.unpackb(elf[q:q + descs])["amdhsa.kernels"])
            q += (descs + 3) // 4 * 4
    return out


def test_no_kernel_spills_vector_registers():
    spilled = {n: k[".vgpr_spill_count"] for n, k in _kernels().items() if k[".vgpr_spill_count"]}
    assert not spilled, spilled


def test_narrow_pq_decode_leaves_room_for_two_workgroups():
    """The D = 64 general PQ kernel (eight waves a workgroup) with at most 4
    outlier channels: four waves to a SIMD, and twice its LDS, fit a CU."""
    seen = 0
    for n, k in _kernels().items():
        m = re.search(r"pq_decode_kernelILi64ELb\dELb\dELb\dELi([04])E", n)
        if m:
            seen += 1
            regs = -(-(k[".vgpr_count"] + k.get(".agpr_count", 0)) // 8) * 8
            assert regs <= 128 and 2 * k[".group_segment_fixed_size"] <= 160 * 1024, n
    assert seen
