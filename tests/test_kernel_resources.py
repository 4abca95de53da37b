"""Registers and scratch of the built kernels, from the code objects' own metadata."""
import re
import struct

import msgpack
import pytest

from hqmq_amd import _lib as L


def _kernels():
    """name -> metadata of every gfx950 kernel in the library (its fat binary: offload bundles that hold one ELF file per target)."""
    blob, found, at = L.library_path().read_bytes(), {}, 0
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    while (at := blob.find(magic, at)) >= 0:
        base, p = at, at + 24
        (entries,) = struct.unpack_from("<Q", blob, p)
        p += 8
        for _ in range(entries):
            offset, size, n = struct.unpack_from("<QQQ", blob, p)
            target = blob[p + 24:p + 24 + n]
            p += 24 + n
            if b"gfx950" in target and size:
                found.update(_metadata(blob[base + offset:base + offset + size]))
        at += 24
    return found


def _metadata(elf):
    (phoff,), (phentsize, phnum) = struct.unpack_from("<Q", elf, 32), struct.unpack_from("<HH", elf, 54)
    for i in range(phnum):
        kind, _, offset, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phentsize)
        p, end = offset, offset + size
        while kind == 4 and p < end:                            # PT_NOTE
            name, desc, note = struct.unpack_from("<III", elf, p)
            p += 12
            if elf[p:p + name].rstrip(b"\0") == b"AMDGPU" and note == 32:
                p += (name + 3) // 4 * 4
                return {k[".name"]: k for k in msgpack.unpackb(elf[p:p + desc])["amdhsa.kernels"]}
            p += (name + 3) // 4 * 4 + (desc + 3) // 4 * 4
    return {}


@pytest.fixture(scope="module")
def fast():
    """(chunks per lane, main, aux and index bits, dtype, outliers, wavefronts, column groups, float8) -> metadata of attn_fast_kernel"""
    out = {}
    for name, k in _kernels().items():
        m = re.search(r"attn_fast_kernelI" + r"Li(\d+)E" * 5 + r"Lb(\d)E" + r"Li(\d+)E" * 2 + r"Lb(\d)E", name)
        if m:
            out[tuple(int(g) for g in m.groups())] = k
    assert len(out) > 100
    return out


def test_decode_kernels_use_no_scratch(fast):
    assert {k: m[".private_segment_fixed_size"] for k, m in fast.items() if m[".private_segment_fixed_size"]} == {}


def test_two_blocks_of_plain_heads_of_64_fit_a_compute_unit(fast):
    """Eight wavefronts a block, four per SIMD: 512 / 4 registers each.  (Tables multiplied out fill the LDS with one block.)"""
    seen = 0
    for (cpl, mb, ab, ib, _, flags, waves, groups, _), m in fast.items():
        if cpl == 4 and not flags and waves == 8 and groups == 1 and (mb, ab, ib) != (12, 1, 10):
            seen += 1
            assert m[".vgpr_count"] <= 128, (mb, ab, ib, m[".vgpr_count"])
    assert seen == 18           # 16+0 (index width known or not), 16+1, 16+2, 16+3 (twice), 12+1, 12+2, 12+3, in both types


def test_prefill_kernels_spill_no_more_registers():
    """Vector registers that attn_prefill_kernel puts into scratch, by head size and outliers: few enough for the time they were measured with."""
    spilled, seen = {}, 0
    for name, k in _kernels().items():
        m = re.search(r"attn_prefill_kernelILi(\d+)ELi(\d+)ELb(\d)ELi(\d)ELi(\d)ELb(\d)E", name)
        if m:
            d_h, _, aux, _, _, flags = (int(g) for g in m.groups())
            seen += 1
            if k[".vgpr_spill_count"] > (0 if d_h == 64 else 3 if not flags else 21 if aux else 14):
                spilled[name] = k[".vgpr_spill_count"]
    assert seen == 36 and spilled == {}
