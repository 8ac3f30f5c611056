"""Registers of the built kernels whose speed hangs on how many of their workgroups a CU holds, read from the library's own metadata."""

from __future__ import annotations

import re
import struct

import msgpack

from pygpukit_amd import _hip


def _kernels():
    """name -> metadata of every kernel: the AMDGPU notes of the code objects inside the library"""
    _hip.load()
    with open(_hip.LIB_PATH, "rb") as f:
        b = f.read()
    out = {}
    for m in re.finditer(rb"\x7fELF\x02\x01\x01\x40", b):        # an ELF file for AMD's HSA
        at = m.start()
        table, count = struct.unpack_from("<Q", b, at + 0x28)[0], struct.unpack_from("<H", b, at + 0x3C)[0]
        for i in range(count):
            head = at + table + 64 * i
            if struct.unpack_from("<I", b, head + 4)[0] != 7:    # a note
                continue
            off = at + struct.unpack_from("<Q", b, head + 24)[0]
            name, size = struct.unpack_from("<II", b, off)
            start = off + 12 + (name + 3 & ~3)
            out.update({k[".name"]: k for k in msgpack.unpackb(b[start:start + size])["amdhsa.kernels"]})
    return out


def test_windowed_attention_of_head_dim_64_leaves_room_for_three_workgroups():
    """Four waves each, one on every SIMD, whose 512 registers hold three of up to 168; nothing of them spilled."""
    got = {n: k for n, k in _kernels().items() if "flash_fwd_kernel" in n and "Li64ELb1E" in n}
    assert len(got) == 2, list(got)                              # without and with slopes
    for n, k in got.items():
        assert k[".vgpr_count"] <= 168 and k[".private_segment_fixed_size"] == 0, (n, k[".vgpr_count"], k[".private_segment_fixed_size"])


def test_merge_and_o_proj_of_four_heads_leaves_room_for_four_workgroups():
    """One wave on every SIMD, whose 512 registers hold four of up to 128: two sequences launch more than two workgroups to a CU."""
    got = {n: k for n, k in _kernels().items() if "attn_merge_oproj_kernelILi128ELi4E" in n}
    assert len(got) == 4, list(got)                              # bf16 and e4m3 weights, up to 16 slices and more
    for n, k in got.items():
        assert k[".vgpr_count"] <= 128 and k[".private_segment_fixed_size"] == 0, (n, k[".vgpr_count"], k[".private_segment_fixed_size"])
