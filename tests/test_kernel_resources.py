"""What the built library says of its backward kernels: no parameter of theirs
lies in a private array.  Such an array is scratch, or 16 bytes of LDS per
thread that are no tile, and each workgroup waits for it before its sweep.
"""
from __future__ import annotations

import re
import struct

import msgpack

from cmpext3 import abi


def _kernels(path):
    """{kernel name: metadata} of every code object in the library."""
    data, out = open(path, "rb").read(), {}
    for m in re.finditer(b"AMDGPU\0\0", data):
        namesz, descsz, kind = struct.unpack_from("<III", data, m.start() - 12) if m.start() >= 12 else (0, 0, 0)
        if namesz == 7 and kind == 32:  # NT_AMDGPU_METADATA
            meta = msgpack.unpackb(data[m.end():m.end() + descsz])
            out.update({k[".name"]: k for k in meta["amdhsa.kernels"]})
    return out


def test_backward_kernels_keep_their_parameters_in_registers():
    seen = 0
    for name, k in _kernels(abi.LIB_PATH).items():
        f32 = re.search(r"attn_bwd32_gradsILi(\d+)ELb\dELi(\d)E", name)
        f16 = re.search(r"attn_bwd_gradsIDF16b?_?Li(\d+)ELb(\d)ELb(\d)ELi\dE", name)
        if f32:
            dk, sweep = int(f32[1]), int(f32[2])
            tiles = 2 * 2 * 32 * ((dk + 15) // 16 * 16 + 4) * 4  # [slot][operand][row][col]
            assert k[".private_segment_fixed_size"] == 0, name
            assert k[".group_segment_fixed_size"] == tiles + (0 if sweep == 2 else 512), name
        elif f16:
            # masked, not causal, D <= 64 spills a few registers for its third wave
            spills = (int(f16[1]), f16[2], f16[3]) == (64, "0", "1")
            assert k[".private_segment_fixed_size"] <= (20 if spills else 0), name
        seen += bool(f32 or f16)
    assert seen >= 40
