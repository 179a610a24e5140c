"""Registers of the built decode-attention kernels, from the metadata notes of
the gfx950 code objects in libglacier_hip.so (no GPU needed).

A SIMD has 512 vector registers a lane, given out in eights: a kernel of up to
96 runs five waves there, up to 168 three. The one-item fp16 kernels of
contexts up to 256, with planes in Q8 or none, keep these whatever the other
layouts' conversions take."""
import os
import re
import struct
import subprocess

import msgpack
import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "glacier-engine_amd", "libglacier_hip.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + n]:
                yield data[at + off:at + off + size]
            p += 24 + n
        at = data.find(MAGIC, p)


def _kernels(elf):
    """amdhsa.kernels of an ELF64 code object's AMDGPU metadata note (type 32)."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    size, count = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        _, kind, _, _, off, length = struct.unpack_from("<IIQQQQ", elf, shoff + i * size)
        p = off
        while kind == 7 and p < off + length:  # SHT_NOTE
            n, d, note = struct.unpack_from("<III", elf, p)
            desc = p + 12 + (n + 3) // 4 * 4
            if note == 32:
                yield from msgpack.unpackb(elf[desc:desc + d])["amdhsa.kernels"]
            p = desc + (d + 3) // 4 * 4


@pytest.fixture(scope="module")
def resources():
    with open(LIB, "rb") as f:
        kernels = [k for o in _code_objects(f.read()) for k in _kernels(o)]
    names = subprocess.run(["c++filt"], input="\n".join(k[".name"] for k in kernels), text=True,
                           capture_output=True, check=True).stdout.split("\n")
    return {re.sub(r"^void |\(.*\)$", "", n): k for n, k in zip(names, kernels)}


@pytest.mark.parametrize("args,most", [("64, 2, 8, false, true", 96), ("128, 2, 8, false, true", 144)])
def test_short_context_attention_registers(resources, args, most):
    k = resources["gk::attn_list_kernel<%s>" % args]
    assert k[".vgpr_count"] <= most and k[".vgpr_spill_count"] == 0
