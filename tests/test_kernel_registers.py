"""Registers and scratch memory of the stage kernels, from the metadata of the
code objects in the built library.  A SIMD has 512 registers per lane,
allocated by eights: three waves take at most 168 each, two 256.  The
ensemble's one-material form is held to two."""
import os
import re
import struct
import subprocess

import msgpack
import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "m2c_amd", "libm2c_amd.so")
pytestmark = pytest.mark.skipif(not os.path.exists(LIB), reason="libm2c_amd.so not built")
SHT_NOTE, NT_AMDGPU_METADATA = 7, 32


def _elf_kernels(e):
    shoff, = struct.unpack_from("<Q", e, 0x28)
    size, count = struct.unpack_from("<HH", e, 0x3A)
    for s in range(count):
        h = shoff + s * size
        if struct.unpack_from("<I", e, h + 4)[0] != SHT_NOTE:
            continue
        q, length = struct.unpack_from("<QQ", e, h + 0x18)
        end = q + length
        while q < end:
            name, desc, kind = struct.unpack_from("<III", e, q)
            at = q + 12 + (name + 3) // 4 * 4
            if kind == NT_AMDGPU_METADATA:
                return msgpack.unpackb(e[at:at + desc])["amdhsa.kernels"]
            q = at + (desc + 3) // 4 * 4
    return []


@pytest.fixture(scope="module")
def kernels():
    """{demangled name: (registers, scratch bytes)}, one bundle per unit."""
    d = open(LIB, "rb").read()
    found, pos = [], d.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while pos >= 0:
        entries, p = struct.unpack_from("<Q", d, pos + 24)[0], pos + 32
        for _ in range(entries):
            off, size, n = struct.unpack_from("<QQQ", d, p)
            if b"gfx950" in d[p + 24:p + 24 + n]:
                found += _elf_kernels(d[pos + off:pos + off + size])
            p += 24 + n
        pos = d.find(b"__CLANG_OFFLOAD_BUNDLE__", pos + 24)
    names = subprocess.run(["c++filt"], input="\n".join(k[".name"] for k in found), capture_output=True, text=True,
                           check=True).stdout.split("\n")
    return {n.split("(")[0]: (k[".vgpr_count"], k[".private_segment_fixed_size"]) for k, n in zip(found, names)}


# kernel<mode, tile, ...>; the last two of k_stage_u: HLLC, any variables
@pytest.mark.parametrize("pattern,count,waves", [
    (r"k_stage_u<\d, \d+, \d+, \d+, true, false>", 24, 3),
    (r"k_stage_u_multi<\d, \d+, \d+, \d+, (true|false), false>", 32, 2),
    (r"k_stage_u<\d, \d+, \d+, \d+, (true, true|false, (true|false))>", 36, 2),
    (r"k_stage<\d, \d+, \d+, \d+, false>", 24, 3),
    (r"k_stage_multi<\d, \d+, \d+, \d+>", 16, 3),
])
def test_waves_of_the_stage_kernels(kernels, pattern, count, waves):
    found = {n: k for n, k in kernels.items() if re.search(r"::%s$" % pattern, n)}
    assert len(found) == count
    least, most = {2: (169, 256), 3: (129, 168)}[waves]
    assert {n: k for n, k in found.items() if not least <= k[0] <= most or k[1] > 0} == {}
