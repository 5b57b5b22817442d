"""Registers of compiled kernels whose speed hangs on how many waves a SIMD
holds: read from the metadata notes of the device code in the built library
(amdhsa.kernels of the NT_AMDGPU_METADATA note), no GPU needed.

A SIMD of gfx950 has 512 vector registers a lane, given out in blocks of 8,
and at most 8 waves."""
import re
import struct
import subprocess

import pytest

from amrsolver_amd import capi

msgpack = pytest.importorskip("msgpack")


def _code_objects(blob):
    """The gfx950 ELF images of the offload bundles in the library."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    pos = blob.find(magic)
    while pos >= 0:
        n, p = struct.unpack_from("<Q", blob, pos + 24)[0], pos + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, p)
            name = blob[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in name and size:
                yield blob[pos + off:pos + off + size]
        pos = blob.find(magic, pos + 1)


def _kernels(elf):
    shoff, = struct.unpack_from("<Q", elf, 40)
    entsize, num = struct.unpack_from("<HH", elf, 58)
    for i in range(num):
        kind, _, _, off, size = struct.unpack_from("<IQQQQ", elf, shoff + i * entsize + 4)
        if kind != 7:  # SHT_NOTE
            continue
        p = off
        while p < off + size:
            namesz, descsz, ntype = struct.unpack_from("<III", elf, p)
            desc = p + 12 + (namesz + 3) // 4 * 4
            if ntype == 32:
                yield from msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]
            p = desc + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    with open(capi.LIBPATH, "rb") as f:
        blob = f.read()
    ks = [k for elf in _code_objects(blob) for k in _kernels(elf)]
    names = subprocess.run(["c++filt"], input="\n".join(k[".name"] for k in ks), capture_output=True, text=True,
                           check=True).stdout.splitlines()
    out = {}
    for name, k in zip(names, ks):
        out[re.sub(r"\(anonymous namespace\)::|amr::|^void ", "", name.replace("void amr", "amr")).split("(")[0]] = k
    return out


def _waves(k):
    regs = k[".vgpr_count"]  # accumulation registers included
    return min(8, 512 // ((regs + 7) // 8 * 8))


def test_inviscid_order_2_with_neighbour_reads_keeps_three_waves(kernels):
    """Boxes with equal strides, KEEP order 2 without viscosity, 16x16 columns:
    at two waves (170 registers or more) 128x100x100 in 64x20x10 boxes takes
    224 us a step, at three 209."""
    k = kernels["k_fused<1, false, 16, 16, false, false, 2, false>"]
    assert _waves(k) >= 3 and k[".vgpr_spill_count"] == 0


def test_pass_structured_order_4_keeps_to_four_waves(kernels):
    """Five waves (96 registers or fewer) take 60 us on 96^3, four 57."""
    assert _waves(kernels["k_keep<2>"]) == 4
