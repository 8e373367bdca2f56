"""Registers of the step kernels in the built library.

A SIMD holds 512 vector registers per lane: a kernel of up to 128 runs four
wavefronts on it, one of 129 three, and one that does not fit keeps values in
scratch memory.  The counts are those that the compiler wrote beside each
kernel of libborn_hip.so (the metadata note of its gfx950 code objects)."""
import os
import struct
import subprocess

import pytest

from conftest import PKG

msgpack = pytest.importorskip("msgpack")


def _code_objects(path):
    """the gfx950 entries of every offload bundle in a host library"""
    data = open(path, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, p)
            if size and b"gfx950" in data[p + 24:p + 24 + length]:
                yield data[at + off:at + off + size]
            p += 24 + length
        at = data.find(magic, at + 24)


def _metadata(elf):
    """the NT_AMDGPU_METADATA (32) notes of a code object"""
    shoff, = struct.unpack_from("<Q", elf, 40)
    entry, count = struct.unpack_from("<HH", elf, 58)
    for k in range(count):
        kind, = struct.unpack_from("<I", elf, shoff + k * entry + 4)
        if kind != 7:  # SHT_NOTE
            continue
        p, size = struct.unpack_from("<QQ", elf, shoff + k * entry + 24)
        end = p + size
        while p < end:
            name, desc, kind = struct.unpack_from("<III", elf, p)
            p += 12 + (name + 3) // 4 * 4
            if kind == 32:
                yield msgpack.unpackb(elf[p:p + desc])
            p += (desc + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    """{"kernel<op, rows, waves, cells, lookahead, lanes>": its metadata}"""
    found = {}
    for elf in _code_objects(os.path.join(PKG, "libborn_hip.so")):
        for m in _metadata(elf):
            for k in m["amdhsa.kernels"]:
                found[k[".name"]] = k
    names = list(found)
    plain = subprocess.run(["c++filt"], input="\n".join(names), text=True, check=True,
                           capture_output=True).stdout.split("\n")
    return {p.split("(")[0].replace("born::", "").replace("void ", ""): found[n]
            for p, n in zip(plain, names)}


# two rows per lane, one cell per lane: the shapes whose rows and fields were
# held in registers together (128 registers: four wavefronts a SIMD)
@pytest.mark.parametrize("op,shape", [
    ("FwdOp<0, float, true, false, false>", "2, 4, 1, 1, 64"),
    ("FwdOp<0, float, true, false, false>", "2, 8, 1, 1, 64"),
    ("FwdOp<0, __half, true, true, false>", "2, 4, 1, 1, 64"),
    ("FwdOp<0, __half, true, true, false>", "2, 8, 1, 2, 64")])
def test_four_wavefronts_per_simd(kernels, op, shape):
    k = kernels["march_kernel<%s, %s>" % (op, shape)]
    assert k[".private_segment_fixed_size"] == 0
    assert k[".vgpr_count"] <= 128, k[".vgpr_count"]


def test_fp32_levels_apart_do_not_spill(kernels):
    some = [n for n in kernels if n.startswith("march_kernel<FwdOp<") and "float, true, false" in n]
    assert len(some) == 68
    assert [n for n in some if kernels[n][".private_segment_fixed_size"]] == []
