"""Registers of the library's kernels where a wave per SIMD hangs on them, from
the metadata of the code object that the build put into the library."""
import os
import re
import struct

import msgpack
import pytest

from nemaktis_amd import _lib

NT_AMDGPU_METADATA = 32


def _code_objects(data):
    """gfx950 code objects of every offload bundle in the file."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(magic))
        pos = at + len(magic) + 8
        for _ in range(n):
            off, size, tlen = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24:pos + 24 + tlen]
            pos += 24 + tlen
            if b"gfx950" in triple:
                yield data[at + off:at + off + size]
        at = data.find(magic, at + 1)


def _kernels(elf):
    shoff, = struct.unpack_from("<Q", elf, 40)
    entsize, num = struct.unpack_from("<HH", elf, 58)
    for i in range(num):
        kind, = struct.unpack_from("<I", elf, shoff + i * entsize + 4)
        off, size = struct.unpack_from("<QQ", elf, shoff + i * entsize + 24)
        end = off + size
        while kind == 7 and off < end:  # SHT_NOTE
            namesz, descsz, note = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (namesz + 3) // 4 * 4
            if note == NT_AMDGPU_METADATA:
                for k in msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]:
                    yield k
            off = desc + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    with open(_lib.LIB_PATH, "rb") as f:
        data = f.read()
    return [k for elf in _code_objects(data) for k in _kernels(elf)]


# a SIMD has 512 vector registers a lane: 128 for four waves
@pytest.mark.parametrize("kernel,most", [("k_fft_rowsILi[0-9]+ELi1E", 128)])
def test_registers(kernels, kernel, most):
    hits = [k for k in kernels if re.search(kernel, k[".name"])]
    assert hits
    for k in hits:
        assert k[".vgpr_count"] <= most and k[".vgpr_spill_count"] == 0, (k[".name"], k[".vgpr_count"])
