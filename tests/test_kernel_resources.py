"""CPU: registers of the built kernels, read from the metadata of the gfx950 code objects in
puter_amd/libputer_hip.so.  A kernel whose time is its passes over memory must not add
passes of its own by spilling registers."""
import os
import struct

import msgpack
import pytest

from puter_amd import build

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
NT_AMDGPU_METADATA = 32


def _code_objects(blob):
    at = blob.find(BUNDLE)
    while at >= 0:
        n, = struct.unpack_from("<Q", blob, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", blob, p)
            if b"gfx950" in blob[p + 24:p + 24 + length] and size:
                yield blob[at + off:at + off + size]
            p += 24 + length
        at = blob.find(BUNDLE, at + 24)


def _kernels(elf):
    """The kernels of the metadata note of an ELF64 code object."""
    phoff, = struct.unpack_from("<Q", elf, 32)
    phentsize, phnum = struct.unpack_from("<HH", elf, 54)
    for i in range(phnum):
        kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phentsize)
        if kind != 4:   # PT_NOTE
            continue
        end = off + size
        while off < end:
            namesz, descsz, ntype = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (namesz + 3) // 4 * 4
            if ntype == NT_AMDGPU_METADATA:
                yield from msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]
            off = desc + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(build.LIBRARY):
        build.build()
    with open(build.LIBRARY, "rb") as f:
        blob = f.read()
    found = {k[".name"]: k for elf in _code_objects(blob) for k in _kernels(elf)}
    assert len(found) > 100
    return found


@pytest.mark.parametrize("name", ["norm_line_kernel"])
def test_kernels_spill_no_registers(kernels, name):
    mine = {n: k for n, k in kernels.items() if name in n}
    assert mine
    assert not {n: k[".vgpr_spill_count"] for n, k in mine.items() if k[".vgpr_spill_count"]}
