"""Resources of the built kernels, read from the code objects in
libereb_hip.so: kernels that the hot calls launch keep everything in registers
and LDS.  Scratch memory costs its traffic on every launch, and the runtime
allocates it at the first dispatch of such a kernel on a queue.  It comes in
unnoticed: a select among members of a by-reference argument, or two branches
merged into one access through a pointer, put whole structures there."""
from __future__ import annotations

import struct

import msgpack
import pytest

import ereb.lib

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _kernels(elf: bytes):
    """The kernel entries of a code object's metadata note."""
    assert elf[:5] == b"\x7fELF\x02"
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    out = []
    for k in range(shnum):
        _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + k * shentsize)
        if kind != 7:  # SHT_NOTE
            continue
        namesz, descsz, ntype = struct.unpack_from("<III", elf, off)
        name = elf[off + 12:off + 12 + namesz].rstrip(b"\0")
        if name == b"AMDGPU" and ntype == 32:
            at = off + 12 + (namesz + 3) // 4 * 4
            out += msgpack.unpackb(elf[at:at + descsz])["amdhsa.kernels"]
    return out


@pytest.fixture(scope="module")
def scratch():
    """{mangled kernel name: bytes of scratch a lane}"""
    with open(ereb.lib.LIB_PATH, "rb") as f:
        lib = f.read()
    out, at = {}, lib.find(MAGIC)
    while at >= 0:
        p = at + len(MAGIC)
        n, = struct.unpack_from("<Q", lib, p)
        p += 8
        for _ in range(n):
            off, size, tl = struct.unpack_from("<QQQ", lib, p)
            triple = lib[p + 24:p + 24 + tl]
            p += 24 + tl
            if b"gfx950" in triple and size:
                for k in _kernels(lib[at + off:at + off + size]):
                    out[k[".name"]] = k[".private_segment_fixed_size"]
        at = lib.find(MAGIC, p)
    assert len(out) > 60
    return out


@pytest.mark.parametrize("kernel", ["k_rk4_coef", "k_fine_place_tables", "k_rk4_pullback",
                                    "k_scatter"])
def test_no_scratch(scratch, kernel):
    found = {k: v for k, v in scratch.items() if f"{len(kernel)}{kernel}" in k}
    assert found
    assert not any(found.values()), found
