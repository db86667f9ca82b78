"""What the compiler made of the built library's kernels, from their metadata: none keeps
registers in scratch memory. (A spill in a GEMM's epilogue cost 5 us a tile before it was
seen: every result was right.)"""

import os
import struct

import pytest

from bux_amd import _lib

msgpack = pytest.importorskip("msgpack")


def _kernels(image: bytes):
    """The kernels of each gfx code object in a library's image: the AMDGPU metadata note
    (type 32, MessagePack) of every ELF embedded in it."""
    at = image.find(b"\x7fELF", 1)  # the library itself is the first
    while at >= 0:
        shoff, = struct.unpack_from("<Q", image, at + 0x28)
        size, count = struct.unpack_from("<HH", image, at + 0x3A)
        for i in range(count):
            kind, = struct.unpack_from("<I", image, at + shoff + i * size + 4)
            where, length = struct.unpack_from("<QQ", image, at + shoff + i * size + 24)
            if kind != 7:  # SHT_NOTE
                continue
            note = image[at + where:at + where + length]
            name_size, desc_size, note_type = struct.unpack_from("<III", note)
            start = 12 + -(-name_size // 4) * 4
            if note_type == 32 and note[12:18] == b"AMDGPU":
                yield from msgpack.unpackb(note[start:start + desc_size])["amdhsa.kernels"]
        at = image.find(b"\x7fELF", at + 1)


def test_no_kernel_spills():
    if not os.path.exists(_lib.PATH):
        pytest.fail(f"{_lib.PATH} is not built: run python -m bux_amd.build")
    with open(_lib.PATH, "rb") as f:
        kernels = list(_kernels(f.read()))
    assert len(kernels) > 60
    spilled = {k[".name"]: k[".private_segment_fixed_size"] for k in kernels
               if k[".private_segment_fixed_size"]}
    assert not spilled
