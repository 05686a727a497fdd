"""Registers of the kernels in librsgpu.so, read from the metadata of its
gfx950 code objects: what a kernel's occupancy rests on and no result shows.
No GPU is needed."""
import os
import re
import struct

import pytest

from rockseis_amd import _lib as R

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _notes(elf):
    """Payloads of the SHT_NOTE sections of a 64-bit little-endian ELF."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    size, num = struct.unpack_from("<HH", elf, 58)
    for i in range(num):
        kind, = struct.unpack_from("<I", elf, shoff + i * size + 4)
        off, n = struct.unpack_from("<QQ", elf, shoff + i * size + 24)
        if kind == 7:
            namesz, descsz, _ = struct.unpack_from("<III", elf, off)
            at = off + 12 + (namesz + 3) // 4 * 4
            yield elf[at:at + descsz]


@pytest.fixture(scope="module")
def kernels():
    msgpack = pytest.importorskip("msgpack")
    R.lib()
    lib = open(os.path.join(os.path.dirname(R.__file__), "librsgpu.so"), "rb").read()
    out = {}
    for m in re.finditer(re.escape(MAGIC), lib):
        n, = struct.unpack_from("<Q", lib, m.end())
        at = m.end() + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", lib, at)
            triple = lib[at + 24:at + 24 + idlen]
            at += 24 + idlen
            if b"gfx950" in triple and size:
                for note in _notes(lib[m.start() + off:m.start() + off + size]):
                    for k in msgpack.unpackb(note, strict_map_key=False).get("amdhsa.kernels", []):
                        out[k[".name"]] = k
    assert len(out) > 300, len(out)
    return out


def test_adjoint_velocity_2d_keeps_its_waves(kernels):
    """Elastic 2D adjoint-state velocity, two rows a thread: the strips' loads
    of boundary tiles must not take registers from interior tiles.  Six waves a
    SIMD need at most 80 VGPRs of the 512."""
    for kind in ("e2d_velocity_kernel", "e2d_velocity_ragged_kernel"):
        for order in range(1, 9):
            name = f"{kind}ILi{order}ELi2ELb1EE"
            found = [k for n, k in kernels.items() if name in n]
            assert len(found) == 1, name
            assert found[0][".vgpr_count"] <= 80, (name, found[0][".vgpr_count"])
