"""Registers of the built sweep kernels, from the code objects' own metadata in
libmlau_hip.so: the sweeps of whole grids fit two wavefronts to a SIMD (256 VGPRs and
AGPRs a lane); with one, the SIMD idles while the wavefront waits on its loads."""
import os
import re
import struct

import pytest

msgpack = pytest.importorskip("msgpack")
LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mlau_amd", "_lib", "libmlau_hip.so")


def kernels():
    """(name, metadata) of every kernel in the library's embedded AMDGPU code objects."""
    data = open(LIB, "rb").read()
    for m in re.finditer(rb"\x7fELF\x02\x01", data):
        o = m.start()
        if struct.unpack_from("<H", data, o + 18)[0] != 224:  # EM_AMDGPU
            continue
        shoff, = struct.unpack_from("<Q", data, o + 40)
        size, num = struct.unpack_from("<HH", data, o + 58)
        for k in range(num):
            h = o + shoff + k * size
            kind, = struct.unpack_from("<I", data, h + 4)
            off, length = struct.unpack_from("<QQ", data, h + 24)
            if kind != 7:  # SHT_NOTE
                continue
            at, end = o + off, o + off + length
            while at + 12 <= end:
                n, d, t = struct.unpack_from("<III", data, at)
                desc = at + 12 + (n + 3) // 4 * 4
                if t == 32 and data[at + 12:at + 18] == b"AMDGPU":  # NT_AMDGPU_METADATA
                    for e in msgpack.unpackb(data[desc:desc + d], strict_map_key=False)["amdhsa.kernels"]:
                        yield e[".name"], e
                at = desc + (d + 3) // 4 * 4


def test_sweeps_fit_two_wavefronts():
    # the marches' choice (last template argument 1) is for grids too small to need them; a
    # kernel over the limit needs its form held to it, which large grids take
    regs = {}
    for name, e in kernels():
        m = re.search(r"k_(sweeps2d|sweeps2d_inl|sweeps3d)(_two)?(ILi.*ELb0EE)", name)
        if m:
            regs[m.group(1), m.group(3), m.group(2)] = e[".vgpr_count"] + e.get(".agpr_count", 0)
    free = {k: v for k, v in regs.items() if not k[2]}
    held = {k: v for k, v in regs.items() if k[2]}
    assert len(free) == 4 * 4 * 3 * (1 + 2 + 1), len(free)
    assert all(v <= 256 for v in held.values()), held
    assert not [k for k, v in free.items() if v > 256 and (k[0], k[1], "_two") not in held]
