"""Registers and scratch of kernels whose speed hangs on the number of waves per SIMD, read from the metadata of the code
objects in the built library (a compiler's choice that no value test sees)."""
import os
import struct

import pytest

msgpack = pytest.importorskip("msgpack")

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "corefl-cpc_amd", "libcorefl_amd.so")
EM_AMDGPU, NT_AMDGPU_METADATA, PT_NOTE = 224, 32, 4


def kernels():
    data = open(LIB, "rb").read()
    out, at = {}, data.find(b"\x7fELF")
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == EM_AMDGPU:
            phoff, = struct.unpack_from("<Q", data, at + 32)
            phentsize, phnum = struct.unpack_from("<HH", data, at + 54)
            for h in range(phnum):
                kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", data, at + phoff + h * phentsize)
                if kind != PT_NOTE:
                    continue
                namesz, descsz, ntype = struct.unpack_from("<III", data, at + off)
                if ntype == NT_AMDGPU_METADATA:
                    desc = at + off + 12 + (namesz + 3) // 4 * 4
                    for k in msgpack.unpackb(data[desc:desc + descsz])["amdhsa.kernels"]:
                        out[k[".name"]] = k
        at = data.find(b"\x7fELF", at + 1)
    return out


# (kernel, arguments of the template as mangled, waves per SIMD of its 512 registers a lane, scratch bytes a lane)
@pytest.mark.parametrize("name,args,waves,scratch", [("k_mix_viscous_node", "ILi8EE", 2, 0)])
def test_waves_per_simd(name, args, waves, scratch):
    if not os.path.exists(LIB):
        pytest.skip("the library is not built")
    found = [k for n, k in kernels().items() if "%d%s%s" % (len(name), name, args) in n]
    assert len(found) == 1, name
    k = found[0]
    registers = (k[".vgpr_count"] + 7) // 8 * 8  # vector and accumulation registers together, in granules of 8
    assert 512 // registers >= waves, (name, registers)
    assert k[".private_segment_fixed_size"] <= scratch, name
