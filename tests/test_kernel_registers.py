"""Registers of the built kernels: those whose speed rests on a number of waves
per SIMD stay within that share of its 512 vector registers (with 258 of them
k_shade_ad had one wave, with 256 two: the full gradient of 3 x 100k rays in the
shoebox took 24.6 ms for 19.5).  Read from the code objects' own metadata."""
import os
import struct

import pytest

msgpack = pytest.importorskip("msgpack")
LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ear_amd", "libear_hip.so")


def _kernels():
    """{mangled name: registers a wave takes} of every device ELF in the library."""
    data = open(LIB, "rb").read()
    out, at = {}, data.find(b"\x7fELF", 1)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == 224:  # EM_AMDGPU
            shoff, = struct.unpack_from("<Q", data, at + 40)
            shsize, shnum = struct.unpack_from("<HH", data, at + 58)
            for i in range(shnum):
                h = at + shoff + i * shsize
                if struct.unpack_from("<I", data, h + 4)[0] != 7:  # SHT_NOTE
                    continue
                off, size = struct.unpack_from("<QQ", data, h + 24)
                p = at + off
                while p < at + off + size:
                    nn, nd, kind = struct.unpack_from("<III", data, p)
                    desc = p + 12 + (nn + 3) // 4 * 4
                    if kind == 32:  # the kernels' metadata
                        for k in msgpack.unpackb(data[desc:desc + nd])["amdhsa.kernels"]:
                            out[k[".name"]] = k[".vgpr_count"]
                    p = desc + (nd + 3) // 4 * 4
        at = data.find(b"\x7fELF", at + 4)
    return out


@pytest.mark.parametrize("kernel,waves", [("10k_shade_ad", 3), ("11k_adj_paths", 3), ("7k_shade", 6),
                                          ("6k_tailILi256ELi16", 4), ("10k_shadow_fILi256ELi16", 6)])
def test_waves_per_simd(kernel, waves):
    if not os.path.exists(LIB):
        pytest.skip("the library is not built")
    regs = {n: r for n, r in _kernels().items() if kernel in n}
    assert regs
    # (given out in eights)
    assert not {n: r for n, r in regs.items() if (r + 7) // 8 * 8 * waves > 512}
