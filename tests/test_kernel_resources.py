"""Registers of the kernels whose speed is their occupancy, from the metadata of the
built library: a SIMD's 512 vector registers per lane hold 512 / n waves of a kernel
with n of them."""
import os
import struct

import msgpack
import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "mctomo_amd", "libmctomo_hip.so")


def kernels():
    """name -> (vector registers, spilled ones) from the code objects' AMDGPU notes"""
    b = open(LIB, "rb").read()
    out, i = {}, b.find(b"AMDGPU\0\0")
    while i >= 0:
        namesz, descsz, kind = struct.unpack("<III", b[i - 12:i])
        if namesz == 7 and kind == 32:
            note = msgpack.unpackb(b[i + 8:i + 8 + descsz], strict_map_key=False)
            for k in note["amdhsa.kernels"]:
                out[k[".name"]] = (k[".vgpr_count"], k[".vgpr_spill_count"])
        i = b.find(b"AMDGPU\0\0", i + 8)
    return out


@pytest.mark.skipif(not os.path.exists(LIB), reason="library not built")
@pytest.mark.parametrize("kernel,count,waves,spilled", [
    ("12k_dispersion12mct_dsp_args", 1, 2, 32), ("17k_dispersion_lane", 1, 2, 48), ("19k_dispersion_layers", 1, 2, 24),
    ("15k_dispersion_sm", 4, 3, 24), ("12k_fm2d_stripILi0E", 1, 3, 0), ("12k_fm2d_stripILi1E", 1, 2, 0)])
def test_waves_per_simd(kernel, count, waves, spilled):
    found = {k: v for k, v in kernels().items() if kernel in k}
    assert len(found) == count
    for name, (regs, spills) in found.items():
        assert 512 // ((regs + 7) // 8 * 8) >= waves, (name, regs)
        assert spills <= spilled, (name, spills)
