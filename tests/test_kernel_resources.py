"""Registers of the built library's persistent kernels: with at most 64 VGPRs
and 80 SGPRs a SIMD holds eight waves, so every workgroup of a full launch (2048
of 256 lanes, eight per CU) is resident at once."""
import os
import re
import struct

import msgpack
import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "taichi-ferrofluid_amd", "libmgpcg.so")


def _kernels():
    """{symbol: metadata} of the gfx950 code objects in the library: each is an
    ELF image whose AMDGPU note (type 32) holds the kernels' metadata."""
    if not os.path.exists(LIB):
        import __graft_entry__

        __graft_entry__.build()
    with open(LIB, "rb") as fh:
        data = fh.read()
    out = {}
    for m in re.finditer(rb"AMDGPU\0\0", data):
        namesz, descsz, kind = struct.unpack_from("<III", data, m.start() - 12)
        if namesz != 7 or kind != 32:
            continue
        meta = msgpack.unpackb(data[m.end():m.end() + descsz])
        out.update({k[".name"]: k for k in meta["amdhsa.kernels"]})
    return out


@pytest.mark.parametrize("kernel", ["k_stage", "k_residual", "k_smooth0_dot", "k_cg_xr",
                                    "k_cg_ap_only", "k_cg_update_p", "k_true_residual"])
def test_fp32_persistent_kernels_fill_the_simds(kernel):
    ks = {n: k for n, k in _kernels().items() if f"{len(kernel)}{kernel}If" in n}
    assert ks
    for n, k in ks.items():
        assert k[".vgpr_count"] <= 64 and k[".sgpr_count"] <= 80, (n, k[".vgpr_count"],
                                                                   k[".sgpr_count"])
