"""Register use of built kernels, from the metadata of libp4g.so's gfx950 code
object (no GPU needed)."""
import struct

import msgpack
import pytest

from p4pdes_amd import capi


def _kernels():
    """{mangled name: metadata} of every kernel in libp4g.so."""
    blob = open(capi.LIBP4G, "rb").read()
    out, at = {}, blob.find(b"\x7fELF", 4)
    while at >= 0:
        if struct.unpack_from("<H", blob, at + 18)[0] == 224:          # EM_AMDGPU
            phoff, = struct.unpack_from("<Q", blob, at + 32)
            phsize, phnum = struct.unpack_from("<HH", blob, at + 54)
            for h in range(phnum):
                kind, = struct.unpack_from("<I", blob, at + phoff + h * phsize)
                off, = struct.unpack_from("<Q", blob, at + phoff + h * phsize + 8)
                if kind != 4:                                          # PT_NOTE
                    continue
                nsize, dsize, _ = struct.unpack_from("<III", blob, at + off)
                d = at + off + 12 + (nsize + 3) // 4 * 4
                for k in msgpack.unpackb(blob[d:d + dsize])["amdhsa.kernels"]:
                    out[k[".name"]] = k
        at = blob.find(b"\x7fELF", at + 4)
    return out


@pytest.fixture(scope="module")
def kernels():
    return _kernels()


# FP64 passes over cell coefficients whose output loads arrays ahead: held to
# four waves with whole cell layers in registers they spilled 7-39 of them,
# and a V(2,2) solve took up to 11 % longer
@pytest.mark.parametrize("out", ["8OutResidIdLi0EE", "8OutResidIdLi1EE", "11OutResidCvtIdfE", "13OutResidNormsIdE",
                                 "7OutChebIdLb0ELi0EE", "7OutChebIdLb0ELi2EE", "7OutChebIdLb1ELi0EE",
                                 "7OutChebIdLb1ELi2EE"])
def test_cell_passes_with_operands_ahead_do_not_spill(kernels, out):
    mine = [k for n, k in kernels.items() if "k_stencilIdLi3ENS_5OpVarIdE" in n and out in n and "OutScaleU" not in n]
    assert mine
    for k in mine:
        assert k[".vgpr_spill_count"] == 0, (k[".name"], k[".vgpr_spill_count"])
