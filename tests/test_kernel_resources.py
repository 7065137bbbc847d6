"""Register use and instructions of built kernels, from the metadata and the
disassembly of libp4g.so's gfx950 code object (no GPU needed)."""
import os
import re
import struct
import subprocess

import msgpack
import pytest

from p4pdes_amd import capi


OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")


def _code_objects():
    """The AMDGPU ELF images in libp4g.so."""
    blob = open(capi.LIBP4G, "rb").read()
    at = blob.find(b"\x7fELF", 4)
    while at >= 0:
        if struct.unpack_from("<H", blob, at + 18)[0] == 224:          # EM_AMDGPU
            shoff, = struct.unpack_from("<Q", blob, at + 40)
            shsize, shnum = struct.unpack_from("<HH", blob, at + 58)
            yield blob[at:at + shoff + shsize * shnum]
        at = blob.find(b"\x7fELF", at + 4)


def _kernels():
    """{mangled name: metadata} of every kernel in libp4g.so."""
    out = {}
    for elf in _code_objects():
        phoff, = struct.unpack_from("<Q", elf, 32)
        phsize, phnum = struct.unpack_from("<HH", elf, 54)
        for h in range(phnum):
            kind, = struct.unpack_from("<I", elf, phoff + h * phsize)
            off, = struct.unpack_from("<Q", elf, phoff + h * phsize + 8)
            if kind != 4:                                              # PT_NOTE
                continue
            nsize, dsize, _ = struct.unpack_from("<III", elf, off)
            d = off + 12 + (nsize + 3) // 4 * 4
            for k in msgpack.unpackb(elf[d:d + dsize])["amdhsa.kernels"]:
                out[k[".name"]] = k
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


def _vgprs(operand):
    m = re.match(r"v\[(\d+):(\d+)\]$|v(\d+)$", operand)
    if not m:
        return set()
    return {int(m[3])} if m[3] else set(range(int(m[1]), int(m[2]) + 1))


# A store of more than 8 bytes reads its data late: the instruction right
# behind it must not write one of its data registers.  The compiler leaves that
# wait state out where a buffer store's offset is in a scalar register, and
# the sweeps' sums were then at times stored with the next instruction's result
# in them.
def test_wide_stores_are_not_followed_by_a_write_of_their_data(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    stores = 0
    for i, elf in enumerate(_code_objects()):
        path = tmp_path / ("co%d" % i)
        path.write_bytes(elf)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], check=True, capture_output=True,
                              text=True).stdout
        where, data = "", set()
        for line in text.splitlines():
            m = re.match(r"[0-9a-f]+ <(\w+)>:", line)
            if m:
                where, data = m[1], set()
                continue
            ins = line.split("//")[0].strip()
            m = re.match(r"(\w+)\s*(.*)", ins)
            if not m:
                continue
            ops = [o.strip() for o in m[2].split(",")]
            if m[1].startswith("v_") and _vgprs(ops[0]) & data:
                pytest.fail("%s: %s overwrites the data of the store before it" % (where, ins))
            wide = re.match(r"(buffer|global|flat)_store_dwordx[34]$", m[1])
            data = _vgprs(ops[0] if m[1].startswith("buffer") else ops[1]) if wide else set()
            stores += bool(wide)
    assert stores > 100
