"""No kernel of the library parks registers in scratch memory: what the compiler wrote beside each kernel in the built library.
(CPU only; reads the notes of this repository's own build.)"""
import os
import re
import struct
import subprocess

import pytest

from galois_amd import _abi

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    """The gfx950 code objects of every bundle in the library: a count, then per entry offset, size and a name."""
    at = blob.find(MAGIC)
    while at >= 0:
        n, p = struct.unpack_from("<Q", blob, at + len(MAGIC))[0], at + len(MAGIC) + 8
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", blob, p)
            name = blob[p + 24:p + 24 + length]
            p += 24 + length
            if b"gfx950" in name:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, at + 1)


def _kernels(tmp_path):
    """(name, its entry in the notes) of every kernel of the library."""
    with open(_abi.LIB_PATH, "rb") as f:
        blob = f.read()
    for i, code in enumerate(_code_objects(blob)):
        path = tmp_path / ("%d.co" % i)
        path.write_bytes(code)
        notes = subprocess.check_output([READELF, "--notes", str(path)], text=True)
        for kernel in re.split(r"\n  - (?=\.)", notes)[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel)
            if name and ".vgpr_count:" in kernel:
                yield name.group(1), kernel


def _field(kernel, name):
    return int(re.search(r"\.%s:\s+(\d+)" % name, kernel).group(1))


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_no_kernel_spills_registers(tmp_path):
    kernels = list(_kernels(tmp_path))
    assert len(kernels) >= 200, "the library's kernels were not found"
    spilled = {name: _field(k, "vgpr_spill_count") for name, k in kernels if _field(k, "vgpr_spill_count")}
    assert not spilled, spilled


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_few_rows_tiles_of_two_by_four_keep_three_waves_a_simd(tmp_path):
    """However the weights arrive: 168 registers are what a SIMD's 512 have for each of three waves (in eights)."""
    regs = {name: _field(k, "vgpr_count") for name, k in _kernels(tmp_path) if "gemm_q4_0_skinnyILi2ELi4E" in name}
    assert len(regs) >= 6, regs
    assert max(regs.values()) <= 168, regs
