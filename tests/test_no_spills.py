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


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_no_kernel_spills_registers(tmp_path):
    with open(_abi.LIB_PATH, "rb") as f:
        blob = f.read()
    seen, spilled = 0, {}
    for i, code in enumerate(_code_objects(blob)):
        path = tmp_path / ("%d.co" % i)
        path.write_bytes(code)
        notes = subprocess.check_output([READELF, "--notes", str(path)], text=True)
        for kernel in re.split(r"\n  - (?=\.)", notes)[1:]:
            name, count = re.search(r"\.name:\s+(\S+)", kernel), re.search(r"\.vgpr_spill_count:\s+(\d+)", kernel)
            if name and count:
                seen += 1
                if int(count.group(1)):
                    spilled[name.group(1)] = int(count.group(1))
    assert seen >= 200, "the library's kernels were not found"
    assert not spilled, spilled
