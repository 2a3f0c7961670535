"""The matrix-free apply reads its LDS tables by absolute address, from 0 on: no
apply kernel may have static LDS, which would come before the dynamic one.  Read
from the kernels' metadata in the built library."""
import os
import re
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qrusty_amd", "libqrhip.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    at = blob.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", blob, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(count if count < 16 else 0):
            off, size, n = struct.unpack_from("<QQQ", blob, p)
            if b"gfx950" in blob[p + 24:p + 24 + n] and size:
                yield blob[at + off:at + off + size]
            p += 24 + n
        at = blob.find(MAGIC, at + 1)


def test_apply_kernels_have_no_static_lds(tmp_path):
    if not os.path.exists(LIB) or not os.path.exists(READELF):
        pytest.skip("no built library or no llvm-readelf")
    lds = {}
    with open(LIB, "rb") as f:
        blob = f.read()
    for code in _code_objects(blob):
        path = tmp_path / "code.elf"
        path.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for kernel in notes.split("- .agpr_count")[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel)[1]
            lds[name] = int(re.search(r"\.group_segment_fixed_size:\s+(\d+)", kernel)[1])
    apply = {k: v for k, v in lds.items() if "k_apply_" in k}
    assert len(apply) > 50 and not any(apply.values()), apply


def test_apply_kernels_keep_four_waves_per_simd(tmp_path):
    """Kernels over tiles of 2^11 rows: at most 128 VGPRs, nothing spilled."""
    if not os.path.exists(LIB) or not os.path.exists(READELF):
        pytest.skip("no built library or no llvm-readelf")
    regs = {}
    with open(LIB, "rb") as f:
        blob = f.read()
    for code in _code_objects(blob):
        path = tmp_path / "code.elf"
        path.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for kernel in notes.split("- .agpr_count")[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel)[1]
            if "k_apply_" in name and "Li11E" in name:
                regs[name] = tuple(int(re.search(rf"\.{f}:\s+(\d+)", kernel)[1])
                                   for f in ("vgpr_count", "vgpr_spill_count"))
    assert len(regs) > 12 and all(v <= 128 and spilled == 0 for v, spilled in regs.values()), regs
