"""The built 4-wave kernels keep every value in registers (csrc/gemm4w.h).

Their statements use fixed registers that are free to the compiler in between. A spilled register tuple that is reloaded there
and used in part is waited for in part: the rest arrives while a statement has the registers in use. So nothing may be
spilled to memory, which the code object's metadata tells."""
import os
import re
import struct
import subprocess

import pytest

from comfyui_amd import _lib

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def code_objects(path):
    """The AMDGPU ELF files inside a shared library."""
    blob = open(path, "rb").read()
    at = blob.find(b"\x7fELF", 1)
    while at >= 0:
        if struct.unpack_from("<H", blob, at + 18)[0] == 224:   # EM_AMDGPU
            yield blob[at:]
        at = blob.find(b"\x7fELF", at + 4)


@pytest.mark.skipif(not os.path.exists(READELF), reason="needs llvm-readelf")
def test_no_kernel_of_the_4_wave_gemm_spills(tmp_path):
    seen = 0
    for i, obj in enumerate(code_objects(_lib.LIB_PATH)):
        f = tmp_path / f"{i}.o"
        f.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True, check=True).stdout
        for kernel in notes.split("- .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel).group(1)
            if "gemm4w_kernel" in name:
                seen += 1
                assert int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", kernel).group(1)) == 0, name
                assert int(re.search(r"\.vgpr_spill_count:\s+(\d+)", kernel).group(1)) == 0, name
    assert seen >= 10
