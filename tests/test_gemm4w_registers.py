"""The built 4-wave kernels keep every value in registers (csrc/gemm4w.h, csrc/swiglu224.h, csrc/swiglu4w.h).

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
            if "gemm4w_kernel" in name or "swiglu224_kernel" in name or "swiglu4w_kernel" in name:
                seen += 1
                assert int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", kernel).group(1)) == 0, name
                assert int(re.search(r"\.vgpr_spill_count:\s+(\d+)", kernel).group(1)) == 0, name
    assert seen >= 16   # 14 forms of the first, the other two


OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs llvm-objdump")
def test_no_fragment_of_the_8_wave_kernels_is_spilled(tmp_path):
    """grouped_gemm_kernel keeps LDS reads in flight in v[200:255] from one statement of its fp8 loop to the next. The 320-token forms
    spill other registers (28 and 48 accesses); a spilled fragment would be stored before it has arrived."""
    seen = 0
    for i, obj in enumerate(code_objects(_lib.LIB_PATH)):
        f = tmp_path / f"{i}.o"
        f.write_bytes(obj)
        text = subprocess.run([OBJDUMP, "-d", str(f)], capture_output=True, text=True, check=True).stdout
        kernel = ""
        for line in text.splitlines():
            head = re.match(r"[0-9a-f]+ <(\S+)>:", line)
            if head:
                kernel = head.group(1)
                seen += "grouped_gemm_kernel" in kernel
            elif "scratch_" in line and "grouped_gemm_kernel" in kernel:
                for lo, hi in re.findall(r"\bv\[?(\d+)(?::(\d+))?\]?", line.split("//")[0]):
                    assert int(hi or lo) < 200, (kernel, line)
    assert seen >= 10
