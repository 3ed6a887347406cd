"""The first requests of a block of the built 4-wave kernels (csrc/gemm4w.h, csrc/swiglu224.h).

A block waits for its first K step by the number of requests behind that step's, so nothing else may be requested between them: the row
indices in front, then two K steps of direct-to-LDS loads, the wait for all but half of them, and the barrier."""
import os
import re
import subprocess

import pytest

from comfyui_amd import _lib
from tests.test_gemm4w_registers import OBJDUMP, code_objects


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs llvm-objdump")
def test_requests_in_front_of_the_first_wait(tmp_path):
    seen = 0
    for i, obj in enumerate(code_objects(_lib.LIB_PATH)):
        f = tmp_path / f"{i}.o"
        f.write_bytes(obj)
        text = subprocess.run([OBJDUMP, "-d", str(f)], capture_output=True, text=True, check=True).stdout
        kernel, requests, checked = "", [], True
        for line in text.splitlines():
            head = re.match(r"[0-9a-f]+ <(\S+)>:", line)
            ins = line.split("//")[0].strip()
            if head:
                assert checked, kernel
                kernel, requests = head.group(1), []
                checked = not ("gemm4w_kernel" in kernel or "swiglu224_kernel" in kernel)
            elif not checked and re.match(r"(buffer|global|scratch|flat)_", ins):
                requests.append(ins.endswith(" lds"))
            elif not checked and requests and requests[-1] and ins.startswith("s_barrier"):
                half = 15 if "swiglu224" in kernel else 16
                assert previous == f"s_waitcnt vmcnt({half})", (kernel, previous)
                assert sum(requests) == 2 * half and all(requests[-2 * half:]), kernel
                checked, seen = True, seen + 1
            previous = ins
        assert checked, kernel
    assert seen >= 15
