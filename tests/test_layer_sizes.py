"""Sizes that the layer does not take (csrc/gemm.hip, hdmoe_down_parts): the layout and the workspace answer, whatever the widths."""
import subprocess
import sys

import pytest

from comfyui_amd import _lib

CODES = [_lib.W_BF16, _lib.W_E4M3FN, _lib.W_E4M3FN_UPCAST]


@pytest.mark.parametrize("code", CODES)
@pytest.mark.parametrize("h,hs", [(32, 3584), (6912, 32), (32, 32), (1, 1), (1, 3584), (6912, 0), (32, 0)])
def test_a_width_under_one_k_step(code, h, hs):
    """In a process of its own: an integer division by zero would end this one."""
    run = ("from comfyui_amd import _lib\n"
           "from comfyui_amd import functional as HF\n"
           "for tokens in (0, 1, 64, 128, 200, 256, 300, 600, 1500):\n"
           "    for experts in (1, 2, 4, 16):\n"
           f"        lay = HF.layer_layout(tokens, 2560, {h}, {hs}, experts, {code})\n"
           f"        assert lay.total == _lib.lib.hdmoe_layer_workspace_bytes(tokens, 2560, {h}, {hs}, experts, {code}) > 0\n"
           f"    _lib.lib.hdmoe_ffn_workspace_bytes(tokens, 2560, {h}, {code})\n")
    assert subprocess.run([sys.executable, "-c", run]).returncode == 0
