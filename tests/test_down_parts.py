"""The cut along K of a dense fp8 down projection (csrc/gemm.hip, hdmoe_down_parts), as the working memory shows it."""
import pytest

from comfyui_amd import _lib

D, H = 2560, 6912


def parts(rows, dim=D, hidden=H):
    align = lambda n: -(-n // 256) * 256
    room = _lib.lib.hdmoe_ffn_workspace_bytes(rows, dim, hidden, _lib.W_E4M3FN) - align(rows * dim) - align(rows * hidden)
    assert room % (rows * dim * 4) < 256 or room % (rows * dim * 4) == 0
    return room // (rows * dim * 4) or 1


@pytest.mark.parametrize("rows,want", [(300, 6), (512, 4), (768, 3), (1024, 3), (1280, 2), (1536, 2), (1600, 2), (1700, 2), (1900, 2), (2048, 2), (2560, 1), (4096, 1)])
def test_parts(rows, want):
    """Whole tiles take their K steps one after the other while cold weights arrive: two parts up to 2048 rows."""
    assert parts(rows) == want


def test_few_steps_are_not_cut():
    assert parts(1700, 512, 1280) == 1   # 5 pairs of K steps: no part has three
