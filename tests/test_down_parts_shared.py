"""The parts of the shared expert's tiles in the down projection of a few tokens (csrc/gemm.hip, hdmoe_down_parts, which the library does not declare)."""
import ctypes

import pytest

from comfyui_amd import _lib

MOST = 12


class Plan(ctypes.Structure):   # HdmoeSplitPlan, csrc/common.h
    _fields_ = [("n", ctypes.c_int), ("pd", ctypes.c_int * MOST), ("ps", ctypes.c_int * MOST), ("bm", ctypes.c_int), ("bm_else", ctypes.c_int),
                ("max_tiles", ctypes.c_int), ("fixed_pd", ctypes.c_int), ("fixed_ps", ctypes.c_int)]


@pytest.mark.parametrize("code", [_lib.W_BF16, _lib.W_E4M3FN, _lib.W_E4M3FN_UPCAST])
@pytest.mark.parametrize("experts,tokens,want", [(4, 64, (5, 3)), (4, 128, (5, 3)), (4, 130, (3, 2)), (4, 256, (3, 2)), (8, 128, (2, 2)), (8, 200, (2, 2)),
                                                 (8, 256, (2, 2)), (10, 130, (2, 2))])
def test_parts(code, experts, tokens, want):
    """Fewer parts of the shared expert's tiles than make them as long as the experts' only where those gain a part."""
    plan = Plan()
    parts = _lib.lib._Z16hdmoe_down_partsiiiiiiiP14HdmoeSplitPlanb(2 * tokens, experts, tokens, 2560, 6912, 3584, code, ctypes.byref(plan), False)
    assert (plan.n, plan.pd[0], plan.ps[0]) == (1, *want) and parts == want[0]
