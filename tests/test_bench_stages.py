"""bench.py names the stages that run: up to 512 slots of an fp8 layer the dispatch is part of the gate/up GEMM."""
import pytest

import bench
from comfyui_amd import synth


@pytest.mark.parametrize("tokens,fp8,inside", [(16, True, True), (64, True, True), (256, True, True), (257, True, False), (1024, True, False),
                                               (64, False, False), (256, False, False)])
def test_dispatch_inside(tokens, fp8, inside):
    kernel = bench.gate_up_kernel_name(tokens, synth.DIM, synth.H_ROUTED, synth.H_SHARED, synth.NUM_EXPERTS, fp8=fp8)
    assert kernel and bench.dispatch_inside(kernel, tokens) is inside
