"""The down projection of a layer whose experts and shared expert have different K, on tiles of several heights dealt out by their length
(csrc/gemm4w.h, g4_two_lengths; up to 448 tiles of the long kind): rows come out as they do among more tokens, where whole tiles are dealt out
in eighths, and for fp8 as on the 8-wave kernels."""
import pytest
import torch

from comfyui_amd import _lib, ops, synth
from comfyui_amd import functional as HF
from comfyui_amd.hidream import FeedForwardSwiGLU, MOEFeedForwardSwiGLU
from tests.helpers import saved_forms, set_form

pytestmark = pytest.mark.gpu
BF16, FP8 = torch.bfloat16, torch.float8_e4m3fn
MOST = 6400   # 520 tiles of the longer kind


@pytest.fixture
def forms():
    yield from saved_forms()


def layer(dev, kind, experts=4, longer_shared=False):
    g = torch.Generator(device=dev).manual_seed(7)
    o = {"fp8": lambda: ops.scaled_fp8_ops(fp8_matrix_mult=True, scale_input=True, override_dtype=FP8),
         "upcast": lambda: ops.scaled_fp8_ops(fp8_matrix_mult=False, scale_input=False, override_dtype=FP8), "bf16": lambda: ops.disable_weight_init}[kind]()
    m = MOEFeedForwardSwiGLU(synth.DIM, 4 * synth.DIM, experts, 2, dtype=BF16, device=dev, operations=o).eval()
    if longer_shared:   # 3584 and 6912 the other way round
        m.experts, m.shared_experts = torch.nn.ModuleList(
            [FeedForwardSwiGLU(synth.DIM, 2 * synth.DIM, dtype=BF16, device=dev, operations=o) for _ in range(experts)]), m.experts[0]
    for f in [*m.experts, m.shared_experts]:
        for lin in (f.w1, f.w2, f.w3):
            w = torch.randn(tuple(lin.weight.shape), generator=g, device=dev) * 0.02
            if kind == "bf16":
                lin.weight = torch.nn.Parameter(w.to(BF16), requires_grad=False)
                continue
            w8, s = synth.quantize_per_tensor(w)
            lin.weight, lin.scale_weight = torch.nn.Parameter(w8, requires_grad=False), torch.nn.Parameter(s, requires_grad=False)
            if kind == "fp8":
                lin.scale_input = torch.nn.Parameter(torch.ones((), device=dev), requires_grad=False)
    gate = torch.randn(tuple(m.gate.weight.shape), generator=g, device=dev) * 0.02
    gate[0, :64] += 0.02   # uneven segments
    m.gate.weight = torch.nn.Parameter(gate.to(BF16), requires_grad=False)
    return m, torch.randn((1, MOST, synth.DIM), generator=g, device=dev).add_(0.2).to(BF16)


@pytest.mark.parametrize("kind", ["fp8", "upcast", "bf16"])
def test_rows_are_those_of_a_larger_call(dev, forms, kind):
    m, x = layer(dev, kind)
    m.batch_invariant = True   # no sums cut along K by the segments' sizes
    with torch.no_grad():
        full = m(x)
        assert bool(torch.isfinite(full.float()).all()) and float(full.float().std()) > 0
        for tokens in (1100, 1801, 2049, 2100, 2300, 2560, 2600, 3000, 4096, 4500, 5400):
            if kind == "fp8":
                assert _lib.lib.hdmoe_plain_kernel_name(2 * tokens, 4, synth.H_ROUTED, tokens, synth.H_SHARED, synth.DIM, 1, 0) == b"gemm4w_kernel<F8, PLAIN>"
            assert torch.equal(m(x[:, :tokens]), full[:, :tokens]), tokens
        if kind == "fp8":
            set_form("HDMOE_SWIGLU4W", "0")
            assert torch.equal(m(x[:, :3000]), full[:, :3000])


@pytest.mark.parametrize("kind", ["fp8", "upcast", "bf16"])
@pytest.mark.parametrize("experts,longer_shared", [(8, False), (2, False), (4, True), (8, True)])
def test_other_numbers_of_experts_and_a_longer_shared_one(dev, forms, kind, experts, longer_shared):
    """More tokens than 448 tiles of the longer kind take: 12000, with a longer shared expert (10 tiles along the features)."""
    m, x = layer(dev, kind, experts, longer_shared)
    m.batch_invariant = True
    H, Hs = m.experts[0].w1.weight.shape[0], m.shared_experts.w1.weight.shape[0]
    assert (H, Hs) == ((3584, 6912) if longer_shared else (6912, 3584))
    x = torch.cat([x, x.flip(1)], 1)[:, :12000 if longer_shared else MOST]
    code = {"fp8": _lib.W_E4M3FN, "upcast": _lib.W_E4M3FN_UPCAST, "bf16": _lib.W_BF16}[kind]
    with torch.no_grad():
        full = m(x)
        assert bool(torch.isfinite(full.float()).all()) and float(full.float().std()) > 0
        for tokens in (2300, 2900, 4096, 5000):
            lay = HF.layer_layout(tokens, synth.DIM, H, Hs, experts, code)
            assert lay.flags == lay.partials   # not cut along K
            y = m(x[:, :tokens])
            if kind == "fp8":
                assert _lib.lib.hdmoe_plain_kernel_name(2 * tokens, experts, H, tokens, Hs, synth.DIM, 1, 0) == b"gemm4w_kernel<F8, PLAIN>"
            assert torch.equal(y, full[:, :tokens]), tokens
