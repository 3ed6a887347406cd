"""The 192-token tile of the fp8 gate/up contraction of a dense feed-forward (csrc/gemm.hip, short_tile_pays): the intermediate it
leaves is that of the other kernels byte for byte, for every form of its epilogue's cast. (Widths are multiples of 256, so K steps come in pairs.)"""
import ctypes

import pytest
import torch

from comfyui_amd import _lib, synth

BF16, FP8 = torch.bfloat16, torch.float8_e4m3fn
H = 6912
SHORT = "grouped_gemm_kernel<FP8_SWIGLU, 3>"


def kernel(rows, D, scale_in2):
    return _lib.lib.hdmoe_gate_up_kernel_name(_lib.W_E4M3FN, rows, 0, D, 256, H, scale_in2).decode()


@pytest.mark.gpu
@pytest.mark.parametrize("D", [256, 768, 2560])            # 2, 6 and 20 K steps
@pytest.mark.parametrize("scale_in2", [None, 1.0, 0.37])   # clamped, cast as it is, scaled
@pytest.mark.parametrize("rows", [300, 577, 768])          # remainders of a tile: 108 rows, 1 row, none
def test_intermediate_is_that_of_the_other_kernels(dev, D, scale_in2, rows):
    from comfyui_amd import functional as HF
    assert kernel(rows, D, scale_in2 is not None) == SHORT and kernel(3000, D, scale_in2 is not None) != SHORT
    g = torch.Generator(device=dev).manual_seed(D + rows)
    ws, scales = [], {}
    for name, shape in (("1", (H, D)), ("2", (D, H)), ("3", (H, D))):
        w, scales["scale_w" + name] = synth.quantize_per_tensor(torch.randn(shape, generator=g, device=dev) * (2.0 / D ** 0.5))
        ws.append(w)
    one = torch.ones((), device=dev)
    if scale_in2 is not None:
        scales.update(scale_in1=one, scale_in3=one, scale_in2=torch.tensor(scale_in2, device=dev))
    fw = HF.make_ffn_weights(*ws, scales)
    x = torch.randn((3000, D), generator=g, device=dev).to(BF16) * 12

    def h(n):
        work = torch.empty(_lib.lib.hdmoe_ffn_workspace_bytes(n, D, H, _lib.W_E4M3FN), dtype=torch.uint8, device=dev)
        out = torch.empty((n, D), dtype=BF16, device=dev)
        _lib.check(_lib.lib.hdmoe_ffn_swiglu(_lib.W_E4M3FN, x.data_ptr(), n, D, H, ctypes.byref(fw), out.data_ptr(), work.data_ptr(),
                                             work.numel(), torch.cuda.current_stream().cuda_stream))
        at = (n * D + 255) // 256 * 256
        return work[at:at + n * H].view(n, H)
    full, part = h(3000), h(rows)
    assert torch.equal(part, full[:rows])
    if scale_in2 is None:
        assert bool((full & 0x7F == 0x7E).any())           # some values are at the limit
