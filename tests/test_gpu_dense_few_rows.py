"""A dense feed-forward in bf16 on up to 128 rows (csrc/gemm.hip, swiglu_on_g4): its gate/up contraction, cut along K where the working memory has
room for the parts, against 64-bit sums with the contract's roundings."""
import ctypes

import pytest
import torch

from comfyui_amd import _lib
from comfyui_amd import functional as HF

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize("D,H", [(2560, 6912), (512, 256)])
@pytest.mark.parametrize("rows", [1, 17, 64, 127, 128])
def test_intermediate(dev, D, H, rows):
    assert _lib.lib.hdmoe_gate_up_kernel_name(_lib.W_BF16, rows, 0, D, 256, H, 0) == b"gemm4w_kernel<SWIGLU>"
    g = torch.Generator(device=dev).manual_seed(rows)
    ws = [(torch.randn(s, generator=g, device=dev) * 0.02).to(BF16) for s in ((H, D), (D, H), (H, D))]
    fw = HF.make_ffn_weights(*ws)
    x = torch.randn((rows, D), generator=g, device=dev).to(BF16)
    work = torch.empty(_lib.lib.hdmoe_ffn_workspace_bytes(rows, D, H, _lib.W_BF16), dtype=torch.uint8, device=dev)
    out = torch.empty((rows, D), dtype=BF16, device=dev)
    _lib.check(_lib.lib.hdmoe_ffn_swiglu(_lib.W_BF16, x.data_ptr(), rows, D, H, ctypes.byref(fw), out.data_ptr(), work.data_ptr(), work.numel(),
                                         torch.cuda.current_stream().cuda_stream))
    h = work[:rows * H * 2].view(BF16).view(rows, H).double()
    bf = lambda t: t.to(BF16).double()
    h1, h3 = bf(x.double() @ ws[0].double().T), bf(x.double() @ ws[2].double().T)
    want = bf(bf(torch.nn.functional.silu(h1)) * h3)
    # fp32 sums in another order are off by about 1e-6 of the magnitudes added and round to another bf16 (2^-8 at most) in under one case of a
    # hundred: for w1 x, w3 x and silu a 2-norm of 3 * 2^-8 * sqrt(1e-2) at the most
    assert float((h - want).norm() / want.norm()) < 1.2e-3
