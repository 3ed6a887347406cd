"""Which kernel a dense bf16 gate/up contraction of up to 128 rows runs on (csrc/gemm.hip, swiglu_on_g4): the 4-wave one where it cuts the tiles along
K, else the three-stage ring, and the room for the parts is asked for where they are cut."""
import ctypes

import pytest
import torch

from comfyui_amd import _lib

RING, G4 = b"grouped_gemm_kernel<BF16_SWIGLU, 2, LIGHT>", b"gemm4w_kernel<SWIGLU>"


@pytest.mark.parametrize("D,H,rows,kernel", [
    (2560, 6912, 1, G4), (2560, 6912, 128, G4), (4096, 11008, 64, G4), (5120, 13824, 128, G4), (2560, 16384, 1, G4),
    (2560, 16384, 64, RING), (2560, 32768, 1, RING), (2560, 32768, 128, RING), (512, 6912, 1, RING), (512, 6912, 128, RING), (512, 1024, 17, RING)])
def test_kernel(D, H, rows, kernel):
    assert _lib.lib.hdmoe_gate_up_kernel_name(_lib.W_BF16, rows, 0, D, 256, H, 0) == kernel


@pytest.mark.gpu
@pytest.mark.parametrize("D,H,rows", [(2560, 6912, 64), (2560, 6912, 1), (512, 6912, 128), (2560, 1024, 17)])
def test_without_the_room_for_the_parts(dev, D, H, rows):
    """The same rows with the whole workspace and with the least that the call takes: sums in another order at most."""
    from comfyui_amd import functional as HF
    g = torch.Generator(device=dev).manual_seed(rows)
    ws = [(torch.randn(s, generator=g, device=dev) * 0.02).to(torch.bfloat16) for s in ((H, D), (D, H), (H, D))]
    fw = HF.make_ffn_weights(*ws)
    x = torch.randn((rows, D), generator=g, device=dev).to(torch.bfloat16)
    bf = lambda t: t.to(torch.bfloat16).double()
    h1, h3 = bf(x.double() @ ws[0].double().T), bf(x.double() @ ws[2].double().T)
    want = bf(bf(torch.nn.functional.silu(h1)) * h3)
    full = _lib.lib.hdmoe_ffn_workspace_bytes(rows, D, H, _lib.W_BF16)
    sizes = {full}
    size = -(-rows * H * 2 // 256) * 256
    while size < full:   # the first that the call takes
        work = torch.empty(size, dtype=torch.uint8, device=dev)
        out = torch.empty((rows, D), dtype=torch.bfloat16, device=dev)
        if _lib.lib.hdmoe_ffn_swiglu(_lib.W_BF16, x.data_ptr(), rows, D, H, ctypes.byref(fw), out.data_ptr(), work.data_ptr(), size,
                                     torch.cuda.current_stream().cuda_stream) == 0:
            sizes.add(size)
            break
        size += rows * D * 4
    for n in sizes:
        work = torch.empty(n, dtype=torch.uint8, device=dev)
        out = torch.empty((rows, D), dtype=torch.bfloat16, device=dev)
        _lib.check(_lib.lib.hdmoe_ffn_swiglu(_lib.W_BF16, x.data_ptr(), rows, D, H, ctypes.byref(fw), out.data_ptr(), work.data_ptr(), n,
                                             torch.cuda.current_stream().cuda_stream))
        h = work[:rows * H * 2].view(torch.bfloat16).view(rows, H).double()
        # fp32 sums in another order are off by about 1e-6 of the magnitudes added and round to another bf16 (2^-8 at most) in under one case of a
        # hundred: for w1 x, w3 x and silu a 2-norm of 3 * 2^-8 * sqrt(1e-2) at the most
        assert float((h - want).norm() / want.norm()) < 1.2e-3, n
