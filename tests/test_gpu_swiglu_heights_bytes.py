"""Gate/up on 16-bit activations on tiles of every height (csrc/gemm4w.h, tile_mix and the texts of 4 to 8 token blocks): a row's K steps are the same,
and at this K no tile is cut along it, so the intermediate is byte for byte that of a call whose tiles are all whole."""
import ctypes

import pytest
import torch

from comfyui_amd import _lib
from tests.test_gpu_swiglu_heights import BF16, D, H, WHOLE, weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("code", [_lib.W_BF16, _lib.W_E4M3FN_UPCAST])
def test_every_height(dev, code):
    g = torch.Generator(device=dev).manual_seed(6)
    fw, *keep = weights(g, dev, code)
    x = torch.randn((WHOLE, D), generator=g, device=dev).to(BF16)

    def h(n):
        room = _lib.lib.hdmoe_ffn_workspace_bytes(n, D, H, code)
        work, out = torch.empty(room, dtype=torch.uint8, device=dev), torch.empty((n, D), dtype=BF16, device=dev)
        _lib.check(_lib.lib.hdmoe_ffn_swiglu(code, x.data_ptr(), n, D, H, ctypes.byref(fw), out.data_ptr(), work.data_ptr(), room,
                                             torch.cuda.current_stream().cuda_stream))
        return work[:n * H * 2].view(BF16).view(n, H)
    full = h(WHOLE)
    assert bool(torch.isfinite(full.float()).all()) and float(full.float().std()) > 0
    for rows in (129, 160, 161, 193, 225, 256, 257, 384, 385, 400, 417, 449, 512, 513, 641, 1000, 1300, 1500, 2000):
        assert torch.equal(h(rows), full[:rows]), rows
