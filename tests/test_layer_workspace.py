"""A layer's workspace that holds fewer parts of the down projection of a few tokens than it is cut into with the whole of it (csrc/layer.hip,
hdmoe_moe_ffn): the call is taken with those parts."""
import ctypes

import pytest
import torch

from comfyui_amd import _lib, synth
from comfyui_amd import functional as HF

CODES = [_lib.W_BF16, _lib.W_E4M3FN, _lib.W_E4M3FN_UPCAST]
D, H, HS, E = synth.DIM, synth.H_ROUTED, synth.H_SHARED, 4


def with_parts(tokens, code, parts):
    """The workspace with room for that many parts of every row."""
    lay = HF.layer_layout(tokens, D, H, HS, E, code)
    return lay.partials + -(-parts * 3 * tokens * D * 4 // 256) * 256 + 256


@pytest.mark.parametrize("code", CODES)
@pytest.mark.parametrize("tokens,parts", [(1, 3), (16, 3), (64, 3), (128, 3), (150, 3), (180, 2), (200, 2), (256, 2)])
def test_taken(code, tokens, parts):
    """What such a call is refused for here is its missing modulation, which is looked at behind the workspace."""
    t = torch.zeros(64, dtype=torch.uint8)
    p = t.data_ptr()
    args = _lib.LayerArgs()
    args.T, args.D, args.H, args.Hs, args.E, args.weight_dtype = tokens, D, H, HS, E, code
    args.x = args.gate_w = args.out = args.mod_scale = p
    args.experts = (_lib.FfnWeights * E)()
    args.shared = ctypes.pointer(_lib.FfnWeights())
    args.workspace = 256   # never read: aligned is all it has to be
    for size, rc in ((with_parts(tokens, code, parts), _lib.E_NULL), (with_parts(tokens, code, parts) - 256, _lib.E_WORKSPACE),
                     (with_parts(150, code, 3) if tokens <= 150 else with_parts(256, code, 2), _lib.E_NULL)):
        args.workspace_bytes = size
        assert _lib.lib.hdmoe_moe_ffn(ctypes.byref(args), None) == rc, size


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["fp8", "upcast", "bf16"])
def test_results(dev, kind):
    from tests.test_gpu_two_lengths import layer
    m, x = layer(dev, kind)
    wdt, experts, shared, keep = m._collect(x)
    code = HF.weight_dtype_code(wdt)
    for tokens, parts in ((16, 3), (128, 3), (200, 2), (256, 2)):
        xs = x.reshape(-1, D)[:tokens].contiguous()
        full = HF.moe_ffn(xs, m.gate.weight, experts, shared, H, HS, wdt)
        size = with_parts(tokens, code, parts)
        assert size < _lib.lib.hdmoe_layer_workspace_bytes(tokens, D, H, HS, E, code)
        work = torch.zeros(size + 4096, dtype=torch.uint8, device=dev)
        y = torch.empty_like(full)
        args = _lib.LayerArgs()
        args.T, args.D, args.H, args.Hs, args.E, args.weight_dtype = tokens, D, H, HS, E, code
        args.x, args.gate_w, args.experts = xs.data_ptr(), m.gate.weight.data_ptr(), (_lib.FfnWeights * E)(*experts)
        sh = _lib.FfnWeights.from_buffer_copy(shared)
        args.shared = ctypes.pointer(sh)
        args.out, args.workspace, args.workspace_bytes, args.fixed_k_cut = y.data_ptr(), work.data_ptr(), size, 0
        _lib.check(_lib.lib.hdmoe_moe_ffn(ctypes.byref(args), torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert int(work[size:].max()) == 0, tokens   # nothing behind its end is touched
        # sums in another order move a value by a bf16 step of 2^-8 at most here and there: all of them together stay under that in the 2-norm
        assert float((y.float() - full.float()).norm() / full.float().norm()) < 2.0 ** -8, tokens
    del keep
