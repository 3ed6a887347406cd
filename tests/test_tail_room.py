"""Working memory of contractions on 16-bit activations: asked for where the plan of the tail tiles uses it, and only there; the sizes
that hold everything but the parts of tail tiles are taken as well, for the same results but for the order of fp32 sums."""
import ctypes

import pytest
import torch

from comfyui_amd import _lib, synth

BF16 = torch.bfloat16
TILE = 256 * 256 * 4
SCRATCH = lambda: groups(rows_static=3000, act=1) - groups(rows_static=3000, act=0)


def groups(act=0, weight=_lib.W_BF16, K=2560, N=2560, E=0, rows=0, rows_static=0, fixed=0):
    a = _lib.LinearArgs()
    a.act_dtype, a.weight_dtype, a.K, a.N, a.act = _lib.W_BF16, weight, K, N, act
    a.E, a.rows, a.rows_static, a.fixed_k_cut = E, rows, rows_static, fixed
    return _lib.lib.hdmoe_linear_groups_workspace_bytes(ctypes.byref(a))


def parts(tiles, K, rows_per_tile, code=_lib.W_BF16):
    return _lib.lib.hdmoe_tail_plan(code, tiles, K, tiles * (256 - rows_per_tile), None, None)


@pytest.mark.parametrize("code", [_lib.W_BF16, _lib.W_E4M3FN_UPCAST])
def test_linears_ask_for_what_their_plan_uses(code):
    assert groups(weight=code, rows_static=1) == 10 * parts(10, 2560, 1, code) * TILE > 0
    assert groups(weight=code, rows_static=512) == 20 * parts(20, 2560, 256, code) * TILE > 0
    assert groups(weight=code, rows_static=3000) == 0                 # 120 tiles: not cut
    assert groups(weight=code, rows_static=3000, N=256, K=256) == 0   # too short
    assert groups(weight=code, rows_static=512, fixed=1) == 0
    assert groups(weight=code, rows_static=512, K=2496) == 0          # not a length of the kernel that cuts
    assert groups(weight=code, E=8, rows=400, N=512) == 256 * TILE    # by segment sizes that the device knows
    assert groups(weight=code, E=8, rows=8 * 40000, rows_static=0) == 0   # more than 24 rounds


def test_room_for_the_activation_only_where_it_hides():
    assert SCRATCH() > 0 and groups(act=1, rows_static=1) == SCRATCH() + groups(rows_static=1)
    assert groups(act=1, rows_static=3000, K=320) == 0
    assert groups(act=1, E=8, rows=400, N=512, fixed=1) == SCRATCH()


def ffn_bytes(rows, code=_lib.W_BF16, D=2560, H=6912):
    return _lib.lib.hdmoe_ffn_workspace_bytes(rows, D, H, code)


def test_feed_forwards_ask_for_what_their_plans_use():
    h = lambda rows: rows * 6912 * 2
    # gate/up 24 x 54 tiles, 16 left over; down projection 240 tiles, not cut. 4400 rows: 972 tiles, 204 left over, not cut
    assert ffn_bytes(6000) == h(6000) + 16 * parts(1296, 2560, 250) * TILE > h(6000)
    assert ffn_bytes(4400) == h(4400)
    lay = lambda T, code=_lib.W_BF16: (lambda l: (_lib.lib.hdmoe_layer_layout_get(T, 2560, 6912, 3584, 4, code, ctypes.byref(l)), l)[1])(_lib.LayerLayout())
    for T in (64, 128):                                      # the three-stage ring: nothing of this kind is cut
        assert lay(T).total == lay(T).flags + 256
    l = lay(960)
    assert max(l.total - l.flags - 256, l.flags - l.partials) >= 256 * TILE
    assert lay(4000).total - lay(4000).flags - 256 in (0, 256 * TILE) and lay(2100).total == lay(2100).flags + 256 + 256 * TILE
    for T in (64, 960, 2100):
        assert lay(T, _lib.W_E4M3FN).total == lay(T, _lib.W_E4M3FN).flags + 256


@pytest.mark.gpu
@pytest.mark.parametrize("code", [_lib.W_BF16, _lib.W_E4M3FN_UPCAST])
def test_feed_forward_with_the_smaller_workspace(dev, code):
    from comfyui_amd import functional as HF
    rows, D, H = 6000, 2560, 6912
    g = torch.Generator(device=dev).manual_seed(1)
    ws, scales = [], {}
    for name, shape in (("1", (H, D)), ("2", (D, H)), ("3", (H, D))):
        w = torch.randn(shape, generator=g, device=dev) * 0.02
        if code == _lib.W_BF16:
            ws.append(w.to(BF16))
        else:
            w, scales["scale_w" + name] = synth.quantize_per_tensor(w)
            ws.append(w)
    fw = HF.make_ffn_weights(*ws, scales)
    x = torch.randn((rows, D), generator=g, device=dev).to(BF16)
    full = HF.ffn_swiglu(x, fw, H, BF16 if code == _lib.W_BF16 else HF.FP8_UPCAST)
    small = rows * H * 2                                      # what the size was without the room for tail tiles
    assert small < ffn_bytes(rows, code)
    work = torch.zeros(small + 4096, dtype=torch.uint8, device=dev)
    y = torch.empty_like(full)
    call = lambda n: _lib.lib.hdmoe_ffn_swiglu(code, x.data_ptr(), rows, D, H, ctypes.byref(fw), y.data_ptr(), work.data_ptr(), n,
                                               torch.cuda.current_stream().cuda_stream)
    _lib.check(call(small))
    assert int(work[small:].max()) == 0                       # nothing behind its end is touched
    d = (y.float() - full.float()).norm() / full.float().norm()
    assert float(d) <= 1e-3                                   # a bf16 rounding here and there falls the other way
    assert not torch.equal(y, full)                           # its tail tiles were not cut
    assert call(small - 256) != 0


@pytest.mark.gpu
def test_layer_with_the_smaller_workspace(dev):
    from comfyui_amd import functional as HF
    T = 2100
    sd = synth.to_state_dict(synth.make_weights(7, device=dev)[0], "bf16")
    m = synth.build_module(sd, "bf16", dev)
    x = torch.randn((T, synth.DIM), generator=torch.Generator(device=dev).manual_seed(3), device=dev).to(BF16)
    wdt, experts, shared, keep = m._collect(x)
    lay = HF.layer_layout(T, synth.DIM, synth.H_ROUTED, synth.H_SHARED, 4, _lib.W_BF16)
    work = torch.zeros(lay.total, dtype=torch.uint8, device=dev)
    full = HF.moe_ffn(x, m.gate.weight, experts, shared, synth.H_ROUTED, synth.H_SHARED, wdt, workspace=work)
    args = _lib.LayerArgs()
    args.T, args.D, args.H, args.Hs, args.E, args.weight_dtype = T, synth.DIM, synth.H_ROUTED, synth.H_SHARED, 4, _lib.W_BF16
    args.x, args.gate_w, args.experts = x.data_ptr(), m.gate.weight.data_ptr(), (_lib.FfnWeights * 4)(*experts)
    sh = _lib.FfnWeights.from_buffer_copy(shared)
    args.shared = ctypes.pointer(sh)
    y = torch.empty_like(full)
    args.out, args.workspace, args.workspace_bytes = y.data_ptr(), work.data_ptr(), lay.flags + 256
    args.fixed_k_cut = 0
    stream = torch.cuda.current_stream().cuda_stream
    work.zero_()
    _lib.check(_lib.lib.hdmoe_moe_ffn(ctypes.byref(args), stream))
    assert float((y.float() - full.float()).norm() / full.float().norm()) <= 1e-3
    assert int(work[lay.flags + 256:].max()) == 0             # nothing behind its end is touched
    args.workspace_bytes = lay.flags
    assert _lib.lib.hdmoe_moe_ffn(ctypes.byref(args), stream) != 0 and b"workspace" in _lib.lib.hdmoe_last_error()
    del keep
