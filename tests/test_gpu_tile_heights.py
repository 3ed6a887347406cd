"""Tiles of fewer than 256 rows in the 16-bit Linears (csrc/gemm4w.h, g4_cap): every height, segments that end anywhere in one, and
tiles of different heights behind each other in a block, for each way a tile is finished.

Bound: fp32 sums (K terms, each rounding at most 2^-24 of the running sum of magnitudes) rounded once to 16 bits; the activation is
compared behind that rounding, with one more step for its own."""
import ctypes

import pytest
import torch

from comfyui_amd import _lib, synth

pytestmark = pytest.mark.gpu
BF16, F16 = torch.bfloat16, torch.float16
STEP = {BF16: 2.0 ** -8, F16: 2.0 ** -11}


def within(y, a, w, bias, scale, act, dt):
    ref = a.double() @ w.double().t() * scale + (0.0 if bias is None else bias.double())
    lim = (a.double().abs() @ w.double().abs().t()) * abs(scale) * (a.shape[1] * 2.0 ** -24) + STEP[dt] * ref.abs() + 1e-7
    if act == "gelu":   # slope at most 1.13
        ref = torch.nn.functional.gelu(ref)
        lim = 1.13 * lim + STEP[dt] * ref.abs() + 1e-7
    err = (y.double() - ref).abs()
    assert bool((err <= lim).all()), float((err / lim).max())


# 10 n-tiles: 1 to 52 m-tiles
@pytest.mark.parametrize("rows,K,height", [(129, 640, 128), (1690, 640, 128), (3100, 640, 128), (3333, 640, 160), (4161, 640, 192), (4801, 2560, 224),
                                           (5249, 640, 256), (6500, 640, 128), (10209, 2560, 224), (11111, 640, 256)])
@pytest.mark.parametrize("kind", ["bf16", "f16", "upcast"])
def test_linear(dev, rows, K, height, kind):
    from comfyui_amd import functional as HF
    N = 2560
    code = {"bf16": _lib.W_BF16, "f16": _lib.W_F16, "upcast": _lib.W_E4M3FN_UPCAST}[kind]
    assert _lib.lib.hdmoe_linear_tile_rows(code, rows, K, N) == height
    g = torch.Generator(device=dev).manual_seed(rows)
    dt = F16 if kind == "f16" else BF16
    a = torch.randn((rows, K), generator=g, device=dev).to(dt)
    b = torch.randn(N, generator=g, device=dev).to(dt)
    w = torch.randn((N, K), generator=g, device=dev) / K ** 0.5
    if kind == "upcast":
        w, s = synth.quantize_per_tensor(w)
        within(HF.linear_upcast(a, w, s, b), a, w, b, float(s.to(BF16)), "none", dt)
        within(HF.linear_upcast(a, w), a, w, None, 1.0, "none", dt)
    else:
        w = w.to(dt)
        for bias in (None, b):
            y = HF.linear(a, w, bias=bias)
            within(y, a, w, bias, 1.0, "none", dt)


@pytest.mark.parametrize("code", [_lib.W_BF16, _lib.W_E4M3FN_UPCAST])
def test_dense_down_projection(dev, code):
    """The contraction without a bias: rows of a dense feed-forward on lower tiles are those of one on whole tiles (no working memory for
    parts, and sizes at which the down projection is not cut)."""
    D = H = 2560
    g = torch.Generator(device=dev).manual_seed(code)
    fw, keep = _lib.FfnWeights(), []
    for i in (1, 2, 3):
        w = torch.randn((D, H), generator=g, device=dev) * 0.02
        if code == _lib.W_BF16:
            keep.append(w.to(BF16))
        else:
            w8, s = synth.quantize_per_tensor(w)
            keep += [s, w8]
            setattr(fw, f"scale_w{i}", s.data_ptr())
        setattr(fw, f"w{i}", keep[-1].data_ptr())
    x = torch.randn((11999, D), generator=g, device=dev).to(BF16)

    def run(rows):
        ws = torch.empty(-(-rows * H * 2 // 256) * 256, dtype=torch.uint8, device=dev)
        y = torch.full((rows + 1, D), 7.0, dtype=BF16, device=dev)
        _lib.check(_lib.lib.hdmoe_ffn_swiglu(code, x.data_ptr(), rows, D, H, ctypes.byref(fw), y.data_ptr(), ws.data_ptr(), ws.numel(), None))
        torch.cuda.synchronize()
        assert bool((y[rows] == 7.0).all())
        return y[:rows]
    full = run(11999)
    assert bool(torch.isfinite(full.float()).all()) and float(full.float().std()) > 0
    for rows, height in ((11999, 256), (3073, 128), (3115, 128), (3627, 160), (8171, 192), (9803, 224)):
        assert _lib.lib.hdmoe_linear_tile_rows(code, rows, H, D) == height
        assert torch.equal(run(rows), full[:rows]), rows


@pytest.mark.parametrize("sizes", [
    (161, 193, 129, 225, 97, 33, 1, 0), (384, 385, 352, 416, 340, 410, 375, 338), (300, 20, 700, 130, 250, 190, 0, 160),
    (224, 224, 224, 224, 224, 224, 224, 225),
])
@pytest.mark.parametrize("act", ["none", "gelu"])
@pytest.mark.parametrize("dt", [BF16, F16])
def test_grouped_linears(dev, sizes, act, dt):
    from comfyui_amd import functional as HF
    K, N, shared = 2048, 4096, 700   # 16 pairs of K steps: the activation hides behind the next tile
    g = torch.Generator(device=dev).manual_seed(sum(sizes))
    rows = sum(sizes)
    ws = [((torch.randn((N, K), generator=g, device=dev) / K ** 0.5).to(dt), torch.randn(N, generator=g, device=dev).to(dt)) for _ in range(9)]
    a = torch.randn((rows, K), generator=g, device=dev).to(dt)
    st = torch.randn((shared, K), generator=g, device=dev).to(dt)
    offsets = torch.tensor([0, *torch.tensor(sizes).cumsum(0).tolist()], dtype=torch.int32, device=dev)
    y, ys = HF.grouped_linear(a, offsets, ws[:8], a_static=st, shared=ws[8], act=act)
    at = 0
    for n, (w, b) in zip(sizes, ws):
        within(y[at:at + n], a[at:at + n], w, b, 1.0, act, dt)
        at += n
    within(ys, st, *ws[8], 1.0, act, dt)
