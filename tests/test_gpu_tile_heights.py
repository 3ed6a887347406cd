"""Tiles of fewer than 256 rows in the 16-bit Linears (csrc/gemm4w.h, g4_cap): every height, segments that end anywhere in one, and
tiles of different heights behind each other in a block, for each way a tile is finished.

Bound: fp32 sums (K terms, each rounding at most 2^-24 of the running sum of magnitudes) rounded once to 16 bits; the activation is
compared behind that rounding, with one more step for its own."""
import pytest
import torch

from comfyui_amd import synth

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


# rows of one Linear at 10 n-tiles: the caps come to 1 to 52 m-tiles of 4 to 8 blocks of 32 rows
@pytest.mark.parametrize("rows", [129, 1690, 3100, 3333, 4161, 5249, 6500, 11111])
@pytest.mark.parametrize("kind", ["bf16", "f16", "upcast"])
def test_linear(dev, rows, kind):
    from comfyui_amd import functional as HF
    K, N = 640, 2560
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
