"""The entry points of the grouped Linears that bring no working memory (hdmoe_grouped_linear, hdmoe_grouped_linear_f16,
hdmoe_grouped_linear_tokens, hdmoe_grouped_swiglu with a width that the 4-wave kernel does not take), called as a program in C calls
them: on the kernels with 256- and with 320-token tiles, routed rows gathered or not.

Bounds: products summed in fp32 (K terms, 2^-24 of the sum of magnitudes each), bias, one rounding to 16 bits (half a step); with
GELU the rounded sum's activation (slope at most 1.13) is rounded again."""
import ctypes

import pytest
import torch

from comfyui_amd import _lib

BF16, F16 = torch.bfloat16, torch.float16
HALF_STEP = {BF16: 2.0 ** -8, F16: 2.0 ** -11}
LW = _lib.LinearWeights


def test_gate_up_of_a_width_off_128_takes_the_taller_tile_where_it_saves_a_round():
    name = lambda rows, D: _lib.lib.hdmoe_gate_up_kernel_name(_lib.W_BF16, rows // 2, 4, D, 6912, 0, 0).decode()
    # 640 rows per expert: 4 x 3 x 54 tiles of 256 rows (three rounds), 4 x 2 x 54 of 320 (two)
    assert name(2560, 2624) == "grouped_gemm_kernel<BF16_SWIGLU, 5>"
    assert name(2000, 2624) == "grouped_gemm_kernel<BF16_SWIGLU, 4>"
    assert name(2560, 2560) == "gemm4w_kernel<SWIGLU>"


def check(y, a, w, b, dt, gelu):
    h = a.double() @ w.double().t() + (0.0 if b is None else b.double())
    acc = (a.double().abs() @ w.double().abs().t()) * (a.shape[1] * 2.0 ** -24)
    lim, ref = acc, h
    if gelu:
        ref = torch.nn.functional.gelu(h)
        lim = 1.13 * (acc + HALF_STEP[dt] * h.abs())
    err = (y.double() - ref).abs()
    lim = lim + HALF_STEP[dt] * ref.abs() + 1e-7
    assert bool((err <= lim).all()), float((err / lim).max())


COUNTS = {
    "few": [3, 0, 40, 1],             # a few rows per expert, one empty
    "mid": [300, 257, 256, 0],        # edges of the 256-token tile
    "tall": [1281, 1280, 1279, 1300], # 320-token tiles: 20 m-tiles of 320 and 24 of 256, by 16 n-tiles and the shared expert's
}


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("K", [192, 256, 320])     # 192, 320: no multiple of 128; 256: two pairs of K steps
@pytest.mark.parametrize("counts", list(COUNTS))
def test_entries_without_working_memory(dev, dt, act, K, counts):
    counts, N = COUNTS[counts], 4096
    E, rows, T = len(counts), sum(counts), sum(counts) // 2
    g = torch.Generator(device=dev).manual_seed(K + rows)
    rnd = lambda *s, sc=1.0: (torch.randn(s, generator=g, device=dev) * sc).to(dt)
    ws, bs = [rnd(N, K, sc=K ** -0.5) for _ in range(E + 1)], [rnd(N) for _ in range(E)] + [None]
    offsets = torch.tensor([0] + torch.tensor(counts).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    p = lambda t: None if t is None else t.data_ptr()
    arr = (LW * E)(*[LW(p(w), p(b)) for w, b in zip(ws[:E], bs)])
    shared = LW(p(ws[E]), p(bs[E]))
    s = torch.cuda.current_stream().cuda_stream
    a, a_sh = rnd(rows, K), rnd(T, K)
    out, out_sh = torch.empty((rows, N), dtype=dt, device=dev), torch.empty((T, N), dtype=dt, device=dev)
    fn = _lib.lib.hdmoe_grouped_linear if dt == BF16 else _lib.lib.hdmoe_grouped_linear_f16
    _lib.check(fn(p(a), p(offsets), rows, E, arr, p(out), p(a_sh), T, ctypes.byref(shared), p(out_sh), K, N, act, s))
    for e, lo, hi in zip(range(E), offsets.tolist(), offsets.tolist()[1:]):
        check(out[lo:hi], a[lo:hi], ws[e], bs[e], dt, act)
    check(out_sh, a_sh, ws[E], None, dt, act)
    # gathered: the same rows read through a permutation of the tokens' slots
    perm = torch.randperm(rows // 2 * 2, generator=torch.Generator().manual_seed(1)).to(torch.int32).to(dev)
    offsets = torch.clamp(offsets, max=2 * T)
    out2 = torch.empty((2 * T, N), dtype=dt, device=dev)
    _lib.check(_lib.lib.hdmoe_grouped_linear_tokens(_lib.W_BF16 if dt == BF16 else _lib.W_F16, p(a_sh), T, p(perm), p(offsets), E, arr,
                                                    p(out2), ctypes.byref(shared), p(out_sh), K, N, act, s))
    a2 = a_sh[(perm // 2).long()]
    for e, lo, hi in zip(range(E), offsets.tolist(), offsets.tolist()[1:]):
        check(out2[lo:hi], a2[lo:hi], ws[e], bs[e], dt, act)
    check(out_sh, a_sh, ws[E], None, dt, act)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [7, 2000, 2560])
def test_gate_up_of_a_width_off_128(dev, rows):
    """256- and 320-token tiles of the 8-wave kernel: the same bytes for a row, and silu(w1 x) * (w3 x) rounded as the modules do."""
    from comfyui_amd import functional as HF
    D, H, E = 320, 6912, 4
    g = torch.Generator(device=dev).manual_seed(rows)
    x = torch.randn((rows, D), generator=g, device=dev).to(BF16)
    w = [(torch.randn((H, D), generator=g, device=dev) / D ** 0.5).to(BF16) for _ in range(2)]
    ex = [HF.make_ffn_weights(w[0], w[0], w[1])] * E
    cut = [rows * i // E for i in range(E + 1)]
    h = HF.grouped_swiglu(x, torch.tensor(cut, dtype=torch.int32, device=dev), ex, H)
    lo = rows // 2
    few = HF.grouped_swiglu(x[lo:lo + 3].contiguous(), torch.tensor([0, 3, 3, 3, 3], dtype=torch.int32, device=dev), ex, H)
    assert torch.equal(h[lo:lo + 3], few)
    a, b = x.double() @ w[0].double().t(), x.double() @ w[1].double().t()
    ref = torch.nn.functional.silu(a) * b
    # roundings of both sums, of silu and of the product (half a step each), of which the first reaches silu with a slope of at most 1.1
    lim = 2.0 ** -8 * (1.1 * a.abs() * b.abs() + 3 * ref.abs()) + 1e-5 * (1 + a.abs()) * (1 + b.abs())
    assert bool(((h.double() - ref).abs() <= lim).all())
