"""fp8 contractions on the 4-wave kernel (csrc/gemm4w.h) against 64-bit arithmetic on the same fp8 operands.

The bound: one rounding to bf16 (2^-9 of the value, 2^-8 with the bias' own) and what the fp8 matrix instruction leaves out of an exact sum, 1e-5 of the
sum of the terms' magnitudes (measured on exactly representable sums; doubled here)."""
import ctypes

import pytest
import torch

from comfyui_amd import _lib

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn


def operands(rows, n, k, seed, dev):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn((rows, k), generator=g).to(FP8)
    w = (torch.randn((n, k), generator=g) * 40).to(FP8)
    return a.to(dev), w.to(dev)


def check(y, a, w, scale, bias=None):
    exact = (a.double() @ w.double().T) * scale
    mag = (a.double().abs() @ w.double().abs().T) * scale
    if bias is not None:
        exact += bias.double()
    err = (y.double() - exact).abs()
    assert bool((err <= 2.0 ** -8 * exact.abs() + 2e-5 * mag).all()), float((err / (exact.abs() + 1e-3 * mag)).max())


@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("rows,k", [(1281, 512), (1300, 768), (1536, 2560), (2500, 512)])
def test_linear(dev, rows, k, with_bias):
    """Row counts where 256-token tiles are taken: the last tile of one row, ragged, full, more tiles than CUs."""
    n = 10240
    name = _lib.lib.hdmoe_plain_kernel_name(0, 0, 0, rows, k, n, 1, int(with_bias))
    assert name == (b"gemm4w_kernel<F8, BIAS>" if with_bias else b"gemm4w_kernel<F8, PLAIN>")
    a, w = operands(rows, n, k, rows + k, dev)
    bias = torch.randn(n, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).to(dev)
    sw, si = torch.tensor(0.0007, device=dev), torch.tensor(0.6, device=dev)
    y = torch.full((rows + 1, n), 7.0, dtype=torch.bfloat16, device=dev)
    _lib.check(_lib.lib.hdmoe_linear_bias(_lib.W_E4M3FN, a.data_ptr(), rows, k, n, w.data_ptr(), sw.data_ptr(), si.data_ptr(),
                                          bias.data_ptr() if with_bias else None, y.data_ptr(), None))
    torch.cuda.synchronize()
    assert bool((y[rows] == 7.0).all())
    check(y[:rows], a, w, float(sw * si), bias if with_bias else None)


@pytest.mark.parametrize("sizes,k", [((1, 0, 700, 499), 512), ((256, 512, 257, 1), 1280), ((1500, 1500, 1500, 1500), 768)])
def test_grouped_down(dev, sizes, k):
    """Expert segments of one row, none, whole tiles and one row more."""
    n, rows = 512, sum(sizes)
    assert _lib.lib.hdmoe_plain_kernel_name(rows, len(sizes), k, 0, 0, n, 1, 0) == b"gemm4w_kernel<F8, PLAIN>"
    off = torch.tensor([0] + list(torch.tensor(sizes).cumsum(0)), dtype=torch.int32)
    a, _ = operands(rows, 256, k, rows, dev)
    ws = [operands(1, n, k, 50 + e, dev)[1] for e in range(len(sizes))]
    sw = [torch.tensor(0.0005 * (e + 1), device=dev) for e in range(len(sizes))]
    si = torch.tensor(0.5, device=dev)
    arr = (_lib.FfnWeights * len(sizes))()
    for e in range(len(sizes)):
        arr[e].w2, arr[e].scale_w2, arr[e].scale_in2 = ws[e].data_ptr(), sw[e].data_ptr(), si.data_ptr()
    y = torch.full((rows + 1, n), 7.0, dtype=torch.bfloat16, device=dev)
    offsets = off.to(dev)
    _lib.check(_lib.lib.hdmoe_grouped_down(_lib.W_E4M3FN, a.data_ptr(), offsets.data_ptr(), rows, len(sizes), k, n, arr, y.data_ptr(), None))
    torch.cuda.synchronize()
    assert bool((y[rows] == 7.0).all())
    for e in range(len(sizes)):
        if sizes[e]:
            check(y[off[e]:off[e + 1]], a[off[e]:off[e + 1]], ws[e], float(sw[e] * si))


@pytest.mark.parametrize("rows,dim,hidden", [(768, 2560, 6912), (300, 2560, 6912), (257, 512, 3584), (1000, 1024, 2560)])
def test_cut_down_projection(dev, rows, dim, hidden):
    """A dense feed-forward whose down projection is cut along K, against the product of the h that it left in its workspace."""
    L = _lib.lib
    aligned = -(-rows * dim // 256) * 256, -(-rows * hidden // 256) * 256
    nbytes = L.hdmoe_ffn_workspace_bytes(rows, dim, hidden, _lib.W_E4M3FN)
    parts, left = divmod(nbytes - sum(aligned), rows * dim * 4)
    assert parts >= 2 and left < 256
    assert L.hdmoe_plain_kernel_name(0, 0, 0, rows, hidden, dim, parts, 0) == b"gemm4w_kernel<F8, PARTIAL>"
    g = torch.Generator().manual_seed(rows)
    x = torch.randn((rows, dim), generator=g).to(torch.bfloat16).to(dev)
    w1, w3 = ((torch.randn((hidden, dim), generator=g) * 40).to(FP8).to(dev) for _ in range(2))
    w2 = (torch.randn((dim, hidden), generator=g) * 40).to(FP8).to(dev)
    scales = torch.tensor([0.0006, 0.0005, 0.0007, 0.5], device=dev)
    one = torch.ones((), device=dev)
    fw = _lib.FfnWeights()
    fw.w1, fw.w2, fw.w3 = w1.data_ptr(), w2.data_ptr(), w3.data_ptr()
    fw.scale_w1, fw.scale_w2, fw.scale_w3 = (scales[i:].data_ptr() for i in range(3))
    fw.scale_in1 = fw.scale_in3 = one.data_ptr()
    fw.scale_in2 = scales[3:].data_ptr()
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    y = torch.full((rows + 1, dim), 7.0, dtype=torch.bfloat16, device=dev)
    _lib.check(L.hdmoe_ffn_swiglu(_lib.W_E4M3FN, x.data_ptr(), rows, dim, hidden, ctypes.byref(fw), y.data_ptr(), ws.data_ptr(), nbytes, None))
    torch.cuda.synchronize()
    assert bool((y[rows] == 7.0).all())
    h = ws[aligned[0]:aligned[0] + rows * hidden].view(FP8).view(rows, hidden)
    assert bool(torch.isfinite(h.float()).all()) and float(h.float().std()) > 0.1
    check(y[:rows], h, w2, float(scales[1]) * 0.5)
