"""fp8 contractions on tiles of fewer than 256 tokens (csrc/gen_gemm4w.py, step8): every height, behind each other in a block, few and many
K steps, against 64-bit arithmetic on the same operands (the bound of test_gpu_gemm4w_fp8.py), and a row's bytes in tiles of other heights."""
import pytest
import torch

from comfyui_amd import _lib
from tests.test_gpu_gemm4w_fp8 import check, operands

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


HEIGHTS = {(3333, 512, 2560): 160, (4161, 768, 2560): 192, (4480, 2560, 2560): 192, (9001, 512, 2560): 192, (5600, 2560, 2560): 224, (1185, 512, 10240): 256,
           (1300, 768, 10240): 256, (5000, 512, 2560): 256, (6305, 768, 2560): 256}   # the others 128


# (up to 256 rows without a bias are the 8-wave kernel's) 10 or 40 n-tiles; the heights that the cost model picks (csrc/gemm4w.h, g4_best_cap), the last tile's may be lower
@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("rows,k,n", [(5600, 2560, 2560), (1, 512, 2560), (128, 768, 2560), (129, 512, 2560), (257, 2560, 10240), (700, 768, 2560), (1185, 512, 10240),
                                      (1300, 768, 10240), (2000, 2560, 2560), (3333, 512, 2560), (4161, 768, 2560), (4480, 2560, 2560),
                                      (5000, 512, 2560), (6305, 768, 2560), (9001, 512, 2560)])
def test_linear(dev, rows, k, n, with_bias):
    from comfyui_amd import functional as HF
    assert _lib.lib.hdmoe_fp8_linear_tile_rows(rows, k, n) == HEIGHTS.get((rows, k, n), 128)
    name = "gemm4w_kernel<F8, BIAS>" if with_bias else "gemm4w_kernel<F8, PLAIN>" if rows > 256 else "grouped_gemm_kernel<FP8_PLAIN, 4, LIGHT>"
    assert _lib.lib.hdmoe_plain_kernel_name(0, 0, 0, rows, k, n, 1, int(with_bias)).decode() == name
    a, w = operands(rows, n, k, rows + k, dev)
    bias = torch.randn(n, generator=torch.Generator().manual_seed(3)).to(BF16).to(dev) if with_bias else None
    sw, si = torch.tensor(0.0007, device=dev), torch.tensor(0.6, device=dev)
    y = HF.linear(a, w, sw, si, bias=bias)
    check(y, a, w, float(sw * si), bias)
    some = min(rows, 96)
    assert torch.equal(HF.linear(a[-some:].contiguous(), w, sw, si, bias=bias), y[-some:])


@pytest.mark.parametrize("sizes,k", [((129, 161, 193, 225, 256, 33, 0, 1), 512), ((400, 416, 450, 480, 511, 513, 300, 290), 768),
                                     ((1000, 20, 2100, 257), 2560)])
def test_segments(dev, sizes, k):
    n, rows = 2560, sum(sizes)
    off = torch.tensor([0] + list(torch.tensor(sizes).cumsum(0)), dtype=torch.int32)
    a, _ = operands(rows, 256, k, rows, dev)
    ws = [operands(1, n, k, 50 + e, dev)[1] for e in range(len(sizes))]
    sw, si = torch.tensor(0.0005, device=dev), torch.tensor(0.5, device=dev)
    arr = (_lib.FfnWeights * len(sizes))()
    for e in range(len(sizes)):
        arr[e].w2, arr[e].scale_w2, arr[e].scale_in2 = ws[e].data_ptr(), sw.data_ptr(), si.data_ptr()
    y = torch.full((rows + 1, n), 7.0, dtype=BF16, device=dev)
    offsets = off.to(dev)
    _lib.check(_lib.lib.hdmoe_grouped_down(_lib.W_E4M3FN, a.data_ptr(), offsets.data_ptr(), rows, len(sizes), k, n, arr, y.data_ptr(), None))
    torch.cuda.synchronize()
    assert bool((y[rows] == 7.0).all())
    for e in range(len(sizes)):
        if sizes[e]:
            check(y[off[e]:off[e + 1]], a[off[e]:off[e + 1]], ws[e], float(sw * si))


@pytest.mark.parametrize("rows,dim,hidden", [(257, 2560, 6912), (300, 512, 3584), (513, 2560, 6912), (768, 2560, 2560), (1300, 2560, 6912), (1700, 2560, 6912), (2048, 2560, 6912),
                                             (2600, 2560, 6912), (1700, 4096, 11008)])
def test_dense_feed_forward(dev, rows, dim, hidden):
    """Down projections in parts of 128-, 160-, 192- and 224-token tiles and whole, against the product of the h left in the workspace."""
    import ctypes
    L = _lib.lib
    FP8 = torch.float8_e4m3fn
    g = torch.Generator(device=dev).manual_seed(rows)
    x = torch.randn((rows, dim), generator=g, device=dev).to(BF16)
    w1, w3 = ((torch.randn((hidden, dim), generator=g, device=dev) * 40).to(FP8) for _ in range(2))
    w2 = (torch.randn((dim, hidden), generator=g, device=dev) * 40).to(FP8)
    scales = torch.tensor([0.0006, 0.0005, 0.0007, 0.5, 1.0], device=dev)
    fw = _lib.FfnWeights()
    fw.w1, fw.w2, fw.w3 = w1.data_ptr(), w2.data_ptr(), w3.data_ptr()
    fw.scale_w1, fw.scale_w2, fw.scale_w3 = (scales[i:].data_ptr() for i in range(3))
    fw.scale_in1 = fw.scale_in3 = scales[4:].data_ptr()
    fw.scale_in2 = scales[3:].data_ptr()
    nbytes = L.hdmoe_ffn_workspace_bytes(rows, dim, hidden, _lib.W_E4M3FN)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    y = torch.full((rows + 1, dim), 7.0, dtype=BF16, device=dev)
    _lib.check(L.hdmoe_ffn_swiglu(_lib.W_E4M3FN, x.data_ptr(), rows, dim, hidden, ctypes.byref(fw), y.data_ptr(), ws.data_ptr(), nbytes, None))
    torch.cuda.synchronize()
    assert bool((y[rows] == 7.0).all())
    at = -(-rows * dim // 256) * 256
    h = ws[at:at + rows * hidden].view(FP8).view(rows, hidden)
    assert float(h.float().std()) > 0.1
    check(y[:rows], h, w2, float(scales[1]) * 0.5)
