"""The fp8 contractions come out the same bit for bit whichever kernel runs them: the 8-wave ones on 64-product matrix instructions and the
4-wave ones on 128-product ones (csrc/gemm4w.h, f8_chunk, has the order of the products). Operands of every e4m3fn code, so that sums
lose bits all along; with the products in ascending order one output in 1e4 differed."""
import pytest
import torch

from comfyui_amd import _lib
from tests.helpers import saved_forms, set_form

pytestmark = pytest.mark.gpu
BF16, FP8 = torch.bfloat16, torch.float8_e4m3fn


@pytest.fixture
def forms():
    yield from saved_forms()


def codes(shape, g, dev):
    c = torch.randint(0, 256, shape, generator=g, device=dev, dtype=torch.int32).to(torch.uint8)
    c[(c & 0x7F) == 0x7F] = 0   # no NaN
    return c.view(FP8)


@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("K,N,sizes", [
    (2560, 2560, (1, 300, 4800, 4801, 6400, 6401)),     # tiles of 128 to 256 tokens of the 4-wave kernel; test_forms has the 8-wave ones
    (512, 10240, (100, 1100, 1281, 2300)),
    (4096, 2560, (200, 6400, 6401)),
])
def test_rows_of_a_linear(dev, K, N, sizes, with_bias):
    """A row has the same bytes whatever rows come with it."""
    from comfyui_amd import functional as HF
    g = torch.Generator(device=dev).manual_seed(K + N)
    a, w = codes((sizes[-1], K), g, dev), codes((N, K), g, dev)
    s, one = torch.tensor(2.0 ** -12, device=dev), torch.ones((), device=dev)
    bias = torch.randn(N, generator=g, device=dev).to(BF16) if with_bias else None
    full = HF.linear(a, w, s, one, bias=bias)
    assert bool(torch.isfinite(full.float()).all())
    for rows in sizes[:-1]:
        assert torch.equal(HF.linear(a[:rows].contiguous(), w, s, one, bias=bias), full[:rows]), rows


def grouped(dev, sizes, K, N, swiglu, seed, scale=2.0 ** -17):
    g = torch.Generator(device=dev).manual_seed(seed)
    E, rows = len(sizes), sum(sizes)
    a = codes((rows, K), g, dev)
    offsets = torch.tensor([0] + list(torch.tensor(sizes).cumsum(0)), dtype=torch.int32, device=dev)
    ws = [[codes((N, K), g, dev) for _ in range(2)] for _ in range(E)]
    scales = torch.tensor([scale, 2 * scale, 0.75, 0.5], device=dev)
    arr = (_lib.FfnWeights * E)()
    for e in range(E):
        if swiglu:
            arr[e].w1, arr[e].w3 = ws[e][0].data_ptr(), ws[e][1].data_ptr()
            arr[e].scale_w1, arr[e].scale_w3 = scales[0:].data_ptr(), scales[1:].data_ptr()
            arr[e].scale_in1 = arr[e].scale_in3 = scales[2:].data_ptr()
            arr[e].scale_in2 = scales[3:].data_ptr()
        else:
            arr[e].w2, arr[e].scale_w2, arr[e].scale_in2 = ws[e][0].data_ptr(), scales[0:].data_ptr(), scales[2:].data_ptr()

    def run():
        out = torch.empty((rows, N), dtype=torch.uint8 if swiglu else BF16, device=dev)
        call = _lib.lib.hdmoe_grouped_swiglu if swiglu else _lib.lib.hdmoe_grouped_down
        _lib.check(call(_lib.W_E4M3FN, a.data_ptr(), offsets.data_ptr(), rows, E, K, N, arr, out.data_ptr(), None))
        torch.cuda.synchronize()
        return out
    run.keep = (a, offsets, ws, scales)
    run.operands = a, ws
    return run


@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("sizes,K,N", [((1500, 1500), 2048, 2560), ((1, 0, 700, 2299), 2560, 2560), ((2048, 2100), 6912, 512)])
def test_forms(dev, forms, sizes, K, N, swiglu):
    """What the launcher picks against the 8-wave kernels."""
    run = grouped(dev, sizes, K, N, swiglu, sum(sizes) + K)
    got = run()
    set_form("HDMOE_SWIGLU4W", "0")
    assert torch.equal(run(), got) and got.float().std() > 0


def test_forms_beyond_the_range(dev, forms):
    """Outputs above 448, infinite sums' products and NaN operands: the same bytes as well."""
    run = grouped(dev, (700, 900), 2048, 2560, True, 5, scale=2.0 ** -9)
    a, ws = run.operands
    a.view(torch.uint8)[::97, 5] = 0x7F
    ws[1][0].view(torch.uint8)[3] = 0xFF
    assert _lib.lib.hdmoe_gate_up_kernel_name(_lib.W_E4M3FN, 800, 2, 2048, 2560, 0, 1) == b"swiglu224_kernel"
    got = run()
    nan = (got & 0x7F) == 0x7F
    assert 0.01 < float(nan.float().mean()) < 0.99
    set_form("HDMOE_SWIGLU4W", "0")
    assert torch.equal(run() & 0x7F, got & 0x7F) and torch.equal(run()[~nan], got[~nan])   # the sign of a NaN is nobody's
