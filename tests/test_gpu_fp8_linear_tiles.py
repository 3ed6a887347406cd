"""The fp8 Linear on tiles of several heights (csrc/gemm.hip, hdmoe_launch_linear_bias): a row's bytes do not depend on the
tile it falls into, and are the scaled product with the bias, rounded once.

K = 384, no multiple of 256, runs on the 8-wave kernel: 9000 rows by 10240 features on 256-token tiles, 1 to 1100 rows on 192-token ones. K = 2560
runs on the 4-wave kernel, whose tiles are 128 tokens and more (test_gpu_fp8_tile_heights.py).
Operands on which the kernels' sums would differ if their products came in another order: test_gpu_fp8_same_sums.py."""
import pytest
import torch

from comfyui_amd import _lib, synth

pytestmark = pytest.mark.gpu
BF16, FP8 = torch.bfloat16, torch.float8_e4m3fn


def kernel(rows, K, N):
    return _lib.lib.hdmoe_plain_kernel_name(0, 0, 0, rows, K, N, 1, 1).decode()


@pytest.mark.parametrize("K", [384, 2560])   # three K steps (an odd number), twenty
def test_rows_do_not_depend_on_the_tile(dev, K):
    from comfyui_amd import functional as HF
    g = torch.Generator(device=dev).manual_seed(K)
    a = torch.randn((9000, K), generator=g, device=dev).to(FP8)
    w, s = synth.quantize_per_tensor(torch.randn((10240, K), generator=g, device=dev) * 0.02)
    b = (torch.randn(10240, generator=g, device=dev) * 0.1).to(BF16)
    one = torch.ones((), device=dev)
    full = HF.linear(a, w, s, one, bias=b)
    for rows in (1, 31, 64, 191, 192, 193, 385, 1100):
        assert kernel(rows, K, 10240) == ("gemm4w_kernel<F8, BIAS>" if K == 2560 else "grouped_gemm_kernel<FP8_PLAIN_BIAS, 3>")
        y = HF.linear(a[:rows].contiguous(), w, s, one, bias=b)
        assert torch.equal(y, full[:rows]), rows
    # fp32 sums of K exact products (2^-24 of the sum of magnitudes each), scaled, biased and rounded to bf16 (half a step)
    x, v = a[:1100].double(), w.double()
    want = (x @ v.t()) * s.double() + b.double()
    lim = (x.abs() @ v.abs().t()) * s.double() * (K + 2) * 2.0 ** -24 + want.abs() * 2.0 ** -8 + 1e-7
    assert bool(((full[:1100].double() - want).abs() <= lim).all())


@pytest.mark.parametrize("K", [512, 640])   # the 4-wave and the 8-wave kernel
def test_last_round_of_many_rows(dev, K):
    """9000 rows by 2560 features: 470 tiles of 192 tokens instead of 360 of 256 (two rounds either way)."""
    from comfyui_amd import functional as HF
    if K == 512:
        assert _lib.lib.hdmoe_fp8_linear_tile_rows(9000, K, 2560) == 192
    else:
        assert kernel(9000, K, 2560) == "grouped_gemm_kernel<FP8_PLAIN_BIAS, 3>"
    g = torch.Generator(device=dev).manual_seed(3)
    a = torch.randn((9000, K), generator=g, device=dev).to(FP8)
    w, s = synth.quantize_per_tensor(torch.randn((2560, K), generator=g, device=dev) * 0.02)
    b = torch.zeros(2560, dtype=BF16, device=dev)
    one = torch.ones((), device=dev)
    y = HF.linear(a, w, s, one, bias=b)
    for lo in (0, 4400, 8500):   # 500 rows at a time: other tiles
        assert torch.equal(y[lo:lo + 500], HF.linear(a[lo:lo + 500].contiguous(), w, s, one, bias=b))
