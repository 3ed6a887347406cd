"""The fp8 Linear on its 192- and 256-token tiles (csrc/gemm.hip, hdmoe_launch_linear_bias): a row's bytes do not depend on the
tile it falls into, and are the scaled product with the bias, rounded once.

9000 rows by 10240 features take 256-token tiles (of the 4-wave kernel; K = 384 of the 8-wave one), 1 to 1100 rows the 192-token ones.
Operands on which the kernels' sums would differ if their products came in another order: test_gpu_fp8_same_sums.py."""
import pytest
import torch

from comfyui_amd import synth

pytestmark = pytest.mark.gpu
BF16, FP8 = torch.bfloat16, torch.float8_e4m3fn


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
        y = HF.linear(a[:rows].contiguous(), w, s, one, bias=b)
        assert torch.equal(y, full[:rows]), rows
    # fp32 sums of K exact products (2^-24 of the sum of magnitudes each), scaled, biased and rounded to bf16 (half a step)
    x, v = a[:1100].double(), w.double()
    want = (x @ v.t()) * s.double() + b.double()
    lim = (x.abs() @ v.abs().t()) * s.double() * (K + 2) * 2.0 ** -24 + want.abs() * 2.0 ** -8 + 1e-7
    assert bool(((full[:1100].double() - want).abs() <= lim).all())


def test_last_round_of_many_rows(dev):
    """9000 rows by 2560 features: 470 tiles of 192 tokens instead of 360 of 256 (two rounds either way)."""
    from comfyui_amd import functional as HF
    g = torch.Generator(device=dev).manual_seed(3)
    a = torch.randn((9000, 512), generator=g, device=dev).to(FP8)
    w, s = synth.quantize_per_tensor(torch.randn((2560, 512), generator=g, device=dev) * 0.02)
    b = torch.zeros(2560, dtype=BF16, device=dev)
    one = torch.ones((), device=dev)
    y = HF.linear(a, w, s, one, bias=b)
    for lo in (0, 4400, 8500):   # 500 rows at a time: other tiles
        assert torch.equal(y[lo:lo + 500], HF.linear(a[lo:lo + 500].contiguous(), w, s, one, bias=b))
