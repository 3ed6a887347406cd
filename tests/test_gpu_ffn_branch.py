"""hdmoe_ffn_branch against the three calls it stands for (hdmoe_ln_modulate_bf16, hdmoe_ffn_swiglu, hdmoe_gated_residual_bf16): the same
bytes, with the down projection cut along K and not, for every weight type, for widths with and without a register form of the LayerNorm."""
import pytest
import torch

from comfyui_amd import functional as HF, hidream, ops, synth

pytestmark = pytest.mark.gpu
BF16, FP8 = torch.bfloat16, torch.float8_e4m3fn


def feed_forward(dim, hidden, weights, dev, seed, scale_in=0.5):
    cls = {"bf16": ops.disable_weight_init, "fp8": ops.scaled_fp8_ops(fp8_matrix_mult=True, scale_input=True, override_dtype=FP8),
           "dequant": ops.scaled_fp8_ops(fp8_matrix_mult=False, scale_input=False, override_dtype=FP8)}[weights]
    ff = hidream.FeedForwardSwiGLU(dim, hidden, dtype=BF16, device=dev, operations=cls).eval()
    g = torch.Generator().manual_seed(seed)
    for lin in (ff.w1, ff.w2, ff.w3):
        w = torch.randn(tuple(lin.weight.shape), generator=g) * 0.03
        if weights == "bf16":
            lin.weight = torch.nn.Parameter(w.to(BF16).to(dev), requires_grad=False)
            continue
        w8, sw = synth.quantize_per_tensor(w)
        lin.weight = torch.nn.Parameter(w8.to(dev), requires_grad=False)
        lin.scale_weight = torch.nn.Parameter(sw.to(dev), requires_grad=False)
        if weights == "fp8":
            lin.scale_input = torch.nn.Parameter(torch.tensor(scale_in, device=dev), requires_grad=False)
    return ff


@pytest.mark.parametrize("weights", ["bf16", "fp8", "dequant"])
@pytest.mark.parametrize("dim,hidden,batch,tokens", [(2560, 10240, 2, 77), (2560, 10240, 1, 700), (512, 1024, 3, 65), (2560, 1536, 2, 2500), (768, 768, 1, 1)])
def test_same_bytes_as_the_three_calls(dev, weights, dim, hidden, batch, tokens):
    ff = feed_forward(dim, hidden, weights, dev, seed=dim + tokens)
    g = torch.Generator().manual_seed(tokens)
    x = torch.randn((batch, tokens, dim), generator=g).to(BF16).to(dev)
    shift, scale, gate = ((torch.randn((batch, 1, dim), generator=g) * 0.3).to(BF16).to(dev) for _ in range(3))
    y = ff.forward_branch(x, shift, scale, gate)
    x2 = x.view(-1, dim)
    n = HF.ln_modulate(x2, scale, shift, tokens)
    want = HF.gated_residual(ff(n.view(batch, tokens, dim)).view(-1, dim), gate, x2, tokens).view(batch, tokens, dim)
    assert bool(torch.isfinite(want.float()).all()) and float(want.float().std()) > 0
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))


def test_scales_that_one_cast_cannot_serve(dev):
    """w1 and w3 change apart behind the caller's back: NaN rows, as hdmoe_ffn_swiglu writes them, never a cast with the wrong factor."""
    ff = feed_forward(512, 1024, "fp8", dev, seed=3)
    x = torch.randn((1, 40, 512), device=dev).to(BF16)
    mods = [torch.zeros((1, 1, 512), dtype=BF16, device=dev) + 0.5 for _ in range(3)]
    assert bool(torch.isfinite(ff.forward_branch(x, *mods).float()).all())
    ff.w3.scale_input.data.fill_(0.25)
    assert bool(torch.isnan(ff.forward_branch(x, *mods).float()).all())   # (written through .data: the cached comparison still stands)


def test_a_forward_of_ones_own_is_called(dev):
    ff = feed_forward(512, 1024, "bf16", dev, seed=4)
    x = torch.randn((1, 33, 512), device=dev).to(BF16)
    mods = [torch.zeros((1, 1, 512), dtype=BF16, device=dev) + 0.5 for _ in range(3)]
    ff.forward = lambda n: torch.zeros_like(n)
    assert torch.equal(ff.forward_branch(x, *mods), x)
