"""With `batch_invariant` (fixed_k_cut of the C interface) a row's bytes do not depend on how the other rows of a call are routed, on
the paths with 16-bit activations, whose last round of tiles is otherwise cut along K by the experts' segment sizes. Without it
they do at these sizes, which says that the cut ran."""
import pytest
import torch

from comfyui_amd import _lib, hunyuan3d, ops, synth

pytestmark = pytest.mark.gpu
BF16, F16, FP8 = torch.bfloat16, torch.float16, torch.float8_e4m3fn
SAME = 100      # tokens at the end of both batches


def tail(tiles, K):
    return _lib.lib.hdmoe_tail_plan(_lib.W_BF16, tiles, K, 0, None, None)


def outcome(call):
    """Whether the shared tokens come out the same in both batches, with and without the flag."""
    return {flag: all(torch.equal(a, b) for a, b in zip(call(flag, 0), call(flag, 1))) for flag in (False, True)}


@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("act", ["none", "gelu"])
def test_grouped_linears(dev, dt, act):
    from comfyui_amd import functional as HF
    T, E, K, N = 3000, 8, 4096, 2048
    g = torch.Generator(device=dev).manual_seed(1)
    x = torch.randn((T, K), generator=g, device=dev).to(dt)
    ws = [((torch.randn((N, K), generator=g, device=dev) / K ** 0.5).to(dt), torch.randn(N, generator=g, device=dev).to(dt))
          for _ in range(E + 1)]
    t = torch.arange(T, device=dev)
    even = torch.stack([t % E, (t + 1) % E], 1)
    two = even.clone()
    two[:-SAME] = torch.tensor([0, 1], device=dev)
    # 3 m-tiles of 8 n-tiles for each expert, 12 for the shared one: 288 tiles; 12 for two experts, 1 for the others: 336
    assert tail(288, K) != tail(336, K)

    def call(flag, batch, sorted_rows=False):
        _, offsets, perm, inv = HF.dispatch([even, two][batch].to(torch.int32).contiguous(), E)
        if sorted_rows:
            y, ys = HF.grouped_linear(x[(perm // 2).long()].contiguous(), offsets, ws[:E], a_static=x, shared=ws[E], act=act, fixed_k_cut=flag)
        else:
            y, ys = HF.grouped_linear_tokens(x, perm, offsets, ws[:E], shared=ws[E], act=act, fixed_k_cut=flag)
        return y[inv.long()].view(T, 2, N)[-SAME:], ys[-SAME:]
    assert outcome(call) == {False: False, True: True}
    assert outcome(lambda f, b: call(f, b, True)) == {False: False, True: True}


def batches(x):
    """Two batches that share their last tokens; in the second one the others are copies of one token."""
    y = x.clone()
    y[:, :-SAME] = x[:, :1]
    return x, y


@pytest.mark.parametrize("dt", [BF16, F16])
def test_gelu_block(dev, dt):
    g = torch.Generator(device=dev).manual_seed(2)
    m = hunyuan3d.MoEBlock(2048, num_experts=8, moe_top_k=2, ff_inner_dim=4096, dtype=dt, device=dev).eval()
    with torch.no_grad():
        for p in m.parameters():
            p.copy_(torch.randn(p.shape, generator=g, device=dev) * (p.shape[-1] ** -0.5 if p.dim() > 1 else 0.2))
    xs = batches(torch.randn((1, 3000, 2048), generator=g, device=dev).to(dt))

    def call(flag, batch):
        m.batch_invariant = flag
        return [m(xs[batch])[0, -SAME:]]
    assert outcome(call) == {False: False, True: True}


@pytest.mark.parametrize("weights", ["bf16", "fp8"])
def test_layer_with_16_bit_activations(dev, weights):
    """960 tokens at the model's width: 544 tiles of an evenly routed gate/up contraction, 32 left over and cut in 4; 652 tiles with
    two experts taking nearly all of them, 140 left over and not cut."""
    assert tail(544, 2560) == 4 and tail(652, 2560) == 1
    sd = synth.to_state_dict(synth.make_weights(7, device=dev)[0], weights, scale_input=False)
    m = synth.build_module(sd, weights, dev, fp8_matrix_mult=False, scale_input=False)
    xs = batches(torch.randn((1, 960, synth.DIM), generator=torch.Generator(device=dev).manual_seed(3), device=dev).to(BF16))
    assert m._collect(xs[0][0]) is not None

    def call(flag, batch):
        m.batch_invariant = flag
        return [m(xs[batch])[0, -SAME:]]
    with torch.no_grad():
        assert outcome(call) == {False: False, True: True}


@pytest.mark.parametrize("weights", ["bf16", "fp8", "fp16"])
def test_linear(dev, weights):
    """700 rows by 2560 features are 30 tiles cut along K, 3000 rows 120 that are not."""
    g = torch.Generator(device=dev).manual_seed(4)
    dt = F16 if weights == "fp16" else BF16
    x = torch.randn((3000, 2560), generator=g, device=dev).to(dt)
    w = torch.randn((2560, 2560), generator=g, device=dev) * 0.02
    if weights == "fp8":
        m = ops.scaled_fp8_ops(fp8_matrix_mult=False, override_dtype=FP8).Linear(2560, 2560, bias=False, device=dev)
        w8, s = synth.quantize_per_tensor(w)
        m.weight, m.scale_weight = torch.nn.Parameter(w8, requires_grad=False), torch.nn.Parameter(s, requires_grad=False)
    else:
        m = ops.disable_weight_init.Linear(2560, 2560, bias=False, dtype=dt, device=dev)
        m.weight = torch.nn.Parameter(w.to(dt), requires_grad=False)
    assert tail(30, 2560) > 1 and tail(120, 2560) == 1

    def call(flag, batch):
        m.batch_invariant = flag
        return [m(x[:[700, 3000][batch]])[:700]]
    with torch.no_grad():
        assert outcome(call) == {False: False, True: True}
