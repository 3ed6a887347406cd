"""Linears that keep fp8 weights and multiply in bf16 are called one by one wherever a call does more than the class says: forward
hooks (what a calibration of scale_input hangs on), a forward set on the instance, a subclass with its own."""
import pytest
import torch

from comfyui_amd import hidream, ops, synth

FP8 = torch.float8_e4m3fn
DIM = 512


def linear(cls, mm=False):
    class_ = ops.scaled_fp8_ops(fp8_matrix_mult=mm, scale_input=False, override_dtype=FP8).Linear if cls is None else cls
    return class_(DIM, DIM, bias=False, dtype=FP8)


def ffn(**kw):
    return hidream.FeedForwardSwiGLU(DIM, 4 * DIM, dtype=FP8, operations=ops.scaled_fp8_ops(override_dtype=FP8, **kw))


def test_plain_linears_are_one_call():
    assert hidream._own_forward(linear(None)) and hidream._own_forward(linear(ops.manual_cast.Linear))
    assert hidream._fusable_dtype([ffn()]) == hidream.HF.FP8_UPCAST


def test_what_calls_do_beyond_the_class_keeps_the_calls():
    base = ops.scaled_fp8_ops(fp8_matrix_mult=False, override_dtype=FP8).Linear

    class Forward(base):
        def forward(self, x):
            return super().forward(x) * 2

    class Cast(base):
        def forward_comfy_cast_weights(self, x):
            return super().forward_comfy_cast_weights(x) * 2

    assert not hidream._own_forward(linear(Forward)) and not hidream._own_forward(linear(Cast))
    for change in (lambda l: l.register_forward_hook(lambda *a: None), lambda l: l.register_forward_pre_hook(lambda *a: None),
                   lambda l: setattr(l, "forward", lambda x: x)):
        f = ffn()
        change(f.w2)
        assert hidream._fusable_dtype([f]) is None
    # the flag of an instance does not change what its class computes
    l = linear(None, mm=True)
    l.hdmoe_fp8_matrix_mult = False
    assert hidream._upcasts(l) and not hidream._own_forward(l)


def test_the_key_of_a_packed_layer_sees_a_new_hook():
    fs = [ffn(), ffn()]
    dev = fs[0].w1.weight.device
    keys = [hidream._pack_key(fs, dev)]
    hook = fs[1].w3.register_forward_hook(lambda *a: None)
    keys.append(hidream._pack_key(fs, dev))
    hook.remove()
    assert keys[0] is not None and keys[0] != keys[1] and keys[0] == hidream._pack_key(fs, dev)
    fs[0].register_forward_pre_hook(lambda *a: None)
    assert hidream._pack_key(fs, dev) != keys[0]


@pytest.mark.gpu
def test_hooks_of_a_layer_run(dev):
    from tests.helpers import small_layer
    sd, x = small_layer(seed=3, dim=DIM, tokens=200, weights="fp8")
    sd = {k: v.to(dev) for k, v in sd.items() if not k.endswith("scale_input")}
    m = synth.build_module(sd, "fp8", dev, dim=DIM, fp8_matrix_mult=False, scale_input=False)
    xd = x.to(dev)
    y = m(xd)                                  # one call; its structures are kept
    seen = []
    hooks = [l.register_forward_hook(lambda mod, args, out: seen.append(args[0].shape[0]))
             for l in (m.experts[0].w2, m.shared_experts.w1)]
    z = m(xd)
    assert len(seen) == 2 and x.reshape(-1, DIM).shape[0] in seen
    for h in hooks:
        h.remove()
    hook = m.experts[1].register_forward_hook(lambda mod, args, out: seen.append(-1))
    m(xd)
    hook.remove()
    assert seen[-1] == -1
    assert torch.equal(m(xd), y) and float((z - y).float().norm() / y.float().norm()) <= 1e-3   # other order of fp32 sums


def test_a_scale_that_is_no_fp32_scalar_is_not_read_as_one():
    f = ffn()
    x = torch.zeros((1, DIM), dtype=torch.bfloat16)
    assert hidream._pack_ffn(f, x, hidream.HF.FP8_UPCAST, []) is not None
    for bad in (torch.ones((), dtype=torch.bfloat16), torch.ones(2)):
        f.w3.scale_weight = torch.nn.Parameter(bad, requires_grad=False)
        assert hidream._pack_ffn(f, x, hidream.HF.FP8_UPCAST, []) is None


def test_what_does_not_start_on_16_bytes_is_not_loaded_as_it_lies():
    """The kernel that multiplies stored fp8 weights in bf16 loads 16 bytes at a time into LDS; the conversion in front of the other
    kernels, which such Linears went through before, writes aligned copies."""
    f = ffn()
    x = torch.zeros((2, DIM), dtype=torch.bfloat16)
    odd = torch.zeros(DIM * DIM * 4 + 16, dtype=torch.uint8)[1:]
    w = odd[: f.w3.weight.numel()].view(FP8).view(f.w3.weight.shape)
    off = torch.zeros(2 * DIM + 8, dtype=torch.bfloat16)[1:2 * DIM + 1].view(2, DIM)
    assert ops._upcast_ready(f.w3, x) and hidream._pack_ffn(f, x, hidream.HF.FP8_UPCAST, []) is not None
    assert not ops._upcast_ready(f.w3, off) and hidream._pack_ffn(f, off, hidream.HF.FP8_UPCAST, []) is None
    f.w3.weight = torch.nn.Parameter(w, requires_grad=False)
    assert not ops._upcast_ready(f.w3, x) and hidream._pack_ffn(f, x, hidream.HF.FP8_UPCAST, []) is None
    # a copy is made of what is not contiguous
    assert hidream.HF.linear_upcast_aligned(off[:, ::2])
