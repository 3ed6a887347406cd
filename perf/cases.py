"""The measured workloads of this package: what a program that uses it has it do, through its public entry points.

A case is a dict of plain values. `listed()` names the fixed ones, `draw(rng)` makes further ones of the same ranges,
`prepare` builds what the caller's program holds before the call (modules with loaded weights, activations on the
device), `run` makes one pass, `work` says what the pass cannot do without and `tolerance` how far another correct
implementation of the same precision may be from it.

The paths ("path" of a case):

  layer     hidream.MOEFeedForwardSwiGLU.forward, one layer of the model (width 2560, 4 routed experts of hidden 6912,
            top-2, shared expert of hidden 3584) on [batch, tokens, width] activations
  branch    the same module's forward_branch: the feed-forward branch of a transformer block (LayerNorm, modulation,
            layer, gate, residual), which is how the blocks use the layer
  text      hidream.FeedForwardSwiGLU.forward_branch: the dense feed-forward branch of the text stream
  linear    the Linear of an operation class with a bias on its own (the attention projections of a scaled-fp8 model)
  gelu_moe  hunyuan3d.MoEBlock.forward (width 2048, 8 GELU experts of hidden 8192, top-2, shared expert)
  patch     Linear.set_weight of a scaled-fp8 class: a patched weight goes back to fp8 by stochastic rounding

How the weights are kept ("weights" of a case):

  fp8       scaled fp8 with fp8 matrix multiply (optimisations on); "scales": "ones" = every scale_input 1.0,
            "calibrated" = every Linear has its own value, w1 and w3 of a feed-forward the same one
  clamp     fp8 without scales and with fp8 matrix multiply (fp8_ops): activations are clamped to the fp8 range
  dequant   scaled fp8 without fp8 matrix multiply, the default policy for such a checkpoint: bf16 arithmetic
  bf16, fp16
"""
import math

import torch

from comfyui_amd import hidream, hunyuan3d, ops, synth

BF16 = torch.bfloat16
FP8 = torch.float8_e4m3fn
DIM, H_ROUTED, H_SHARED, EXPERTS = synth.DIM, synth.H_ROUTED, synth.H_SHARED, synth.NUM_EXPERTS
GELU_DIM, GELU_HIDDEN, GELU_EXPERTS = 2048, 8192, 8


def listed():
    return [
        # the smallest calls (a thumbnail preview): weights have to be read for a few tokens, and five launches made
        dict(name="layer-fp8-64", path="layer", weights="fp8", scales="ones", batch=1, tokens=64, skew=False, outliers=False),
        # a 256 x 256 image, most tokens on one expert, exact ties between two others
        dict(name="layer-fp8-256-skew", path="layer", weights="fp8", scales="ones", batch=1, tokens=256, skew=True, outliers=False),
        # a 512 x 512 image with bf16 weights
        dict(name="layer-bf16-1024", path="layer", weights="bf16", scales="ones", batch=1, tokens=1024, skew=False, outliers=False),
        # a 1024 x 1024 image, every Linear with its own scale_input
        dict(name="layer-fp8-4096", path="layer", weights="fp8", scales="calibrated", batch=1, tokens=4096, skew=False, outliers=False),
        # the headline: a 1024 x 1024 image with classifier-free guidance, outlier channels
        dict(name="layer-fp8-8192", path="layer", weights="fp8", scales="ones", batch=2, tokens=4096, skew=False, outliers=True),
        # a block's whole feed-forward branch at the largest batch
        dict(name="branch-fp8-32768", path="branch", weights="fp8", scales="ones", batch=2, tokens=16384, skew=False, outliers=False),
        # a 1360 x 768 image with the default policy for a scaled-fp8 checkpoint (bf16 arithmetic on fp8 weights)
        dict(name="layer-dequant-4080", path="layer", weights="dequant", scales="none", batch=1, tokens=4080, skew=False, outliers=False),
        # the text stream: a few hundred tokens of two prompts
        dict(name="text-fp8-768", path="text", weights="fp8", scales="ones", batch=2, tokens=384),
        # an attention projection over image and text tokens together
        dict(name="linear-fp8-4480", path="linear", weights="fp8", scales="calibrated", batch=1, tokens=4480, k=2560, n=2560),
        # the sibling model's block, in the type it runs in by default, at two times 4096 latent tokens
        dict(name="gelu-moe-fp16-8192", path="gelu_moe", weights="fp16", batch=2, tokens=4096),
        # and in bf16 on a small ragged batch
        dict(name="gelu-moe-bf16-1500", path="gelu_moe", weights="bf16", batch=1, tokens=1500),
        # a patched expert weight going back to fp8 (done for every Linear when a patch is applied to a model)
        dict(name="patch-f32-6912x2560", path="patch", weights="fp32", n=6912, k=2560),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["layer", "layer", "layer", "layer", "branch", "text", "linear", "linear", "gelu_moe", "gelu_moe", "patch"])
    batch = rng.choice([1, 1, 2])
    if path in ("layer", "branch"):
        weights = rng.choice(["fp8", "fp8", "clamp", "dequant", "bf16"])
        most = 16384 if weights in ("fp8", "clamp") else 8192
        return dict(path=path, weights=weights, scales=rng.choice(["ones", "calibrated"]) if weights == "fp8" else "none",
                    batch=batch, tokens=_log_int(rng, 32, most) // batch, skew=rng.random() < 0.25, outliers=rng.random() < 0.25)
    if path == "text":
        weights = rng.choice(["fp8", "fp8", "dequant", "bf16"])
        return dict(path=path, weights=weights, scales=rng.choice(["ones", "calibrated"]) if weights == "fp8" else "none",
                    batch=batch, tokens=_log_int(rng, 64, 1024))
    if path == "linear":
        weights = rng.choice(["fp8", "fp8", "clamp", "dequant", "bf16"])
        k, n = rng.choice([(DIM, DIM), (DIM, DIM), (DIM, 4 * DIM), (GELU_DIM, GELU_DIM), (4096, DIM)])
        return dict(path=path, weights=weights, scales="calibrated" if weights == "fp8" else "none", batch=batch,
                    tokens=_log_int(rng, 64, 9000) // batch, k=k, n=n)
    if path == "gelu_moe":
        return dict(path=path, weights=rng.choice(["fp16", "bf16"]), batch=batch, tokens=_log_int(rng, 128, 8192) // batch)
    n, k = rng.choice([(H_ROUTED, DIM), (DIM, H_ROUTED), (H_SHARED, DIM), (DIM, H_SHARED), (DIM, DIM), (4 * DIM, DIM)])
    return dict(path="patch", weights=rng.choice(["fp32", "fp32", "bf16"]), n=n, k=k + 8 * rng.randrange(8))


# ---- inputs -----------------------------------------------------------------------------------------------------


def _tokens(g, batch, tokens, width, dtype, outliers=False):
    """Activations behind a LayerNorm: N(0,1), optionally 1 % of the channels twenty times as large."""
    x = torch.randn((batch * tokens, width), generator=g, device="cuda")
    if outliers:
        x[:, torch.randperm(width, generator=g, device="cuda")[: width // 100]] *= 20.0
    return x.to(dtype).view(batch, tokens, width)


def _scale_input(g, case):
    """A stored scale_input: 1.0, or what a calibration run leaves, the largest activation (27 to 45 here, five times
    that with outlier channels) over 448."""
    if case["scales"] == "ones":
        return torch.ones((), device="cuda")
    return (torch.rand((), generator=g, device="cuda") * 0.04 + 0.06) * (5.0 if case.get("outliers") else 1.0)


def _weight(g, n, k, sigma=0.02):
    return torch.randn((n, k), generator=g, device="cuda") * sigma


def _fill_fp8(lin, w, kind, scale_input):
    """Store fp32 master weights in a Linear of an fp8 operation class, as loading a checkpoint leaves them."""
    if kind == "clamp":
        lin.weight = torch.nn.Parameter(w.to(FP8), requires_grad=False)
        return
    w8, s = synth.quantize_per_tensor(w)
    lin.weight = torch.nn.Parameter(w8, requires_grad=False)
    lin.scale_weight = torch.nn.Parameter(s, requires_grad=False)
    if kind == "fp8":
        lin.scale_input = torch.nn.Parameter(scale_input, requires_grad=False)


def _operations(weights):
    if weights == "fp8":
        return ops.scaled_fp8_ops(fp8_matrix_mult=True, scale_input=True, override_dtype=FP8)
    if weights == "dequant":
        return ops.scaled_fp8_ops(fp8_matrix_mult=False, scale_input=False, override_dtype=FP8)
    return ops.fp8_ops if weights == "clamp" else ops.disable_weight_init


def _fill_ffn(ffn, g, case):
    fp8 = case["weights"] == "fp8"
    s13 = _scale_input(g, case) if fp8 else None
    for name in ("w1", "w2", "w3"):
        lin = getattr(ffn, name)
        w = _weight(g, *lin.weight.shape)
        if case["weights"] == "bf16":
            lin.weight = torch.nn.Parameter(w.to(BF16), requires_grad=False)
        elif name == "w2":
            _fill_fp8(lin, w, case["weights"], _scale_input(g, case) if fp8 else None)
        else:   # w1 and w3 read the same activations
            _fill_fp8(lin, w, case["weights"], s13.clone() if fp8 else None)


def _moe_layer(g, case):
    m = hidream.MOEFeedForwardSwiGLU(DIM, 4 * DIM, EXPERTS, 2, dtype=FP8 if case["weights"] == "clamp" else BF16, device="cuda",
                                     operations=_operations(case["weights"]))
    for f in list(m.experts) + [m.shared_experts]:
        _fill_ffn(f, g, case)
    wg = _weight(g, EXPERTS, DIM, 1.0 / math.sqrt(DIM))
    if case["skew"]:
        wg[:, 0] = torch.tensor([0.1875, 0.0, 0.0, -3.0], device="cuda")
    m.gate.weight = torch.nn.Parameter(wg.to(BF16), requires_grad=False)
    return m.eval()


def _modulation(g, batch):
    return [(torch.randn((batch, 1, DIM), generator=g, device="cuda") * 0.3).to(BF16) for _ in range(3)]


@torch.no_grad()
def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    path = case["path"]
    if path in ("layer", "branch"):
        m = _moe_layer(g, case)
        x = _tokens(g, case["batch"], case["tokens"], DIM, BF16, case["outliers"])
        if case["skew"]:   # channel 0 carries the gate's bias; every 64th token is nothing else (experts 1 and 2 tie)
            x[..., 0] = 1.0
            x.view(-1, DIM)[::64, 1:] = 0.0
        return dict(path=path, module=m, x=x, mods=_modulation(g, case["batch"]) if path == "branch" else None)
    if path == "text":
        f = hidream.FeedForwardSwiGLU(DIM, 4 * DIM, dtype=BF16, device="cuda", operations=_operations(case["weights"]))
        _fill_ffn(f, g, case)
        return dict(path=path, module=f.eval(), x=_tokens(g, case["batch"], case["tokens"], DIM, BF16), mods=_modulation(g, case["batch"]))
    if path == "linear":
        kind = case["weights"]
        lin = _operations(kind).Linear(case["k"], case["n"], bias=True, dtype=FP8 if kind == "clamp" else BF16, device="cuda")
        w = _weight(g, case["n"], case["k"])
        if kind == "bf16":
            lin.weight = torch.nn.Parameter(w.to(BF16), requires_grad=False)
        else:
            _fill_fp8(lin, w, kind, _scale_input(g, case) if kind == "fp8" else None)
        lin.bias = torch.nn.Parameter((torch.randn(case["n"], generator=g, device="cuda") * 0.1).to(BF16), requires_grad=False)
        return dict(path=path, module=lin.eval(), x=_tokens(g, case["batch"], case["tokens"], case["k"], BF16))
    if path == "gelu_moe":
        dtype = torch.float16 if case["weights"] == "fp16" else BF16
        m = hunyuan3d.MoEBlock(GELU_DIM, num_experts=GELU_EXPERTS, moe_top_k=2, ff_inner_dim=GELU_HIDDEN, dtype=dtype, device="cuda")
        for p in m.parameters():
            p.copy_(_weight(g, 1, p.numel(), 1.0 / math.sqrt(p.shape[-1]) if p.dim() > 1 else 0.2).view(p.shape))
        return dict(path=path, module=m.eval(), x=_tokens(g, case["batch"], case["tokens"], GELU_DIM, dtype))
    if path == "patch":
        lin = _operations("fp8").Linear(case["k"], case["n"], bias=False, dtype=BF16, device="cuda")
        w = _weight(g, case["n"], case["k"])
        _fill_fp8(lin, w, "fp8", torch.ones((), device="cuda"))
        # the dequantised weight plus a low-rank update, which is what reaches set_weight
        up, down = _weight(g, case["n"], 16), _weight(g, 16, case["k"])
        patched = (w + up @ down).to(torch.float32 if case["weights"] == "fp32" else BF16)
        return dict(path=path, module=lin, x=patched, seed=seed & 0x7FFFFFFF)
    raise ValueError(path)


@torch.no_grad()
def run(state):
    m, x, path = state["module"], state["x"], state["path"]
    if path in ("branch", "text"):
        return m.forward_branch(x, *state["mods"])
    if path == "patch":
        m.set_weight(x, inplace_update=True, seed=state["seed"])
        return m.weight
    return m(x)


# ---- bounds -----------------------------------------------------------------------------------------------------


def work(case):
    path, weight_bytes = case["path"], {"bf16": 2, "fp16": 2}.get(case["weights"], 1)
    if path == "patch":
        return {"bytes": case["n"] * case["k"] * ({"fp32": 4, "bf16": 2}[case["weights"]] + 1), "flops": 0}
    rows = case["batch"] * case["tokens"]
    if path == "linear":
        k, n = case["k"], case["n"]
        return {"bytes": rows * (k + n) * 2 + n * k * weight_bytes + n * 2, "flops": 2 * rows * k * n}
    if path == "text":
        return {"bytes": rows * DIM * 4 + 3 * H_ROUTED * DIM * weight_bytes + 3 * case["batch"] * DIM * 2,
                "flops": 6 * rows * DIM * H_ROUTED}
    if path == "gelu_moe":
        return {"bytes": rows * GELU_DIM * 4 + (GELU_EXPERTS + 1) * (2 * GELU_DIM * GELU_HIDDEN + GELU_DIM + GELU_HIDDEN) * 2,
                "flops": rows * (3 * 4 * GELU_DIM * GELU_HIDDEN + 2 * GELU_DIM * GELU_EXPERTS)}
    return {"bytes": rows * DIM * 4 + 3 * DIM * (EXPERTS * H_ROUTED + H_SHARED) * weight_bytes + EXPERTS * DIM * 2
            + (3 * case["batch"] * DIM * 2 if path == "branch" else 0),
            "flops": rows * (6 * DIM * (2 * H_ROUTED + H_SHARED) + 2 * DIM * EXPERTS)}


def tolerance(case):
    """About four times the distance between the path and its dataflow in 64 bits, or with fp32 sums in another order
    (the figures in the comments: relative 2-norm, largest difference over the larger of the value and the rms)."""
    path, weights = case["path"], case["weights"]
    if path == "patch":
        return "exact"                          # the same draws give the same bytes
    if path == "linear":
        # one rounding to bf16 at the end (1.7e-3, 0.008); dequant rounds a scaled operand as well (3.0e-3, 0.011)
        return {"rel": 1.2e-2, "max": 0.05} if weights == "dequant" else {"rel": 6e-3, "max": 0.03}
    if weights in ("fp8", "clamp"):
        # a bf16 rounding of an intermediate that falls the other way moves an fp8 value by one step of 6 %
        # (2.4e-3 to 3.7e-3, 0.04 to 0.09)
        return {"rel": 1.2e-2, "max": 0.36}
    if weights == "fp16":
        return {"rel": 2e-3, "max": 0.012}      # 4.5e-4, 0.003
    if weights == "dequant":
        return {"rel": 2e-2, "max": 0.18}       # 5.8e-3, 0.046
    return {"rel": 1.6e-2, "max": 0.12}         # 3.6e-3 to 4.5e-3, 0.018 to 0.030
