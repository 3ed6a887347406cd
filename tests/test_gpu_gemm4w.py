"""The 4-wave 16-bit GEMM (csrc/gemm4w.h) behind the Linears: edges of its 256 x 256 tiles, the cut of tail tiles along K,
the activation hidden behind the next tile, fp8 weights multiplied in bf16.

Bounds: the kernel adds products in fp32 (K terms, each rounding at most 2^-24 of the running sum of magnitudes) and rounds
once to the 16-bit format (half a step: 2^-9 of the value in bf16, 2^-12 in fp16)."""
import pytest
import torch

from comfyui_amd import synth
from oracle import hidream_moe_oracle as O

pytestmark = pytest.mark.gpu
BF16, F16, FP8 = torch.bfloat16, torch.float16, torch.float8_e4m3fn
HALF_STEP = {BF16: 2.0 ** -8, F16: 2.0 ** -11}   # a step's width over the smallest value of a binade, halved, times 2 for slack


def reference(a, w, bias, scale=1.0):
    """float64 result and the bound on the fp32 sum of products."""
    r = a.double() @ w.double().t()
    mag = a.double().abs() @ w.double().abs().t()
    b = 0.0 if bias is None else bias.double()
    return r * scale + b, mag * abs(scale) * (a.shape[1] * 2.0 ** -24)


def within(y, ref, acc, dt):
    err = (y.double() - ref).abs()
    lim = acc + HALF_STEP[dt] * ref.abs() + 1e-7
    assert bool((err <= lim).all()), float((err / lim).max())


def planned(rows, N, K, code=0):
    """Parts that the tail tiles of one Linear are cut into."""
    from comfyui_amd import _lib
    mt = -(-rows // 256)
    return _lib.lib.hdmoe_tail_plan(code, mt * (N // 256), K, (mt * 256 - rows) * (N // 256), None, None)


@pytest.mark.parametrize("rows,N,K,parts", [
    (1, 256, 256, 1),          # one tile, two pairs of K steps, no middle pair: too short to be cut
    (255, 512, 384, 1),        # an odd number of pairs, the last row of a tile missing
    (257, 256, 2560, 10),      # one row in a second m-tile
    (700, 2560, 2560, 4),      # 30 tiles
    (1750, 10240, 2560, 5),    # 280 tiles: one whole round, 24 cut ones
    (2000, 10240, 512, 1),     # 320 tiles, the second round of 64 not cut
    (66000, 256, 256, 1),      # 258 tiles of two pairs
])
@pytest.mark.parametrize("dt", [BF16, F16])
def test_linear(dev, rows, N, K, parts, dt):
    from comfyui_amd import functional as HF
    assert planned(rows, N, K) == parts
    g = torch.Generator(device=dev).manual_seed(rows + K)
    a = torch.randn((rows, K), generator=g, device=dev).to(dt)
    w = (torch.randn((N, K), generator=g, device=dev) / K ** 0.5).to(dt)
    b = torch.randn(N, generator=g, device=dev).to(dt)
    for bias in (None, b):
        y = HF.linear(a, w, bias=bias)
        within(y, *reference(a, w, bias), dt)
        assert torch.equal(y, HF.linear(a, w, bias=bias))


@pytest.mark.parametrize("rows,N,K,parts", [
    (1, 256, 384, 1), (300, 512, 640, 1),
    (1000, 2560, 2560, 4),     # 40 tiles
    (1750, 10240, 2560, 5),    # one whole round, 24 cut tiles
    (4480, 2560, 2560, 1), (513, 1024, 4096, 8),
])
def test_fp8_weight_in_bf16(dev, rows, N, K, parts):
    from comfyui_amd import functional as HF
    assert planned(rows, N, K, 3) == parts
    g = torch.Generator(device=dev).manual_seed(rows + K)
    a = torch.randn((rows, K), generator=g, device=dev).to(BF16)
    w, s = synth.quantize_per_tensor(torch.randn((N, K), generator=g, device=dev) * 0.02)
    b = torch.randn(N, generator=g, device=dev).to(BF16)
    within(HF.linear_upcast(a, w, s, b), *reference(a, w, b, float(s.to(BF16))), BF16)
    within(HF.linear_upcast(a, w), *reference(a, w, None), BF16)


@pytest.mark.parametrize("rows,N,K", [(16, 2560, 2560), (4480, 2560, 2560), (7000, 2560, 4096)])
def test_scale_on_the_sum_is_no_further_from_64_bits(dev, rows, N, K):
    """Against the product with the unrounded scale in 64 bits: scaling the fp32 sum, and scaling the smaller operand first (rounded to
    bf16) with the sum itself exact."""
    from comfyui_amd import functional as HF
    g = torch.Generator(device=dev).manual_seed(rows)
    a = torch.randn((rows, K), generator=g, device=dev).to(BF16)
    w, s = synth.quantize_per_tensor(torch.randn((N, K), generator=g, device=dev) * 0.02)
    true = a.double() @ (w.double() * s.double()).t()
    sb = s.to(BF16)
    first = (a.double() @ (w.to(BF16) * sb).double().t()) if N < rows else ((a * sb).double() @ w.double().t())
    far = lambda y: float((y.double() - true).norm() / true.norm())
    assert far(HF.linear_upcast(a, w, s)) <= far(first.to(BF16))


@pytest.mark.parametrize("rows", [700, 3000])     # cut tiles (their biases are read by the second kernel), whole ones
@pytest.mark.parametrize("dt", [BF16, F16])
def test_bias_that_starts_anywhere(dev, rows, dt):
    from comfyui_amd import functional as HF
    g = torch.Generator(device=dev).manual_seed(rows)
    a = torch.randn((rows, 2560), generator=g, device=dev).to(dt)
    w = (torch.randn((2560, 2560), generator=g, device=dev) * 0.02).to(dt)
    store = torch.randn(2560 + 8, generator=g, device=dev).to(dt)
    for at in (1, 2, 4):
        b = store[at:at + 2560]
        within(HF.linear(a, w, bias=b), *reference(a, w, b), dt)
    if dt == BF16:
        w8, s = synth.quantize_per_tensor(w.float())
        assert torch.equal(HF.linear_upcast(a, w8, s, store[1:2561]), HF.linear_upcast(a, w8, s, store[1:2561].clone()))


def test_every_fp8_code_becomes_its_bf16_value(dev):
    """Each of the 256 codes at every place of a row's first eight (the places that one conversion handles)."""
    from comfyui_amd import functional as HF
    codes = torch.arange(256, dtype=torch.uint8, device=dev).view(FP8)
    a = torch.zeros((8, 384), dtype=BF16, device=dev)
    a[torch.arange(8), torch.arange(8)] = 1.0
    for at in range(8):
        w = torch.zeros((256, 384), device=dev).to(FP8)
        w.view(torch.uint8)[:, at] = codes.view(torch.uint8)
        y = HF.linear_upcast(a, w)[at]
        want = codes.to(BF16)
        assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.equal(torch.nan_to_num(y), torch.nan_to_num(want))


@pytest.mark.parametrize("T,E,K,N", [
    (40, 8, 2048, 256),      # a few rows per expert: every tile cut
    (1500, 8, 2048, 4096),   # ragged segments, one or two whole tiles per block: activation deferred, hidden or drained
    (700, 5, 512, 1024),     # K too short to hide the activation behind
    (3000, 4, 2176, 2048),   # 17 pairs: one more than the deferred activation takes
])
@pytest.mark.parametrize("dt", [BF16, F16])
def test_experts_with_gelu(dev, T, E, K, N, dt):
    from comfyui_amd import functional as HF
    g = torch.Generator(device=dev).manual_seed(T + N)
    x = torch.randn((T, K), generator=g, device=dev).to(dt)
    ws = [((torch.randn((N, K), generator=g, device=dev) / K ** 0.5).to(dt), (torch.randn(N, generator=g, device=dev) * 0.3).to(dt))
          for _ in range(E + 1)]
    ws[1] = (ws[1][0], None)
    idx, _ = HF.gate_top2(x, (torch.randn((E, K), generator=g, device=dev) / K ** 0.5).to(dt))
    _, offsets, perm, _ = HF.dispatch(idx, E)
    rows = x[(perm // 2).long()].contiguous()
    y, ys = HF.grouped_linear_tokens(x, perm, offsets, ws[:E], shared=ws[E], act="gelu")
    y2, ys2 = HF.grouped_linear(rows, offsets, ws[:E], a_static=x, shared=ws[E], act="gelu")
    assert torch.equal(y, y2) and torch.equal(ys, ys2)          # gathered or not: the same tiles
    bounds = offsets.tolist()
    for out, a, (w, b) in [(y[lo:hi], rows[lo:hi], ws[e]) for e, (lo, hi) in enumerate(zip(bounds, bounds[1:]))] + [(ys, x, ws[E])]:
        h, acc = reference(a, w, b)
        # the sum is rounded, then its GELU (slope at most 1.13) is
        ref = torch.nn.functional.gelu(h)
        within(out, ref, 1.13 * (acc + HALF_STEP[dt] * h.abs()), dt)


@pytest.mark.parametrize("dt", [BF16, F16])
def test_gelu_of_special_values(dev, dt):
    """Infinities, NaN, the far tails and the largest values come out as 0.5 h (1 + erf(h / sqrt 2)) has them, from wherever a tile
    is activated: its first token block in the epilogue, the others behind the next tile's K loop, the last whole tile of a block
    without one, cut tiles in the kernel that adds the parts up."""
    from comfyui_amd import _lib
    from comfyui_amd import functional as HF
    K, N = 2048, 256
    tiles = 2 * 256 + 20                                          # 16 pairs of K steps: as many as the hidden activation takes
    assert _lib.lib.hdmoe_tail_plan(_lib.W_BF16, tiles, K, 0, None, None) > 1
    big = [60000.0] if dt == F16 else [60000.0, 1e30, 1.5e38, 1.8e38, 3.38e38]
    vals = [0.0, -0.0, 1.0, -1.0, 5.0, -5.0, 9.0, -9.0, float("inf"), float("-inf"), float("nan")] + big + [-v for v in big]
    a = torch.zeros((256 * tiles, K), dtype=dt, device=dev)
    w = torch.zeros((N, K), dtype=dt, device=dev)
    b = torch.tensor(vals, dtype=torch.float64).to(dt).repeat(N // len(vals) + 1)[:N].contiguous().to(dev)
    _, y = HF.grouped_linear(a[:0], None, [], a_static=a, shared=(w, b), act="gelu")
    want = 0.5 * b.double() * torch.special.erfc(b.double() * -0.5 ** 0.5)
    assert bool(torch.isnan(want[9])) and float(want[8]) == float("inf")
    assert bool((torch.isnan(y) == torch.isnan(want)).all())
    near = b.abs() < 8
    # the approximation is within 7e-7 of the value, so at most the next 16-bit number (fp16: also a subnormal one); in cut tiles
    # 1 + erf cancels: erff is good to an ulp or two of 1 (2^-24 each), times |h| / 2
    lim = 2 * HALF_STEP[dt] * want.abs() + 2.0 ** -24 * (dt == F16) + b.double().abs() * 2.0 ** -23
    assert bool(((y[:, near].double() - want[near]).abs() <= lim[near]).all())
    up, down = ~near & (b > 0), ~near & (b < 0) & ~torch.isinf(b)
    assert bool((y[:, up] == b[up]).all())
    assert bool(((y[:, down] <= 0) & (y[:, down].double() >= want[down] * (1 + 2 * HALF_STEP[dt]))).all())


@pytest.mark.parametrize("tokens", [1, 70, 300, 900, 2100])
def test_layer_without_fp8_matrix_multiply(dev, tokens):
    """The one-call layer on fp8 weights and bf16 arithmetic against the composition of its Linears (their own forward,
    checked above), and against the oracle."""
    from comfyui_amd import functional as HF
    from tests.helpers import oracle_params, small_layer
    dim = 512
    sd, x = small_layer(seed=tokens, dim=dim, tokens=tokens, weights="fp8")
    sd = {k: v for k, v in sd.items() if not k.endswith("scale_input")}
    m = synth.build_module({k: v.to(dev) for k, v in sd.items()}, "fp8", dev, dim=dim, fp8_matrix_mult=False, scale_input=False)
    xd = x.to(dev)
    x2 = xd.reshape(-1, dim)
    assert m._collect(x2) is not None
    y = m(xd)
    composed = m._forward_composed(x2, m.gate.weight).view_as(xd)
    d = O.error_metrics(y.cpu(), composed.cpu())
    assert d["rel_rms"] <= 1e-3, d      # a bf16 rounding here and there falls the other way
    idx, w, _, _ = O.gate_fixed_order(x.reshape(-1, dim), sd["gate.weight"])
    ref = O.moe_forward(x, oracle_params(sd, 4), "upcast", gate_result=(idx, w))
    d = O.error_metrics(y.cpu(), ref)
    assert d["rel_rms"] <= 1e-2, d
    f = m.experts[1]
    d = O.error_metrics(f(xd).cpu(), f.w2(HF.silu_mul(f.w1(xd), f.w3(xd))).cpu())
    assert d["rel_rms"] <= 1e-3, d


def ffn_reference(x, w1, w2, w3, s1, s2, s3):
    """The feed-forward's dataflow with 64-bit sums: one rounding of every scaled sum, of silu and of the product."""
    lin = lambda a, w, s: (a.double() @ w.double().t() * float(s.to(BF16))).to(BF16)
    h = (torch.nn.functional.silu(lin(x, w1, s1).double()).to(BF16).double() * lin(x, w3, s3).double()).to(BF16)
    return lin(h, w2, s2)


def dequant_weights(dev, seed, D, H):
    """w1, w2, w3 and scales that are far apart (a mixed-up pair is off by a factor)."""
    g = torch.Generator(device=dev).manual_seed(seed)
    out = [synth.quantize_per_tensor(torch.randn(s, generator=g, device=dev) * 0.02) for s in ((H, D), (D, H), (H, D))]
    return [w for w, _ in out], [s * f for (_, s), f in zip(out, (1.0, 0.7, 2.9))]


def test_dense_feed_forward_without_fp8_matrix_multiply_with_cut_tiles(dev):
    """6000 rows at the model's width: 1296 gate/up tiles, the 16 left over cut along K and finished by the kernel that adds up."""
    from comfyui_amd import _lib
    from comfyui_amd import functional as HF
    D, H = synth.DIM, synth.H_ROUTED
    assert _lib.lib.hdmoe_tail_plan(_lib.W_E4M3FN_UPCAST, 24 * 54, D, 144 * 54, None, None) > 1
    ws, ss = dequant_weights(dev, 1, D, H)
    x = torch.randn((6000, D), generator=torch.Generator(device=dev).manual_seed(2), device=dev).to(BF16)
    y = HF.ffn_swiglu(x, HF.make_ffn_weights(*ws, dict(zip(("scale_w1", "scale_w2", "scale_w3"), ss))), H, HF.FP8_UPCAST)
    ref = ffn_reference(x, *ws, *ss)
    for lo in (0, 3000, 5800):          # the last rows lie in the cut tiles
        d = O.error_metrics(y[lo:lo + 200].cpu(), ref[lo:lo + 200].cpu())
        assert d["rel_rms"] <= 1e-3 and d["max_over_rms"] <= 0.05, (lo, d)     # a bf16 rounding here and there falls the other way


def test_layer_without_fp8_matrix_multiply_with_cut_tiles(dev):
    """960 tokens at the model's width: two m-tiles per expert and four of the shared one, 544 gate/up tiles, the last 32 (of the shared
    expert) cut in 4."""
    from comfyui_amd import _lib
    from comfyui_amd import functional as HF
    D, H, Hs, E, T = synth.DIM, synth.H_ROUTED, synth.H_SHARED, 4, 960
    assert _lib.lib.hdmoe_tail_plan(_lib.W_E4M3FN_UPCAST, 544, D, 0, None, None) == 4
    g = torch.Generator(device=dev).manual_seed(3)
    parts = [dequant_weights(dev, 10 + e, D, H if e < E else Hs) for e in range(E + 1)]
    fw = [HF.make_ffn_weights(*ws, dict(zip(("scale_w1", "scale_w2", "scale_w3"), ss))) for ws, ss in parts]
    x = torch.randn((T, D), generator=g, device=dev).to(BF16)
    gate = (torch.randn((E, D), generator=g, device=dev) / D ** 0.5).to(BF16)
    y, idx, w = HF.moe_ffn(x, gate, fw[:E], fw[E], H, Hs, HF.FP8_UPCAST, want_routing=True)
    counts = torch.bincount(idx.flatten().long(), minlength=E)
    assert bool(((counts > 256) & (counts <= 512)).all()), counts
    terms = torch.zeros((T, 2, D), device=dev, dtype=BF16)
    for e in range(E):
        t, slot = (idx == e).nonzero(as_tuple=True)
        terms[t, slot] = ffn_reference(x[t], *parts[e][0], *parts[e][1])
    terms = (terms * w.view(T, 2, 1)).to(BF16)
    ref = (terms[:, 0] + terms[:, 1]) + ffn_reference(x, *parts[E][0], *parts[E][1])
    d = O.error_metrics(y.cpu(), ref.cpu())
    assert d["rel_rms"] <= 1e-3 and d["max_over_rms"] <= 0.05, d


@pytest.mark.parametrize("tokens", [
    77_700,    # routed rows of hidden 6912 (their h is the largest operand) just above 2 GiB
    155_400,   # above 4 GiB: more than one call takes, composed per expert
])
def test_layer_without_fp8_matrix_multiply_of_many_tokens(dev, tokens):
    """fp8 weights multiplied in bf16, up to where an expert's rows fit the Linears. A token's output is that of a small batch
    but for the order of fp32 sums (the K cut goes by the batch)."""
    from comfyui_amd import functional as HF
    dim, hidden_arg = 512, 10240
    sd = synth.to_state_dict(synth.make_weights(5, dim=dim, hidden_arg=hidden_arg, device=dev)[0], "fp8", scale_input=False)
    m = synth.build_module(sd, "fp8", dev, dim=dim, hidden_arg=hidden_arg, fp8_matrix_mult=False, scale_input=False)
    assert m.experts[0].w1.weight.shape[0] == 6912
    assert HF.moe_ffn_rows_fit(tokens, dim, 6912, 3584) == (tokens < 100_000)
    x = torch.randn((1, tokens, dim), generator=torch.Generator(device=dev).manual_seed(5), device=dev).to(BF16)
    with torch.no_grad():
        y = m(x)
        for lo in (0, tokens // 2, tokens - 300):
            d = O.error_metrics(y[:, lo:lo + 300].cpu(), m(x[:, lo:lo + 300].contiguous()).cpu())
            assert d["rel_rms"] <= 1e-3, (lo, d)     # a bf16 rounding here and there falls the other way


def test_dense_feed_forward_without_fp8_matrix_multiply_of_many_rows(dev):
    """155 400 rows: h of hidden 6912 just above 2 GiB."""
    from comfyui_amd import functional as HF
    g = torch.Generator(device=dev).manual_seed(6)
    ws, scales = [], {}
    for name, shape in (("1", (6912, 512)), ("2", (512, 6912)), ("3", (6912, 512))):
        w, s = synth.quantize_per_tensor(torch.randn(shape, generator=g, device=dev) * 0.02)
        ws.append(w)
        scales["scale_w" + name] = s
    fw = HF.make_ffn_weights(*ws, scales)
    x = torch.randn((155_400, 512), generator=g, device=dev).to(BF16)
    y = HF.ffn_swiglu(x, fw, 6912, HF.FP8_UPCAST)
    for lo in (0, 155_100):
        d = O.error_metrics(y[lo:lo + 300].cpu(), HF.ffn_swiglu(x[lo:lo + 300].contiguous(), fw, 6912, HF.FP8_UPCAST).cpu())
        assert d["rel_rms"] <= 1e-3, (lo, d)


@pytest.mark.parametrize("dt", [BF16, F16])
def test_graph_replays_with_cut_tiles_and_hidden_activation(dev, dt):
    """Experts with GELU (deferred, drained and cut tiles) and a second Linear with cut tiles, captured once and replayed on new inputs
    in place, with the same calls made eagerly on other data in between."""
    from comfyui_amd import functional as HF
    T, E, D, H = 3000, 8, 2048, 4096
    g = torch.Generator(device=dev).manual_seed(9)
    rnd = lambda *s: (torch.randn(s, generator=g, device=dev) / s[-1] ** 0.5).to(dt)
    first, second = [(rnd(H, D), rnd(H)) for _ in range(E + 1)], [(rnd(D, H), rnd(D)) for _ in range(E + 1)]
    gate = rnd(E, D)

    def block(x):
        idx, _ = HF.gate_top2(x, gate)
        _, offsets, perm, _ = HF.dispatch(idx, E)
        h, hs = HF.grouped_linear_tokens(x, perm, offsets, first[:E], shared=first[E], act="gelu")
        return HF.grouped_linear(h, offsets, second[:E], a_static=hs, shared=second[E])
    xs = [torch.randn((T, D), generator=g, device=dev).to(dt) for _ in range(4)]
    want = [block(x) for x in xs]
    x = xs[0].clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        block(x)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            out = block(x)
    torch.cuda.current_stream().wait_stream(s)
    for i in (1, 2, 3, 0, 2):
        x.copy_(xs[i])
        graph.replay()
        torch.cuda.synchronize()
        other = block(xs[(i + 1) % 4])
        assert all(torch.equal(a, b) for a, b in zip(out, want[i])) and all(torch.equal(a, b) for a, b in zip(other, want[(i + 1) % 4]))
