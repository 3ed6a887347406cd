"""Gate/up on 16-bit activations with low tiles behind whole ones (csrc/gemm4w.h, tile_mix): a row's K steps are the same on a tile of any height, so
the intermediate is byte for byte that of a call whose tiles are all whole."""
import ctypes

import pytest
import torch

from comfyui_amd import _lib, synth
from comfyui_amd import functional as HF

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16
D, H, WHOLE = 512, 6912, 256 * 29   # 54 tiles along the features by 29: more than low tiles are looked for at


def weights(g, dev, code):
    ws, scales = [], {}
    for name, shape in (("1", (H, D)), ("2", (D, H)), ("3", (H, D))):
        w = torch.randn(shape, generator=g, device=dev) * 0.05
        if code == _lib.W_BF16:
            ws.append(w.to(BF16))
            continue
        w8, scales["scale_w" + name] = synth.quantize_per_tensor(w)
        ws.append(w8)
    return HF.make_ffn_weights(*ws, scales or None), ws, scales


@pytest.mark.parametrize("code", [_lib.W_BF16, _lib.W_E4M3FN_UPCAST])
def test_dense(dev, code):
    g = torch.Generator(device=dev).manual_seed(5)
    fw, *keep = weights(g, dev, code)
    x = torch.randn((WHOLE, D), generator=g, device=dev).to(BF16)

    def h(n):
        # (the least workspace that the call takes: no tile is cut along K)
        least = n * H * 2 + 256
        out = torch.empty((n, D), dtype=BF16, device=dev)
        for room in (least, _lib.lib.hdmoe_ffn_workspace_bytes(n, D, H, code)):
            work = torch.empty(room, dtype=torch.uint8, device=dev)
            if _lib.lib.hdmoe_ffn_swiglu(code, x.data_ptr(), n, D, H, ctypes.byref(fw), out.data_ptr(), work.data_ptr(), room,
                                         torch.cuda.current_stream().cuda_stream) == 0:
                return work[:n * H * 2].view(BF16).view(n, H)
        raise AssertionError(n)
    full = h(WHOLE)
    assert bool(torch.isfinite(full.float()).all()) and float(full.float().std()) > 0
    for rows in (129, 160, 256, 257, 384, 400, 512, 513, 641, 1000, 1300, 1500, 2000):
        part = h(rows)
        same = torch.equal(part, full[:rows])
        # a tile that is cut along K (where the parts' room comes with that of a cut down projection) ends on sums in another order
        err = (part.float() - full[:rows].float()).norm() / full[:rows].float().norm()
        assert same or float(err) < 2.0 ** -9, rows
    assert torch.equal(h(1300), full[:1300]) and torch.equal(h(2000), full[:2000])


@pytest.mark.parametrize("sizes", [(300, 1, 513), (260, 520, 0, 131), (700, 255)])
def test_experts(dev, sizes):
    """Segments of one call, each against a call of its own."""
    g = torch.Generator(device=dev).manual_seed(sum(sizes))
    sets = [weights(g, dev, _lib.W_BF16) for _ in sizes]
    a = torch.randn((sum(sizes), D), generator=g, device=dev).to(BF16)

    def run(rows, counts, members):
        offsets = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device=dev)
        arr = (_lib.FfnWeights * len(members))(*[sets[m][0] for m in members])
        out = torch.full((rows.shape[0] + 1, H), 7.0, dtype=BF16, device=dev)
        _lib.check(_lib.lib.hdmoe_grouped_swiglu(_lib.W_BF16, rows.data_ptr(), offsets.data_ptr(), rows.shape[0], len(members), D, H, arr, out.data_ptr(),
                                                 torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert bool((out[-1] == 7.0).all())
        return out[:-1]
    got, at = run(a, sizes, range(len(sizes))), 0
    for e, n in enumerate(sizes):
        if n > 128:   # (up to 128 rows alone run on another kernel)
            assert torch.equal(got[at:at + n], run(a[at:at + n].contiguous(), (n,), (e,))), (e, n)
        at += n
