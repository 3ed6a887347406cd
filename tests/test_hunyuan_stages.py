"""What hunyuan3d.FeedForward offers of its Linears: its methods, a module list with more than its three modules, modules with methods of their own."""
import torch

from comfyui_amd import hunyuan3d

BF16 = torch.bfloat16


def feed_forward(cls=hunyuan3d.FeedForward):
    return cls(64, inner_dim=128, dtype=BF16).eval()


def same(a, b):
    return all(p is q for pair, other in zip(a, b) for p, q in zip(pair, other))


def test_methods():
    f, x = feed_forward(), torch.zeros((2, 64), dtype=BF16)
    want = (f.net[0].proj.weight, f.net[0].proj.bias), (f.net[2].weight, f.net[2].bias)
    assert same(f.stage_weights(), want) and same(f.stages(x), want) and f.fusable(x)
    assert f.stages(x.half()) is None and not f.fusable(x.half())


def test_a_further_module_in_the_list():
    f, x = feed_forward(), torch.zeros((2, 64), dtype=BF16)
    f.net.append(torch.nn.Identity())
    assert f.fusable(x) and same(f.stages(x), f.stage_weights())


def test_modules_with_methods_of_their_own():
    class Never(hunyuan3d.FeedForward):
        def fusable(self, x):
            return False

    x = torch.zeros((2, 64), dtype=BF16)
    assert hunyuan3d._stages(feed_forward(Never), x) is None
    f = feed_forward()
    assert same(hunyuan3d._stages(f, x), f.stage_weights())
    f.fusable = lambda x: False
    assert hunyuan3d._stages(f, x) is None
