"""fp8 layers whose down projection is cut in (2, 1) parts on tiles of 128, 160 and 256 tokens (csrc/tail_units.h, g4_cut_height): the parts are the
same, so a token's bytes are too, with three experts above 256 rows as well (a second round of 128-token tiles)."""
import pytest
import torch

from tests.test_gpu_two_lengths import layer

pytestmark = pytest.mark.gpu


def m_tiles(m, x, bm):
    top = (x[0].float() @ m.gate.weight.float().t()).topk(2).indices
    return sum(-(-int(c) // bm) for c in torch.bincount(top.reshape(-1), minlength=4))


def test_rows_in_tiles_of_other_heights(dev):
    m, _ = layer(dev, "fp8")
    m.gate.weight.data[0, :64] -= 0.02   # even
    g = torch.Generator(device=dev).manual_seed(11)
    tiles = set()
    with torch.no_grad():
        for _ in range(40):
            x = torch.randn((1, 640, m.gate.weight.shape[1]), generator=g, device=dev).to(torch.bfloat16)
            n = m_tiles(m, x[:, :512], 128)
            if n in tiles:
                continue
            tiles.add(n)
            full = m(x)
            assert bool(torch.isfinite(full.float()).all()) and float(full.float().std()) > 0
            for tokens in (475, 484, 500, 512, 530):
                assert torch.equal(m(x[:, :tokens]), full[:, :tokens]), (tokens, n)
    assert 11 in tiles and len(tiles) >= 2, tiles
