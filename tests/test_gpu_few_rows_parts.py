"""Layers of up to 256 tokens, whose down projection is cut along K by the sizes alone (csrc/gemm.hip, hdmoe_down_parts; five to three parts of the
experts' tiles, fewer of the shared expert's): the sums are those of whole tiles in another order, and a token's do not depend on the
routing of the others, also where all of them go to the same two experts."""
import pytest
import torch

from tests.test_gpu_two_lengths import layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["fp8", "upcast", "bf16"])
def test_cut_rows_against_whole_tiles(dev, kind):
    m, x = layer(dev, kind)
    m.batch_invariant = True
    with torch.no_grad():
        full = m(x[:, :2400]).float()   # whole tiles
        same_two = x[:, :1].expand(1, 256, x.shape[2])
        for tokens in (1, 16, 64, 128, 129, 200, 256):
            y = m(x[:, :tokens])
            # Intermediates are the same bytes (16-bit activations: or a rounding of a differently ordered sum apart), sums in another order move a
            # row of the down projection by a bf16 step of 2^-8 at most here and there: all of them together stay under that in the 2-norm.
            ref = full[:, :tokens]
            assert float((y.float() - ref).norm() / ref.norm()) < 2.0 ** -8, tokens
            if tokens > 1:
                half = tokens // 2
                z = m(torch.cat([x[:, :half], same_two[:, :tokens - half]], 1))
                assert torch.equal(z[:, :half], y[:, :half]), tokens
                assert torch.equal(z[:, half:], z[:, half:half + 1].expand_as(z[:, half:])), tokens
