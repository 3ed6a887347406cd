"""The row kernel of the gate at D = 2048 (csrc/gate.hip, KERNEL_ROUTE4): bit for bit what the fixed-order checker says, for every number
of experts it takes (experts 5 to 8 sit in a second register), both 16-bit types, fewer tokens than waves, exact ties."""
import pytest
import torch

from comfyui_amd import functional as HF
from oracle import hidream_moe_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,E", [(1, 2), (7, 5), (17, 8), (300, 3), (1500, 7), (2049, 6), (5000, 8), (64, 4), (33, 9)])
def test_gate_is_bit_exact(dev, dtype, T, E):
    g = torch.Generator().manual_seed(T + E)
    x = torch.randn((T, 2048), generator=g).to(dtype)
    wg = (torch.randn((E, 2048), generator=g) / 2048 ** 0.5).to(dtype)
    if T > 16:
        wg[E - 1] = wg[0]               # the last and the first expert tie on every token
        x[5] = 0.0                      # all experts tie
        x[9] = x[3] * 64.0              # a softmax with one expert left
    idx_ref, w_ref, _, _ = O.gate_fixed_order(x, wg)
    idx, w = HF.gate_top2(x.to(dev), wg.to(dev))
    assert torch.equal(idx.cpu(), idx_ref)
    assert torch.equal(w.cpu().view(torch.int16), w_ref.view(torch.int16))
