"""The dispatch of up to 512 slots inside the gate/up contraction (csrc/gemm.hip, HdmoeRoute): the results that it leaves, at the numbers of
slots and experts where a wave or the block is just full."""
import pytest

from tests import test_gpu_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,E,T", [(256, 4, 31), (256, 4, 32), (256, 4, 33), (256, 2, 128), (256, 4, 255), (256, 4, 256), (256, 8, 256), (256, 16, 256),
                                     (2560, 4, 64), (2560, 4, 256)])
def test_dispatch(dev, dim, E, T):
    test_gpu_layer.test_layer_dispatch_from_gate_histograms(dev, "fp8", dim, E, T)
