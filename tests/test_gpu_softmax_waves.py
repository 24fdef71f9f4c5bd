"""The number of waves that a softmax launch keeps on a compute unit (an LDS
reservation next to the LDS the kernel itself uses, which holds the draws of
ragged rows with dropout) must not change a bit of the results."""
import pytest
import torch

from helpers import randn
from oslo_amd.torch import _C

pytestmark = pytest.mark.gpu


# (values that leave at least three workgroups of 1, 2, 1 and 6 waves on a compute
#  unit: below that a launch is not limited)
CASES = [(sk, dtype, waves)
         for sk, dtype, values in [(2048, torch.bfloat16, (3, 12, 20, 28)), (1531, torch.float16, (6, 12, 20, 28)),
                                   (260, torch.float32, (3, 12, 20, 28)), (4100, torch.bfloat16, (18, 24, 31))]
         for waves in values]


@pytest.mark.parametrize("sk,dtype,waves", CASES)
def test_waves_per_compute_unit_keep_the_bits(device, sk, dtype, waves):
    k = _C.get_softmax_kernel()
    x, g = randn((2, 37, sk), dtype, 1).to(device), randn((2, 37, sk), dtype, 2).to(device)

    def run():
        y = k.fused_scaled_upper_triang_masked_softmax_forward(x, 0.25)
        out, stats = k.softmax_dropout_forward(x, None, 0.25, 0.1, 5, 8)
        return (y, k.fused_scaled_upper_triang_masked_softmax_backward(g, y, 0.25), out, stats,
                k.softmax_dropout_backward(g, x, stats, None, 0.25, 0.1, 5, 8))

    want = run()
    _C.tune("softmax_waves_per_cu", waves)
    try:
        got = run()
    finally:
        _C.tune("softmax_waves_per_cu", 0)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
