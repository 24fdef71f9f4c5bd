"""The reductions inside a wavefront and the packed keep decisions, at the
sizes where they can go wrong: every lane-group size after every kind of
instruction that can produce the operand (a float16 dot product, an
exponential), and thresholds at both ends of their range."""
import numpy as np
import pytest
import torch

from helpers import check, f64, randn
from oracle import closed_form as cf
from oracle import philox
from oslo_amd.torch import _C

pytestmark = pytest.mark.gpu

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16


# thresholds 0 (keeps everything), 1, 2, 65535 and 65536 (keeps nothing)
@pytest.mark.parametrize("p", [1e-6, 1.0 / 65536, 2.0 / 65536, 65535.0 / 65536, 1.0 - 2.0 ** -24])
def test_keep_decisions_at_the_ends_of_the_threshold(device, p):
    got = _C.get_fused_elementwise_kernel().philox_mask(1 << 21, p, 4321, 12, device).cpu().numpy()
    assert np.array_equal(got, philox.keep_mask(1 << 21, p, 4321, 12))


# lanes that hold a row: 8, 16, 32, a wave, two waves; aligned and ragged rows
@pytest.mark.parametrize("sk", [8, 64, 61, 128, 124, 256, 251, 512, 509, 1024, 1021, 5120, 5117])
@pytest.mark.parametrize("dtype", [F16, BF16, F32])
def test_sums_and_maxima_of_every_lane_group(device, sk, dtype):
    k = _C.get_softmax_kernel()
    x = randn((3, 5, sk), dtype, seed=sk, std=4.0)
    g = randn((3, 5, sk), dtype, seed=sk + 1)
    # the maximum sits at another lane in every row
    for r in range(15):
        x.view(15, sk)[r, (r * 37 + 5) % sk] = 20.0
    none = torch.zeros(3, 1, 1, sk, dtype=torch.bool, device=device)
    y = k.fused_scaled_masked_softmax_forward(x.view(3, 1, 5, sk).to(device), none, 0.5)
    hidden = np.zeros((3, 5, sk), dtype=bool)
    check(y.view(3, 5, sk), cf.softmax_masked_fwd(f64(x), hidden, 0.5), "forward", atol=1e-9)
    # (no mask: the dense kernel, whose float16 sum is a chain of dot products)
    dx = k.fused_scaled_masked_softmax_backward(g.view(3, 1, 5, sk).to(device), y, 0.5)
    check(dx.view(3, 5, sk), cf.softmax_bwd(f64(g), f64(y.view(3, 5, sk)), 0.5), "backward", atol=2e-7)
