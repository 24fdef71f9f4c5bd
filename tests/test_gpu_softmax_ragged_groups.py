"""Softmax rows of two and three chunks per lane in lane groups: lengths on both
sides of every change of the group that depends on the type, the mask or the
pass, ragged and whole chunks, through the checks (and tolerances) of the other
ragged rows."""
import pytest
import torch

from test_gpu_softmax import test_masked as check_masked
from test_gpu_softmax_bias import test_bias_softmax as check_bias
from test_gpu_softmax_bias import test_bias_softmax_dropout as check_bias_dropout
from test_gpu_softmax_causal_masked import test_causal_masked as check_causal_masked
from test_gpu_softmax_dropout import test_causal_dropout as check_causal_dropout
from test_gpu_softmax_dropout import test_masked_dropout as check_masked_dropout
from test_gpu_softmax import test_causal as check_causal
from test_gpu_softmax_ragged import BF16, F16, F32
from test_gpu_softmax_ragged import test_hidden_keys_held_twice as check_held_twice
from test_gpu_softmax_ragged import test_lengths as check_length
from test_gpu_softmax_ragged import test_the_sign_of_a_zero_held_twice as check_zero_held_twice
from helpers import randn
from oslo_amd.torch import _C

pytestmark = pytest.mark.gpu

# chunks: the most that a group takes in some type, mask or pass
EDGES = [9, 10, 12, 17, 18, 19, 25, 28, 33, 36, 40, 44, 50, 63]
LENGTHS = [(d, n * e + r) for d, e in ((BF16, 8), (F16, 8), (F32, 4)) for n in EDGES for r in (-1, 1)]


@pytest.mark.parametrize("dtype,sk", LENGTHS)
def test_lengths(device, dtype, sk):
    check_length(device, dtype, sk)


@pytest.mark.parametrize("chunks", [9, 10, 16, 17, 20, 21, 33, 34, 44, 45, 49, 63])
@pytest.mark.parametrize("dtype", [BF16, F16, F32])
def test_whole_chunks(device, dtype, chunks):
    check_length(device, dtype, chunks * (4 if dtype == F32 else 8))


@pytest.mark.parametrize("dtype,sk", [c for c in LENGTHS if c[0] != F16])
def test_keys_held_twice(device, dtype, sk):
    check_held_twice(device, dtype, sk)
    check_zero_held_twice(device, dtype, sk)


@pytest.mark.parametrize("dtype,sk", [(BF16, n) for n in (85, 133, 149, 251, 301, 389)] + [(F32, n) for n in (37, 79, 131, 171, 253)])
def test_rounds_of_workgroups(device, dtype, sk):
    """Enough rows that the launch limits the waves on a CU and that the last
    workgroup is partly empty: the rows are those of a launch of few."""
    k = _C.get_softmax_kernel()
    per, b = 61, 1 + (1 << 19) // (61 * 32)
    x = randn((1, per, sk), dtype, 5).to(device)
    xs = x.expand(b, per, sk).contiguous()
    y = k.fused_scaled_upper_triang_masked_softmax_forward(xs, 0.5)
    assert torch.equal(y, k.fused_scaled_upper_triang_masked_softmax_forward(x, 0.5).expand_as(y))
    dx = k.fused_scaled_upper_triang_masked_softmax_backward(xs, y, 0.5)
    assert torch.equal(dx, dx[:1].expand_as(dx))
    _, stats = k.softmax_dropout_forward(xs, None, 0.5, 0.0, 5, 8)
    _, first = k.softmax_dropout_forward(x, None, 0.5, 0.0, 5, 8)
    assert torch.equal(stats.view(b, per, 2), first.view(1, per, 2).expand(b, per, 2))
    dd = k.softmax_dropout_backward(xs, xs, stats, None, 0.5, 0.0, 5, 8)
    assert torch.equal(dd, dd[:1].expand_as(dd))


@pytest.mark.parametrize("dtype,sk", [(d, n) for d in (BF16, F16) for n in (71, 199, 257)] + [(F32, n) for n in (35, 99, 129)])
def test_a_term_shared_by_the_batch(device, dtype, sk):
    """... keeps other groups."""
    check_bias(device, 3, 2, 9, sk, dtype, 0.25, "t5", False)
    check_bias_dropout(device, 3, 2, 9, sk, dtype, 0.25, "t5", False, 0.1)


@pytest.mark.parametrize("dtype", [BF16, F16])
def test_two_row_sets_of_one_chunk(device, dtype):
    """25 whole chunks, one per lane of 32, and two row sets to a wave."""
    _C.tune("softmax_rows_per_wave", 2)
    try:
        check_causal(device, 2, 7, 200, dtype, 0.25)
        check_causal_dropout(device, 2, 7, 200, dtype, 0.25, 0.1)
        check_masked(device, 2, 2, 7, 200, dtype, 0.25, "padding")
        check_masked_dropout(device, 2, 2, 7, 200, dtype, 0.25, "full", 0.1)
        check_bias(device, 2, 2, 7, 200, dtype, 0.25, "t5", False)
        check_bias_dropout(device, 2, 2, 7, 200, dtype, 0.25, "perq", True, 0.1)
        check_causal_masked(device, 2, 2, 7, 200, dtype, 0.25, "holes")
    finally:
        _C.tune("softmax_rows_per_wave", 0)
