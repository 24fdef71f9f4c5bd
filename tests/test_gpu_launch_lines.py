"""The lines of the launch rules that row counts, the mask and the type move:
each side of them against the float64 oracle, through the checks (and
tolerances) of the per-op tests."""
import pytest
import torch

from helpers import check, f64, randn
from oracle import closed_form as cf
from oracle import philox
from oslo_amd.torch import _C
from test_gpu_norm import test_layer_norm as check_layer_norm
from test_gpu_norm import test_rms_norm as check_rms_norm
from test_gpu_residual_norm import test_fused_vs_oracle as check_fused
from test_gpu_softmax import test_masked as check_masked
from test_gpu_softmax_bias import test_bias_softmax as check_bias
from test_gpu_softmax_bias import test_bias_softmax_dropout as check_bias_dropout
from test_gpu_softmax_causal_masked import test_causal_masked as check_causal_masked

pytestmark = pytest.mark.gpu

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16


@pytest.mark.parametrize("sk", [132, 136, 140, 156, 172, 176, 180])
@pytest.mark.parametrize("sq", [1, 7])
def test_fp32_rows_with_a_term_in_two_row_sets(device, sq, sk):
    """34 to 44 chunks: two sets of rows to a wave, the last one partly empty."""
    check_bias(device, 3, 1, sq, sk, F32, 0.25, "t5", False)
    check_bias(device, 1, 3, sq, sk, F32, 0.25, "perq", True)
    check_bias_dropout(device, 3, 1, sq, sk, F32, 0.25, "t5", False, 0.1)


@pytest.mark.parametrize("sk", [121, 128, 129, 137, 143, 145, 329, 336, 337, 343, 345])
@pytest.mark.parametrize("dtype", [BF16, F16])
def test_backward_of_ragged_rows_without_a_diagonal(device, dtype, sk):
    """16, 18, 42 and 43 chunks, which rows under the diagonal hold otherwise."""
    check_masked(device, 2, 2, 9, sk, dtype, 0.25, "padding")
    check_causal_masked(device, 2, 2, 9, sk, dtype, 0.25, "padding")


@pytest.mark.parametrize("dtype,sk", [(F32, 97), (F32, 397), (F32, 1111), (BF16, 389), (BF16, 1003), (F16, 2049)])
def test_blocks_of_a_term_shared_by_the_batch(device, dtype, sk):
    """More than 64 blocks of ragged rows, in lane groups and in whole waves."""
    check_bias(device, 3, 2, 96, sk, dtype, 0.25, "t5", False)
    check_bias_dropout(device, 3, 2, 96, sk, dtype, 0.25, "t5", False, 0.1)


# rows of a whole workgroup, one and up to two of them to a CU, and beyond
@pytest.mark.parametrize("n1,n2,dtype", [
    (255, 6144, F32), (257, 6144, F32), (511, 8192, F32), (513, 8192, F32), (300, 12288, BF16), (515, 12288, BF16)])
def test_two_rows_to_a_workgroup(device, n1, n2, dtype):
    check_layer_norm(device, n1, n2, dtype, dtype, True)
    check_rms_norm(device, n1, n2, dtype, dtype, True)
    check_fused(device, n1, n2, dtype, 0.1, False)
    check_fused(device, n1, n2, dtype, 0.1, True)


# bias-dropout-add: steps that fill the finer slots, one too many, two each
@pytest.mark.parametrize("rows,cols,dtype", [
    (256, 5120, BF16), (258, 5120, BF16), (300, 6144, F16), (800, 5120, BF16), (1500, 5120, BF16), (1500, 5120, F32)])
def test_column_sums_of_a_few_steps(device, rows, cols, dtype):
    g = randn((rows, cols), dtype, rows + cols)
    dx, db = _C.get_fused_elementwise_kernel().bias_dropout_add_backward(g.to(device), 0.2, 9, 4)
    keep = torch.from_numpy(philox.keep_mask(rows * cols, 0.2, 9, 4)).view(rows, cols).bool()
    check(dx, cf.bias_dropout_add_bwd(f64(g), keep.numpy(), 0.2)[0], "dx", atol=1e-6)
    # (the sum of dx as stored, in float32: relative 2^-24 of each of `rows` terms of order one)
    check(db, dx.double().sum(0).cpu().numpy(), "dbias", atol=1e-5 * rows ** 0.5 + 1e-6, min_exact=0.97)
