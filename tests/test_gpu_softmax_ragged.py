"""Softmax rows whose length is no multiple of a 16-byte chunk, or whose
operands lie off the 16-byte grid: the last chunk of a row overlaps the one
before it, and a chunk straddles two dropout groups.  Lengths on both sides of
every change of the lane groups and wave counts, all four masks, with and
without dropout, against the float64 oracle through the checks (and tolerances)
of the per-op test files."""
import pytest
import torch

from helpers import check, f64, randn
from oracle import closed_form as cf
from oslo_amd.torch import _C
from test_gpu_softmax import test_causal as check_causal
from test_gpu_softmax import test_masked as check_masked
from test_gpu_softmax_bias import test_bias_softmax as check_bias
from test_gpu_softmax_bias import test_bias_softmax_dropout as check_bias_dropout
from test_gpu_softmax_causal_masked import test_causal_masked as check_causal_masked
from test_gpu_softmax_dropout import test_causal_dropout as check_causal_dropout
from test_gpu_softmax_dropout import test_masked_dropout as check_masked_dropout

pytestmark = pytest.mark.gpu

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16

# chunks of a row: the largest number that each lane group or wave count holds
EDGES = [1, 8, 16, 24, 32, 48, 64, 96, 128, 192, 256, 512, 1024]


def _lengths(dtype):
    e = 4 if dtype == F32 else 8
    out = [1, e - 1]                                 # shorter than a chunk
    for n in EDGES:
        out += [n * e - 1, n * e + 1]                # the row's last chunk almost full, almost empty
    out += [5 * e + e // 2, 4096 * e + 1]            # half full; beyond sixteen waves
    return sorted(set(out))


@pytest.mark.parametrize("dtype,sk", [(d, n) for d in (BF16, F32) for n in _lengths(d)] +
                         [(F16, n) for n in (7, 63, 381, 1003, 2049)])
def test_lengths(device, dtype, sk):
    sq = min(sk, 7 if sk < 5000 else 3)
    check_causal(device, 2, sq, sk, dtype, 0.25)
    check_causal_dropout(device, 2, sq, sk, dtype, 0.25, 0.1)
    check_masked(device, 2, 2, sq, sk, dtype, 0.25, "padding")
    check_masked_dropout(device, 2, 2, sq, sk, dtype, 0.25, "full", 0.1)
    check_bias(device, 2, 2, sq, sk, dtype, 0.25, "t5", False)
    check_bias_dropout(device, 2, 2, sq, sk, dtype, 0.25, "perq", True, 0.1)
    check_causal_masked(device, 2, 2, sq, sk, dtype, 0.25, "holes")


@pytest.mark.parametrize("dtype", [F32, F16, BF16])
@pytest.mark.parametrize("sk", [64, 333, 2048])
def test_operands_off_the_vector_grid(device, dtype, sk):
    """Every operand one element past a 16-byte boundary, whole and odd rows."""
    ab, sq, scale = 3, 9, 0.5
    x, g = randn((ab, sq, sk), dtype, 1), randn((ab, sq, sk), dtype, 2)

    def shifted(t):
        flat = torch.empty(t.numel() + 1, dtype=dtype, device=device)
        flat[1:].copy_(t.reshape(-1))
        return flat[1:].view(t.shape)

    lib = _C.load_library()
    code = {F32: 0, F16: 1, BF16: 2}[dtype]
    st = torch.cuda.current_stream().cuda_stream
    xd, gd = shifted(x), shifted(g)
    y, dx = shifted(torch.zeros_like(x)), shifted(torch.zeros_like(x))
    assert lib.oslo_softmax_causal_fwd(xd.data_ptr(), y.data_ptr(), ab, sq, sk, scale, code, st) == 0
    assert lib.oslo_softmax_causal_bwd(gd.data_ptr(), y.data_ptr(), dx.data_ptr(), ab, sq, sk, scale, code, st) == 0
    check(y, cf.softmax_causal_fwd(f64(x), scale), "causal fwd", atol=1e-9)
    check(dx, cf.softmax_bwd(f64(g), f64(y), scale), "causal bwd", atol=1e-7)


@pytest.mark.parametrize("sk", [77, 1531])
def test_backward_in_place(device, sk):
    """The input gradient may overwrite the incoming gradient: the chunk that
    overlaps its neighbour is read before either is stored."""
    x, g = randn((2, 33, sk), BF16, 3), randn((2, 33, sk), BF16, 4)
    k = _C.get_softmax_kernel()
    y = k.fused_scaled_upper_triang_masked_softmax_forward(x.to(device), 0.5)
    want = k.fused_scaled_upper_triang_masked_softmax_backward(g.to(device), y, 0.5)
    gd = g.to(device)
    got = k.fused_scaled_upper_triang_masked_softmax_backward(gd, y, 0.5, inplace=True)
    assert got.data_ptr() == gd.data_ptr() and torch.equal(got, want)
    _, stats = k.softmax_dropout_forward(x.to(device), None, 0.5, 0.1, 9, 8)
    want = k.softmax_dropout_backward(g.to(device), x.to(device), stats, None, 0.5, 0.1, 9, 8)
    got = k.softmax_dropout_backward(g.to(device), x.to(device), stats, None, 0.5, 0.1, 9, 8, inplace=True)
    assert torch.equal(got, want)
