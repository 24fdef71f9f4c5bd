"""Column sums of the element-wise backwards with few rows: every tile width
(8 to 128 lanes), slots of one step, the change to slots of 16 rows at 128
partial rows, and a workspace that holds the coarse partial rows only."""
import pytest
import torch

from helpers import check, f64, randn
from oracle import closed_form as cf
from oracle import philox
from oslo_amd.torch import _C

pytestmark = pytest.mark.gpu

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16

SHAPES = [(rows, cols, dtype) for cols, dtype in (
    (8, F16), (64, BF16), (120, F16), (256, BF16), (448, F16), (768, BF16), (1000, BF16), (2048, F16),
    (4, F32), (100, F32), (768, F32), (1024, F32)) for rows in (1, 2, 17, 255, 257)]
SHAPES += [(2047, 768, BF16), (2049, 768, F16), (300, 4096, BF16), (1025, 1024, F32)]


@pytest.mark.parametrize("rows,cols,dtype", SHAPES)
def test_column_sums(device, rows, cols, dtype):
    x, g = randn((rows, cols), dtype, rows + cols), randn((rows, cols), dtype, rows + cols + 1)
    b = randn((cols,), dtype, 5, std=0.3)
    k = _C.get_fused_elementwise_kernel()
    dx, db = k.bias_gelu_backward(g.to(device), x.to(device), b.to(device))
    check(dx, cf.bias_gelu_bwd(f64(g), f64(x), f64(b))[0], "gelu dx", atol=2e-6, min_exact=0.99)
    # the sum of dx as stored, in float32: relative 2^-24 of each of `rows` terms of order one
    check(db, dx.double().sum(0).cpu().numpy(), "gelu dbias", atol=1e-5 * rows ** 0.5 + 1e-6, min_exact=0.97)
    dx, db = k.bias_dropout_add_backward(g.to(device), 0.2, 9, 4)
    keep = torch.from_numpy(philox.keep_mask(rows * cols, 0.2, 9, 4)).view(rows, cols).bool()
    assert int(dx.cpu()[~keep].count_nonzero()) == 0
    check(dx, cf.bias_dropout_add_bwd(f64(g), keep.numpy(), 0.2)[0], "dropout dx", atol=1e-6)
    check(db, dx.double().sum(0).cpu().numpy(), "dropout dbias", atol=1e-5 * rows ** 0.5 + 1e-6, min_exact=0.97)


@pytest.mark.parametrize("have", ["coarse", "between", "all", "too few"])
def test_a_workspace_of_the_coarse_partial_rows_is_enough(device, have):
    rows, cols = 64, 512
    x, g, b = (randn(s, BF16, i).to(device) for i, s in ((1, (rows, cols)), (2, (rows, cols)), (3, (cols,))))
    lib = _C.load_library()
    full = lib.oslo_workspace_bytes(_C.OSLO_OP_BIAS_GELU_BWD, rows, cols) // (4 * cols)
    parts = {"coarse": rows // 16, "between": rows // 16 + 3, "all": full, "too few": rows // 16 - 1}[have]
    assert full > rows // 16 + 3
    ws = torch.full((full * cols,), float("nan"), device=device)
    dx, db = torch.empty_like(x), torch.empty_like(b)
    rc = lib.oslo_bias_gelu_bwd(g.data_ptr(), x.data_ptr(), b.data_ptr(), dx.data_ptr(), db.data_ptr(), ws.data_ptr(),
                                parts * cols * 4, rows, cols, 2, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    if have == "too few":
        assert rc < 0
        return
    assert rc == 0 and int((~ws[parts * cols:].isnan()).sum()) == 0
    check(db, dx.double().sum(0).cpu().numpy(), "dbias", atol=1e-4, min_exact=0.97)


def test_a_norm_workspace_of_the_wider_slots_is_enough(device):
    """[300, 4096] bf16: two row slots gave 150 partial rows, one gives 256."""
    n1, n2 = 300, 4096
    x, dy, w = (randn(s, BF16, i).to(device) for i, s in ((1, (n1, n2)), (2, (n1, n2)), (3, (n2,))))
    k = _C.get_layernorm_kernel()
    y, mean, inv = k.layer_norm_forward_affine(x, (n2,), w, w, 1e-5)
    want = k.layer_norm_backward_affine(dy, mean, inv, x, (n2,), w, w, 1e-5)
    ws = torch.full((2 * 256 * n2,), float("nan"), device=device)
    dx, dg, db = torch.empty_like(x), torch.empty_like(w), torch.empty_like(w)
    lib = _C.load_library()
    rc = lib.oslo_ln_bwd(dy.data_ptr(), x.data_ptr(), mean.data_ptr(), inv.data_ptr(), w.data_ptr(), dx.data_ptr(),
                         dg.data_ptr(), db.data_ptr(), ws.data_ptr(), 2 * 150 * n2 * 4, n1, n2, 2, 2,
                         torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rc == 0 and int((~ws[2 * 150 * n2:].isnan()).sum()) == 0
    assert torch.equal(dx, want[0])
    for a, b in ((dg, want[1]), (db, want[2])):  # another order of the same sum
        assert torch.allclose(a.float(), b.float(), rtol=2.0 ** -7, atol=1e-3)
