"""How a norm launch splits few rows, fp32 rows with the fused prologue and the
rows of a backward: batches on both sides of each line of the launch rules,
against the float64 oracle (plain) and, with the prologue, against the two
plain launches it replaces."""
import pytest
import torch

from helpers import check, f64, randn
from oracle import closed_form as cf
from oslo_amd.torch import _C

pytestmark = pytest.mark.gpu

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16


def operands(n1, n2, dtype, device):
    x, dy = randn((n1, n2), dtype, n1 + n2, mean=0.5), randn((n1, n2), dtype, n1 + n2 + 1)
    gamma, beta = randn((n2,), dtype, 3, std=0.1, mean=1.0), randn((n2,), dtype, 4, std=0.1)
    return x, dy, gamma, beta


# forward: one, two or more chunks per lane (at most two waves per SIMD), one or
# two row groups (three workgroups per CU); backward: 3, 7 and 12 rows per CU
@pytest.mark.parametrize("n1,n2,dtype", [
    (1, 6144, BF16), (171, 6144, BF16), (255, 4096, F16), (257, 4096, F16), (513, 2048, BF16),
    (769, 4096, BF16), (1537, 4096, F16), (1790, 4096, BF16), (3048, 1024, BF16), (3073, 1024, F16),
    (128, 4096, F32), (129, 4096, F32), (1025, 1024, F32), (2305, 768, F32),
])
def test_plain_norm_against_the_oracle(device, n1, n2, dtype):
    x, dy, gamma, beta = operands(n1, n2, dtype, device)
    k = _C.get_layernorm_kernel()
    xd, gd, bd = x.to(device), gamma.to(device), beta.to(device)
    y, mean, invvar = k.layer_norm_forward_affine(xd, (n2,), gd, bd, 1e-5)
    oy, omean, oinv = cf.layer_norm_fwd(f64(x), f64(gamma), f64(beta), 1e-5)
    check(y, oy, "forward", atol=2e-6)
    dx, dg, db = k.layer_norm_backward_affine(dy.to(device), mean, invvar, xd, (n2,), gd, bd, 1e-5)
    odx, odg, odb = cf.layer_norm_bwd(f64(dy), f64(x), f64(mean), f64(invvar), f64(gamma))
    check(dx, odx, "dx", atol=4e-6)
    # (sums of n1 terms of order one: their float32 rounding is absolute)
    for got, want, what in ((dg, odg, "dgamma"), (db, odb, "dbeta")):
        check(got, want, what, atol=2e-6 * n1 ** 0.5, min_exact=0.97)
    # (two roundings: a neighbour after the first, one ulp, is multiplied by a
    # gamma of up to 1.5 and rounded again: two ulp of the result)
    yr, inv = k.rms_norm_forward_affine(xd, (n2,), gd, 1e-5)
    check(yr, cf.rms_norm_fwd(f64(x), f64(gamma), 1e-5, out={F32: "f64", F16: "f16", BF16: "bf16"}[dtype])[0],
          "rms forward", atol=2e-6, max_ulp=2)


# fp32: 4096, 8192 (the longest row of two chunks per lane) and beyond, 5 waves
# of the former split (4672), 16-bit rows of 16 and 8 elements per lane
@pytest.mark.parametrize("p", [0.0, 0.1])
@pytest.mark.parametrize("n1,n2,dtype", [
    (40, 4672, F32), (700, 4672, F32), (60, 8192, F32), (60, 8196, F32), (1030, 2048, F32), (90, 4092, F32),
    (3, 2944, BF16), (260, 2048, F16), (2100, 2048, BF16), (1200, 1024, F32),
])
def test_fused_norm_against_the_two_launches(device, n1, n2, dtype, p):
    x, dy, gamma, beta = (t.to(device) for t in operands(n1, n2, dtype, device))
    res, dh = randn((n1, n2), dtype, 9).to(device), randn((n1, n2), dtype, 10).to(device)
    bias = randn((n2,), dtype, 11, std=0.1).to(device)
    k, ek = _C.get_layernorm_kernel(), _C.get_fused_elementwise_kernel()
    y, h, mean, invvar = k.bias_dropout_add_norm_forward(False, x, bias, res, (n2,), gamma, beta, 1e-5, p, 77, 8)
    h2 = ek.bias_dropout_add_forward(x, bias, res, p, 77, 8)
    assert torch.equal(h, h2)
    y2, mean2, invvar2 = k.layer_norm_forward_affine(h2, (n2,), gamma, beta, 1e-5)
    # one dtype, two orders of summation of the statistics (relative 2^-22)
    assert torch.allclose(mean, mean2, rtol=1e-5, atol=1e-6) and torch.allclose(invvar, invvar2, rtol=2e-6)
    if dtype == F32:
        assert torch.allclose(y, y2, rtol=1e-5, atol=1e-5)
    else:
        # (an ulp, or the float32 rounding of the statistics where (h - mean) * rs
        # and beta cancel: 2^-22 of terms of at most eight)
        assert ((y.float() - y2.float()).abs() <= 2.0 ** -7 * y2.float().abs() + 1e-5).all()
        assert float((y == y2).double().mean()) > 0.998
    g_res, g_in, g_gamma, g_beta, g_bias = k.bias_dropout_add_norm_backward(
        False, dy, dh, h, mean, invvar, (n2,), gamma, p, 77, 8)
    _, dg2, db2 = k.layer_norm_backward_affine(dy, mean, invvar, h, (n2,), gamma, beta, 1e-5)
    tol = dict(rtol=1e-5, atol=2e-5 * n1 ** 0.5) if dtype == F32 else dict(rtol=2.0 ** -7, atol=1e-3)
    assert torch.allclose(g_gamma, dg2, **tol) and torch.allclose(g_beta, db2, **tol)
    kept = ek.philox_mask(n1 * n2, p, 77, 8, device).view(n1, n2).bool() if p > 0 else torch.ones_like(h, dtype=torch.bool)
    g_in = g_res if p == 0.0 and g_in is None else g_in
    assert int(g_in[~kept].count_nonzero()) == 0
    want = g_res.float() / (1.0 - p)
    ulp = 1e-6 if dtype == F32 else 2.0 ** -7 if dtype == BF16 else 2.0 ** -10
    assert ((g_in.float() - want)[kept].abs() <= ulp * want[kept].abs() + 1e-6).all()
    check(g_bias, g_in.double().sum(0).cpu().numpy(), "dbias", atol=1e-5 * n1 ** 0.5, min_exact=0.97)
