"""The row slots of a norm-backward workgroup: column sums folded through LDS,
slots traded for workgroups when the rows are few, one chunk per lane in fp32,
and prefetches that stop at the last row.  Row counts around the number of
compute units (256) times the slots, row lengths around a whole number of waves
and half-waves; bounds as in tests/test_gpu_norm.py (the sums are fp32 and
their order does not depend on the values)."""
import pytest
import torch

from helpers import NP_NAME, check, f64, randn
from oracle import closed_form as cf
from oracle import philox
from oslo_amd.torch import _C

from test_gpu_norm import test_layer_norm as check_layer_norm
from test_gpu_norm import test_rms_norm as check_rms_norm
from test_gpu_residual_norm import test_fused_vs_oracle as check_fused

pytestmark = pytest.mark.gpu

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16

CASES = [(n1, n2, dt)
         for n2, dt in [(768, F32), (772, F32), (4096, F32), (4100, F32), (100, F32), (768, BF16), (1280, F16),
                        (1032, F16), (2048, BF16), (64, F16)]
         for n1 in ((1, 2, 255, 257, 513, 2049) if n2 < 1000 else (3, 257, 700))]


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("n1,n2,dtype", CASES)
def test_slots(device, n1, n2, dtype, fused):
    x, dy, dh = (randn((n1, n2), dtype, n1 + n2 + i) for i in range(3))
    gamma = randn((n2,), dtype, 9, std=0.1, mean=1.0)
    h64 = f64(x)
    _, mean, inv = cf.layer_norm_fwd(h64, f64(gamma), f64(gamma), 1e-5)
    mean, inv = (torch.from_numpy(a).float().reshape(-1) for a in (mean, inv))
    dev = [t.to(device) for t in (dy, dh, x, mean, inv, gamma)]
    k = _C.get_layernorm_kernel()
    atol = 2e-5 * n1 ** 0.5  # sums over n1 rows, as in tests/test_gpu_norm.py
    if fused:
        keep = philox.keep_mask(n1 * n2, 0.1, 3, 8).reshape(n1, n2).astype(bool)
        got = k.bias_dropout_add_norm_backward(False, *dev[:5], (n2,), dev[5], 0.1, 3, 8)
        want = cf.bias_dropout_add_norm_bwd(f64(dy), f64(dh), h64, f64(mean), f64(inv), f64(gamma), keep, 0.1, False,
                                            NP_NAME[dtype])
        want = list(want[:4]) + [f64(got[1]).sum(0)]  # dbias: of dx as stored
    else:
        got = k.layer_norm_backward_affine(dev[0], *dev[3:5], dev[2], (n2,), dev[5], dev[5], 1e-5)
        want = cf.layer_norm_bwd(f64(dy), h64, f64(mean), f64(inv), f64(gamma))
    tensors = 2 if fused else 1
    for i, (g, w) in enumerate(zip(got, want)):
        check(g, w, "output %d" % i, atol=2e-6 if i < tensors else atol, max_ulp=1 if i < tensors else 2)


@pytest.mark.parametrize("prefetch", [1, 2])
@pytest.mark.parametrize("tin,tout", [(F32, F32), (F16, F16), (BF16, BF16), (F32, F16), (F32, BF16)])
def test_sixteen_slots_of_sixteen_elements_per_lane(device, tin, tout, prefetch):
    """Rows that one wave holds with 16 elements a lane, the last ones idle, and
    enough of them that a workgroup keeps its sixteen slots."""
    n1, n2 = 15 * 256 + 10, 800
    _C.tune("norm_bwd_vpl", 4)
    _C.tune("norm_bwd_prefetch", prefetch)
    try:
        check_layer_norm(device, n1, n2, tin, tout, True)
        check_rms_norm(device, n1, n2, tin, tout, True)
        if tin == tout:
            check_fused(device, n1, n2, tin, 0.1, False)
            check_fused(device, n1, n2, tin, 0.1, True)
    finally:
        _C.tune("norm_bwd_vpl", 0)
        _C.tune("norm_bwd_prefetch", 0)
