"""The arithmetic of the Adam kernel (products by split reciprocals, square root
and quotient by one Newton step) over the range of float32, and the tensor
table at its edges.

Bound: update = (m / bc1) / (sqrt(v / bc2) + eps) with every operation within
0.51 ulp of float32 gives a relative error of at most 5 * 0.51 * 2^-24 * 2 <
4e-7; p and the decay are zero here, so p = -lr * update shows it."""
import numpy as np
import pytest
import torch

from helpers import check, f64, randn
from oracle import closed_form as cf
from oslo_amd.torch import _C

pytestmark = pytest.mark.gpu

F32 = torch.float32


@pytest.mark.parametrize("step", [1, 3, 100000])
def test_update_over_the_range_of_float32(device, step):
    n = 1 << 14
    v = torch.exp2(torch.linspace(-126, 100, n, dtype=torch.float64)).float()
    m = torch.exp2(torch.linspace(-50, 40, n, dtype=torch.float64)).float() * randn((n,), F32, 1).sign()
    g, p = torch.zeros(n), torch.zeros(n)
    lists = [[t.to(device)] for t in (g, p, m, v)]
    _C.get_adam_kernel().multi_tensor_adam(0, None, lists, 1.0, 0.9, 0.999, 1e-8, step, 1, 1, 0.0)
    want, _, _ = cf.adam_step(f64(g), f64(p), f64(m), f64(v), 1.0, 0.9, 0.999, 1e-8, step, 1, 1, 0.0)
    got = f64(lists[1][0])
    assert np.all(np.abs(got - want) <= 4e-7 * np.abs(want))


def test_special_values(device):
    """Zero and infinite moments as the plain quotient has them: an overflowed
    second moment leaves the parameter where it is, 0 / eps is 0."""
    inf = float("inf")
    m = torch.tensor([0.0, 1.0, -2.0, inf, inf, 0.0, float("nan"), 1.0])
    v = torch.tensor([0.0, inf, inf, 1.0, inf, 1e-45, 1.0, 0.0])
    for bias_correction in (0, 1):
        lists = [[t.to(device)] for t in (torch.zeros(8), torch.ones(8), m, v)]
        _C.get_adam_kernel().multi_tensor_adam(0, None, lists, 0.5, 0.9, 0.999, 0.25, 2, 1, bias_correction, 0.0)
        p = lists[1][0].cpu()
        assert p[[0, 1, 2, 5]].tolist() == [1.0, 1.0, 1.0, 1.0]
        assert p[3] == -inf and p[4].isnan() and p[6].isnan() and p[7] < 0.0


def test_quotients_at_the_ends_of_the_range(device):
    """update = m / (sqrt(v) + eps) where it overflows (loaded moments; it is
    infinite, not NaN), and with divisors that have no normal reciprocal."""
    inf = float("inf")
    cases = [(1e35, 0.0, 1e-8), (-3e38, 1e-30, 0.0), (3e38, 0.25, 0.5), (-3.4e38, 0.2, 0.5), (1e-10, 0.0, 1e-40),
             (1.0, 0.0, 1e-45), (-1e-44, 0.0, 1e-44), (0.0, 0.0, 1e-40), (1e38, 0.0, 2e38), (-3e38, 0.0, 3.3e38),
             (1e-38, 0.0, 1e38), (1e-30, 1e-45, 0.0), (1e30, 3e38, 0.0), (inf, 0.0, 1e-40), (2e38, 0.0, 0.5)]
    for m, v, eps in cases:
        host = [torch.tensor([t], dtype=F32) for t in (0.0, 0.0, m, v)]
        lists = [[t.to(device)] for t in host]
        _C.get_adam_kernel().multi_tensor_adam(0, None, lists, 1.0, 1.0, 1.0, eps, 1, 1, 0, 0.0)
        got = float(lists[1][0])
        denom = np.float32(np.float32(np.sqrt(f64(host[3])[0])) + np.float32(eps))
        with np.errstate(over="ignore"):
            want = -float(np.float32(f64(host[2])[0] / np.float64(denom)))
        if np.isinf(want):
            assert got == want, (m, v, eps, got)
        else:
            # (a subnormal quotient is rounded once more)
            assert abs(got - want) <= 4e-7 * abs(want) + 1.5e-45, (m, v, eps, got, want)


@pytest.mark.parametrize("dtype", [F32, torch.bfloat16])
@pytest.mark.parametrize("count", [1, 2, 87, 88, 89, 177])
def test_tensor_table(device, dtype, count):
    """Tensors of zero to three workgroups around the 88 that one launch takes."""
    piece = 256 * (4 if dtype == F32 else 8)
    sizes = [(i * 7) % 4 * piece // 2 + i % 3 for i in range(count)]
    host = [[randn((n,), dtype, 4 * i + j, std=0.1).abs() for i, n in enumerate(sizes)] for j in range(4)]
    devl = [[t.to(device) for t in lst] for lst in host]
    _C.get_adam_kernel().multi_tensor_adam(0, None, devl, 1e-2, 0.9, 0.999, 1e-8, 7, 1, 1, 0.01)
    kw = {} if dtype == F32 else {"min_exact": 0.99}
    for i, n in enumerate(sizes):
        if n:
            want = cf.adam_step(*(f64(host[j][i]) for j in range(4)), 1e-2, 0.9, 0.999, 1e-8, 7, 1, 1, 0.01)
            for j, floor in ((1, 5e-7), (2, 1e-7), (3, 1e-8)):
                check(devl[j][i], want[j - 1], "list %d tensor %d" % (j, i), atol=floor, **kw)
