"""bias-GeLU backward around the tensor size at which the launch shape changes
(256 MB in a 16-bit type): the same values on both sides, row by row, and the
bias gradient as the sum of dx as stored."""
import pytest
import torch

from helpers import check, f64, randn, ulp_distance
from oracle import closed_form as cf
from oslo_amd.torch import _C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [32767, 32768, 32769])   # 256 MB at 4096 columns
def test_both_launch_shapes(device, dtype, rows):
    cols = 4096
    el = _C.get_fused_elementwise_kernel()
    x, g, b = (randn((65, cols), dtype, i).to(device) for i in (1, 2, 3))
    rep = -(-rows // 65)
    X, G = x.repeat(rep, 1)[:rows].contiguous(), g.repeat(rep, 1)[:rows].contiguous()
    bias = b[0].contiguous()
    dx, db = el.bias_gelu_backward(G, X, bias)
    want, _ = cf.bias_gelu_bwd(f64(g), f64(x), f64(bias))
    check(dx[:65], want, "first rows", atol=1e-6, min_exact=0.995)
    # equal rows give equal results but for a float16 product that one of the
    # unrolled steps rounds once (multiply and convert in one instruction) and
    # another twice: one ulp, where the float32 value lies within 2^-13 of an ulp
    # of a tie, so in less than 2^-12 of the elements, with a margin of 4
    first = dx[:65].cpu()
    for i in range(0, rows, 65 * 37):
        part = dx[i:i + 65].cpu()
        d = ulp_distance(part, first[:part.shape[0]])
        assert int(d.max()) <= 1 and int((d != 0).sum()) <= 2 ** -10 * d.numel()
    tail = dx[rows - rows % 65:].cpu()
    assert int(ulp_distance(tail, first[:tail.shape[0]]).max()) <= 1
    # fp32 sums of `rows` terms of size one: 2^-24 * sqrt(rows) * the sum of magnitudes' rms, with a margin of 8
    total = dx.double().sum(0)
    bound = 8 * 2 ** -24 * rows ** 0.5 * dx.double().square().sum(0).sqrt() + torch.finfo(dtype).eps * total.abs()
    assert ((db.double() - total).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("chunks", [2, 8])
def test_the_override_reaches_the_build(device, dtype, chunks):
    """eltwise_unroll below the 256 MB: a workgroup of four rows of lanes takes
    4 * chunks rows a step, and a small problem has one partial row per step."""
    rows, cols = 64, 512
    x, g = (randn((rows, cols), dtype, i).to(device) for i in (1, 2))
    bias = torch.zeros(cols, dtype=dtype, device=device)
    dx, db = torch.empty_like(x), torch.empty_like(bias)
    lib = _C.load_library()
    _C.tune("eltwise_unroll", chunks)
    try:
        nbytes = lib.oslo_workspace_bytes(_C.OSLO_OP_BIAS_GELU_BWD, rows, cols)
        ws = torch.full((nbytes // 4,), float("nan"), device=device)
        assert lib.oslo_bias_gelu_bwd(g.data_ptr(), x.data_ptr(), bias.data_ptr(), dx.data_ptr(), db.data_ptr(),
                                      ws.data_ptr(), nbytes, rows, cols, 1 if dtype == torch.float16 else 2,
                                      torch.cuda.current_stream().cuda_stream) == 0
    finally:
        _C.tune("eltwise_unroll", 0)
    torch.cuda.synchronize()
    written = int((~ws.isnan()).sum())
    assert written == min(rows // 16, rows // (4 * chunks)) * cols
