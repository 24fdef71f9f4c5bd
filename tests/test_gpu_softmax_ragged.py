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


@pytest.mark.parametrize("dtype,sk", [(d, n) for d in (BF16, F16, F32) for n in _lengths(d)] + [(F16, 1003)])
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


# lengths whose last chunk and the one before it lie in one lane group, in one
# wave (same slot and different slots of it) and in two waves
OVERLAPS = [(BF16, n) for n in (77, 381, 513, 1531, 2049, 4099)] + [(F16, 2051), (F32, 39), (F32, 1027)]


def _overlap(dtype, sk):
    """First key of the row's last chunk, first key that only it holds, and the
    first key of the chunk before it."""
    e = 4 if dtype == F32 else 8
    own = (sk - 1) // e * e
    return sk - e, own, own - e


@pytest.mark.parametrize("dtype,sk", OVERLAPS)
def test_hidden_keys_held_twice(device, dtype, sk):
    """The last two chunks of a row differ in being read: the chunk before the
    last is hidden altogether (mask, absorbing term).  Whatever gradient its keys
    carry, also those that the last chunk holds and reads, they get zeros and the
    row does not see them.  (The plain backward of shorter rows does not look at
    the mask: a gradient that is not finite then shows in both chunks.)"""
    dup, own, before = _overlap(dtype, sk)
    b, h, sq, scale, p = 2, 2, 9, 0.25, 0.1
    x, g = randn((b, h, sq, sk), dtype, 1).to(device), randn((b, h, sq, sk), dtype, 2).to(device)
    hidden = torch.zeros(b, 1, 1, sk, dtype=torch.bool, device=device)
    hidden[..., before:own] = True
    term = torch.zeros(b, 1, 1, sk, dtype=dtype, device=device).masked_fill_(hidden, float("-inf"))
    bad = g.clone()
    bad[..., dup:own] = float("nan")
    k = _C.get_softmax_kernel()
    y = k.fused_scaled_masked_softmax_forward(x, hidden, scale)
    outs = []
    for grad in (g, bad):
        _, st = k.softmax_dropout_forward(x, hidden, scale, p, 3, 8)
        _, st_term = k.softmax_bias_dropout_forward(x, term, scale, p, 3, 8)
        chunks = -(-sk // (4 if dtype == F32 else 8))
        masked, biased = (grad if chunks > most else g for most in (48, 64 if dtype == F32 else 128))
        outs.append((k.fused_scaled_masked_softmax_backward(masked, y, scale, hidden),
                     k.softmax_bias_backward(biased, y, scale, term),
                     k.softmax_dropout_backward(grad, x, st, hidden, scale, p, 3, 8),
                     k.softmax_bias_dropout_backward(grad, x, term, st_term, scale, p, 3, 8)))
    for i, (clean, dirty) in enumerate(zip(*outs)):
        assert torch.equal(clean, dirty), "output %d" % i   # (false for a NaN)
        assert (dirty[..., before:own] == 0).all(), "output %d" % i


@pytest.mark.parametrize("dtype,sk", OVERLAPS)
def test_the_sign_of_a_zero_held_twice(device, dtype, sk):
    """The other way round: the chunk before the last is read for its first key,
    the last one lies beyond the diagonal.  A hidden key that both hold gets the
    same zero from either, scale * (0 * (0 - s))."""
    dup, own, before = _overlap(dtype, sk)
    scale, ab = 0.25, 64
    # the first of sk - before queries sees `before + 1` keys; the others are not looked at
    xq, gq = (torch.zeros(ab, sk - before, sk, dtype=dtype, device=device) for _ in range(2))
    xq[:, 0], gq[:, 0] = (randn((ab, sk), dtype, seed).to(device) for seed in (1, 2))
    g = gq[:, 0].double()
    k = _C.get_softmax_kernel()
    y = k.fused_scaled_upper_triang_masked_softmax_forward(xq, scale)
    assert (y[:, 0, before + 1:] == 0).all() and (y[:, 0, before] > 0).all()
    dx = k.fused_scaled_upper_triang_masked_softmax_backward(gq, y, scale)[:, 0].float()
    s = (y[:, 0].double() * g).sum(-1, keepdim=True)
    first = max(dup, before + 1)
    assert (dx[:, first:own] == 0).all()
    sure = (s.abs() > 1e-3).expand(-1, own - first)   # (an fp32 sum of terms below 5)
    assert torch.equal(torch.signbit(dx[:, first:own])[sure], (s > 0).expand(-1, own - first)[sure])


@pytest.mark.parametrize("dtype,sk", OVERLAPS)
def test_hidden_keys_of_a_row_of_nan(device, dtype, sk):
    """Forward: a NaN among the logits of a row leaves NaN at the keys that the
    row sees and zeros at the others, however its chunks lie; with dropout a key
    that is seen may be dropped."""
    dup, own, before = _overlap(dtype, sk)
    b, h, sq, scale, p = 2, 2, 3, 0.25, 0.1
    x = randn((b, h, sq, sk), dtype, 1).to(device)
    hidden = torch.zeros(b, 1, 1, sk, dtype=torch.bool, device=device)
    hidden[..., dup:own] = True
    hidden[1, ..., before:] = True
    x[:, :, 1, 0] = float("nan")
    k = _C.get_softmax_kernel()
    y = k.fused_scaled_masked_softmax_forward(x, hidden, scale)
    z, _ = k.softmax_dropout_forward(x, hidden, scale, p, 3, 8)
    h4 = hidden.expand_as(x)
    assert (y[h4] == 0).all() and (z[h4] == 0).all()
    assert y[:, :, 1][~h4[:, :, 1]].isnan().all() and not y[:, :, 0].isnan().any()
    seen = z[:, :, 1][~h4[:, :, 1]]
    assert (seen.isnan() | (seen == 0)).all()
    # causal: the row of the NaN sees `before + 1` keys
    xq = torch.zeros(2, sk - before, sk, dtype=dtype, device=device)
    xq[:, 0, 0] = float("nan")
    y = k.fused_scaled_upper_triang_masked_softmax_forward(xq, scale)[:, 0]
    z, _ = k.softmax_dropout_forward(xq, None, scale, p, 3, 8)
    assert y[:, :before + 1].isnan().all()
    assert (y[:, before + 1:] == 0).all() and (z[:, 0, before + 1:] == 0).all()


@pytest.mark.parametrize("dtype,sk", [(BF16, 2049), (BF16, 4099), (F32, 1027)])
def test_backward_in_place_over_several_waves(device, dtype, sk):
    """In place where the chunk that overlaps its neighbour is held by another
    wave: every wave has read its chunks before one of them stores."""
    b, h, sq, scale, p = 2, 3, 11, 0.25, 0.1
    x, g = randn((b, h, sq, sk), dtype, 3).to(device), randn((b, h, sq, sk), dtype, 4).to(device)
    hidden = (torch.arange(sk, device=device) % 5 == 1).expand(b, 1, 1, sk).contiguous()
    hidden[1, ..., sk // 2:] = True
    term = torch.zeros(b, 1, 1, sk, dtype=dtype, device=device).masked_fill_(hidden, float("-inf"))
    k = _C.get_softmax_kernel()
    for causal in (False, True):
        y = k.fused_scaled_masked_softmax_forward(x, hidden, scale, causal=causal)
        z = k.softmax_bias_forward(x, term, scale, causal=causal)
        _, st = k.softmax_dropout_forward(x, hidden, scale, p, 3, 8, causal=causal)
        _, st_term = k.softmax_bias_dropout_forward(x, term, scale, p, 3, 8, causal=causal)
        for run in (lambda t, ip: k.fused_scaled_masked_softmax_backward(t, y, scale, hidden, ip, causal),
                    lambda t, ip: k.softmax_bias_backward(t, z, scale, term, causal, inplace=ip),
                    lambda t, ip: k.softmax_dropout_backward(t, x, st, hidden, scale, p, 3, 8, ip, causal),
                    lambda t, ip: k.softmax_bias_dropout_backward(t, x, term, st_term, scale, p, 3, 8, causal,
                                                                  inplace=ip)):
            want = run(g.clone(), False)
            buf = g.clone()
            got = run(buf, True)
            assert got.data_ptr() == buf.data_ptr() and torch.equal(got, want)


@pytest.mark.parametrize("dtype,chunks", [(BF16, 48), (BF16, 49), (BF16, 128), (BF16, 129), (F32, 48), (F32, 49),
                                          (F32, 64), (F32, 65)])
@pytest.mark.parametrize("causal", [False, True])
def test_plain_backward_with_and_without_a_look_at_the_mask(device, dtype, chunks, causal):
    """Around the row lengths at which the plain backward starts to look at the
    mask or at the additive term: padding, a row of which every key is hidden
    (uniform under the mask, over all keys), per-query masks, absorbing terms."""
    e = 4 if dtype == F32 else 8
    sk = chunks * e - 3
    check_causal_masked(device, 2, 2, 9, sk, dtype, 0.25, "holes")
    check_masked(device, 2, 2, 9, sk, dtype, 0.25, "full")
    b, h, sq, scale = 2, 2, 9, 0.25
    x, g = randn((b, h, sq, sk), dtype, 1), randn((b, h, sq, sk), dtype, 2)
    hidden = torch.arange(sk).expand(b, 1, 1, sk) >= torch.tensor([sk, sk // 2]).view(b, 1, 1, 1)
    k = _C.get_softmax_kernel()
    for fill in (-10000.0, float("-inf"), torch.finfo(dtype).min):
        term = torch.zeros(b, 1, 1, sk, dtype=dtype).masked_fill_(hidden, fill)
        y = k.softmax_bias_forward(x.to(device), term.to(device), scale, causal)
        for skip in (None, True):
            dx = k.softmax_bias_backward(g.to(device), y, scale, term.to(device), causal, skip)
            check(dx, cf.softmax_bwd(f64(g), f64(y), scale), "additive %g" % fill, atol=1e-7)
