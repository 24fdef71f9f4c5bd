"""The native autograd Functions against the Python ones that they stand in for
on eager GPU calls: outputs and gradients bit for bit over operand layouts and
requires-grad subsets, and the parts of torch that look at an autograd node
(saved-tensor hooks, version counters, second derivatives, tracing, vmap, forward
mode, several threads, a second stream)."""
import threading

import pytest
import torch

from oslo_amd.torch.nn.modules import functional as F

pytestmark = pytest.mark.gpu

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16


def rnd(*shape, dtype, device, seed, std=1.0, mean=0.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * std + mean).to(dtype).to(device)


# name -> (operands, call through the user function, call of the Python Function);
# `s` is the seed and offset of the dropout
def norm_operands(dtype, device, n=48, w=BF16):
    return [rnd(7, 5, n, dtype=dtype, device=device, seed=1, mean=0.3), rnd(n, dtype=w, device=device, seed=2, mean=1.0),
            rnd(n, dtype=w, device=device, seed=3)]


def scores(dtype, device, sk=40):
    return rnd(2, 3, 24, sk, dtype=dtype, device=device, seed=4, std=3.0)


OPS = {
    "layer_norm_affine": (lambda t, d: norm_operands(t, d, w=t),
                          lambda x, w, b, s: F.fused_layer_norm_affine(x, w, b, (48,), 1e-5),
                          lambda x, w, b, s: F._FusedLayerNormAffineFunction.apply(x, w, b, (48,), 1e-5)),
    "layer_norm": (lambda t, d: norm_operands(t, d)[:1],
                   lambda x, s: F.fused_layer_norm(x, (5, 48), 1e-5),
                   lambda x, s: F._FusedLayerNormFunction.apply(x, (5, 48), 1e-5)),
    "rms_norm_affine": (lambda t, d: norm_operands(t, d, w=t)[:2],
                        lambda x, w, s: F.fused_rms_norm_affine(x, w, (48,), 1e-5),
                        lambda x, w, s: F._FusedRMSNormAffineFunction.apply(x, w, (48,), 1e-5)),
    "rms_norm": (lambda t, d: norm_operands(t, d)[:1],
                 lambda x, s: F.fused_rms_norm(x, (48,), 1e-5),
                 lambda x, s: F._FusedRMSNormFunction.apply(x, (48,), 1e-5)),
    "mixed_layer_norm": (lambda t, d: norm_operands(F32, d),
                         lambda x, w, b, s: F.mixed_dtype_fused_layer_norm_affine(x, w, b, (48,), 1e-5),
                         lambda x, w, b, s: F._FusedLayerNormAffineMixedDtypesFunction.apply(x, w, b, (48,), 1e-5)),
    "mixed_rms_norm": (lambda t, d: norm_operands(F32, d)[:2],
                       lambda x, w, s: F.mixed_dtype_fused_rms_norm_affine(x, w, (48,), 1e-5),
                       lambda x, w, s: F._FusedRMSNormAffineMixedDtypesFunction.apply(x, w, (48,), 1e-5)),
    "bias_gelu": (lambda t, d: norm_operands(t, d, w=t)[:2],
                  lambda x, b, s: F.fused_bias_gelu(x, b),
                  lambda x, b, s: F._FusedBiasGeLUFunction.apply(x, b)),
    "bias_dropout_add": (lambda t, d: norm_operands(t, d, w=t)[:2] + [rnd(7, 5, 48, dtype=t, device=d, seed=9)],
                         lambda x, b, r, s: F.fused_bias_dropout_add(x, b, r, 0.3, True),
                         lambda x, b, r, s: F._FusedBiasDropoutAddFunction.apply(x, b, r, 0.3, *s, False)),
    "dropout_only": (lambda t, d: norm_operands(t, d, w=t)[:1],
                     lambda x, s: F.fused_bias_dropout_add(x, None, None, 0.3, True),
                     lambda x, s: F._FusedBiasDropoutAddFunction.apply(x, None, None, 0.3, *s, False)),
    "dropout_residual": (lambda t, d: [norm_operands(t, d, w=t)[0], rnd(7, 5, 48, dtype=t, device=d, seed=9)],
                         lambda x, r, s: F.fused_bias_dropout_add(x, None, r, 0.3, True),
                         lambda x, r, s: F._FusedBiasDropoutAddFunction.apply(x, None, r, 0.3, *s, False)),
    "causal": (lambda t, d: [scores(t, d)[0]],
               lambda x, s: F.scaled_upper_triang_masked_softmax(x, 0.5),
               lambda x, s: F._ScaledUpperTriangMaskedSoftmax.apply(x, 0.5)),
    "causal_dropout": (lambda t, d: [scores(t, d)[0]],
                       lambda x, s: F.scaled_upper_triang_masked_softmax_dropout(x, 0.5, 0.3),
                       lambda x, s: F._ScaledMaskedSoftmaxDropout.apply(x, None, 0.5, 0.3, *s)),
    "term": (lambda t, d: [scores(t, d), rnd(1, 3, 24, 40, dtype=t, device=d, seed=5)],
             lambda x, m, s: F.scaled_bias_softmax(x, m, 0.5, causal=True),
             lambda x, m, s: F._ScaledBiasSoftmax.apply(x, m, 0.5, True)),
    "term_dropout": (lambda t, d: [scores(t, d), rnd(2, 1, 1, 40, dtype=F32, device=d, seed=5)],
                     lambda x, m, s: F.scaled_bias_softmax_dropout(x, m, 0.5, 0.3),
                     lambda x, m, s: F._ScaledBiasSoftmaxDropout.apply(x, m, 0.5, 0.3, *s, False)),
}
for causal in (False, True):
    def masked(x, s, causal=causal, native=True, p=0.0):
        m = torch.arange(40, device=x.device).view(1, 1, 1, 40) >= torch.tensor([40, 13], device=x.device).view(2, 1, 1, 1)
        if native:
            return F.scaled_masked_softmax_dropout(x, m, 0.5, p, True, causal=causal)
        if p:
            return F._ScaledMaskedSoftmaxDropout.apply(x, m, 0.5, p, *s, causal)
        return F._ScaledMaskedSoftmax.apply(x, m, 0.5, causal)
    for p in (0.0, 0.3):
        OPS["masked%s%s" % ("_causal" if causal else "", "_dropout" if p else "")] = (
            lambda t, d: [scores(t, d)],
            lambda x, s, f=masked, p=p: f(x, s, p=p), lambda x, s, f=masked, p=p: f(x, s, native=False, p=p))
for rms in (False, True):
    for p in (0.0, 0.3):
        def ops(t, d, rms=rms):
            x, w, b = norm_operands(t, d, w=t)
            return [x, rnd(48, dtype=t, device=d, seed=6), rnd(7, 5, 48, dtype=t, device=d, seed=7), w] + ([] if rms else [b])
        OPS["residual_%s_%s" % ("rms" if rms else "layer_norm", p)] = (
            ops,
            lambda x, b, r, w, nb=None, s=None, rms=rms, p=p:
                F._bias_dropout_add_norm(rms, x, b, r, w, nb, (48,), 1e-5, p, True, True),
            lambda x, b, r, w, nb=None, s=None, rms=rms, p=p:
                F._FusedBiasDropoutAddNormFunction.apply(x, b, r, w, nb, (48,), 1e-5, p, *(s if p else (0, 0)), rms))


def random_state(device):
    gen = torch.cuda.default_generators[torch.cuda.current_device()]
    return gen.initial_seed(), gen.get_offset()


def evaluate(call, operands, mask, layout, device):
    """Outputs, gradients and the call's node, on fresh leaves; `mask` says which
    operands require a gradient, `layout` whether the first is a transposed view."""
    leaves = [t.detach().clone().requires_grad_(bool(mask >> k & 1)) for k, t in enumerate(operands)]
    args = list(leaves)
    if layout == "strided":
        args[0] = args[0].transpose(0, 1).contiguous().transpose(0, 1)
        assert args[0].shape[0] < 2 or not args[0].is_contiguous()
    torch.manual_seed(11)
    s = random_state(device)
    out = call(*args, s=s)
    outs = out if isinstance(out, tuple) else (out,)
    grads = [rnd(*o.shape, dtype=o.dtype, device=device, seed=20 + k) for k, o in enumerate(outs)]
    if mask:
        torch.autograd.backward(outs, grads)
    return [o.detach() for o in outs], [t.grad for t in leaves], outs[0].grad_fn


def equal(a, b):
    return (a is None) == (b is None) and (a is None or (a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)))


@pytest.mark.parametrize("layout", ["contiguous", "strided"])
@pytest.mark.parametrize("dtype", [F32, F16, BF16])
@pytest.mark.parametrize("name", sorted(OPS))
def test_native_and_python_functions_agree(device, name, dtype, layout):
    make, native, python = OPS[name]
    operands = make(dtype, device)
    for mask in range(1 << len(operands)):
        on, gn, node = evaluate(native, operands, mask, layout, device)
        op, gp, _ = evaluate(python, operands, mask, layout, device)
        assert all(equal(a, b) for a, b in zip(on, op)), (name, mask)
        assert all(equal(a, b) for a, b in zip(gn, gp)), (name, mask)
        assert (node is not None) == bool(mask) and (node is None or "CppFunction" in type(node).__name__)


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("name", ["layer_norm_affine", "mixed_layer_norm", "rms_norm_affine", "mixed_rms_norm"])
def test_a_norm_without_a_weight(device, name, bias, dtype):
    """The norm without parameters, in the input's dtype; a bias is not looked at."""
    _, native, python = OPS[name]
    if bias and "rms" in name:
        pytest.skip("RMSNorm has no bias")
    operands = norm_operands(dtype, device, w=BF16)[::2] if bias else norm_operands(dtype, device)[:1]
    rest = () if "rms" in name or bias else (None,)
    for mask in range(1 << len(operands)):
        got = [evaluate(lambda x, *b, s, f=f: f(x, None, *b, *rest, s), operands, mask, "contiguous", device)
               for f in (native, python)]
        assert all(equal(a, b) for k in (0, 1) for a, b in zip(got[0][k], got[1][k])), mask
        assert got[0][0][0].dtype == dtype and (got[0][2] is None) == (got[1][2] is None)


def test_a_layer_norm_with_a_weight_needs_a_bias(device):
    x, w, _ = norm_operands(F32, device, w=F32)
    for call in (F.fused_layer_norm_affine, F.mixed_dtype_fused_layer_norm_affine):
        before = torch.cuda.memory_stats(device)["allocation.all.allocated"]
        with pytest.raises(RuntimeError, match="needs a bias"):
            call(x, w, None, (48,))
        assert torch.cuda.memory_stats(device)["allocation.all.allocated"] == before


def test_only_the_sum_of_a_residual_norm_is_used(device):
    """No gradient arrives at the normalised output: the norm's parameters get none."""
    make, native, python = OPS["residual_layer_norm_0.3"]
    for call in (native, python):
        leaves = [t.requires_grad_() for t in make(BF16, device)]
        torch.manual_seed(5)
        s = random_state(device)
        _, h = call(*leaves, s=s)
        h.backward(torch.ones_like(h))
        assert leaves[3].grad is None and leaves[4].grad is None
        if call is native:
            want = [t.grad for t in leaves]
        else:
            assert all(equal(a, t.grad) for a, t in zip(want, leaves))


@pytest.mark.parametrize("n2,dtype", [(12296, BF16), (6148, F32)])
def test_rows_whose_backward_is_composed(device, n2, dtype):
    x, r, dy = (rnd(6, n2, dtype=dtype, device=device, seed=k) for k in (1, 2, 3))
    b, w, nb = (rnd(n2, dtype=dtype, device=device, seed=k) for k in (4, 5, 6))
    got = []
    for native in (True, False):
        leaves = [t.clone().requires_grad_() for t in (x, b, r, w, nb)]
        torch.manual_seed(5)
        s = random_state(device)
        if native:
            y, h = F._bias_dropout_add_norm(False, *leaves, (n2,), 1e-5, 0.2, True, True)
        else:
            y, h = F._FusedBiasDropoutAddNormFunction.apply(*leaves, (n2,), 1e-5, 0.2, *s, False)
        torch.autograd.backward([y, h], [dy, dy])
        got.append([t.grad for t in leaves])
    assert all(equal(a, b) for a, b in zip(*got))


def test_saved_tensor_hooks_see_the_saved_tensors(device):
    x = rnd(4, 5, 16, 16, dtype=BF16, device=device, seed=1).requires_grad_()
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.to(device)):
        y = F.scaled_masked_softmax(x, torch.zeros(1, 1, 1, 16, dtype=torch.bool, device=device), 0.5)
    assert sorted(map(tuple, packed)) == [(1, 1, 1, 16), (4, 5, 16, 16)]
    g = rnd(4, 5, 16, 16, dtype=BF16, device=device, seed=2)
    y.backward(g)
    z = x.detach().clone().requires_grad_()
    F.scaled_masked_softmax(z, torch.zeros(1, 1, 1, 16, dtype=torch.bool, device=device), 0.5).backward(g)
    assert torch.equal(x.grad, z.grad)


@pytest.mark.parametrize("name", ["causal", "bias_gelu", "layer_norm_affine"])
def test_a_saved_tensor_changed_in_place_is_noticed(device, name):
    make, native, _ = OPS[name]
    leaves = [t.requires_grad_() for t in make(BF16, device)]
    x = leaves[0] * 1.0
    y = native(x, *leaves[1:], s=None)
    (y if name == "causal" else x).data_ptr()
    with torch.no_grad():
        (y if name == "causal" else x).add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()


def test_large_outputs_that_are_placed_in_a_larger_allocation(device):
    """From 64 MiB on the probabilities are a view of their allocation."""
    x = rnd(9, 1024, 4096, dtype=BF16, device=device, seed=1).requires_grad_()
    y = F.scaled_upper_triang_masked_softmax(x, 1.0)
    g = torch.ones_like(y)
    y.backward(g)
    z = x.detach().clone().requires_grad_()
    w = F._ScaledUpperTriangMaskedSoftmax.apply(z, 1.0)
    w.backward(g)
    assert torch.equal(y, w) and torch.equal(x.grad, z.grad)
    # (in place on the output itself: refused by torch for a view that a Function returns)
    for out in (y, w):
        with pytest.raises(RuntimeError, match="modified inplace|modified in-place"):
            out.mul_(2.0)
    y.detach().mul_(2.0)  # (an ordinary tensor to its user)
    small = F.scaled_upper_triang_masked_softmax(x[:1, :8, :8], 1.0)
    assert torch.equal(small.mul_(2.0), 2.0 * F.scaled_upper_triang_masked_softmax(x[:1, :8, :8], 1.0))


@pytest.mark.parametrize("name", sorted(OPS))
def test_second_derivatives_are_as_absent_as_in_python(device, name):
    """A backward pass that is asked for its own graph: the gradients, and whether
    they carry one, as the Python Function gives them."""
    make, native, python = OPS[name]
    got = []
    for call in (native, python):
        leaves = [t.requires_grad_() for t in make(BF16, device)]
        torch.manual_seed(11)
        out = call(*leaves, s=random_state(device))
        outs = list(out) if isinstance(out, tuple) else [out]
        dys = [rnd(*o.shape, dtype=o.dtype, device=device, seed=20 + k).requires_grad_() for k, o in enumerate(outs)]
        got.append(torch.autograd.grad(outs, leaves, dys, create_graph=True, allow_unused=True))
    for a, b in zip(*got):
        assert equal(a, b) and (a is None or a.requires_grad == b.requires_grad)


def test_a_method_replaced_on_the_kernel_object_is_called(device, monkeypatch):
    from oslo_amd.torch import _C

    k = _C.get_softmax_kernel()
    real, seen = k.fused_scaled_upper_triang_masked_softmax_backward, []
    x = scores(BF16, device)[0].requires_grad_()
    with monkeypatch.context() as m:
        m.setattr(k, "fused_scaled_upper_triang_masked_softmax_backward", lambda *a: seen.append(1) or real(*a))
        F.scaled_upper_triang_masked_softmax(x).sum().backward()
    assert seen == [1] and not k.replaced()
    F.scaled_upper_triang_masked_softmax(x).sum().backward()
    assert seen == [1]


def test_tracing_records_the_function(device):
    from oslo_amd.torch.nn import FusedLayerNorm

    m = FusedLayerNorm(32).to(device)
    x = rnd(4, 32, dtype=F32, device=device, seed=1)
    with torch.no_grad():
        traced = torch.jit.trace(m, x, check_trace=False)
        other = rnd(4, 32, dtype=F32, device=device, seed=2)
        assert torch.equal(traced(other), m(other))


def test_transforms_that_a_function_without_rules_refuses(device):
    """The calls go to the native node, which refuses them as torch does of a C++ Function."""
    x = rnd(3, 4, 32, dtype=F32, device=device, seed=1)
    with pytest.raises(RuntimeError, match="functorch transforms"):
        torch.vmap(lambda t: F.fused_rms_norm(t, (32,)))(x)
    with pytest.raises(RuntimeError, match="functorch transforms"):
        torch.func.grad(lambda t: F.fused_rms_norm(t, (32,)).sum())(x)
    import torch.autograd.forward_ad as fwad

    with fwad.dual_level(), pytest.raises((RuntimeError, NotImplementedError), match="jvp"):
        F.fused_rms_norm(fwad.make_dual(x.requires_grad_(), torch.ones_like(x)), (32,))


def test_no_grad_inference_and_autocast(device):
    x, w, b = norm_operands(F32, device, w=F32)
    for ctx in (torch.no_grad(), torch.inference_mode()):
        with ctx:
            y = F.fused_layer_norm_affine(x, w.requires_grad_() if not torch.is_inference_mode_enabled() else w, b, (48,))
        assert not y.requires_grad and y.grad_fn is None
    with torch.autocast("cuda", dtype=BF16):
        y = F.fused_layer_norm_affine(x.requires_grad_(), w, b, (48,))
    assert y.dtype == BF16
    y.float().sum().backward()
    assert x.grad is not None and x.grad.dtype == F32


def test_threads_and_a_second_stream(device):
    """Backward passes of several threads, one of them on a stream of its own:
    the same gradients as alone."""
    def work(out, k, stream):
        with torch.cuda.stream(stream):
            x = rnd(64, 768, dtype=BF16, device=device, seed=k).requires_grad_()
            w, b = (rnd(768, dtype=BF16, device=device, seed=k + j).requires_grad_() for j in (50, 60))
            for _ in range(20):
                x.grad = w.grad = b.grad = None
                y = F.fused_layer_norm_affine(x, w, b, (768,))
                F.fused_bias_gelu(y, b).float().square().sum().backward()
            stream.synchronize()
            out[k] = [t.grad.clone() for t in (x, w, b)]
            stream.synchronize()

    alone, together = {}, {}
    for k in range(3):
        work(alone, k, torch.cuda.current_stream())
    streams = [torch.cuda.current_stream(), torch.cuda.current_stream(), torch.cuda.Stream()]
    threads = [threading.Thread(target=work, args=(together, k, streams[k])) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(3):
        assert all(torch.equal(a, b) for a, b in zip(alone[k], together[k]))
