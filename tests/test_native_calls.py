"""The native side of the kernel objects (checks, allocation, launch): what it
refuses without a GPU, and where it places the large softmax outputs."""
import pytest
import torch

from oslo_amd.torch import _C

X, B = torch.zeros(2, 8), torch.zeros(8)
X3, X4, M4 = torch.zeros(2, 3, 8), torch.zeros(1, 2, 3, 8), torch.zeros(1, 1, 1, 8)
STATS = torch.zeros(6, 2)

CALLS = [
    lambda ln, sm, el: ln.layer_norm_forward_affine(X, (8,), B, B, 1e-5),
    lambda ln, sm, el: ln.layer_norm_backward_affine(X, B, B, X, (8,), B, B, 1e-5),
    lambda ln, sm, el: ln.bias_dropout_add_norm_forward(True, X, B, X, (8,), B, None, 1e-5, 0.1, 2 ** 64 - 1, 0),
    lambda ln, sm, el: ln.bias_dropout_add_norm_backward(False, X, None, X, B, B, (8,), B, 0.1, 1, 0),
    lambda ln, sm, el: sm.fused_scaled_upper_triang_masked_softmax_forward(X3, 1.0),
    lambda ln, sm, el: sm.fused_scaled_upper_triang_masked_softmax_backward(X3, X3, 1),
    lambda ln, sm, el: sm.fused_scaled_masked_softmax_forward(X4, M4.bool(), 1.0, causal=True),
    lambda ln, sm, el: sm.fused_scaled_masked_softmax_backward(X4, X4, 1.0),
    lambda ln, sm, el: sm.softmax_dropout_forward(X3, None, 1.0, 0.1, 1, 0),
    lambda ln, sm, el: sm.softmax_dropout_backward(X4, X4, STATS, M4.bool(), 1.0, 0.1, 1, 0),
    lambda ln, sm, el: sm.softmax_bias_forward(X4, M4, 1.0),
    lambda ln, sm, el: sm.softmax_bias_backward(X4, X4, 1.0, M4),
    lambda ln, sm, el: sm.softmax_bias_dropout_forward(X4, M4, 1.0, 0.1, 1, 0),
    lambda ln, sm, el: sm.softmax_bias_dropout_backward(X4, X4, M4, STATS, 1.0, 0.1, 1, 0),
    lambda ln, sm, el: el.bias_gelu_forward(X, None),
    lambda ln, sm, el: el.bias_gelu_backward(X, X, B),
    lambda ln, sm, el: el.bias_dropout_add_forward(X, B, X, 0.1, 1, 0, return_mask=True),
    lambda ln, sm, el: el.bias_dropout_add_backward(X, 0.1, 1, 0),
]


@pytest.mark.parametrize("call", range(len(CALLS)))
def test_tensors_off_the_gpu_are_refused(call):
    kernels = _C.get_layernorm_kernel(), _C.get_softmax_kernel(), _C.get_fused_elementwise_kernel()
    with pytest.raises(RuntimeError, match="must be a CUDA tensor"):
        CALLS[call](*kernels)


def test_other_arguments_are_refused():
    calls = _C.load_calls()
    with pytest.raises(TypeError, match="must be a Tensor"):
        calls.gelu_forward(3, None)
    with pytest.raises(TypeError, match="too few"):
        calls.gelu_forward(X)
    with pytest.raises(TypeError):
        calls.bias_forward(X4, M4, "scale", False, None)
    with pytest.raises(TypeError):
        calls.norm_forward(False, X, 8, None, None, 1e-5, False)


def _backwards(device, n1, n2, other):
    """The four backwards that take a workspace, on [n1, n2] with an incoming
    gradient of `other` columns."""
    ln, _, el = _C.get_layernorm_kernel(), None, _C.get_fused_elementwise_kernel()
    x, g = torch.randn(n1, n2, device=device), torch.randn(n1, other, device=device)
    w, stat = torch.ones(n2, device=device), torch.ones(n1, device=device)
    return [lambda: ln.layer_norm_backward_affine(g, stat, stat, x, (n2,), w, w, 1e-5),
            lambda: ln.rms_norm_backward_affine(g, stat, x, (n2,), w, 1e-5),
            lambda: ln.bias_dropout_add_norm_backward(False, g, None, x, stat, stat, (n2,), w, 0.1, 1, 0),
            lambda: el.bias_gelu_backward(g, x, w)]


def _cached():
    return {key: slot.tensor for key, slot in _C._ws_cache.slots.items()}


@pytest.mark.gpu
def test_a_refused_backward_leaves_the_workspaces_alone(device):
    before = _cached()
    for call in _backwards(device, 2048, 8192, 8):   # (larger than what other tests leave there)
        with pytest.raises(RuntimeError):
            call()
    after = _cached()
    assert after.keys() == before.keys() and all(after[k] is before[k] for k in after)


@pytest.mark.gpu
def test_a_failed_allocation_of_a_workspace(device, monkeypatch):
    """The error comes through as it is, and the slot is free for the next call."""
    def fail(nbytes, index):
        raise MemoryError("no workspace")

    with torch.cuda.stream(torch.cuda.Stream()):      # (a stream without cached workspaces)
        calls = _backwards(device, 64, 128, 128)
        with monkeypatch.context() as m:
            m.setattr(_C._ws_cache, "allocate", fail)
            for call in calls:
                with pytest.raises(MemoryError, match="no workspace"):
                    call()
        for call in calls:
            assert all(torch.isfinite(t).all() for t in call())
    torch.cuda.synchronize()


@pytest.mark.gpu
def test_large_softmax_outputs_are_staggered(device):
    sm = _C.get_softmax_kernel()
    x = torch.randn(1, 4096, 8192, dtype=torch.bfloat16, device=device)
    y = sm.fused_scaled_upper_triang_masked_softmax_forward(x, 1.0)
    dx = sm.fused_scaled_upper_triang_masked_softmax_backward(x, y, 1.0)
    for t, k in ((y, 1), (dx, 2)):   # 64 MiB each
        assert t.is_contiguous() and t.shape == x.shape
        assert t.data_ptr() % (2 << 20) == k * _C.STAGGER_STEP % (2 << 20)
