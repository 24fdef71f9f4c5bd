"""Loader and thin bindings for ``liboslo_hip.so`` (the C ABI in ``include/oslo_hip.h``).

Mirrors the role of the reference's ``oslo/torch/_C/__init__.py``: lazily
obtained kernel objects (``get_layernorm_kernel()`` at ``_C/__init__.py:193-206``
there) whose methods have the signatures of the reference's pybind modules
(``FusedLayerNormBinder.cpp:404-424``, ``FusedScaleMaskSoftmaxBinder.cpp:111-127``).
Instead of JIT-compiling CUDA through ``torch.utils.cpp_extension`` the shared
library is built ahead of time by ``hipcc`` for gfx950 and bound with ctypes;
tensors cross the boundary as raw device pointers and every output and
workspace is allocated on this side, by torch's caching allocator.  The methods
of the layer ops do that in native code (``csrc/torch_calls.cpp``: checks,
allocation, launch): in Python they cost three times the launch itself.

A missing or unloadable library raises ``EnvironmentError`` (the reference's
exception type, ``_C/__init__.py:200-204``); there is no fallback for GPU
tensors.
"""
import ctypes
import importlib.machinery
import importlib.util
import os
import subprocess
import sys
import threading

import torch

_CSRC_DIR = os.path.normpath(
    os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "..", "csrc")
)
LIBRARY_PATH = os.path.join(_CSRC_DIR, "liboslo_hip.so")
CALLS_PATH = os.path.join(_CSRC_DIR, "oslo_torch_calls.so")

OSLO_OP_LN_BWD = 1
OSLO_OP_RMS_BWD = 2
OSLO_OP_BIAS_GELU_BWD = 3
OSLO_OP_BIAS_DROPOUT_ADD_BWD = 4
OSLO_OP_BIAS_DROPOUT_ADD_NORM_BWD = 5

ABI_VERSION = 1

_DTYPE_CODE = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}
OSLO_DTYPE_F64 = 3  # LayerNorm / RMSNorm only
OSLO_LN_BWD_STATIC_SCRATCH_BYTES = 16 * 1024 * 1024

_lib = None
_calls = None
_lib_lock = threading.Lock()

_p = ctypes.c_void_p
_i64 = ctypes.c_int64
_u64 = ctypes.c_uint64
_int = ctypes.c_int
_f32 = ctypes.c_float
_f64 = ctypes.c_double

# name -> (restype, argtypes); one entry per declaration in include/oslo_hip.h and
# include/oslo_hip_testing.h
_SIGNATURES = {
    "oslo_hip_last_error": (ctypes.c_char_p, []),
    "oslo_hip_arch": (ctypes.c_char_p, []),
    "oslo_hip_abi_version": (_int, []),
    "oslo_workspace_bytes": (_i64, [_int, _i64, _i64]),
    "oslo_ln_fwd": (_int, [_p, _p, _p, _p, _p, _p, _i64, _i64, _f64, _int, _int, _p]),
    "oslo_ln_bwd": (
        _int,
        [_p, _p, _p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _int, _int, _p],
    ),
    "oslo_ln_bwd_static": (
        _int,
        [_p, _p, _p, _p, _p, _p, _p, _p, _i64, _i64, _int, _int, _p],
    ),
    "oslo_rms_fwd": (_int, [_p, _p, _p, _p, _i64, _i64, _f64, _int, _int, _p]),
    "oslo_rms_bwd": (
        _int,
        [_p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _int, _int, _p],
    ),
    "oslo_softmax_causal_fwd": (_int, [_p, _p, _i64, _i64, _i64, _f32, _int, _p]),
    "oslo_softmax_causal_bwd": (_int, [_p, _p, _p, _i64, _i64, _i64, _f32, _int, _p]),
    "oslo_softmax_masked_fwd": (
        _int,
        [_p, _p, _p, _i64, _i64, _i64, _i64, _i64, _i64, _f32, _int, _p],
    ),
    "oslo_softmax_masked_bwd": (
        _int,
        [_p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _i64, _f32, _int, _p],
    ),
    "oslo_softmax_causal_masked_fwd": (
        _int,
        [_p, _p, _p, _i64, _i64, _i64, _i64, _i64, _i64, _f32, _int, _p],
    ),
    "oslo_softmax_causal_masked_bwd": (
        _int,
        [_p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _i64, _f32, _int, _p],
    ),
    "oslo_softmax_causal_masked_dropout_fwd": (
        _int,
        [_p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _i64, _f32, _f32, _u64, _u64,
         _int, _p],
    ),
    "oslo_softmax_causal_masked_dropout_bwd": (
        _int,
        [_p, _p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _i64, _f32, _f32, _u64,
         _u64, _int, _p],
    ),
    "oslo_softmax_batch_per_block": (_int, [_i64, _i64, _i64, _i64]),
    "oslo_softmax_causal_dropout_fwd": (
        _int,
        [_p, _p, _p, _i64, _i64, _i64, _f32, _f32, _u64, _u64, _int, _p],
    ),
    "oslo_softmax_causal_dropout_bwd": (
        _int,
        [_p, _p, _p, _p, _i64, _i64, _i64, _f32, _f32, _u64, _u64, _int, _p],
    ),
    "oslo_softmax_masked_dropout_fwd": (
        _int,
        [_p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _i64, _f32, _f32, _u64, _u64,
         _int, _p],
    ),
    "oslo_softmax_masked_dropout_bwd": (
        _int,
        [_p, _p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _i64, _f32, _f32, _u64,
         _u64, _int, _p],
    ),
    "oslo_softmax_bias_fwd": (
        _int,
        [_p, _p, _p, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _int, _int, _f32, _int, _p],
    ),
    "oslo_softmax_bias_bwd": (
        _int,
        [_p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _int, _int, _f32, _int, _p],
    ),
    "oslo_softmax_bias_dropout_fwd": (
        _int,
        [_p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _int, _int, _f32, _f32,
         _u64, _u64, _int, _p],
    ),
    "oslo_softmax_bias_dropout_bwd": (
        _int,
        [_p, _p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _int, _int, _f32, _f32,
         _u64, _u64, _int, _p],
    ),
    "oslo_bias_gelu_fwd": (_int, [_p, _p, _p, _i64, _i64, _int, _p]),
    "oslo_bias_gelu_bwd": (_int, [_p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _int, _p]),
    "oslo_bias_dropout_add_fwd": (
        _int,
        [_p, _p, _p, _p, _p, _i64, _i64, _f32, _u64, _u64, _int, _p],
    ),
    "oslo_bias_dropout_add_bwd": (
        _int,
        [_p, _p, _p, _p, _i64, _i64, _i64, _f32, _u64, _u64, _int, _p],
    ),
    "oslo_bias_dropout_add_norm_fwd": (
        _int,
        [_p, _p, _p, _p, _p, _p, _p, _p, _p, _i64, _i64, _f64, _f32, _u64, _u64, _int,
         _int, _p],
    ),
    "oslo_bias_dropout_add_norm_bwd": (
        _int,
        [_p, _p, _p, _p, _p, _p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _f32, _u64,
         _u64, _int, _int, _p],
    ),
    "oslo_multi_tensor_adam": (
        _int,
        [_p, _p, _p, _p, _p, _i64, _f32, _f32, _f32, _f32, _int, _int, _int, _f32, _int, _p],
    ),
    "oslo_multi_tensor_sgd": (
        _int,
        [_p, _p, _p, _p, _p, _i64, _f32, _f32, _f32, _f32, _int, _int, _int, _f32, _int, _int,
         _int, _p, _p],
    ),
    "oslo_multi_tensor_adagrad": (_int, [_p, _p, _p, _p, _i64, _f32, _f32, _int, _f32, _int, _p]),
    "oslo_multi_tensor_novograd": (
        _int,
        [_p, _p, _p, _p, _i64, _p, _f32, _f32, _f32, _f32, _int, _int, _f32, _int, _int, _int, _p],
    ),
    "oslo_multi_tensor_lamb_stage1": (
        _int,
        [_p, _p, _p, _p, _p, _i64, _f32, _f32, _f32, _int, _int, _f32, _int, _int, _p, _f32,
         _int, _p],
    ),
    "oslo_multi_tensor_lamb_stage2": (
        _int, [_p, _p, _p, _i64, _p, _p, _f32, _f32, _int, _int, _p],
    ),
    "oslo_multi_tensor_norm_partials": (_i64, [_p, _i64, _int]),
    "oslo_multi_tensor_norm": (
        _int, [_p, _p, _i64, _int, _p, _i64, _p, _p, _int, _int, _f32, _f32, _p, _int, _p],
    ),
    "oslo_multi_tensor_lamb_mp_stage1": (
        _int,
        [_p, _p, _p, _p, _p, _i64, _f32, _f32, _f32, _p, _int, _f32, _int, _int, _p, _p, _p, _p,
         _int, _int, _p],
    ),
    "oslo_multi_tensor_lamb_mp_stage2": (
        _int, [_p, _p, _p, _p, _i64, _p, _p, _p, _f32, _int, _p, _int, _int, _p],
    ),
    "oslo_rng_from_device": (_int, [_p]),
    "oslo_philox_mask": (_int, [_p, _i64, _f32, _u64, _u64, _p]),
    "oslo_philox_words": (_int, [_p, _i64, _i64, _u64, _u64, _p]),
    "oslo_copy_probe": (_int, [_p, _p, _i64, _p]),
    "oslo_colsum_finalize_probe": (_int, [_p, _i64, _i64, _p, _p, _p, _int, _p]),
    "oslo_wave_reduce_selftest": (_int, [_p, _p]),
    "oslo_tune": (_int, [ctypes.c_char_p, _int]),
}

EXPORTED_SYMBOLS = tuple(_SIGNATURES)


def build_library(force=False):
    """Compiles ``liboslo_hip.so`` and the native side of this module in place
    with hipcc (``make`` in ``csrc``)."""
    cmd = ["make", "-C", _CSRC_DIR, "-j8", "PYTHON=" + sys.executable]
    if force:
        subprocess.run(["make", "-C", _CSRC_DIR, "clean"], check=True,
                       stdout=subprocess.DEVNULL)
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        raise EnvironmentError(
            "Failed compiling the HIP kernels for gfx950 (%s):\n%s"
            % (" ".join(cmd), proc.stdout[-4000:])
        )
    return LIBRARY_PATH


def load_library():
    """Returns the ctypes handle, loading (and if absent, building) the library."""
    global _lib
    if _lib is not None:
        return _lib
    with _lib_lock:
        if _lib is not None:
            return _lib
        if not os.path.exists(LIBRARY_PATH):
            build_library()
        try:
            lib = ctypes.CDLL(LIBRARY_PATH)
            for name, (restype, argtypes) in _SIGNATURES.items():
                fn = getattr(lib, name)
                fn.restype = restype
                fn.argtypes = argtypes
            if lib.oslo_hip_abi_version() != ABI_VERSION:
                raise OSError(
                    "ABI version %d, expected %d"
                    % (lib.oslo_hip_abi_version(), ABI_VERSION)
                )
        except (OSError, AttributeError) as exc:
            raise EnvironmentError(
                "Failed loading the HIP kernels (%s): %s. Rebuild with "
                "`make -C %s`." % (LIBRARY_PATH, exc, _CSRC_DIR)
            ) from exc
        _lib = lib
    return _lib


def load_calls():
    """Returns the extension module with the native side of the kernel objects."""
    global _calls
    if _calls is not None:
        return _calls
    load_library()
    with _lib_lock:
        if _calls is not None:
            return _calls
        if not os.path.exists(CALLS_PATH):
            build_library()
        try:
            loader = importlib.machinery.ExtensionFileLoader("oslo_torch_calls", CALLS_PATH)
            module = importlib.util.module_from_spec(
                importlib.util.spec_from_loader("oslo_torch_calls", loader))
            loader.exec_module(module)
        except (ImportError, OSError) as exc:
            raise EnvironmentError(
                "Failed loading the HIP kernels (%s): %s. Rebuild with "
                "`make -C %s`." % (CALLS_PATH, exc, _CSRC_DIR)
            ) from exc
        _calls = module
    return _calls


def _check(rc, lib):
    if rc != 0:
        raise RuntimeError(lib.oslo_hip_last_error().decode("utf-8", "replace"))


def _ptr(t):
    return None if t is None else t.data_ptr()


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream(t):
    """Handle of torch's current stream on the tensor's device."""
    if _raw_stream is not None:
        return _raw_stream(t.device.index)
    return torch.cuda.current_stream(t.device).cuda_stream


class _SameDevice:
    def __enter__(self):
        return None

    def __exit__(self, *exc):
        return False


_SAME_DEVICE = _SameDevice()


def _device_of(t):
    """Context that makes the tensor's device current; nothing to do (and
    nothing allocated) when it already is."""
    if t.device.index == torch.cuda.current_device():
        return _SAME_DEVICE
    return torch.cuda.device_of(t)


def _dtype_code(t, what):
    try:
        return _DTYPE_CODE[t.dtype]
    except KeyError:
        raise RuntimeError(
            "%s: dtype %s is not supported by the HIP kernels "
            "(float32, float16 and bfloat16 are; float64 only by the norms)"
            % (what, t.dtype)
        ) from None


def _check_input(t, name):
    # CHECK_INPUT of FusedLayerNormBinder.cpp:8-14
    if not t.is_cuda:
        raise RuntimeError("%s must be a CUDA tensor" % name)
    if not t.is_contiguous():
        raise RuntimeError("%s must be contiguous" % name)


# Backward workspaces (fp32 partial rows of the parameter gradients).  A backward
# entry point enqueues two launches, the main kernel that writes the partial rows
# and the finalize kernel that reads them, so a workspace must not be handed to
# another call before both launches of this one are on the stream:
#   * eager calls share one workspace per (device, stream, op), grown on demand;
#     the slot's lock is held from the moment the workspace is picked until the C
#     call has returned.  Calls that share a stream are then ordered on it as
#     whole calls (two host threads on one stream cannot interleave their
#     launches); calls on different streams or devices never share a workspace;
#   * a call under stream capture neither reads nor writes the cache: it gets a
#     workspace of its own, which the graph's private pool then owns.  Two graphs
#     never share partial rows, deleting one graph cannot free memory another one
#     points at, and the cached tensors are never referenced by a graph, so
#     replacing one by a larger one is always safe.
class _WorkspaceSlot:
    __slots__ = ("lock", "tensor")

    def __init__(self):
        self.lock = threading.Lock()
        self.tensor = None


class _WorkspaceLease:
    """``with lease as ws:`` -> ``ws.tensor`` (None when the call needs no
    workspace) and ``ws.nbytes`` for the duration of one C call."""

    __slots__ = ("tensor", "nbytes", "_cache", "_key", "_slot")

    def __init__(self, cache=None, key=None, nbytes=0):
        self.tensor, self.nbytes = None, nbytes
        self._cache, self._key, self._slot = cache, key, None

    def __enter__(self):
        cache = self._cache
        if cache is None or self.nbytes <= 0:
            return self
        if cache.capturing():
            self.tensor = cache.allocate(self.nbytes, self._key[0])
            return self
        slot = cache.slots.get(self._key)
        if slot is None:
            slot = cache.slots.setdefault(self._key, _WorkspaceSlot())
        slot.lock.acquire()
        self._slot = slot
        try:
            ws = slot.tensor
            if ws is None or ws.numel() < self.nbytes:
                # (round up so that a sweep over growing shapes settles quickly)
                size = max(self.nbytes, 16)
                if size > (1 << 16):
                    size = (size + (1 << 20) - 1) & ~((1 << 20) - 1)
                ws = slot.tensor = cache.allocate(size, self._key[0])
            self.tensor = ws
        except BaseException:
            self._slot = None
            slot.lock.release()
            raise
        return self

    def __exit__(self, *exc):
        slot, self._slot = self._slot, None
        if slot is not None:
            slot.lock.release()
        return False


class _WorkspaceCache:
    def __init__(self, allocate, capturing):
        self.slots = {}
        self.allocate = allocate    # (nbytes, device index) -> uint8 tensor
        self.capturing = capturing  # () -> bool: the current stream is being captured

    def lease(self, index, stream, op, nbytes):
        return _WorkspaceLease(self, (index, stream, op), nbytes)


def _allocate_workspace(nbytes, index):
    return torch.empty(nbytes, dtype=torch.uint8, device=torch.device("cuda", index))


_ws_cache = _WorkspaceCache(_allocate_workspace, torch.cuda.is_current_stream_capturing)
_ws_bytes_cache = {}
_NO_WORKSPACE = _WorkspaceLease()


def _workspace(lib, op, n1, n2, device):
    """Lease of the workspace of backward op `op` on an [n1, n2] problem."""
    key = (op, n1, n2)
    nbytes = _ws_bytes_cache.get(key)
    if nbytes is None:
        nbytes = int(lib.oslo_workspace_bytes(op, n1, n2))
        if nbytes < 0:
            _check(nbytes, lib)
        if len(_ws_bytes_cache) < 4096:
            _ws_bytes_cache[key] = nbytes
    index = device.index if device.index is not None else torch.cuda.current_device()
    stream = _raw_stream(index) if _raw_stream is not None else torch.cuda.current_stream(device).cuda_stream
    return _ws_cache.lease(index, stream, op, nbytes)


def _leases(lib, op):
    """What a native backward calls for its workspace, once it has checked its
    operands: ``(n1, n2, device)`` -> lease."""
    return lambda n1, n2, device: _workspace(lib, op, n1, n2, device)


class device_rng:
    """Within the block, the dropout entry points called on this host thread
    read (seed, offset) from ``state`` -- two 64-bit integers in device memory --
    when their kernels run, and add their ``offset`` argument to it; their
    ``seed`` argument is ignored.  ``state`` None makes the block a no-op.
    Launches captured in a graph then draw a new mask on every replay."""

    def __init__(self, state):
        if state is not None:
            if not (state.is_cuda and state.is_contiguous() and state.numel() == 2
                    and state.element_size() == 8):
                raise RuntimeError("device_rng: two 64-bit integers on the GPU expected")
        self._state = state

    def __enter__(self):
        if self._state is not None:
            lib = load_library()
            _check(lib.oslo_rng_from_device(self._state.data_ptr()), lib)
        return self

    def __exit__(self, *exc):
        if self._state is not None:
            lib = load_library()
            lib.oslo_rng_from_device(None)
        return False


def tune(key, value):
    """Overrides a launch heuristic of the library (0 restores the default)."""
    lib = load_library()
    _check(lib.oslo_tune(key.encode(), int(value)), lib)
    _ws_bytes_cache.clear()  # workspace sizes depend on the launch shapes


class _Kernel:
    """What the kernel objects of the layer ops share."""

    def __init__(self, lib):
        self._lib = lib
        self._calls = load_calls()
        self._attributes = None

    def replaced(self):
        """Whether a method was replaced on this object (not on its class)."""
        if len(self.__dict__) == self._attributes:
            return False
        # (a method that was put back is an attribute of the object still)
        return any(getattr(v, "__func__", None) is not getattr(type(self), name)
                   for name, v in self.__dict__.items() if hasattr(type(self), name))

    def _built(self):
        self._attributes = len(self.__dict__)


# ---------------------------------------------------------------------------
# LayerNorm / RMSNorm
# ---------------------------------------------------------------------------
class _LayerNormKernel(_Kernel):
    """The ten functions of the reference's ``oslo_fused_layer_norm`` module."""

    def __init__(self, lib):
        super().__init__(lib)
        self._leases = [_leases(lib, op) for op in
                        (OSLO_OP_LN_BWD, OSLO_OP_RMS_BWD, OSLO_OP_BIAS_DROPOUT_ADD_NORM_BWD)]
        self._built()

    # -- forward ----------------------------------------------------------
    def layer_norm_forward(self, input, normalized_shape, eps):
        return self._calls.norm_forward(False, input, normalized_shape, None, None, eps, False)

    def layer_norm_forward_affine(self, input, normalized_shape, gamma, beta, eps):
        return self._calls.norm_forward(False, input, normalized_shape, gamma, beta, eps, False)

    def layer_norm_forward_affine_mixed_dtypes(self, input, normalized_shape, gamma, beta, eps):
        return self._calls.norm_forward(False, input, normalized_shape, gamma, beta, eps, True)

    def rms_norm_forward(self, input, normalized_shape, eps):
        return self._calls.norm_forward(True, input, normalized_shape, None, None, eps, False)

    def rms_norm_forward_affine(self, input, normalized_shape, gamma, eps):
        return self._calls.norm_forward(True, input, normalized_shape, gamma, None, eps, False)

    def rms_norm_forward_affine_mixed_dtypes(self, input, normalized_shape, gamma, eps):
        return self._calls.norm_forward(True, input, normalized_shape, gamma, None, eps, True)

    # -- backward ---------------------------------------------------------
    def _backward(self, rms, dout, mean, invvar, input, normalized_shape, gamma, beta):
        return self._calls.norm_backward(
            rms, dout, mean, invvar, input, normalized_shape, gamma, beta,
            None if gamma is None else self._leases[1 if rms else 0],
        )

    def layer_norm_backward(self, dout, mean, invvar, input, normalized_shape, eps):
        return self._backward(False, dout, mean, invvar, input, normalized_shape, None, None)[0]

    def layer_norm_backward_affine(
        self, dout, mean, invvar, input, normalized_shape, gamma, beta, eps
    ):
        return list(
            self._backward(False, dout, mean, invvar, input, normalized_shape, gamma, beta)
        )

    def rms_norm_backward(self, dout, invvar, input, normalized_shape, eps):
        return self._backward(True, dout, None, invvar, input, normalized_shape, None, None)[0]

    def rms_norm_backward_affine(self, dout, invvar, input, normalized_shape, gamma, eps):
        gi, gg, _ = self._backward(
            True, dout, None, invvar, input, normalized_shape, gamma, None
        )
        return [gi, gg]

    # -- bias-dropout-add fused into the norm (no counterpart in the
    #    reference's module: its models chain FusedBiasDropout, the residual
    #    add and LayerNorm, oslo/transformers/models/bert/modeling_bert.py:
    #    343-346) ----------------------------------------------------------
    def bias_dropout_add_norm_forward(
        self, rms, input, bias, residual, normalized_shape, gamma, beta, eps,
        p, seed, offset, want_h=True,
    ):
        """``h = dropout(input + bias, p) + residual; y = norm(h)``.

        Returns ``[y, h, mean, invvar]`` (``h`` None when ``want_h`` is false,
        ``mean`` None for RMSNorm).  One dtype throughout.
        """
        return self._calls.residual_norm_forward(
            rms, input, bias, residual, normalized_shape, gamma, beta, eps, p, seed, offset, want_h
        )

    def bias_dropout_add_norm_backward(
        self, rms, dout, dh_extra, h, mean, invvar, normalized_shape, gamma,
        p, seed, offset, need_bias_grad=True,
    ):
        """Returns ``(grad_residual, grad_input, grad_gamma, grad_beta, grad_bias)``;
        ``grad_input`` is ``grad_residual`` itself when ``p == 0``."""
        return self._calls.residual_norm_backward(
            rms, dout, dh_extra, h, mean, invvar, normalized_shape, gamma, p, seed, offset,
            need_bias_grad, self._leases[2] if gamma is not None or need_bias_grad else None,
        )


# ---------------------------------------------------------------------------
# scaled masked softmax
# ---------------------------------------------------------------------------
# The softmax backward streams three tensors of gigabytes at identical offsets
# (y, dy -> dx).  torch places large tensors on 2 MiB boundaries; when all three
# start on the same 2 MiB phase their requests meet in the same memory channels
# and the kernel measures 1.5-4 % slower on MI355X than with the starts a little
# over 1 MiB apart.  The tensors this binding allocates for the softmax (the
# probabilities in forward, the input gradient in backward) are therefore placed
# on phase k * (1 MiB + 4 KiB) of their own 2 MiB-rounded allocation, k = 1 for
# forward outputs and k = 2 for backward outputs; operands that torch allocated
# (the scores, the incoming gradient) sit on phase 0.
STAGGER_MIN_BYTES = 64 << 20
STAGGER_STEP = (1 << 20) + 4096
_STAGGER_ROUND = 2 << 20


def empty_staggered(shape, dtype, device, k):
    """An uninitialised contiguous tensor whose first byte lies k * STAGGER_STEP
    (modulo 2 MiB) past a 2 MiB boundary; small tensors and k == 0 are plain
    ``torch.empty``.  Costs 2 MiB of slack per tensor."""
    n = 1
    for d in shape:
        n *= int(d)
    nbytes = n * torch.empty(0, dtype=dtype).element_size()
    if k == 0 or nbytes < STAGGER_MIN_BYTES:
        return torch.empty(tuple(shape), dtype=dtype, device=device)
    base = torch.empty(nbytes + _STAGGER_ROUND, dtype=torch.uint8, device=device)
    off = (k * STAGGER_STEP - base.data_ptr()) % _STAGGER_ROUND
    return base[off:off + nbytes].view(dtype).view(tuple(shape))


class _SoftmaxKernel(_Kernel):
    """The five functions of ``FusedScaleMaskSoftmaxBinder.cpp:111-127``.

    The reference admits fp16 / bf16 only (``:42-44, 84-86``); fp32 is accepted
    here as well.  ``fused_scaled_masked_softmax_backward`` takes an optional
    ``mask`` (not in the reference signature) that lets the kernel skip loads
    of masked keys.
    """

    def __init__(self, lib):
        super().__init__(lib)
        self._built()

    def fused_scaled_masked_softmax_forward(self, input, mask, scale_factor, causal=False):
        """``causal=True`` (not in the reference's shim) hides the keys beyond
        the diagonal as well: causal attention on a padded batch."""
        return self._calls.masked_forward(input, mask, scale_factor, causal)

    def fused_scaled_masked_softmax_backward(
        self, output_grads, softmax_results, scale_factor, mask=None, inplace=False,
        causal=False,
    ):
        # inplace=True overwrites output_grads, as the kernel this shim was
        # written for does
        return self._calls.masked_backward(
            output_grads, softmax_results, scale_factor, mask, inplace, causal
        )

    def get_batch_per_block(self, query_seq_len, key_seq_len, batches, attn_heads):
        lib = self._lib
        rc = lib.oslo_softmax_batch_per_block(
            int(query_seq_len), int(key_seq_len), int(batches), int(attn_heads)
        )
        if rc < 0:
            _check(rc, lib)
        return int(rc)

    def fused_scaled_upper_triang_masked_softmax_forward(self, input, scale_factor):
        return self._calls.causal_forward(input, scale_factor)

    def fused_scaled_upper_triang_masked_softmax_backward(
        self, output_grads, softmax_results, scale_factor, inplace=False
    ):
        return self._calls.causal_backward(output_grads, softmax_results, scale_factor, inplace)

    # -- softmax with the attention dropout fused in (no counterpart in the
    #    reference's shim: the models apply nn.Dropout to the probabilities,
    #    oslo/transformers/models/gpt2/modeling_gpt2.py:138-142) -------------
    def softmax_dropout_forward(self, input, mask, scale_factor, p, seed, offset, causal=False):
        """``dropout(softmax(mask(scale * input)), p)`` -> ``[out, stats]``.

        ``mask=None`` selects the causal form on a 3-D ``[attn_batches, sq, sk]``
        input, otherwise ``input`` is ``[b, np, sq, sk]`` and ``mask`` a 4-D
        padding mask (with ``causal=True`` the keys beyond the diagonal are
        hidden as well).  ``stats`` (float32 ``[rows, 2]``) and ``input`` are
        what the backward pass needs.
        """
        return self._calls.dropout_forward(
            input, mask, scale_factor, p, seed, offset, causal
        )

    def softmax_dropout_backward(
        self, output_grads, input, stats, mask, scale_factor, p, seed, offset,
        inplace=False, causal=False,
    ):
        return self._calls.dropout_backward(
            output_grads, input, stats, mask, scale_factor, p, seed, offset, inplace, causal
        )

    # -- softmax with an additive floating-point term (no counterpart in the
    #    reference's shim; its models add the term to the scores with torch,
    #    oslo/transformers/models/bert/modeling_bert.py:298-306) -------------
    @staticmethod
    def _bias_operand(bias, input):
        """The additive term as the kernel addresses it: ``(tensor, stride_b,
        stride_h, stride_q, dtype_code)``.  ``bias`` broadcasts against the 4-D
        ``input``: up to four dimensions, each of the leading three either 1 or
        the full size (expanded views are fine: their stride is 0), the keys
        contiguous; its dtype becomes the input's or float32."""
        return load_calls().bias_operand(bias, input)

    @staticmethod
    def _bias_flags(causal, skip_hidden, strides, forward):
        return load_calls().bias_flags(causal, skip_hidden, strides[1], strides[2], forward)

    def softmax_bias_forward(self, input, bias, scale_factor, causal=False, skip_hidden=None):
        """``softmax(scale * input + bias)`` over the last dimension of the
        ``[b, np, sq, sk]`` input; ``causal`` hides the keys beyond the diagonal
        as well.  ``skip_hidden`` (default: off in the forward passes, on in the
        backward passes when the term is shared by heads or queries) lets the
        kernel leave logits unread whose term is -inf or the lowest finite value."""
        return self._calls.bias_forward(input, bias, scale_factor, causal, skip_hidden)

    def softmax_bias_backward(
        self, output_grads, softmax_results, scale_factor, bias=None, causal=False,
        skip_hidden=None, inplace=False,
    ):
        """``scale * y * (g - sum(g * y))``; ``bias`` (optional) only lets the
        kernel skip loads, as in the forward pass."""
        return self._calls.bias_backward(
            output_grads, softmax_results, scale_factor, bias, causal, skip_hidden, inplace
        )

    def softmax_bias_dropout_forward(
        self, input, bias, scale_factor, p, seed, offset, causal=False, skip_hidden=None
    ):
        """``dropout(softmax(scale * input + bias), p)`` -> ``[out, stats]``."""
        return self._calls.bias_dropout_forward(
            input, bias, scale_factor, p, seed, offset, causal, skip_hidden
        )

    def softmax_bias_dropout_backward(
        self, output_grads, input, bias, stats, scale_factor, p, seed, offset,
        causal=False, skip_hidden=None, inplace=False,
    ):
        return self._calls.bias_dropout_backward(
            output_grads, input, bias, stats, scale_factor, p, seed, offset, causal, skip_hidden,
            inplace,
        )


# ---------------------------------------------------------------------------
# bias-GeLU and bias-dropout-add (TorchScript in the reference,
# oslo/torch/nn/modules/functional.py:23-50, 295-298; native here)
# ---------------------------------------------------------------------------
class _FusedElementwiseKernel(_Kernel):
    def __init__(self, lib):
        super().__init__(lib)
        self._gelu_leases = _leases(lib, OSLO_OP_BIAS_GELU_BWD)
        self._dropout_leases = _leases(lib, OSLO_OP_BIAS_DROPOUT_ADD_BWD)
        self._built()

    def bias_gelu_forward(self, input, bias):
        return self._calls.gelu_forward(input, bias)

    def bias_gelu_backward(self, grad_output, input, bias, need_bias_grad=True):
        return self._calls.gelu_backward(
            grad_output, input, bias, need_bias_grad,
            self._gelu_leases if bias is not None and need_bias_grad else None,
        )

    def bias_dropout_add_forward(
        self, input, bias, residual, p, seed, offset, out=None, return_mask=False
    ):
        result = self._calls.dropout_add_forward(
            input, bias, residual, p, seed, offset, out, return_mask
        )
        return result if return_mask else result[0]

    def bias_dropout_add_backward(
        self, grad_output, p, seed, offset, need_input_grad=True, need_bias_grad=True
    ):
        return self._calls.dropout_add_backward(
            grad_output, p, seed, offset, need_input_grad, need_bias_grad,
            self._dropout_leases if need_bias_grad else None,
        )

    def philox_mask(self, n, p, seed, offset, device):
        lib = self._lib
        mask = torch.empty(int(n), dtype=torch.uint8, device=device)
        with torch.cuda.device(mask.device):
            rc = lib.oslo_philox_mask(
                _ptr(mask), int(n), float(p), int(seed), int(offset), _stream(mask)
            )
            _check(rc, lib)
        return mask

    def philox_words(self, ngroups, first_group, seed, offset, device):
        lib = self._lib
        out = torch.empty(int(ngroups) * 4, dtype=torch.int32, device=device)
        with torch.cuda.device(out.device):
            rc = lib.oslo_philox_words(
                _ptr(out), int(ngroups), int(first_group), int(seed), int(offset),
                _stream(out),
            )
            _check(rc, lib)
        return out

    def copy_probe(self, src, dst):
        lib = self._lib
        nbytes = src.numel() * src.element_size()
        with _device_of(src):
            _check(lib.oslo_copy_probe(_ptr(src), _ptr(dst), nbytes, _stream(src)), lib)
        return dst

    def wave_reduce_selftest(self, device):
        lib = self._lib
        out = torch.zeros(4, dtype=torch.float32, device=device)
        with torch.cuda.device(out.device):
            _check(lib.oslo_wave_reduce_selftest(_ptr(out), _stream(out)), lib)
        return out


_layernorm_kernel = None
_softmax_kernel = None
_elementwise_kernel = None


def get_layernorm_kernel():
    global _layernorm_kernel
    if _layernorm_kernel is None:
        _layernorm_kernel = _LayerNormKernel(load_library())
    return _layernorm_kernel


def get_softmax_kernel():
    global _softmax_kernel
    if _softmax_kernel is None:
        _softmax_kernel = _SoftmaxKernel(load_library())
    return _softmax_kernel


# ---------------------------------------------------------------------------
# multi-tensor optimizer steps
# ---------------------------------------------------------------------------
def _tensor_tables(tensor_lists, names, dtypes=None):
    """Checks lists of equally long, pairwise equally sized contiguous GPU
    tensors (the checks of the reference's multi_tensor_apply.cuh:44-72) and
    returns ``(pointer tables, sizes, n, first tensor)``; ``dtypes[k]`` None
    means list k follows the dtype of its first tensor."""
    n = len(tensor_lists[0])
    for lst in tensor_lists:
        if len(lst) != n:
            raise RuntimeError("Size mismatch among tensor lists")
    if n == 0:
        return None, None, 0, None
    ref = tensor_lists[0][0]
    device = ref.device
    counts = [t.numel() for t in tensor_lists[0]]
    for k, lst in enumerate(tensor_lists):
        want = lst[0].dtype if dtypes is None or dtypes[k] is None else dtypes[k]
        # one pass per list; the slow loop below only runs to name the offender
        if all(t.is_cuda and t.dtype == want and t.device == device and t.is_contiguous() for t in lst):
            if k == 0 or [t.numel() for t in lst] == counts:
                continue
        for i, t in enumerate(lst):
            _check_input(t, "%s %d" % (names[k], i))
            if t.dtype != want or t.device != device:
                raise RuntimeError(
                    "A tensor was not the same dtype / on the same device as the first tensor"
                )
            if t.numel() != counts[i]:
                raise RuntimeError("Size mismatch among tensor lists")
    arr = ctypes.c_void_p * n
    sizes = (ctypes.c_int64 * n)(*counts)
    tables = [arr(*[t.data_ptr() for t in lst]) for lst in tensor_lists]
    return tables, sizes, n, ref


class _AdamKernel:
    """``multi_tensor_adam`` of the reference's ``oslo_fused_adam`` module
    (``oslo/torch/_C/csrc/FusedAdamBinder.cpp:12-15``), same argument list."""

    def __init__(self, lib):
        self._lib = lib

    def multi_tensor_adam(
        self, chunk_size, noop_flag, tensor_lists, lr, beta1, beta2, epsilon, step,
        mode, bias_correction, weight_decay,
    ):
        """``tensor_lists`` = ``[grads, params, exp_avgs, exp_avg_sqs]``, updated in
        place.  ``chunk_size`` and ``noop_flag`` are accepted for signature
        compatibility; the reference's kernel does not act on them either
        (``multi_tensor_adam.cu:29-31``)."""
        lib = self._lib
        if len(tensor_lists) != 4:
            raise RuntimeError("tensor_lists must hold [grads, params, exp_avgs, exp_avg_sqs]")
        names = ("grad", "param", "exp_avg", "exp_avg_sq")
        ref_dtype = tensor_lists[1][0].dtype if len(tensor_lists[1]) else None
        tables, sizes, n, ref = _tensor_tables(tensor_lists, names, [ref_dtype] * 4)
        if n == 0:
            return
        code = _dtype_code(ref, "params[0]")
        with _device_of(ref):
            rc = lib.oslo_multi_tensor_adam(
                tables[0], tables[1], tables[2], tables[3], sizes, n, float(lr), float(beta1),
                float(beta2), float(epsilon), int(step), int(mode), int(bias_correction),
                float(weight_decay), code, _stream(ref),
            )
            _check(rc, lib)


def _flag_ptr(noop_flag, ref):
    """Device pointer of the overflow flag (an int32 tensor), or None."""
    if noop_flag is None:
        return None
    if not (noop_flag.is_cuda and noop_flag.dtype == torch.int32 and noop_flag.numel() >= 1):
        raise RuntimeError("noop_flag must be an int32 tensor on the GPU")
    if ref is not None and noop_flag.device != ref.device:
        raise RuntimeError("expected noop flag to be on the same device as tensors")
    return noop_flag.data_ptr()


class _SGDKernel:
    """``multi_tensor_sgd`` of ``oslo/torch/_C/csrc/FusedSGDBinder.cpp``."""

    def __init__(self, lib):
        self._lib = lib

    def multi_tensor_sgd(
        self, chunk_size, noop_flag, tensor_lists, wd, momentum, dampening, lr, nesterov,
        first_run, wd_after_momentum, scale,
    ):
        """``tensor_lists`` = ``[grads, weights, momentum buffers]`` or, with a
        fourth list, additionally 16-bit copies of the updated float32 weights
        (``multi_tensor_sgd.cu:139-201``).  Nothing happens while ``noop_flag``
        is non-zero."""
        lib = self._lib
        if len(tensor_lists) not in (3, 4):
            raise RuntimeError("tensor_lists must hold [grads, weights, momentums(, weight copies)]")
        names = ("grad", "weight", "momentum", "weight copy")
        wdtype = tensor_lists[1][0].dtype if len(tensor_lists[1]) else None
        dts = [None, wdtype, wdtype, None][: len(tensor_lists)]
        tables, sizes, n, ref = _tensor_tables(tensor_lists, names, dts)
        if n == 0:
            return
        copy = len(tensor_lists) == 4
        if copy and tensor_lists[3][0].dtype not in (torch.float16, torch.bfloat16):
            raise RuntimeError("Additional output tensors should always be fp16 (or bf16).")
        with _device_of(ref):
            rc = lib.oslo_multi_tensor_sgd(
                tables[0], tables[1], tables[2], tables[3] if copy else None, sizes, n,
                float(wd), float(momentum), float(dampening), float(lr), int(bool(nesterov)),
                int(bool(first_run)), int(bool(wd_after_momentum)), float(scale),
                _dtype_code(tensor_lists[0][0], "grads[0]"),
                _dtype_code(tensor_lists[1][0], "weights[0]"),
                _dtype_code(tensor_lists[3][0], "copies[0]") if copy else 0,
                _flag_ptr(noop_flag, ref), _stream(ref),
            )
            _check(rc, lib)


class _AdagradKernel:
    """``multi_tensor_adagrad`` of ``oslo/torch/_C/csrc/FusedAdagradBinder.cpp``."""

    def __init__(self, lib):
        self._lib = lib

    def multi_tensor_adagrad(self, chunk_size, noop_flag, tensor_lists, lr, epsilon, mode,
                             weight_decay):
        """``tensor_lists`` = ``[grads, params, sums of squares]``, one dtype."""
        lib = self._lib
        if len(tensor_lists) != 3:
            raise RuntimeError("tensor_lists must hold [grads, params, sums]")
        d = tensor_lists[0][0].dtype if len(tensor_lists[0]) else None
        tables, sizes, n, ref = _tensor_tables(tensor_lists, ("grad", "param", "sum"), [d] * 3)
        if n == 0:
            return
        # (an int32 tensor on the GPU, which multi_tensor_apply.cuh:100 takes the pointer
        #  of; the update itself does not read it, multi_tensor_adagrad.cu:26-80)
        _flag_ptr(noop_flag, ref)
        with _device_of(ref):
            rc = lib.oslo_multi_tensor_adagrad(
                tables[0], tables[1], tables[2], sizes, n, float(lr), float(epsilon), int(mode),
                float(weight_decay), _dtype_code(ref, "grads[0]"), _stream(ref),
            )
            _check(rc, lib)


class _L2NormKernel:
    """``multi_tensor_l2norm`` of ``oslo/torch/_C/csrc/FusedL2NormBinder.cpp``,
    and ``norm_out``, the blend into stored per-tensor norms that the
    reference's NovoGrad step calls internally
    (``multi_tensor_l2norm.cu:323-385``)."""

    def __init__(self, lib):
        self._lib = lib

    def _run(self, tensors, out_global, out_per_tensor, norm_type, blend, alpha, beta, noop_flag,
             skip_if_flag=False):
        lib = self._lib
        tables, sizes, n, ref = _tensor_tables([tensors], ("tensor",))
        code = _dtype_code(ref, "tensors[0]")
        need = int(lib.oslo_multi_tensor_norm_partials(sizes, n, code))
        if need < 0:
            _check(need, lib)
        partials = torch.empty(need, dtype=torch.float32, device=ref.device)
        with _device_of(ref):
            rc = lib.oslo_multi_tensor_norm(
                tables[0], sizes, n, code, _ptr(partials), need, _ptr(out_global),
                _ptr(out_per_tensor), int(norm_type), int(blend), float(alpha), float(beta),
                _flag_ptr(noop_flag, ref), int(bool(skip_if_flag)), _stream(ref),
            )
            _check(rc, lib)

    def multi_tensor_l2norm_mp(self, chunk_size, noop_flag, tensor_lists, per_tensor=False):
        """``multi_tensor_l2norm`` that does nothing while ``noop_flag`` is
        raised: the results then hold whatever their memory held
        (``oslo/torch/_C/csrc/FusedMixedPrecisionL2NormBinder.cpp``,
        ``multi_tensor_l2norm_mp.cu:33-35, 113-115``)."""
        if noop_flag is None:
            raise RuntimeError("multi_tensor_l2norm_mp needs the overflow flag")
        return self.multi_tensor_l2norm(chunk_size, noop_flag, tensor_lists, per_tensor,
                                        _skip_if_flag=True)

    def multi_tensor_l2norm(self, chunk_size, noop_flag, tensor_lists, per_tensor=False,
                            _skip_if_flag=False):
        """Returns ``(norm over all tensors [1], norm of each tensor [n] or an
        empty tensor)``, float32.  A sum that is not finite sets ``noop_flag``."""
        if len(tensor_lists) != 1:
            raise RuntimeError("tensor_lists must hold one list")
        tensors = tensor_lists[0]
        if len(tensors) == 0:
            raise RuntimeError("multi_tensor_l2norm: no tensors")
        dev = tensors[0].device
        ret = torch.empty(1, dtype=torch.float32, device=dev)
        ret_per_tensor = torch.empty(len(tensors) if per_tensor else 0, dtype=torch.float32,
                                     device=dev)
        self._run(tensors, ret, ret_per_tensor if per_tensor else None, 2, 0, 0.0, 0.0, noop_flag,
                  _skip_if_flag)
        return ret, ret_per_tensor

    def multi_tensor_norm_out(self, chunk_size, noop_flag, tensor_lists, out, alpha, beta,
                              norm_type):
        """``out[t] = sqrt(alpha * out[t]**2 + beta * |x_t|_2**2)`` (``norm_type``
        2) or ``alpha * out[t] + beta * max|x_t|`` (``norm_type`` 0), in place."""
        tensors = tensor_lists[0]
        if len(tensors) == 0:
            return
        _check_input(out, "out")
        if out.dtype != torch.float32 or out.numel() != len(tensors):
            raise RuntimeError("out must be float32 with one element per tensor")
        if norm_type not in (0, 2):
            raise RuntimeError("only the L2 norm (2) and the max norm (0) are supported")
        self._run(tensors, None, out, norm_type, 1, alpha, beta, noop_flag)


class _NovogradKernel:
    """``multi_tensor_novograd`` of ``oslo/torch/_C/csrc/FusedNovogradBinder.cpp``."""

    def __init__(self, lib):
        self._lib = lib

    def multi_tensor_novograd(
        self, chunk_size, noop_flag, tensor_lists, grad_norms, lr, beta1, beta2, epsilon, step,
        bias_correction, weight_decay, grad_averaging, moment_mode, norm_type,
    ):
        """``tensor_lists`` = ``[grads, params, exp_avgs]``; ``grad_norms`` holds
        one float32 per tensor and is blended with this step's gradient norms
        first, as in the reference's host function
        (``multi_tensor_novograd.cu:131-136``)."""
        lib = self._lib
        if len(tensor_lists) != 3:
            raise RuntimeError("tensor_lists must hold [grads, params, exp_avgs]")
        d = tensor_lists[0][0].dtype if len(tensor_lists[0]) else None
        tables, sizes, n, ref = _tensor_tables(tensor_lists, ("grad", "param", "exp_avg"), [d] * 3)
        if n == 0:
            return
        get_l2norm_kernel().multi_tensor_norm_out(
            chunk_size, noop_flag, [tensor_lists[0]], grad_norms, beta2, 1.0 - beta2, norm_type
        )
        with _device_of(ref):
            rc = lib.oslo_multi_tensor_novograd(
                tables[0], tables[1], tables[2], sizes, n, _ptr(grad_norms), float(lr),
                float(beta1), float(beta2), float(epsilon), int(step), int(bias_correction),
                float(weight_decay), int(grad_averaging), int(moment_mode),
                _dtype_code(ref, "grads[0]"), _stream(ref),
            )
            _check(rc, lib)


class _LambKernel:
    """``multi_tensor_lamb`` of ``oslo/torch/_C/csrc/FusedLambBinder.cpp``."""

    def __init__(self, lib):
        self._lib = lib

    def multi_tensor_lamb(
        self, chunk_size, noop_flag, tensor_lists, lr, beta1, beta2, epsilon, step,
        bias_correction, weight_decay, grad_averaging, mode, global_grad_norm, max_grad_norm,
        use_nvlamb=False,
    ):
        """``tensor_lists`` = ``[grads, params, exp_avgs, exp_avg_sqs]``, one
        dtype; the gradients are overwritten with the update direction
        (``multi_tensor_lamb.cu:313-317``).  ``global_grad_norm`` is a float32
        tensor with the norm of all gradients."""
        lib = self._lib
        if len(tensor_lists) != 4:
            raise RuntimeError("tensor_lists must hold [grads, params, exp_avgs, exp_avg_sqs]")
        names = ("grad", "param", "exp_avg", "exp_avg_sq")
        d = tensor_lists[0][0].dtype if len(tensor_lists[0]) else None
        tables, sizes, n, ref = _tensor_tables(tensor_lists, names, [d] * 4)
        if n == 0:
            return
        _check_input(global_grad_norm, "global_grad_norm")
        if global_grad_norm.dtype != torch.float32 or global_grad_norm.numel() < 1:
            raise RuntimeError("global_grad_norm must be a float32 tensor")
        code = _dtype_code(ref, "grads[0]")
        norms = get_l2norm_kernel()
        _, param_norms = norms.multi_tensor_l2norm(chunk_size, noop_flag, [tensor_lists[1]], True)
        with _device_of(ref):
            rc = lib.oslo_multi_tensor_lamb_stage1(
                tables[0], tables[1], tables[2], tables[3], sizes, n, float(beta1), float(beta2),
                float(epsilon), int(step), int(bias_correction), float(weight_decay),
                int(grad_averaging), int(mode), _ptr(global_grad_norm), float(max_grad_norm),
                code, _stream(ref),
            )
            _check(rc, lib)
        _, update_norms = norms.multi_tensor_l2norm(chunk_size, noop_flag, [tensor_lists[0]], True)
        with _device_of(ref):
            rc = lib.oslo_multi_tensor_lamb_stage2(
                tables[0], tables[1], sizes, n, _ptr(param_norms), _ptr(update_norms), float(lr),
                float(weight_decay), int(bool(use_nvlamb)), code, _stream(ref),
            )
            _check(rc, lib)


def _device_scalar(t, name, dtype, ref):
    """Pointer of a one-element tensor of ``dtype`` on the device of ``ref``."""
    if not (isinstance(t, torch.Tensor) and t.is_cuda and t.dtype == dtype and t.numel() >= 1
            and t.device == ref.device):
        raise RuntimeError("%s must be a %s tensor on %s" % (name, dtype, ref.device))
    return t.data_ptr()


class _LambMpKernel:
    """``multi_tensor_lamb_mp`` of
    ``oslo/torch/_C/csrc/FusedMixedPrecisionLambBinder.cpp``."""

    def __init__(self, lib):
        self._lib = lib

    def multi_tensor_lamb_mp(
        self, chunk_size, noop_flag, tensor_lists, lr, beta1, beta2, epsilon, step,
        bias_correction, weight_decay, grad_averaging, mode, global_grad_norm, max_grad_norm,
        use_nvlamb, found_inf, inv_scale,
    ):
        """``tensor_lists`` = ``[grads, params, exp_avgs, exp_avg_sqs]`` of one
        dtype, or with a fifth list ``[grads, float32 master params, float32
        exp_avgs, float32 exp_avg_sqs, model params of the gradients' dtype]``
        (``multi_tensor_lamb_mp.cu:334-337``).  ``lr``, ``step`` (int32),
        ``global_grad_norm``, ``max_grad_norm`` and ``inv_scale`` are one-element
        tensors on the GPU; nothing is updated while ``noop_flag`` is raised.
        ``found_inf`` is accepted as in the reference, whose kernels do not
        read it either."""
        lib = self._lib
        if len(tensor_lists) not in (4, 5):
            raise RuntimeError("tensor_lists must hold 4 or 5 lists")
        names = ("grad", "param", "exp_avg", "exp_avg_sq", "model param")
        gd = tensor_lists[0][0].dtype if len(tensor_lists[0]) else None
        pd = tensor_lists[1][0].dtype if len(tensor_lists[1]) else None
        master = len(tensor_lists) == 5
        dts = [gd, pd, pd, pd] + ([gd] if master else [])
        tables, sizes, n, ref = _tensor_tables(tensor_lists, names, dts)
        if n == 0:
            return
        if master and pd != torch.float32:
            raise RuntimeError("with five lists the parameters and moments are float32 master values")
        if not master and pd != gd:
            raise RuntimeError("with four lists all tensors share one dtype")
        flag = _flag_ptr(noop_flag, ref)
        if flag is None:
            raise RuntimeError("multi_tensor_lamb_mp needs the overflow flag")
        gcode, pcode = _dtype_code(tensor_lists[0][0], "grads[0]"), _dtype_code(tensor_lists[1][0], "params[0]")
        norms = get_l2norm_kernel()
        _, param_norms = norms.multi_tensor_l2norm_mp(chunk_size, noop_flag, [tensor_lists[1]], True)
        with _device_of(ref):
            rc = lib.oslo_multi_tensor_lamb_mp_stage1(
                tables[0], tables[1], tables[2], tables[3], sizes, n, float(beta1), float(beta2),
                float(epsilon), _device_scalar(step, "step", torch.int32, ref), int(bias_correction),
                float(weight_decay), int(grad_averaging), int(mode),
                _device_scalar(global_grad_norm, "global_grad_norm", torch.float32, ref),
                _device_scalar(max_grad_norm, "max_grad_norm", torch.float32, ref),
                _device_scalar(inv_scale, "inv_scale", torch.float32, ref), flag, gcode, pcode,
                _stream(ref),
            )
            _check(rc, lib)
        _, update_norms = norms.multi_tensor_l2norm_mp(chunk_size, noop_flag, [tensor_lists[0]], True)
        with _device_of(ref):
            rc = lib.oslo_multi_tensor_lamb_mp_stage2(
                tables[0], tables[1], tables[4] if master else None, sizes, n, _ptr(param_norms),
                _ptr(update_norms), _device_scalar(lr, "lr", torch.float32, ref),
                float(weight_decay), int(bool(use_nvlamb)), flag, gcode, pcode, _stream(ref),
            )
            _check(rc, lib)


_optimizer_kernels = {}


def _optimizer_kernel(cls):
    kernel = _optimizer_kernels.get(cls)
    if kernel is None:
        kernel = _optimizer_kernels[cls] = cls(load_library())
    return kernel


def get_adam_kernel():
    return _optimizer_kernel(_AdamKernel)


def get_sgd_kernel():
    return _optimizer_kernel(_SGDKernel)


def get_adagrad_kernel():
    return _optimizer_kernel(_AdagradKernel)


def get_novograd_kernel():
    return _optimizer_kernel(_NovogradKernel)


def get_l2norm_kernel():
    return _optimizer_kernel(_L2NormKernel)


def get_lamb_kernel():
    return _optimizer_kernel(_LambKernel)


def get_l2norm_mp_kernel():
    return _optimizer_kernel(_L2NormKernel)


def get_lamb_mp_kernel():
    return _optimizer_kernel(_LambMpKernel)


def get_fused_elementwise_kernel():
    global _elementwise_kernel
    if _elementwise_kernel is None:
        _elementwise_kernel = _FusedElementwiseKernel(load_library())
    return _elementwise_kernel
