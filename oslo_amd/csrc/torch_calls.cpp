// The per-call host work of the layer ops, in native code, in two layers:
//
// * calls: argument checks, output allocation, the launch through the C ABI
//   (include/oslo_hip.h) and nothing else.  One method per method of the kernel
//   objects in oslo_amd/torch/_C/__init__.py, which document the semantics and
//   own the workspaces of the calls made through them.
// * autograd: the Functions of oslo_amd/torch/nn/modules/functional.py for eager
//   calls on GPU tensors (methods ag_*), on top of the same calls.  That module
//   decides which calls come here; the Python Functions it keeps run the rest
//   (CPU tensors, calls under torch.jit tracing, dropout whose state a captured
//   graph reads from device memory, dropout in place).
//
// Why native: a decoding step or a small layer is bound by the host.  Checks
// and allocations in Python with a ctypes call of twelve to eighteen arguments
// took 9-11 us of a norm's 14.6 us a call, of which the launch is about 3; a
// Python autograd.Function costs another 3 us forward and some 25 us in a
// backward pass, most of them the engine's thread waiting for the GIL.
//
// The GIL is released from the checks to the launch (and taken again around the
// lease of a workspace), so that a launch that blocks (a full queue) does not
// stop other Python threads; a backward pass of an ag_* Function never takes it.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/ExpandUtils.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <optional>
#include <tuple>
#include <vector>

#include "../../include/oslo_hip.h"

namespace {

using at::Tensor;
using Shape = std::vector<int64_t>;

struct Dropout {
  double p;
  uint64_t seed, offset;
};

// ---------------------------------------------------------------- arguments
struct Args {
  PyObject *const *a;
  Py_ssize_t n, i = 0;

  PyObject *next() {
    TORCH_CHECK_TYPE(i < n, "too few arguments");
    return a[i++];
  }
  const Tensor &tensor() {
    PyObject *o = next();
    TORCH_CHECK_TYPE(THPVariable_Check(o), "argument ", i, " must be a Tensor, not ", Py_TYPE(o)->tp_name);
    return THPVariable_Unpack(o);
  }
  // undefined for None
  Tensor optional() {
    if (a[i < n ? i : 0] == Py_None) {
      next();
      return Tensor();
    }
    return tensor();
  }
  bool flag() {
    const int r = PyObject_IsTrue(next());
    if (r < 0) throw python_error();
    return r != 0;
  }
  // None -> -1, else the truth value
  int tristate() {
    if (i < n && a[i] == Py_None) {
      ++i;
      return -1;
    }
    return flag() ? 1 : 0;
  }
  double real() {
    const double v = PyFloat_AsDouble(next());
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return v;
  }
  int64_t integer() {
    const int64_t v = PyLong_AsLongLong(next());
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
  }
  // a callable, null for None
  PyObject *callable() {
    PyObject *o = next();
    return o == Py_None ? nullptr : o;
  }
  // any integer, modulo 2^64
  uint64_t word() {
    PyObject *o = PyNumber_Long(next());
    if (o == nullptr) throw python_error();
    const uint64_t v = PyLong_AsUnsignedLongLongMask(o);
    Py_DECREF(o);
    if (v == (uint64_t)-1 && PyErr_Occurred()) throw python_error();
    return v;
  }
  Dropout dropout() {
    const double p = real();
    const uint64_t seed = word();
    return {p, seed, word()};
  }
  Shape sizes() {
    PyObject *o = PySequence_Fast(next(), "normalized_shape must be a sequence of integers");
    if (o == nullptr) throw python_error();
    Shape v;
    for (Py_ssize_t k = 0; k < PySequence_Fast_GET_SIZE(o); ++k) {
      PyObject *e = PyNumber_Long(PySequence_Fast_GET_ITEM(o, k));
      v.push_back(e != nullptr ? PyLong_AsLongLong(e) : -1);
      Py_XDECREF(e);
      if (PyErr_Occurred()) {
        Py_DECREF(o);
        throw python_error();
      }
    }
    Py_DECREF(o);
    return v;
  }
};

struct NoGil {
  PyThreadState *state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};
struct Gil {
  PyGILState_STATE state = PyGILState_Ensure();
  ~Gil() { PyGILState_Release(state); }
};
template <typename F> auto without_gil(const F &f) {
  const NoGil nogil;
  return f();
}

PyObject *wrap(const Tensor &t) {
  if (t.defined()) return THPVariable_Wrap(t);
  Py_RETURN_NONE;
}

PyObject *wrap_all(std::initializer_list<Tensor> ts, bool list) {
  const Py_ssize_t n = (Py_ssize_t)ts.size();
  PyObject *o = list ? PyList_New(n) : PyTuple_New(n);
  if (o == nullptr) throw python_error();
  Py_ssize_t k = 0;
  for (const Tensor &t : ts) {
    PyObject *e = wrap(t);
    if (e == nullptr) {
      Py_DECREF(o);
      throw python_error();
    }
    if (list) PyList_SET_ITEM(o, k++, e);
    else PyTuple_SET_ITEM(o, k++, e);
  }
  return o;
}

// ---------------------------------------------------------------- checks
std::string dtype_name(at::ScalarType t) { return "torch." + c10::getDtypeNames(t).first; }

int dtype_code(const Tensor &t, const char *what, bool f64 = false) {
  switch (t.scalar_type()) {
    case at::kFloat: return OSLO_DTYPE_F32;
    case at::kHalf: return OSLO_DTYPE_F16;
    case at::kBFloat16: return OSLO_DTYPE_BF16;
    case at::kDouble:
      if (f64) return OSLO_DTYPE_F64;
      break;
    default: break;
  }
  TORCH_CHECK(false, what, ": dtype ", dtype_name(t.scalar_type()),
              " is not supported by the HIP kernels (float32, float16 and bfloat16 are",
              f64 ? "" : "; float64 only by the norms", ")");
}

// CHECK_INPUT of FusedLayerNormBinder.cpp:8-14
void check_input(const Tensor &t, const char *name) {
  TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
}

void check_param(const Tensor &t, const Shape &shape, const char *name) {
  if (t.defined())
    TORCH_CHECK(t.sizes() == at::IntArrayRef(shape), name, " of shape ", t.sizes(),
                " does not match normalized_shape=", at::IntArrayRef(shape));
}

// check_args / compute_n1_n2 of FusedLayerNormBinder.cpp:19-36, 59-93
void rows_and_length(const Tensor &x, const Shape &shape, int64_t &n1, int64_t &n2) {
  const int64_t nd = (int64_t)shape.size();
  TORCH_CHECK(nd >= 1,
              "Expected normalized_shape to be at least 1-dimensional, i.e., containing at "
              "least one element, but got normalized_shape=", at::IntArrayRef(shape));
  TORCH_CHECK(x.dim() >= nd && x.sizes().slice(x.dim() - nd) == at::IntArrayRef(shape),
              "Given normalized_shape=", at::IntArrayRef(shape), ", expected input with shape [*, ",
              c10::Join(", ", shape), "], but got input of size", x.sizes());
  n2 = 1;
  for (int64_t s : shape) n2 *= s;
  n1 = n2 > 0 ? x.numel() / n2 : 0;
}

void check_rc(int rc) { TORCH_CHECK(rc == 0, oslo_hip_last_error()); }

void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }

// FusedLayerNormBinder.cpp:146-152: the statistics are fp32 for 16-bit inputs
// and have the input's type otherwise
at::ScalarType stat_type(const Tensor &t) { return t.scalar_type() == at::kDouble ? at::kDouble : at::kFloat; }

Tensor new_f32(const Tensor &like, at::IntArrayRef shape) { return at::empty(shape, like.options().dtype(at::kFloat)); }

// The operand's device made current for one call, and torch's current stream on it.
struct OnDevice {
  c10::DeviceGuard guard;
  void *stream;
  explicit OnDevice(const Tensor &t)
      : guard(t.device()), stream(c10::hip::getCurrentHIPStream(t.device().index()).stream()) {}
};

// A backward workspace is leased behind the checks, so that a refused call
// leaves the cache as it is, on the operand's device, whose capture decides about
// the cache, and behind the outputs.  The backward calls take the way to get one
// as an argument: (n1, n2, operand) -> an object that holds `tensor` (undefined:
// none) and `nbytes` until the launches are on the stream.

// The lease that a callable of the Python module hands out, held to the end of
// the scope; null: no workspace.
struct PythonLease {
  PyObject *lease = nullptr;
  Tensor tensor;
  int64_t nbytes = 0;

  PythonLease(PyObject *get, int64_t n1, int64_t n2, const Tensor &like) {
    if (get == nullptr) return;
    const Gil gil;
    PyObject *device = THPDevice_New(like.device());
    if (device != nullptr) lease = PyObject_CallFunction(get, "LLN", (long long)n1, (long long)n2, device);
    if (lease == nullptr) throw python_error();
    try {
      PyObject *entered = PyObject_CallMethod(lease, "__enter__", nullptr);
      if (entered == nullptr) throw python_error();
      Py_DECREF(entered);
    } catch (...) {
      Py_CLEAR(lease);
      throw;
    }
    PyObject *t = PyObject_GetAttrString(lease, "tensor");
    PyObject *n = t != nullptr ? PyObject_GetAttrString(lease, "nbytes") : nullptr;
    if (n != nullptr) {
      if (THPVariable_Check(t)) tensor = THPVariable_Unpack(t);
      nbytes = PyLong_AsLongLong(n);
    }
    Py_XDECREF(t);
    Py_XDECREF(n);
    if (PyErr_Occurred()) {
      release();
      throw python_error();
    }
  }
  PythonLease(const PythonLease &) = delete;
  ~PythonLease() {
    if (lease == nullptr) return;
    const Gil gil;
    release();
  }

  void release() {
    PyObject *type, *value, *trace;  // (an error on its way out stays)
    PyErr_Fetch(&type, &value, &trace);
    PyObject *r = PyObject_CallMethod(lease, "__exit__", "OOO", Py_None, Py_None, Py_None);
    if (r == nullptr) PyErr_WriteUnraisable(lease);
    Py_XDECREF(r);
    Py_CLEAR(lease);
    PyErr_Restore(type, value, trace);
  }
};

auto python_lease(PyObject *get) {
  return [get](int64_t n1, int64_t n2, const Tensor &like) { return PythonLease(get, n1, n2, like); };
}

// A workspace of its own for one call from torch's allocator, which orders its
// next use behind the launches on the stream (under capture: in the graph's
// pool).  What an autograd backward takes: no lock and no Python.
struct OwnWorkspace {
  Tensor tensor;
  int64_t nbytes = 0;
  OwnWorkspace(int op, bool wanted, int64_t n1, int64_t n2, const Tensor &like) {
    if (!wanted) return;
    nbytes = oslo_workspace_bytes(op, n1, n2);
    TORCH_CHECK(nbytes >= 0, oslo_hip_last_error());
    if (nbytes > 0) tensor = at::empty({nbytes}, like.options().dtype(at::kByte));
  }
};
auto own_workspace(int op, bool wanted) {
  return [op, wanted](int64_t n1, int64_t n2, const Tensor &like) { return OwnWorkspace(op, wanted, n1, n2, like); };
}

// An output of the softmax: from 64 MiB on it starts k * (1 MiB + 4 KiB) past
// a 2 MiB boundary (empty_staggered of the Python module says why).
Tensor softmax_out(const Tensor &like, int k) {
  constexpr int64_t kMin = 64ll << 20, kStep = (1 << 20) + 4096, kRound = 2 << 20;
  const int64_t nbytes = like.numel() * (int64_t)like.element_size();
  if (nbytes < kMin) return at::empty(like.sizes(), like.options());
  const Tensor base = at::empty({nbytes + kRound}, like.options().dtype(at::kByte));
  const int64_t phase = (int64_t)(reinterpret_cast<uintptr_t>(base.data_ptr()) % kRound);
  const int64_t off = ((k * kStep - phase) % kRound + kRound) % kRound;
  return base.slice(0, off, off + nbytes).view(like.scalar_type()).view(like.sizes());
}

// ---------------------------------------------------------------- norms
struct NormOut {
  Tensor out, mean, inv;
};
NormOut norm_fwd(bool rms, const Tensor &x, const Shape &shape, const Tensor &gamma, const Tensor &beta, double eps,
                 bool mixed) {
  check_input(x, "input");
  int64_t n1, n2;
  rows_and_length(x, shape, n1, n2);
  check_param(gamma, shape, "gamma");
  check_param(beta, shape, "beta");
  const int din = dtype_code(x, "input", true);
  const at::ScalarType out_type = mixed ? gamma.scalar_type() : x.scalar_type();
  const std::pair<const char *, const Tensor *> params[] = {{"gamma", &gamma}, {"beta", &beta}};
  for (const auto &[name, t] : params)
    if (t->defined()) {
      check_input(*t, name);
      TORCH_CHECK(t->scalar_type() == out_type, name, " has dtype ", dtype_name(t->scalar_type()),
                  " but the output dtype is ", dtype_name(out_type));
    }
  const int dout = mixed ? dtype_code(gamma, "output", true) : din;
  const OnDevice on(x);
  NormOut r;
  r.out = at::empty(x.sizes(), x.options().dtype(out_type));
  const auto stats = x.options().dtype(stat_type(x));
  r.inv = at::empty({n1}, stats);
  if (rms) {
    check_rc(oslo_rms_fwd(ptr(x), ptr(gamma), ptr(r.out), ptr(r.inv), n1, n2, eps, din, dout, on.stream));
  } else {
    r.mean = at::empty({n1}, stats);
    check_rc(oslo_ln_fwd(ptr(x), ptr(gamma), ptr(beta), ptr(r.out), ptr(r.mean), ptr(r.inv), n1, n2, eps, din, dout,
                         on.stream));
  }
  return r;
}

// (rms, input, normalized_shape, gamma, beta, eps, mixed) -> [output, (mean,) invvar]
PyObject *norm_forward(Args &g) {
  const bool rms = g.flag();
  const Tensor &x = g.tensor();
  const auto shape = g.sizes();
  const Tensor gamma = g.optional(), beta = g.optional();
  const double eps = g.real();
  const bool mixed = g.flag();
  const NormOut r = without_gil([&] { return norm_fwd(rms, x, shape, gamma, beta, eps, mixed); });
  return rms ? wrap_all({r.out, r.inv}, true) : wrap_all({r.out, r.mean, r.inv}, true);
}

struct NormGrads {
  Tensor dx, dg, db;
};
template <typename Lease>
NormGrads norm_bwd(bool rms, const Tensor &dy, const Tensor &mean, const Tensor &inv, const Tensor &x,
                   const Shape &shape, const Tensor &gamma, const Tensor &beta, const Lease &lease) {
  check_input(dy, "dout");
  check_input(inv, "invvar");
  check_input(x, "input");
  if (!rms) {
    TORCH_CHECK(mean.defined(), "mean is missing");
    check_input(mean, "mean");
  }
  int64_t n1, n2;
  rows_and_length(x, shape, n1, n2);
  TORCH_CHECK(dy.sizes() == x.sizes(), "dout of size ", dy.sizes(), " does not match input of size ", x.sizes());
  const int din = dtype_code(x, "input", true), dcode = dtype_code(dy, "dout", true);
  const std::pair<const char *, const Tensor *> stats[] = {{"invvar", &inv}, {"mean", &mean}};
  for (const auto &[name, t] : stats)
    if (t->defined()) {
      TORCH_CHECK(t->scalar_type() == stat_type(x), name, " has dtype ", dtype_name(t->scalar_type()),
                  ", expected ", dtype_name(stat_type(x)));
      TORCH_CHECK(t->numel() == n1, name, " has ", t->numel(), " elements for ", n1, " rows of input");
    }
  if (gamma.defined()) {
    check_input(gamma, "gamma");
    check_param(gamma, shape, "gamma");
    TORCH_CHECK(gamma.scalar_type() == dy.scalar_type(), "gamma has dtype ", dtype_name(gamma.scalar_type()),
                " but dout has dtype ", dtype_name(dy.scalar_type()));
  }
  const OnDevice on(x);
  NormGrads r;
  r.dx = at::empty(x.sizes(), x.options());
  if (gamma.defined()) {
    r.dg = at::empty_like(gamma);
    if (!rms) r.db = at::empty_like(beta.defined() ? beta : gamma);
  }
  const auto ws = lease(n1, n2, x);
  check_rc(rms ? oslo_rms_bwd(ptr(dy), ptr(x), ptr(inv), ptr(gamma), ptr(r.dx), ptr(r.dg), ptr(ws.tensor), ws.nbytes,
                              n1, n2, din, dcode, on.stream)
               : oslo_ln_bwd(ptr(dy), ptr(x), ptr(mean), ptr(inv), ptr(gamma), ptr(r.dx), ptr(r.dg), ptr(r.db),
                             ptr(ws.tensor), ws.nbytes, n1, n2, din, dcode, on.stream));
  return r;
}

// (rms, dout, mean, invvar, input, normalized_shape, gamma, beta, workspace)
// -> (grad_input, grad_gamma, grad_beta)
PyObject *norm_backward(Args &g) {
  const bool rms = g.flag();
  const Tensor &dy = g.tensor();
  const Tensor mean = g.optional();
  const Tensor &inv = g.tensor();
  const Tensor &x = g.tensor();
  const auto shape = g.sizes();
  const Tensor gamma = g.optional(), beta = g.optional();
  const auto lease = python_lease(g.callable());
  const NormGrads r = without_gil([&] { return norm_bwd(rms, dy, mean, inv, x, shape, gamma, beta, lease); });
  return wrap_all({r.dx, r.dg, r.db}, false);
}

struct ResidualNormOut {
  Tensor y, h, mean, inv;
};
ResidualNormOut residual_norm_fwd(bool rms, const Tensor &x, const Tensor &bias, const Tensor &res,
                                  const Shape &shape, const Tensor &gamma, const Tensor &beta, double eps,
                                  const Dropout &d, bool want_h) {
  check_input(x, "input");
  int64_t n1, n2;
  rows_and_length(x, shape, n1, n2);
  const std::pair<const char *, const Tensor *> ops[] = {
      {"gamma", &gamma}, {"beta", &beta}, {"bias", &bias}, {"residual", &res}};
  for (const auto &[name, t] : ops)
    if (t->defined()) {
      check_input(*t, name);
      if (t != &res) check_param(*t, shape, name);
    }
  TORCH_CHECK(!res.defined() || res.sizes() == x.sizes(), "residual and input differ in shape");
  for (const auto &[name, t] : ops)
    TORCH_CHECK(!t->defined() || t->scalar_type() == x.scalar_type(), name, " has dtype ",
                dtype_name(t->scalar_type()), " but input has dtype ", dtype_name(x.scalar_type()));
  const int code = dtype_code(x, "input");
  const OnDevice on(x);
  ResidualNormOut r;
  r.y = at::empty(x.sizes(), x.options());
  if (want_h) r.h = at::empty(x.sizes(), x.options());
  r.inv = new_f32(x, {n1});
  if (!rms) r.mean = new_f32(x, {n1});
  check_rc(oslo_bias_dropout_add_norm_fwd(ptr(x), ptr(bias), ptr(res), ptr(gamma), ptr(beta), ptr(r.h), ptr(r.y),
                                          (float *)ptr(r.mean), (float *)ptr(r.inv), n1, n2, eps, (float)d.p, d.seed,
                                          d.offset, rms, code, on.stream));
  return r;
}

// (rms, input, bias, residual, normalized_shape, gamma, beta, eps, p, seed, offset, want_h)
// -> [y, h, mean, invvar]
PyObject *residual_norm_forward(Args &g) {
  const bool rms = g.flag();
  const Tensor &x = g.tensor();
  const Tensor bias = g.optional(), res = g.optional();
  const auto shape = g.sizes();
  const Tensor gamma = g.optional(), beta = g.optional();
  const double eps = g.real();
  const Dropout d = g.dropout();
  const bool want_h = g.flag();
  const ResidualNormOut r =
      without_gil([&] { return residual_norm_fwd(rms, x, bias, res, shape, gamma, beta, eps, d, want_h); });
  return wrap_all({r.y, r.h, r.mean, r.inv}, true);
}

struct ResidualNormGrads {
  Tensor dres, dx, dg, db, dbias;  // dx undefined without dropout: it is dres
};
template <typename Lease>
ResidualNormGrads residual_norm_bwd(bool rms, const Tensor &dy, const Tensor &extra, const Tensor &h,
                                    const Tensor &mean, const Tensor &inv, const Shape &shape, const Tensor &gamma,
                                    const Dropout &d, bool want_bias, const Lease &lease) {
  check_input(dy, "dout");
  check_input(h, "h");
  check_input(inv, "invvar");
  int64_t n1, n2;
  rows_and_length(h, shape, n1, n2);
  TORCH_CHECK(dy.sizes() == h.sizes() && dy.scalar_type() == h.scalar_type(), "dout and h differ in shape or dtype");
  if (!rms) {
    TORCH_CHECK(mean.defined(), "mean is missing");
    check_input(mean, "mean");
  }
  const auto check_stat = [&](const Tensor &t, const char *name) {
    TORCH_CHECK(t.scalar_type() == at::kFloat && t.numel() == n1, name,
                " must be float32 with one element per row of h");
  };
  check_stat(inv, "invvar");
  if (!rms) check_stat(mean, "mean");
  if (extra.defined()) {
    check_input(extra, "dh_extra");
    TORCH_CHECK(extra.sizes() == h.sizes() && extra.scalar_type() == h.scalar_type(),
                "dh_extra and h differ in shape or dtype");
  }
  const int code = dtype_code(h, "h");
  if (gamma.defined()) {
    check_input(gamma, "gamma");
    check_param(gamma, shape, "gamma");
    TORCH_CHECK(gamma.scalar_type() == h.scalar_type(), "gamma has dtype ", dtype_name(gamma.scalar_type()),
                " but h has dtype ", dtype_name(h.scalar_type()));
  }
  const OnDevice on(h);
  ResidualNormGrads r;
  r.dres = at::empty(h.sizes(), h.options());
  if (d.p > 0.0) r.dx = at::empty(h.sizes(), h.options());
  if (gamma.defined()) {
    r.dg = at::empty_like(gamma);
    if (!rms) r.db = at::empty_like(gamma);
  }
  if (want_bias) r.dbias = at::empty(shape, h.options());
  const auto ws = lease(n1, n2, h);
  check_rc(oslo_bias_dropout_add_norm_bwd(
      ptr(dy), ptr(extra), ptr(h), rms ? nullptr : (const float *)ptr(mean), (const float *)ptr(inv), ptr(gamma),
      ptr(r.dres), ptr(r.dx), ptr(r.dg), ptr(r.db), ptr(r.dbias), ptr(ws.tensor), ws.nbytes, n1, n2, (float)d.p,
      d.seed, d.offset, rms, code, on.stream));
  return r;
}

// (rms, dout, dh_extra, h, mean, invvar, normalized_shape, gamma, p, seed, offset,
//  need_bias_grad, workspace)
// -> (grad_residual, grad_input, grad_gamma, grad_beta, grad_bias)
PyObject *residual_norm_backward(Args &g) {
  const bool rms = g.flag();
  const Tensor &dy = g.tensor();
  const Tensor extra = g.optional();
  const Tensor &h = g.tensor();
  const Tensor mean = g.optional();
  const Tensor &inv = g.tensor();
  const auto shape = g.sizes();
  const Tensor gamma = g.optional();
  const Dropout d = g.dropout();
  const bool want_bias = g.flag();
  const auto lease = python_lease(g.callable());
  const ResidualNormGrads r = without_gil([&] {
    return residual_norm_bwd(rms, dy, extra, h, mean, inv, shape, gamma, d, want_bias, lease);
  });
  return wrap_all({r.dres, r.dx.defined() ? r.dx : r.dres, r.dg, r.db, r.dbias}, false);
}

// ---------------------------------------------------------------- softmax
void check_same(const Tensor &a, const char *na, const Tensor &b, const char *nb) {
  check_input(a, na);
  check_input(b, nb);
  TORCH_CHECK(a.scalar_type() == b.scalar_type(), na, " and ", nb, " differ in dtype");
  TORCH_CHECK(a.sizes() == b.sizes(), na, " and ", nb, " differ in shape");
}

// A boolean mask (non-zero = hidden) as contiguous bytes.
Tensor mask_bytes(const Tensor &mask, const Tensor &like) {
  TORCH_CHECK(mask.device() == like.device(), "mask is on ", mask.device().str(), " but the softmax operand is on ",
              like.device().str());
  if (mask.scalar_type() == at::kBool || mask.scalar_type() == at::kByte) return mask.contiguous();
  return mask.ne(0).contiguous();
}

void check_mask_dims(const Tensor &x, const Tensor &mask) {
  TORCH_CHECK(x.dim() == 4 && mask.dim() == 4, "expected 4D tensor");
  TORCH_CHECK(mask.size(1) == 1 && mask.size(3) == x.size(3) && (mask.size(0) == 1 || mask.size(0) == x.size(0)) &&
                  (mask.size(2) == 1 || mask.size(2) == x.size(2)),
              "mask of size ", mask.sizes(), " does not broadcast to [", x.size(0), ", 1, ", x.size(2), ", ",
              x.size(3), "]");
}

Tensor causal_fwd(const Tensor &x, float scale) {
  TORCH_CHECK(x.dim() == 3, "expected 3D tensor");
  check_input(x, "input");
  const int code = dtype_code(x, "input");
  const OnDevice on(x);
  const Tensor out = softmax_out(x, 1);
  check_rc(oslo_softmax_causal_fwd(ptr(x), ptr(out), x.size(0), x.size(1), x.size(2), scale, code, on.stream));
  return out;
}

// (input, scale) -> out
PyObject *causal_forward(Args &g) {
  const Tensor &x = g.tensor();
  const float scale = (float)g.real();
  return wrap(without_gil([&] { return causal_fwd(x, scale); }));
}

Tensor causal_bwd(const Tensor &dy, const Tensor &y, float scale, bool inplace) {
  TORCH_CHECK(dy.dim() == 3 && y.dim() == 3, "expected 3D tensor");
  check_same(dy, "output_grads", y, "softmax_results");
  const int code = dtype_code(dy, "output_grads");
  const OnDevice on(dy);
  const Tensor dx = inplace ? dy : softmax_out(dy, 2);
  check_rc(oslo_softmax_causal_bwd(ptr(dy), ptr(y), ptr(dx), y.size(0), y.size(1), y.size(2), scale, code, on.stream));
  return dx;
}

// (output_grads, softmax_results, scale, inplace) -> grad_input
PyObject *causal_backward(Args &g) {
  const Tensor &dy = g.tensor();
  const Tensor &y = g.tensor();
  const float scale = (float)g.real();
  const bool inplace = g.flag();
  return wrap(without_gil([&] { return causal_bwd(dy, y, scale, inplace); }));
}

Tensor masked_fwd(const Tensor &x, const Tensor &mask, float scale, bool causal) {
  check_mask_dims(x, mask);
  check_input(x, "input");
  const int code = dtype_code(x, "input");
  const OnDevice on(x);
  const Tensor m = mask_bytes(mask, x);
  const Tensor out = softmax_out(x, 1);
  check_rc((causal ? oslo_softmax_causal_masked_fwd : oslo_softmax_masked_fwd)(
      ptr(x), (const uint8_t *)ptr(m), ptr(out), x.size(0), x.size(1), x.size(2), x.size(3), mask.size(0),
      mask.size(2), scale, code, on.stream));
  return out;
}

// (input, mask, scale, causal) -> out
PyObject *masked_forward(Args &g) {
  const Tensor &x = g.tensor();
  const Tensor &mask = g.tensor();
  const float scale = (float)g.real();
  const bool causal = g.flag();
  return wrap(without_gil([&] { return masked_fwd(x, mask, scale, causal); }));
}

Tensor masked_bwd(const Tensor &dy, const Tensor &y, float scale, const Tensor &mask, bool inplace, bool causal) {
  TORCH_CHECK(dy.dim() == 4 && y.dim() == 4, "expected 4D tensor");
  check_same(dy, "output_grads", y, "softmax_results");
  if (mask.defined()) check_mask_dims(y, mask);
  const int code = dtype_code(dy, "output_grads");
  const OnDevice on(dy);
  const Tensor m = mask.defined() ? mask_bytes(mask, y) : Tensor();
  const Tensor dx = inplace ? dy : softmax_out(dy, 2);
  check_rc((causal ? oslo_softmax_causal_masked_bwd : oslo_softmax_masked_bwd)(
      ptr(dy), ptr(y), (const uint8_t *)ptr(m), ptr(dx), y.size(0), y.size(1), y.size(2), y.size(3),
      mask.defined() ? mask.size(0) : 1, mask.defined() ? mask.size(2) : 1, scale, code, on.stream));
  return dx;
}

// (output_grads, softmax_results, scale, mask, inplace, causal) -> grad_input
PyObject *masked_backward(Args &g) {
  const Tensor &dy = g.tensor();
  const Tensor &y = g.tensor();
  const float scale = (float)g.real();
  const Tensor mask = g.optional();
  const bool inplace = g.flag(), causal = g.flag();
  return wrap(without_gil([&] { return masked_bwd(dy, y, scale, mask, inplace, causal); }));
}

int64_t row_count(const Tensor &x) { return x.numel() > 0 ? x.numel() / x.size(-1) : 0; }

struct SoftmaxOut {
  Tensor out, stats;
};
SoftmaxOut dropout_fwd(const Tensor &x, const Tensor &mask, float scale, const Dropout &d, bool causal) {
  check_input(x, "input");
  if (mask.defined()) check_mask_dims(x, mask);
  else TORCH_CHECK(x.dim() == 3, "expected 3D tensor");
  const int code = dtype_code(x, "input");
  const OnDevice on(x);
  const Tensor m = mask.defined() ? mask_bytes(mask, x) : Tensor();
  SoftmaxOut r{softmax_out(x, 1), new_f32(x, {row_count(x), 2})};
  float *st = r.stats.data_ptr<float>();
  check_rc(!mask.defined()
               ? oslo_softmax_causal_dropout_fwd(ptr(x), ptr(r.out), st, x.size(0), x.size(1), x.size(2), scale,
                                                 (float)d.p, d.seed, d.offset, code, on.stream)
               : (causal ? oslo_softmax_causal_masked_dropout_fwd : oslo_softmax_masked_dropout_fwd)(
                     ptr(x), (const uint8_t *)ptr(m), ptr(r.out), st, x.size(0), x.size(1), x.size(2), x.size(3),
                     mask.size(0), mask.size(2), scale, (float)d.p, d.seed, d.offset, code, on.stream));
  return r;
}

// (input, mask, scale, p, seed, offset, causal) -> [out, stats]
PyObject *dropout_forward(Args &g) {
  const Tensor &x = g.tensor();
  const Tensor mask = g.optional();
  const float scale = (float)g.real();
  const Dropout d = g.dropout();
  const bool causal = g.flag();
  const SoftmaxOut r = without_gil([&] { return dropout_fwd(x, mask, scale, d, causal); });
  return wrap_all({r.out, r.stats}, true);
}

void check_dropout_operands(const Tensor &dy, const Tensor &x, const Tensor &stats) {
  check_input(dy, "output_grads");
  check_input(x, "input");
  check_input(stats, "stats");
  TORCH_CHECK(dy.scalar_type() == x.scalar_type() && dy.sizes() == x.sizes(),
              "output_grads and input differ in dtype or shape");
  TORCH_CHECK(stats.scalar_type() == at::kFloat && stats.numel() == 2 * row_count(x),
              "stats must be float32 [rows, 2]");
}

Tensor dropout_bwd(const Tensor &dy, const Tensor &x, const Tensor &stats, const Tensor &mask, float scale,
                   const Dropout &d, bool inplace, bool causal) {
  check_dropout_operands(dy, x, stats);
  if (mask.defined()) check_mask_dims(x, mask);
  else TORCH_CHECK(x.dim() == 3, "expected 3D tensor");
  const int code = dtype_code(x, "input");
  const OnDevice on(x);
  const Tensor m = mask.defined() ? mask_bytes(mask, x) : Tensor();
  const Tensor dx = inplace ? dy : softmax_out(dy, 2);
  const float *st = stats.data_ptr<float>();
  check_rc(!mask.defined()
               ? oslo_softmax_causal_dropout_bwd(ptr(dy), ptr(x), st, ptr(dx), x.size(0), x.size(1), x.size(2),
                                                 scale, (float)d.p, d.seed, d.offset, code, on.stream)
               : (causal ? oslo_softmax_causal_masked_dropout_bwd : oslo_softmax_masked_dropout_bwd)(
                     ptr(dy), ptr(x), (const uint8_t *)ptr(m), st, ptr(dx), x.size(0), x.size(1), x.size(2),
                     x.size(3), mask.size(0), mask.size(2), scale, (float)d.p, d.seed, d.offset, code, on.stream));
  return dx;
}

// (output_grads, input, stats, mask, scale, p, seed, offset, inplace, causal) -> grad_input
PyObject *dropout_backward(Args &g) {
  const Tensor &dy = g.tensor();
  const Tensor &x = g.tensor();
  const Tensor &stats = g.tensor();
  const Tensor mask = g.optional();
  const float scale = (float)g.real();
  const Dropout d = g.dropout();
  const bool inplace = g.flag(), causal = g.flag();
  return wrap(without_gil([&] { return dropout_bwd(dy, x, stats, mask, scale, d, inplace, causal); }));
}

// The additive term as the kernel addresses it: four dimensions, its strides
// along batch, heads and queries (0 = broadcast; expanded views have it), the
// keys contiguous, the input's dtype or fp32.
struct Term {
  Tensor t;
  int64_t sb, sh, sq;
  int code;
  Term(const Tensor &term, const Tensor &x) : t(term) {
    while (t.dim() < 4) t = t.unsqueeze(0);
    const int64_t sk = x.size(3);
    if (t.size(3) != sk) t = t.expand({-1, -1, -1, sk}).contiguous();
    if (t.scalar_type() != x.scalar_type() && t.scalar_type() != at::kFloat) t = t.to(at::kFloat);
    if (sk > 1 && t.stride(3) != 1) t = t.contiguous();
    const auto stride = [&](int64_t d) { return t.size(d) == 1 ? 0 : t.stride(d); };
    sb = stride(0), sh = stride(1), sq = stride(2);
    code = dtype_code(t, "the additive term");
  }
  static void check(const Tensor &t, const Tensor &x) {
    TORCH_CHECK(x.dim() == 4, "expected 4D tensor");
    TORCH_CHECK(t.is_floating_point(), "the additive term must be a floating-point tensor");
    TORCH_CHECK(t.device() == x.device(), "the additive term is on ", t.device().str(),
                " but the softmax operand is on ", x.device().str());
    TORCH_CHECK(t.dim() <= 4, "the additive term has more than four dimensions");
    bool fits = true;
    for (int64_t d = 0; d < t.dim(); ++d) fits &= t.size(d) == 1 || t.size(d) == x.size(d + 4 - t.dim());
    TORCH_CHECK(fits, "additive term of size ", t.sizes(), " does not broadcast to ", x.sizes());
  }
};

// `skip` -1 is the default: the test for hidden keys in the backward passes
// only, and there only where the term is small next to the logits (shared by
// the heads or by the queries), where a hidden chunk saves two loads.  (Waiting
// for the term before the logits are requested costs a forward pass more than
// the unread logits save: [16, 16, 1024, 1024] fp16 with 48 % of the keys under
// -inf 159 us with the test, 163 without; with a -10000 mask, which hides
// nothing, 190-210 against 163.)
int term_flags(bool causal, int skip, int64_t sh, int64_t sq, bool forward) {
  const bool test = skip < 0 ? !forward && (sh == 0 || sq == 0) : skip != 0;
  return (causal ? OSLO_SOFTMAX_CAUSAL : 0) | (test ? OSLO_SOFTMAX_SKIP_HIDDEN : 0);
}

// (bias, input) -> (term, stride_b, stride_h, stride_q, dtype code)
PyObject *bias_operand(Args &g) {
  const Tensor &bias = g.tensor();
  const Tensor &x = g.tensor();
  Term::check(bias, x);
  const Term t(bias, x);
  PyObject *o = THPVariable_Wrap(t.t);
  if (o == nullptr) throw python_error();
  return Py_BuildValue("NLLLi", o, (long long)t.sb, (long long)t.sh, (long long)t.sq, t.code);
}

// (causal, skip_hidden, stride_h, stride_q, forward) -> flags
PyObject *bias_flags(Args &g) {
  const bool causal = g.flag();
  const int skip = g.tristate();
  const int64_t sh = g.integer(), sq = g.integer();
  return PyLong_FromLong(term_flags(causal, skip, sh, sq, g.flag()));
}

Tensor bias_fwd(const Tensor &x, const Tensor &bias, float scale, bool causal, int skip) {
  check_input(x, "input");
  Term::check(bias, x);
  const int code = dtype_code(x, "input");
  const OnDevice on(x);
  const Term t(bias, x);
  const int flags = term_flags(causal, skip, t.sh, t.sq, true);
  const Tensor out = softmax_out(x, 1);
  check_rc(oslo_softmax_bias_fwd(ptr(x), ptr(t.t), ptr(out), x.size(0), x.size(1), x.size(2), x.size(3), t.sb, t.sh,
                                 t.sq, t.code, flags, scale, code, on.stream));
  return out;
}

// (input, bias, scale, causal, skip_hidden) -> out
PyObject *bias_forward(Args &g) {
  const Tensor &x = g.tensor();
  const Tensor &bias = g.tensor();
  const float scale = (float)g.real();
  const bool causal = g.flag();
  const int skip = g.tristate();
  return wrap(without_gil([&] { return bias_fwd(x, bias, scale, causal, skip); }));
}

Tensor bias_bwd(const Tensor &dy, const Tensor &y, float scale, const Tensor &bias, bool causal, int skip,
                bool inplace) {
  TORCH_CHECK(dy.dim() == 4 && y.dim() == 4, "expected 4D tensor");
  check_same(dy, "output_grads", y, "softmax_results");
  const int code = dtype_code(y, "softmax_results");
  if (bias.defined()) Term::check(bias, y);
  const OnDevice on(dy);
  std::optional<Term> t;
  int flags = causal ? OSLO_SOFTMAX_CAUSAL : 0;
  if (bias.defined()) {
    t.emplace(bias, y);
    flags = term_flags(causal, skip, t->sh, t->sq, false);
    if (!(flags & OSLO_SOFTMAX_SKIP_HIDDEN)) t.reset();  // (only the test reads the term)
  }
  const Tensor dx = inplace ? dy : softmax_out(dy, 2);
  check_rc(oslo_softmax_bias_bwd(ptr(dy), ptr(y), t ? ptr(t->t) : nullptr, ptr(dx), y.size(0), y.size(1), y.size(2),
                                 y.size(3), t ? t->sb : 0, t ? t->sh : 0, t ? t->sq : 0, t ? t->code : code, flags,
                                 scale, code, on.stream));
  return dx;
}

// (output_grads, softmax_results, scale, bias, causal, skip_hidden, inplace) -> grad_input
PyObject *bias_backward(Args &g) {
  const Tensor &dy = g.tensor();
  const Tensor &y = g.tensor();
  const float scale = (float)g.real();
  const Tensor bias = g.optional();
  const bool causal = g.flag();
  const int skip = g.tristate();
  const bool inplace = g.flag();
  return wrap(without_gil([&] { return bias_bwd(dy, y, scale, bias, causal, skip, inplace); }));
}

SoftmaxOut bias_dropout_fwd(const Tensor &x, const Tensor &bias, float scale, const Dropout &d, bool causal,
                            int skip) {
  check_input(x, "input");
  Term::check(bias, x);
  const int code = dtype_code(x, "input");
  const OnDevice on(x);
  const Term t(bias, x);
  const int flags = term_flags(causal, skip, t.sh, t.sq, true);
  SoftmaxOut r{softmax_out(x, 1), new_f32(x, {x.size(0) * x.size(1) * x.size(2), 2})};
  check_rc(oslo_softmax_bias_dropout_fwd(ptr(x), ptr(t.t), ptr(r.out), r.stats.data_ptr<float>(), x.size(0),
                                         x.size(1), x.size(2), x.size(3), t.sb, t.sh, t.sq, t.code, flags, scale,
                                         (float)d.p, d.seed, d.offset, code, on.stream));
  return r;
}

// (input, bias, scale, p, seed, offset, causal, skip_hidden) -> [out, stats]
PyObject *bias_dropout_forward(Args &g) {
  const Tensor &x = g.tensor();
  const Tensor &bias = g.tensor();
  const float scale = (float)g.real();
  const Dropout d = g.dropout();
  const bool causal = g.flag();
  const int skip = g.tristate();
  const SoftmaxOut r = without_gil([&] { return bias_dropout_fwd(x, bias, scale, d, causal, skip); });
  return wrap_all({r.out, r.stats}, true);
}

Tensor bias_dropout_bwd(const Tensor &dy, const Tensor &x, const Tensor &bias, const Tensor &stats, float scale,
                        const Dropout &d, bool causal, int skip, bool inplace) {
  check_input(dy, "output_grads");
  check_input(x, "input");
  check_input(stats, "stats");
  TORCH_CHECK(dy.scalar_type() == x.scalar_type() && dy.sizes() == x.sizes(),
              "output_grads and input differ in dtype or shape");
  Term::check(bias, x);
  TORCH_CHECK(stats.scalar_type() == at::kFloat && stats.numel() == 2 * x.size(0) * x.size(1) * x.size(2),
              "stats must be float32 [rows, 2]");
  const int code = dtype_code(x, "input");
  const OnDevice on(x);
  const Term t(bias, x);
  const int flags = term_flags(causal, skip, t.sh, t.sq, false);
  const Tensor dx = inplace ? dy : softmax_out(dy, 2);
  check_rc(oslo_softmax_bias_dropout_bwd(ptr(dy), ptr(x), ptr(t.t), stats.data_ptr<float>(), ptr(dx), x.size(0),
                                         x.size(1), x.size(2), x.size(3), t.sb, t.sh, t.sq, t.code, flags, scale,
                                         (float)d.p, d.seed, d.offset, code, on.stream));
  return dx;
}

// (output_grads, input, bias, stats, scale, p, seed, offset, causal, skip_hidden, inplace) -> grad_input
PyObject *bias_dropout_backward(Args &g) {
  const Tensor &dy = g.tensor();
  const Tensor &x = g.tensor();
  const Tensor &bias = g.tensor();
  const Tensor &stats = g.tensor();
  const float scale = (float)g.real();
  const Dropout d = g.dropout();
  const bool causal = g.flag();
  const int skip = g.tristate();
  const bool inplace = g.flag();
  return wrap(
      without_gil([&] { return bias_dropout_bwd(dy, x, bias, stats, scale, d, causal, skip, inplace); }));
}

// ---------------------------------------------------------------- element-wise
void rows_and_cols(const Tensor &x, const Tensor &bias, int64_t &rows, int64_t &cols) {
  cols = x.dim() > 0 ? x.size(-1) : 1;
  if (bias.defined())
    TORCH_CHECK(bias.dim() == 1 && bias.size(0) == cols, "bias of size ", bias.sizes(),
                " does not match the last dimension of input of size ", x.sizes());
  rows = cols > 0 ? x.numel() / cols : 0;
}

void check_bias(const Tensor &bias, const Tensor &x) {
  if (!bias.defined()) return;
  check_input(bias, "bias");
  TORCH_CHECK(bias.scalar_type() == x.scalar_type(), "bias and input differ in dtype");
}

Tensor gelu_fwd(const Tensor &x, const Tensor &bias) {
  check_input(x, "input");
  check_bias(bias, x);
  int64_t rows, cols;
  rows_and_cols(x, bias, rows, cols);
  const int code = dtype_code(x, "input");
  const OnDevice on(x);
  const Tensor out = at::empty(x.sizes(), x.options());
  check_rc(oslo_bias_gelu_fwd(ptr(x), ptr(bias), ptr(out), rows, cols, code, on.stream));
  return out;
}

// (input, bias) -> out
PyObject *gelu_forward(Args &g) {
  const Tensor &x = g.tensor();
  const Tensor bias = g.optional();
  return wrap(without_gil([&] { return gelu_fwd(x, bias); }));
}

struct ColumnGrads {
  Tensor dx, db;
};
template <typename Lease>
ColumnGrads gelu_bwd(const Tensor &dy, const Tensor &x, const Tensor &bias, bool want_bias, const Lease &lease) {
  check_input(dy, "grad_output");
  check_input(x, "input");
  TORCH_CHECK(dy.scalar_type() == x.scalar_type() && dy.sizes() == x.sizes(), "grad_output does not match input");
  check_bias(bias, x);
  int64_t rows, cols;
  rows_and_cols(x, bias, rows, cols);
  const int code = dtype_code(x, "input");
  const OnDevice on(x);
  ColumnGrads r;
  r.dx = at::empty(x.sizes(), x.options());
  if (bias.defined() && want_bias) r.db = at::empty_like(bias);
  const auto ws = lease(rows, cols, x);
  check_rc(oslo_bias_gelu_bwd(ptr(dy), ptr(x), ptr(bias), ptr(r.dx), ptr(r.db), ptr(ws.tensor), ws.nbytes, rows, cols,
                              code, on.stream));
  return r;
}

// (grad_output, input, bias, need_bias_grad, workspace) -> (grad_input, grad_bias)
PyObject *gelu_backward(Args &g) {
  const Tensor &dy = g.tensor();
  const Tensor &x = g.tensor();
  const Tensor bias = g.optional();
  const bool want_bias = g.flag();
  const auto lease = python_lease(g.callable());
  const ColumnGrads r = without_gil([&] { return gelu_bwd(dy, x, bias, want_bias, lease); });
  return wrap_all({r.dx, r.db}, false);
}

struct DropoutAddOut {
  Tensor out, mask;
};
DropoutAddOut dropout_add_fwd(const Tensor &x, const Tensor &bias, const Tensor &res, const Dropout &d, Tensor out,
                              bool want_mask) {
  check_input(x, "input");
  check_bias(bias, x);
  if (res.defined()) {
    check_input(res, "residual");
    TORCH_CHECK(res.scalar_type() == x.scalar_type(), "residual and input differ in dtype");
    TORCH_CHECK(res.sizes() == x.sizes(), "residual does not match input");
  }
  int64_t rows, cols;
  rows_and_cols(x, bias, rows, cols);
  const int code = dtype_code(x, "input");
  const OnDevice on(x);
  Tensor mask;
  if (!out.defined()) out = at::empty(x.sizes(), x.options());
  if (want_mask) mask = at::empty(x.sizes(), x.options().dtype(at::kByte));
  check_rc(oslo_bias_dropout_add_fwd(ptr(x), ptr(bias), ptr(res), ptr(out), (uint8_t *)ptr(mask), rows, cols,
                                     (float)d.p, d.seed, d.offset, code, on.stream));
  return {out, mask};
}

// (input, bias, residual, p, seed, offset, out, return_mask) -> (out, mask or None)
PyObject *dropout_add_forward(Args &g) {
  const Tensor &x = g.tensor();
  const Tensor bias = g.optional(), res = g.optional();
  const Dropout d = g.dropout();
  const Tensor out = g.optional();
  const bool want_mask = g.flag();
  const DropoutAddOut r = without_gil([&] { return dropout_add_fwd(x, bias, res, d, out, want_mask); });
  return wrap_all({r.out, r.mask}, false);
}

template <typename Lease>
ColumnGrads dropout_add_bwd(const Tensor &dy, const Dropout &d, bool want_input, bool want_bias, const Lease &lease) {
  check_input(dy, "grad_output");
  int64_t rows, cols;
  rows_and_cols(dy, Tensor(), rows, cols);
  ColumnGrads r;
  if (want_input || want_bias) {
    const int code = dtype_code(dy, "grad_output");
    const OnDevice on(dy);
    if (want_input) r.dx = at::empty(dy.sizes(), dy.options());
    if (want_bias) r.db = at::empty({cols}, dy.options());
    const auto ws = lease(rows, cols, dy);
    check_rc(oslo_bias_dropout_add_bwd(ptr(dy), ptr(r.dx), ptr(r.db), ptr(ws.tensor), ws.nbytes, rows, cols,
                                       (float)d.p, d.seed, d.offset, code, on.stream));
  }
  return r;
}

// (grad_output, p, seed, offset, need_input_grad, need_bias_grad, workspace)
// -> (grad_input, grad_bias)
PyObject *dropout_add_backward(Args &g) {
  const Tensor &dy = g.tensor();
  const Dropout d = g.dropout();
  const bool want_input = g.flag(), want_bias = g.flag();
  const auto lease = python_lease(g.callable());
  const ColumnGrads r = without_gil([&] { return dropout_add_bwd(dy, d, want_input, want_bias, lease); });
  return wrap_all({r.dx, r.db}, false);
}

// ---------------------------------------------------------------- autograd
// One class per Python Function of functional.py, which documents what is saved
// and why; the numbers a backward needs travel as one list of 64-bit words.
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

Tensor contiguous(const OptTensor &t) { return t.has_value() && t->defined() ? t->contiguous() : Tensor(); }
OptTensor some(const Tensor &t) { return t.defined() ? OptTensor(t) : OptTensor(); }
bool given(const OptTensor &t) { return t.has_value() && t->defined(); }

int64_t word_of(double v) {
  int64_t w;
  std::memcpy(&w, &v, sizeof w);
  return w;
}
double real_of(int64_t w) {
  double v;
  std::memcpy(&v, &w, sizeof v);
  return v;
}
void keep_words(AutogradContext *ctx, Shape words) { ctx->saved_data["words"] = std::move(words); }
Shape words_of(AutogradContext *ctx) { return ctx->saved_data["words"].toIntVector(); }
Shape dropout_words(const Dropout &d) { return {word_of(d.p), (int64_t)d.seed, (int64_t)d.offset}; }
Dropout dropout_of(const Shape &w, size_t at = 0) { return {real_of(w[at]), (uint64_t)w[at + 1], (uint64_t)w[at + 2]}; }

// LayerNorm and RMSNorm, with or without parameters, of one or of mixed dtypes.
// Without a weight it is the norm without parameters, in the input's dtype,
// whatever the bias, which gets no gradient then.
struct NormFunction : Function<NormFunction> {
  static Tensor forward(AutogradContext *ctx, const Tensor &input, const OptTensor &weight, const OptTensor &bias,
                        bool rms, bool mixed, const Shape &shape, double eps) {
    TORCH_CHECK(rms || !given(weight) || given(bias), "LayerNorm with a weight needs a bias");
    const Tensor x = input.contiguous(), w = contiguous(weight), b = w.defined() ? contiguous(bias) : Tensor();
    const NormOut r = norm_fwd(rms, x, shape, w, b, eps, mixed && w.defined());
    ctx->save_for_backward({x, w, b, r.mean, r.inv});
    Shape words{rms};
    words.insert(words.end(), shape.begin(), shape.end());
    keep_words(ctx, std::move(words));
    return r.out;
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const auto saved = ctx->get_saved_variables();
    const Shape words = words_of(ctx), shape(words.begin() + 1, words.end());
    const bool rms = words[0] != 0;
    const Tensor &w = saved[1];
    const NormGrads r =
        norm_bwd(rms, grads[0].contiguous(), saved[3], saved[4], saved[0], shape, w, saved[2],
                 own_workspace(rms ? OSLO_OP_RMS_BWD : OSLO_OP_LN_BWD, w.defined()));
    return {r.dx, r.dg, r.db, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// Rows for which the one-kernel backward of bias-dropout-add + norm spills
// (_fused_norm_backward_spills of functional.py).
bool residual_norm_spills(const Tensor &h, const Shape &shape) {
  int64_t n2 = 1;
  for (int64_t d : shape) n2 *= d;
  return n2 > (h.element_size() == 2 ? 12288 : 6144);
}

// ... and the same gradients from the norm's backward followed by that of
// bias-dropout-add: the gradient of h is rounded to its dtype between the two.
ResidualNormGrads residual_norm_bwd_in_two(bool rms, const Tensor &dy, const Tensor &extra, const Tensor &h,
                                           const Tensor &mean, const Tensor &inv, const Shape &shape,
                                           const Tensor &gamma, const Dropout &d, bool want_input, bool want_bias) {
  const NormGrads n = norm_bwd(rms, dy, mean, inv, h, shape, gamma, rms ? Tensor() : gamma,
                               own_workspace(rms ? OSLO_OP_RMS_BWD : OSLO_OP_LN_BWD, gamma.defined()));
  Tensor dh = n.dx;
  if (extra.defined()) dh += extra;
  const ColumnGrads c = dropout_add_bwd(dh, d, want_input && d.p > 0.0, want_bias,
                                        own_workspace(OSLO_OP_BIAS_DROPOUT_ADD_BWD, want_bias));
  return {dh, d.p > 0.0 ? c.dx : Tensor(), n.dg, n.db, c.db.defined() ? c.db.view(shape) : Tensor()};
}

// (y, h): a gradient that nobody sends stays undefined
struct ResidualNormFunction : Function<ResidualNormFunction> {
  static variable_list forward(AutogradContext *ctx, const Tensor &input, const OptTensor &bias,
                               const OptTensor &residual, const OptTensor &weight, const OptTensor &norm_bias,
                               bool rms, const Shape &shape, double eps, const Dropout &d) {
    ctx->set_materialize_grads(false);
    const Tensor w = contiguous(weight);
    const ResidualNormOut r = residual_norm_fwd(rms, input.contiguous(), contiguous(bias), contiguous(residual),
                                                shape, w, contiguous(norm_bias), eps, d, true);
    ctx->save_for_backward({r.h, r.inv, r.mean, w});
    Shape words = dropout_words(d);
    words.insert(words.end(), {rms, given(bias), given(residual), given(norm_bias)});
    words.insert(words.end(), shape.begin(), shape.end());
    keep_words(ctx, std::move(words));
    return {r.y, r.h};
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &h = saved[0], &inv = saved[1], &mean = saved[2], &w = saved[3];
    const Shape words = words_of(ctx), shape(words.begin() + 7, words.end());
    const Dropout d = dropout_of(words);
    const bool rms = words[3], has_bias = words[4], has_res = words[5], has_norm_bias = words[6];
    const bool want_input = ctx->needs_input_grad(0), want_bias = has_bias && ctx->needs_input_grad(1);
    ResidualNormGrads r;
    if (!grads[0].defined()) {
      // only h was used: the backward of dropout(input + bias) + residual
      if (grads[1].defined()) {
        const ColumnGrads c = dropout_add_bwd(grads[1].contiguous(), d, want_input, want_bias,
                                              own_workspace(OSLO_OP_BIAS_DROPOUT_ADD_BWD, want_bias));
        r.dres = grads[1], r.dx = c.dx, r.dbias = c.db;
      }
    } else {
      const Tensor dy = grads[0].contiguous(), extra = grads[1].defined() ? grads[1].contiguous() : Tensor();
      r = residual_norm_spills(h, shape)
              ? residual_norm_bwd_in_two(rms, dy, extra, h, mean, inv, shape, w, d, want_input, want_bias)
              : residual_norm_bwd(rms, dy, extra, h, mean, inv, shape, w, d, want_bias,
                                  own_workspace(OSLO_OP_BIAS_DROPOUT_ADD_NORM_BWD, w.defined() || want_bias));
      if (d.p == 0.0) r.dx = r.dres;
    }
    return {r.dx,     want_bias ? r.dbias : Tensor(), has_res ? r.dres : Tensor(), r.dg, has_norm_bias ? r.db : Tensor(),
            Tensor(), Tensor(),                       Tensor(),                    Tensor()};
  }
};

struct CausalSoftmaxFunction : Function<CausalSoftmaxFunction> {
  static Tensor forward(AutogradContext *ctx, const Tensor &x, double scale) {
    const Tensor y = causal_fwd(x.contiguous(), (float)scale);
    ctx->save_for_backward({y});
    keep_words(ctx, {word_of(scale)});
    return y;
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const auto saved = ctx->get_saved_variables();
    return {causal_bwd(grads[0].contiguous(), saved[0], (float)real_of(words_of(ctx)[0]), false), Tensor()};
  }
};

struct MaskedSoftmaxFunction : Function<MaskedSoftmaxFunction> {
  static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &mask, double scale, bool causal) {
    const Tensor y = masked_fwd(x.contiguous(), mask, (float)scale, causal);
    ctx->save_for_backward({y, mask});
    keep_words(ctx, {word_of(scale), causal});
    return y;
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const auto saved = ctx->get_saved_variables();
    const Shape w = words_of(ctx);
    return {masked_bwd(grads[0].contiguous(), saved[0], (float)real_of(w[0]), saved[1], false, w[1] != 0), Tensor(),
            Tensor(), Tensor()};
  }
};

struct SoftmaxDropoutFunction : Function<SoftmaxDropoutFunction> {
  static Tensor forward(AutogradContext *ctx, const Tensor &input, const OptTensor &mask, double scale,
                        const Dropout &d, bool causal) {
    const Tensor x = input.contiguous(), m = given(mask) ? *mask : Tensor();
    const SoftmaxOut r = dropout_fwd(x, m, (float)scale, d, causal);
    ctx->save_for_backward({x, r.stats, m});
    Shape words = dropout_words(d);
    words.insert(words.end(), {word_of(scale), causal});
    keep_words(ctx, std::move(words));
    return r.out;
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const auto saved = ctx->get_saved_variables();
    const Shape w = words_of(ctx);
    return {dropout_bwd(grads[0].contiguous(), saved[0], saved[1], saved[2], (float)real_of(w[3]), dropout_of(w),
                        false, w[4] != 0),
            Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// Gradient of an additive term from that of the sum it was added into, summed
// over the dimensions the term was broadcast along.
Tensor term_grad(const Tensor &dt, const Tensor &bias) {
  return at::sum_to(dt, bias.sizes()).to(bias.scalar_type());
}

struct TermSoftmaxFunction : Function<TermSoftmaxFunction> {
  static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &bias, double scale, bool causal) {
    const Tensor y = bias_fwd(x.contiguous(), bias, (float)scale, causal, -1);
    ctx->save_for_backward({y, bias});
    keep_words(ctx, {word_of(scale), causal});
    return y;
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &y = saved[0], &bias = saved[1];
    const Shape w = words_of(ctx);
    const double scale = real_of(w[0]);
    const Tensor g = grads[0].contiguous();
    if (!ctx->needs_input_grad(1))
      return {bias_bwd(g, y, (float)scale, bias, w[1] != 0, -1, false), Tensor(), Tensor(), Tensor()};
    // gradient of the sum first (scale 1), then the two operands' shares
    const Tensor dt = bias_bwd(g, y, 1.0f, bias, w[1] != 0, -1, false);
    Tensor dx;
    if (ctx->needs_input_grad(0)) dx = scale == 1.0 ? dt : dt * scale;
    return {dx, term_grad(dt, bias), Tensor(), Tensor()};
  }
};

struct TermSoftmaxDropoutFunction : Function<TermSoftmaxDropoutFunction> {
  static Tensor forward(AutogradContext *ctx, const Tensor &input, const Tensor &bias, double scale,
                        const Dropout &d, bool causal) {
    const Tensor x = input.contiguous();
    const SoftmaxOut r = bias_dropout_fwd(x, bias, (float)scale, d, causal, -1);
    ctx->save_for_backward({x, r.stats, bias});
    Shape words = dropout_words(d);
    words.insert(words.end(), {word_of(scale), causal});
    keep_words(ctx, std::move(words));
    return r.out;
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &stats = saved[1], &bias = saved[2];
    const Shape w = words_of(ctx);
    const double scale = real_of(w[3]);
    const Tensor dt = bias_dropout_bwd(grads[0].contiguous(), x, bias, stats, (float)scale, dropout_of(w), w[4] != 0,
                                       -1, false);
    if (!ctx->needs_input_grad(1)) return {dt, Tensor(), Tensor(), Tensor(), Tensor()};
    // (the kernel returns scale * d(sum): the term's share is that without the scale)
    return {ctx->needs_input_grad(0) ? dt : Tensor(), term_grad(scale == 1.0 ? dt : dt / scale, bias), Tensor(),
            Tensor(), Tensor()};
  }
};

struct BiasGeluFunction : Function<BiasGeluFunction> {
  static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &bias) {
    ctx->save_for_backward({x, bias});
    return gelu_fwd(x.contiguous(), bias.contiguous());
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const auto saved = ctx->get_saved_variables();
    const bool want_bias = ctx->needs_input_grad(1);
    const ColumnGrads r = gelu_bwd(grads[0].contiguous(), saved[0].contiguous(), saved[1].contiguous(), want_bias,
                                   own_workspace(OSLO_OP_BIAS_GELU_BWD, want_bias));
    return {r.dx, r.db};
  }
};

struct DropoutAddFunction : Function<DropoutAddFunction> {
  static Tensor forward(AutogradContext *ctx, const Tensor &x, const OptTensor &bias, const OptTensor &residual,
                        const Dropout &d) {
    Shape words = dropout_words(d);
    words.insert(words.end(), {given(bias), given(residual)});
    keep_words(ctx, std::move(words));
    return dropout_add_fwd(x.contiguous(), contiguous(bias), contiguous(residual), d, Tensor(), false).out;
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const Shape w = words_of(ctx);
    const bool has_bias = w[3], has_res = w[4];
    // (the operands that were given are numbered among themselves)
    const bool want_bias = has_bias && ctx->needs_input_grad(1);
    const bool want_res = has_res && ctx->needs_input_grad(has_bias ? 2 : 1);
    const Tensor g = grads[0].contiguous();
    const ColumnGrads r = dropout_add_bwd(g, dropout_of(w), ctx->needs_input_grad(0), want_bias,
                                          own_workspace(OSLO_OP_BIAS_DROPOUT_ADD_BWD, want_bias));
    return {r.dx, r.db, want_res ? g : Tensor(), Tensor()};
  }
};

// (rms, mixed, input, weight, bias, normalized_shape, eps) -> out
PyObject *ag_norm(Args &g) {
  const bool rms = g.flag(), mixed = g.flag();
  const Tensor &x = g.tensor();
  const Tensor w = g.optional(), b = g.optional();
  const Shape shape = g.sizes();
  const double eps = g.real();
  return wrap(without_gil([&] { return NormFunction::apply(x, some(w), some(b), rms, mixed, shape, eps); }));
}

// (rms, input, bias, residual, weight, norm_bias, normalized_shape, eps, p, seed, offset) -> (y, h)
PyObject *ag_residual_norm(Args &g) {
  const bool rms = g.flag();
  const Tensor &x = g.tensor();
  const Tensor bias = g.optional(), res = g.optional(), w = g.optional(), b = g.optional();
  const Shape shape = g.sizes();
  const double eps = g.real();
  const Dropout d = g.dropout();
  const variable_list r = without_gil([&] {
    return ResidualNormFunction::apply(x, some(bias), some(res), some(w), some(b), rms, shape, eps, d);
  });
  return wrap_all({r[0], r[1]}, false);
}

// (input, scale) -> probabilities
PyObject *ag_causal(Args &g) {
  const Tensor &x = g.tensor();
  const double scale = g.real();
  return wrap(without_gil([&] { return CausalSoftmaxFunction::apply(x, scale); }));
}

// (input, mask, scale, causal) -> probabilities
PyObject *ag_masked(Args &g) {
  const Tensor &x = g.tensor();
  const Tensor &mask = g.tensor();
  const double scale = g.real();
  const bool causal = g.flag();
  return wrap(without_gil([&] { return MaskedSoftmaxFunction::apply(x, mask, scale, causal); }));
}

// (input, mask or None, scale, p, seed, offset, causal) -> dropped probabilities
PyObject *ag_dropout(Args &g) {
  const Tensor &x = g.tensor();
  const Tensor mask = g.optional();
  const double scale = g.real();
  const Dropout d = g.dropout();
  const bool causal = g.flag();
  return wrap(without_gil([&] { return SoftmaxDropoutFunction::apply(x, some(mask), scale, d, causal); }));
}

// (input, bias, scale, causal) -> probabilities
PyObject *ag_term(Args &g) {
  const Tensor &x = g.tensor();
  const Tensor &bias = g.tensor();
  const double scale = g.real();
  const bool causal = g.flag();
  return wrap(without_gil([&] { return TermSoftmaxFunction::apply(x, bias, scale, causal); }));
}

// (input, bias, scale, p, seed, offset, causal) -> dropped probabilities
PyObject *ag_term_dropout(Args &g) {
  const Tensor &x = g.tensor();
  const Tensor &bias = g.tensor();
  const double scale = g.real();
  const Dropout d = g.dropout();
  const bool causal = g.flag();
  return wrap(without_gil([&] { return TermSoftmaxDropoutFunction::apply(x, bias, scale, d, causal); }));
}

// (input, bias) -> out
PyObject *ag_bias_gelu(Args &g) {
  const Tensor &x = g.tensor();
  const Tensor &bias = g.tensor();
  return wrap(without_gil([&] { return BiasGeluFunction::apply(x, bias); }));
}

// (input, bias or None, residual or None, p, seed, offset) -> out
PyObject *ag_dropout_add(Args &g) {
  const Tensor &x = g.tensor();
  const Tensor bias = g.optional(), res = g.optional();
  const Dropout d = g.dropout();
  return wrap(without_gil([&] { return DropoutAddFunction::apply(x, some(bias), some(res), d); }));
}

// ---------------------------------------------------------------- module
template <PyObject *(*F)(Args &)>
PyObject *entry(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args args{a, n};
  return F(args);
  END_HANDLE_TH_ERRORS
}

#define OSLO_METHOD(F) {#F, (PyCFunction)(void (*)(void))entry<F>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    OSLO_METHOD(norm_forward),
    OSLO_METHOD(norm_backward),
    OSLO_METHOD(residual_norm_forward),
    OSLO_METHOD(residual_norm_backward),
    OSLO_METHOD(causal_forward),
    OSLO_METHOD(causal_backward),
    OSLO_METHOD(masked_forward),
    OSLO_METHOD(masked_backward),
    OSLO_METHOD(dropout_forward),
    OSLO_METHOD(dropout_backward),
    OSLO_METHOD(bias_operand),
    OSLO_METHOD(bias_flags),
    OSLO_METHOD(bias_forward),
    OSLO_METHOD(bias_backward),
    OSLO_METHOD(bias_dropout_forward),
    OSLO_METHOD(bias_dropout_backward),
    OSLO_METHOD(gelu_forward),
    OSLO_METHOD(gelu_backward),
    OSLO_METHOD(dropout_add_forward),
    OSLO_METHOD(dropout_add_backward),
    OSLO_METHOD(ag_norm),
    OSLO_METHOD(ag_residual_norm),
    OSLO_METHOD(ag_causal),
    OSLO_METHOD(ag_masked),
    OSLO_METHOD(ag_dropout),
    OSLO_METHOD(ag_term),
    OSLO_METHOD(ag_term_dropout),
    OSLO_METHOD(ag_bias_gelu),
    OSLO_METHOD(ag_dropout_add),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "oslo_torch_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_oslo_torch_calls() { return PyModule_Create(&module); }
