// Multi-tensor Adam / AdamW step for gfx950.
//
// One launch updates up to kMaxTensors parameter tensors: the tensor table
// (four pointers and a length per tensor, plus the prefix sums of the
// workgroups each tensor takes) travels in the kernel arguments, so nothing
// is staged in device memory.  A workgroup owns one short contiguous piece of
// one tensor -- a 128-bit vector per lane of each of g, p, m, v -- and
// exits: the launch is a plain streaming pass bound by HBM (28 bytes per fp32
// element, 14 per 16-bit element).  Arithmetic follows
// oslo/torch/_C/csrc/multi_tensor_adam.cu:22-110 of the reference: fp32 math,
// mode 0 = L2 regularisation (the decay joins the gradient), mode 1 =
// decoupled weight decay (AdamW).
#include <math.h>

#include "capi.h"
#include "common.hip.h"

namespace oslo {

// 44 bytes a tensor next to the scalars in the 4 KB of kernel arguments
constexpr int kMaxTensors = 88;
constexpr int kAdamThreads = 256;

struct AdamTable {
  void *g[kMaxTensors];
  void *p[kMaxTensors];
  void *m[kMaxTensors];
  void *v[kMaxTensors];
  int64_t n[kMaxTensors];
  int32_t first_block[kMaxTensors + 1];  // prefix sums of workgroups
  int ntensors;
};

// 1 / bc as the sum of two floats: x / bc is then one fused multiply-add on a
// product and lies within 0.5001 ulp of the quotient.  (An infinite x, which an
// overflowed second moment is, enters the small product as the largest float.)
struct Recip {
  float hi, lo;
};

struct AdamArgs {
  float beta1, beta2, eps, lr, decay;
  Recip rbc1, rbc2;
  int mode;
  int scaled;  // eps beyond 2^-96 ... 2^90: see quotient()
};
static_assert(sizeof(AdamTable) + sizeof(AdamArgs) <= 4096, "kernel arguments");

static Recip reciprocal(float bc) {
  const double r = 1.0 / (double)bc;
  Recip q;
  q.hi = (float)r;
  q.lo = (float)(r - (double)q.hi);
  if (!(fabs(r) <= 3.0e38)) q.lo = 0.f;  // bc = 0: x / 0
  return q;
}

__device__ __forceinline__ float times(float x, const Recip &r) {
  return fmaf(x, r.hi, __builtin_amdgcn_fmed3f(x, -__FLT_MAX__, __FLT_MAX__) * r.lo);
}

// sqrt(x), one Newton step on x * v_rsq_f32(x): s + (x - s^2) / (2 sqrt(x)).
// x below 2^-96 is scaled by 2^64, where the residual of the step would lose
// its bits; zero and infinity are their own roots, NaN and negative values
// come out as NaN.
__device__ __forceinline__ float root(float x) {
  const bool small = x < 0x1p-96f;
  const float y = small ? x * 0x1p64f : x;
  const float r = __builtin_amdgcn_rsqf(y);
  const float s = y * r;
  const float t = fmaf(fmaf(-s, s, y), 0.5f * r, s);
  const float u = small ? t * 0x1p-32f : t;
  return x == 0.f || x == __builtin_inff() ? x : u;
}

// a / b, one Newton step on a * v_rcp_f32(b): q + (a - b q) / b, with the
// special values (zero, infinity, NaN) of the exact quotient.  A quotient that
// overflows stays infinite (its residual enters the step as the largest float).
// The divisors that v_rcp_f32 does not take, subnormal ones and those whose
// reciprocal is subnormal, are scaled with the dividend; only an eps of that size
// leads to one (SCALED, a branch of the whole vector: in every step it would cost
// 16-bit tensors of 2 M parameters 5 %).
template <bool SCALED> __device__ __forceinline__ float quotient(float a, float b) {
  if constexpr (SCALED) {
    const float k = fabsf(b) < 0x1p-96f ? 0x1p64f : fabsf(b) > 0x1p96f ? 0x1p-64f : 1.f;
    a *= k;
    b *= k;
  }
  const float r = __builtin_amdgcn_rcpf(b);
  const float q = a * r;
  const float rest = __builtin_amdgcn_fmed3f(fmaf(-b, q, a), -__FLT_MAX__, __FLT_MAX__);
  return __builtin_amdgcn_div_fixupf(fmaf(rest, r, q), b, a);
}

// The update of multi_tensor_adam.cu:78-96, term for term.  Its three
// divisions and the square root as the language defines them are some 145
// instructions an element: bf16 spent 83 % of its time in them.  The two by
// constants are products here, the other two take one Newton step.
template <bool SCALED>
__device__ __forceinline__ void adam_update(float g, float &p, float &m,
                                            float &v, const AdamArgs &a) {
  if (a.mode == 0) g = g + a.decay * p;
  m = a.beta1 * m + (1.f - a.beta1) * g;
  v = a.beta2 * v + (1.f - a.beta2) * g * g;
  const float denom = root(times(v, a.rbc2)) + a.eps;
  float update = quotient<SCALED>(times(m, a.rbc1), denom);
  if (a.mode != 0) update = update + a.decay * p;
  p = p - a.lr * update;
}

template <typename T, int kAdamUnroll>
__global__ __launch_bounds__(kAdamThreads) void multi_tensor_adam_kernel(
    AdamTable tab, AdamArgs a) {
  constexpr int E = io<T>::EPV;
  constexpr int64_t kPiece = (int64_t)kAdamThreads * kAdamUnroll * E;
  // which tensor does this workgroup belong to: the last one that starts at or
  // before it (uniform: scalar loads, a search by halves)
  const int b = (int)blockIdx.x;
  int t = 0;
  for (int end = tab.ntensors; end - t > 1;) {
    const int mid = (t + end) >> 1;
    if (tab.first_block[mid] <= b) t = mid;
    else end = mid;
  }
  const int64_t piece = b - tab.first_block[t];
  const int64_t n = tab.n[t];
  const int64_t start = piece * kPiece;
  const T *g = static_cast<const T *>(tab.g[t]);
  T *p = static_cast<T *>(tab.p[t]);
  T *m = static_cast<T *>(tab.m[t]);
  T *v = static_cast<T *>(tab.v[t]);
  const bool aligned = ((reinterpret_cast<uintptr_t>(g) | reinterpret_cast<uintptr_t>(p) |
                         reinterpret_cast<uintptr_t>(m) | reinterpret_cast<uintptr_t>(v)) &
                        15u) == 0;
  if (aligned && start + kPiece <= n) {
    // full piece: kAdamUnroll vectors per lane and operand, all loads first
    float rg[kAdamUnroll][E], rp[kAdamUnroll][E], rm[kAdamUnroll][E], rv[kAdamUnroll][E];
#pragma unroll
    for (int u = 0; u < kAdamUnroll; ++u) {
      const int64_t i = start + ((int64_t)u * kAdamThreads + threadIdx.x) * E;
      load_chunk<T, E>(g + i, rg[u]);
      load_chunk<T, E>(p + i, rp[u]);
      load_chunk<T, E>(m + i, rm[u]);
      load_chunk<T, E>(v + i, rv[u]);
    }
#pragma unroll
    for (int u = 0; u < kAdamUnroll; ++u) {
      const int64_t i = start + ((int64_t)u * kAdamThreads + threadIdx.x) * E;
      if (a.scaled) {
#pragma unroll
        for (int e = 0; e < E; ++e) adam_update<true>(rg[u][e], rp[u][e], rm[u][e], rv[u][e], a);
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e) adam_update<false>(rg[u][e], rp[u][e], rm[u][e], rv[u][e], a);
      }
      store_chunk<T, E>(p + i, rp[u]);
      store_chunk<T, E>(m + i, rm[u]);
      store_chunk<T, E>(v + i, rv[u]);
    }
    return;
  }
  // last piece of a tensor, or a tensor whose storage is not 16-byte aligned
  const int64_t end = start + kPiece < n ? start + kPiece : n;
  for (int64_t i = start + threadIdx.x; i < end; i += kAdamThreads) {
    const float gg = io<T>::from_scalar(g[i]);
    float pp = io<T>::from_scalar(p[i]);
    float mm = io<T>::from_scalar(m[i]);
    float vv = io<T>::from_scalar(v[i]);
    if (a.scaled)
      adam_update<true>(gg, pp, mm, vv, a);
    else
      adam_update<false>(gg, pp, mm, vv, a);
    p[i] = io<T>::to_scalar(pp);
    m[i] = io<T>::to_scalar(mm);
    v[i] = io<T>::to_scalar(vv);
  }
}

template <typename T, int kAdamUnroll>
static int launch_adam(const void *const *g, void *const *p, void *const *m,
                       void *const *v, const int64_t *sizes, int64_t ntensors,
                       const AdamArgs &a, hipStream_t st) {
  constexpr int64_t kPiece = (int64_t)kAdamThreads * kAdamUnroll * io<T>::EPV;
  AdamTable tab;
  tab.ntensors = 0;
  tab.first_block[0] = 0;
  auto flush = [&]() -> int {
    if (tab.ntensors == 0) return OSLO_OK;
    const int64_t blocks = tab.first_block[tab.ntensors];
    if (blocks > 0) {
      multi_tensor_adam_kernel<T, kAdamUnroll>
          <<<dim3((unsigned)blocks), kAdamThreads, 0, st>>>(tab, a);
      const int rc = check_launch("multi_tensor_adam_kernel");
      if (rc != OSLO_OK) return rc;
    }
    tab.ntensors = 0;
    return OSLO_OK;
  };
  for (int64_t i = 0; i < ntensors; ++i) {
    if (sizes[i] == 0) continue;
    if (sizes[i] < 0)
      return fail(OSLO_ERR_INVALID_ARGUMENT, "multi_tensor_adam: tensor %lld has size %lld",
                  (long long)i, (long long)sizes[i]);
    if (!g[i] || !p[i] || !m[i] || !v[i])
      return fail(OSLO_ERR_INVALID_ARGUMENT, "multi_tensor_adam: tensor %lld has a null pointer",
                  (long long)i);
    // one launch stays below 2^32 work-items
    if (tab.ntensors > 0 &&
        (int64_t)tab.first_block[tab.ntensors] + ceil_div(sizes[i], kPiece) > max_workgroups(kAdamThreads)) {
      const int rc = flush();
      if (rc != OSLO_OK) return rc;
    }
    if (ceil_div(sizes[i], kPiece) > max_workgroups(kAdamThreads))
      return fail(OSLO_ERR_UNSUPPORTED, "multi_tensor_adam: a tensor too large for one launch");
    const int k = tab.ntensors;
    tab.g[k] = const_cast<void *>(g[i]);
    tab.p[k] = p[i];
    tab.m[k] = m[i];
    tab.v[k] = v[i];
    tab.n[k] = sizes[i];
    tab.first_block[k + 1] = tab.first_block[k] + (int32_t)ceil_div(sizes[i], kPiece);
    tab.ntensors = k + 1;
    if (tab.ntensors == kMaxTensors) {
      const int rc = flush();
      if (rc != OSLO_OK) return rc;
    }
  }
  return flush();
}

}  // namespace oslo

extern "C" {

int oslo_multi_tensor_adam(const void *const *g, void *const *p, void *const *m,
                           void *const *v, const int64_t *sizes,
                           int64_t ntensors, float lr, float beta1, float beta2,
                           float eps, int step, int mode, int bias_correction,
                           float weight_decay, int dtype, void *stream) {
  oslo::tune_snapshot();
  using namespace oslo;
  if (!valid_dtype(dtype))
    return fail(OSLO_ERR_INVALID_ARGUMENT, "multi_tensor_adam: unknown dtype %d", dtype);
  OSLO_REQUIRE(ntensors >= 0, "multi_tensor_adam: negative tensor count");
  OSLO_REQUIRE(mode == 0 || mode == 1, "multi_tensor_adam: mode %d is neither 0 (L2) nor 1 (AdamW)",
               mode);
  if (ntensors == 0) return OSLO_OK;
  OSLO_REQUIRE(g && p && m && v && sizes, "multi_tensor_adam: null table pointer");
  AdamArgs a;
  a.beta1 = beta1;
  a.beta2 = beta2;
  a.eps = eps;
  a.lr = lr;
  a.decay = weight_decay;
  a.mode = mode;
  a.scaled = eps != 0.f && !(eps >= 0x1p-96f && eps <= 0x1p90f);
  // multi_tensor_adam.cu:120-125: 1 - beta^step, evaluated by std::pow on the
  // float betas (which promotes to double) and stored as float
  float bc1 = 1.0f, bc2 = 1.0f;
  if (bias_correction == 1) {
    bc1 = (float)(1.0 - pow((double)beta1, (double)step));
    bc2 = (float)(1.0 - pow((double)beta2, (double)step));
  }
  a.rbc1 = reciprocal(bc1);
  a.rbc2 = reciprocal(bc2);
  hipStream_t st = (hipStream_t)stream;
  // 128-bit vectors per lane and operand: short-lived workgroups sweep the
  // seven streams in the tightest window, so one is the fastest for every type
  // and size (with the arithmetic of adam_update; before, four with IEEE
  // divisions).  85 M parameters: fp32 411 -> 396 us (6.0 TB/s), bf16 218 -> 191,
  // fp16 218 -> 192; 1.6 M parameters: 10.2 -> 8.3, 9.5 -> 5.4, 10.0 -> 5.6.
  // Two vectors: 400, 198, 199; 9.0, 6.1, 6.3.
  const int unroll = g_tune.adam_unroll == 2 || g_tune.adam_unroll == 4 ? g_tune.adam_unroll : 1;
#define OSLO_ADAM(T_)                                                           \
  (unroll == 1   ? launch_adam<T_, 1>(g, p, m, v, sizes, ntensors, a, st)       \
   : unroll == 2 ? launch_adam<T_, 2>(g, p, m, v, sizes, ntensors, a, st)       \
                 : launch_adam<T_, 4>(g, p, m, v, sizes, ntensors, a, st))
  if (dtype == OSLO_DTYPE_F32) return OSLO_ADAM(float);
  if (dtype == OSLO_DTYPE_F16) return OSLO_ADAM(_Float16);
  return OSLO_ADAM(__bf16);
#undef OSLO_ADAM
}

}  // extern "C"
