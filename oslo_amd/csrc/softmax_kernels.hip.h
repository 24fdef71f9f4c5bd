// Scaled causal (upper-triangular) and padding-masked softmax, forward and
// backward, for gfx950.
//
// A row of sk keys is held in registers by `wpr` wavefronts (one wavefront
// for sk <= 64 * VPL * E); a wavefront processes RPW rows at once so that
// short rows still keep several 128-bit loads in flight per lane, and rows of
// at most 32 chunks (256 16-bit keys) lie side by side in a wavefront, 8, 16
// or 32 lanes each, so that no lane idles.  Rows whose length is no multiple
// of a chunk, or whose operands are not 16-byte aligned, take the same kernels
// in a build that accesses the chunks where they lie (RAG).  Keys that
// are masked out are never loaded: the causal kernels stop at the diagonal,
// the masked kernels read the mask bytes of a chunk first and skip the chunk
// when all of them are set.  Probabilities of masked keys are written as
// exact zeros.
//
// Semantics: oslo/transformers/models/gpt2/modeling_gpt2.py:116-138 (causal),
// oslo/transformers/models/bert/modeling_bert.py:298-306 (additive padding
// mask); entry-point shapes follow
// oslo/torch/_C/csrc/FusedScaleMaskSoftmaxBinder.cpp:39-105.
#pragma once
#include "capi.h"
#include "common.hip.h"

namespace oslo {

constexpr int kModeCausal = 0;
constexpr int kModeMasked = 1;
constexpr int kModeDense = 2;  // backward without a mask
constexpr int kModeBias = 3;   // additive floating-point term instead of a mask

// An additive term at or below this value (the lowest finite bfloat16; the
// lowest finite float and -inf lie below it) absorbs any logit it is added to:
// the sum is the term itself in float arithmetic, so the logit need not be read.
constexpr float kBiasHidden = -3.38e38f;

constexpr float kLog2e = 1.4426950408889634f;

struct SoftmaxGeom {
  int64_t rows;     // total softmax rows
  int sq, sk;
  int np;           // heads (masked mode)
  int mask_b_stride_rows;  // mask rows per batch entry: mask_sq, or 0 if mask_b == 1
  int mask_per_query;      // 1 if mask_sq == sq else 0
  int wpr, rpb;     // waves per row, rows per workgroup pass (without RPW)
  int causal;       // masked mode: key j of query i is also hidden when j > i + (sk - sq)
  // n / sq and n / np for n < 2^31 as mulhi(n, mul) >> shift (shift == 32: divisor 1),
  // filled in by set_fast_div on the host
  uint32_t sq_mul = 0, sq_shift = 32, np_mul = 0, np_shift = 32;
  float inv_sk = 0.f;  // 1 / sk, the value of a row without a visible key
  // index of the launch's first workgroup among those of the whole problem (a
  // problem beyond 2^32 work-items takes several launches)
  int64_t blk0 = 0;
  // additive term (kModeBias): element strides of its batch, head and query
  // dimensions (0 = broadcast), bytes per element, and whether a chunk whose
  // terms are all <= kBiasHidden skips the load of its logits
  int64_t bias_sb = 0, bias_sh = 0, bias_sq = 0;
  int bias_esize = 0, bias_skip = 0;
  // An additive term shared by the batch (a position bias [1, np, sq, sk]): the
  // rows are visited in runs of 2^group_shift consecutive rows of one batch
  // entry, then the same rows of the next entry, so that the nb rows that read
  // one row of the term run close to each other and the L2 serves it to all
  // but the first of them (measured at [16, 16, 1024, 1024] fp16: 221 us in
  // stored order, 203 us with runs of one row, 169 us with runs of 32, which
  // keep the logits in long contiguous pieces).  With xcd_wpx != 0 workgroup w
  // works on block (w % 8) * xcd_wpx + w / 8, which puts consecutive blocks on
  // one of the eight dies (191 us with runs of one row, 179-181 us with runs
  // of 32-128: not the default).
  int batch_inner = 0, nb = 1;
  int group_shift = 0;   // the batch index advances after 2^group_shift rows
  uint32_t nb_mul = 0, nb_shift = 32;
  int64_t hq_rows = 0;   // np * sq
  int64_t xcd_wpx = 0;   // 0: blocks in launch order
  int64_t die_end = 0;   // ragged rows: end of the blocks dealt out by die (work_block)
  // Order of the queries of one attention matrix under the diagonal: 0 = long
  // rows first, 1 = as stored, 2 = long and short rows in turn (the k-th row
  // visited is sq - 1 - k / 2 for even k and k / 2 for odd k), so that any run
  // of consecutive rows moves the same number of bytes.
  int causal_order = 0;
};

// Query index of the k-th row visited in an attention matrix of sq queries.
__device__ __forceinline__ int causal_query(const SoftmaxGeom &g, int k) {
  if (g.causal_order == 2) return (k & 1) ? (k >> 1) : g.sq - 1 - (k >> 1);
  return g.causal_order == 1 ? k : g.sq - 1 - k;
}

// The block of rows a workgroup works on.
template <bool RAG = false>
__device__ __forceinline__ int64_t work_block(const SoftmaxGeom &g) {
  if (g.xcd_wpx != 0) return (int64_t)(blockIdx.x & 7u) * g.xcd_wpx + (int64_t)(blockIdx.x >> 3);
  const int64_t b = (int64_t)blockIdx.x + g.blk0;
  if constexpr (RAG) {
    // Workgroups go to the eight dies in turn.  Of every 64, each die takes
    // eight consecutive blocks: the cache line that two blocks of ragged rows
    // share is then mostly written through one L2, while the launch still moves
    // through memory in one compact window.  (bf16 causal with dropout
    // [128, 1531, 1531] forward + backward 374 -> 370 us, fp16 [2, 32, 1003,
    // 1003] with a key mask, in its layer, 98 -> 96; runs of 4 and of 16 the
    // same, of 32 slower: 385.)
    if (b < g.die_end) return (b & ~(int64_t)63) | ((b & 7) << 3) | ((b >> 3) & 7);
  }
  return b;
}

// Division of n < 2^31 by a divisor 1 <= d < 2^31 fixed for the launch: with
// l = ceil(log2 d) and mul = ceil(2^(31 + l) / d) < 2^32, floor(n / d) equals
// mulhi(n, mul) >> (l - 1) exactly (the error term n * e / (d * 2^(31 + l)) with
// e < d stays below 2^-l <= 1 / d).  A run-time division costs about as many
// vector instructions as the softmax of a short row.
static inline void fast_div_make(uint32_t d, uint32_t *mul, uint32_t *shift) {
  if (d <= 1) {
    *mul = 0;
    *shift = 32;
    return;
  }
  uint32_t l = 0;
  while ((1ull << l) < d) ++l;
  *mul = (uint32_t)(((1ull << (31 + l)) + d - 1) / d);
  *shift = l - 1;
}

static inline void set_fast_div(SoftmaxGeom &g) {
  fast_div_make((uint32_t)g.sq, &g.sq_mul, &g.sq_shift);
  fast_div_make((uint32_t)g.np, &g.np_mul, &g.np_shift);
  fast_div_make((uint32_t)g.nb, &g.nb_mul, &g.nb_shift);
  g.inv_sk = 1.0f / (float)g.sk;
  g.causal_order = g_tune.softmax_causal_order > 0 ? g_tune.softmax_causal_order - 1 : 0;
}

__device__ __forceinline__ uint32_t fast_div(uint32_t n, uint32_t mul, uint32_t shift) {
  return shift == 32 ? n : __umulhi(n, mul) >> shift;
}

// 1 / s for the row sum s >= 1 of a softmax: the hardware reciprocal refined by
// one Newton step (within an ulp of the quotient; an IEEE division costs ten
// instructions).  Every softmax kernel forms its normaliser with this function.
__device__ __forceinline__ float row_recip(float s) {
  const float r = __builtin_amdgcn_rcpf(s);
  return __builtin_fmaf(r, __builtin_fmaf(-s, r, 1.0f), r);
}

// Reductions over the wpr (<= 16) consecutive waves of a row: lane 0 of each
// wave publishes its wave's value in LDS, lane l < wpr then reads the value of
// wave first + l and one DPP row reduction combines them.  With LPR < 64 a
// row belongs to LPR consecutive lanes of one wave (wpr == 1) and the
// reduction stays inside that group.
template <int LPR = kWave>
__device__ __forceinline__ float row_reduce_sum(float a, float *red, int wave,
                                                int first, int wpr, int lane) {
  if constexpr (LPR < kWave) return group_allreduce<OpSum, LPR>(a);
  a = wave_sum(a);
  if (wpr > 1) {
    if (lane == 0) red[wave] = a;
    __syncthreads();
    const bool own = lane < wpr;
    const float r = red[own ? first + lane : first];
    a = row16_allreduce<OpSum>(own ? r : 0.f);
  }
  return a;
}
template <int LPR = kWave>
__device__ __forceinline__ float row_reduce_max(float a, float *red, int wave,
                                                int first, int wpr, int lane) {
  if constexpr (LPR < kWave) return group_allreduce<OpMax, LPR>(a);
  a = wave_max(a);
  if (wpr > 1) {
    if (lane == 0) red[wave] = a;
    __syncthreads();
    // lanes >= wpr repeat the first wave's value, which leaves the maximum unchanged
    a = row16_allreduce<OpMax>(red[lane < wpr ? first + lane : first]);
  }
  return a;
}

// Mask bytes of one chunk as loaded, and their bits: bit e set when key e of
// the chunk is masked out.  (In two steps, like every operand of these
// kernels: all loads of a row are requested before any is converted.  A
// conversion next to its load, inside the branch that decides about the load,
// makes the wave wait for one chunk before it requests the next.)
template <int E, bool ANY> struct MaskChunk {
  uint32_t w[E / 4];
  __device__ __forceinline__ void load(const uint8_t *p) {
    if constexpr (E == 8) {
      u32x2 m;
      if constexpr (ANY)
        m = *reinterpret_cast<const u32x2_any *>(p);
      else
        m = *reinterpret_cast<const u32x2 *>(p);
      w[0] = m.x;
      w[1] = m.y;
    } else {
      if constexpr (ANY)
        w[0] = *reinterpret_cast<const u32_any *>(p);
      else
        w[0] = *reinterpret_cast<const uint32_t *>(p);
    }
  }
  // bit 7 of every byte that is not zero
  static __device__ __forceinline__ uint32_t nonzero_bytes(uint32_t v) {
    return (((v & 0x7f7f7f7fu) + 0x7f7f7f7fu) | v) & 0x80808080u;
  }
  // (the flags of four bytes at a time, then gathered: 14 instructions where
  //  testing the eight bytes one by one takes 24)
  __device__ __forceinline__ uint32_t bits() const {
    uint32_t x = nonzero_bytes(w[0]) >> 7;
    if constexpr (E == 8) x |= nonzero_bytes(w[1]) >> 3;
    x |= (x >> 7) | (x >> 14) | (x >> 21);
    return x & ((1u << E) - 1u);
  }
};

// All outstanding vector loads have arrived.  The kernels say so once, between
// the loads of a row and their use (and, where they have to look at mask bytes or
// terms before they know which logits to request, between the two): the
// compiler otherwise carries a load inside a branch as possibly outstanding
// through all later branches and waits again in front of each, by then for the
// loads or the stores in between.
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0f70); }

// Bits of the keys i0 .. i0 + E that lie at or beyond `visible`.
template <int E>
__device__ __forceinline__ uint32_t beyond_bits(int i0, int visible) {
  constexpr uint32_t kAllBits = (1u << E) - 1u;
  // keys of the chunk below the diagonal, 0 .. E
  const int left = min(max(visible - i0, 0), E);
  return kAllBits & (kAllBits << left);
}

// Row bookkeeping shared by forward and backward.  Rows are numbered so that
// a workgroup's rows are consecutive; under the diagonal the queries of an
// attention matrix are visited in the order causal_query() gives.
template <int MODE>
__device__ __forceinline__ void row_setup(const SoftmaxGeom &g, int64_t r,
                                          const uint8_t *mask, int64_t &row,
                                          int &visible,
                                          const uint8_t *&mrow) {
  mrow = nullptr;
  visible = g.sk;
  row = r;
  // multiplication by a precomputed reciprocal where the row count allows it
  const bool small = g.rows <= 0x7fffffff;
  if constexpr (MODE == kModeCausal) {
    const int64_t batch =
        small ? (int64_t)fast_div((uint32_t)r, g.sq_mul, g.sq_shift) : r / g.sq;
    const int qi = causal_query(g, (int)(r - batch * g.sq));
    row = batch * g.sq + qi;
    int v = qi + 1 + (g.sk - g.sq);
    visible = v < 0 ? 0 : (v > g.sk ? g.sk : v);
  } else if constexpr (MODE == kModeMasked) {
    const int64_t bh =
        small ? (int64_t)fast_div((uint32_t)r, g.sq_mul, g.sq_shift) : r / g.sq;
    int qi = (int)(r - bh * g.sq);
    if (g.causal) {  // uniform over the launch: the order of causal mode
      qi = causal_query(g, qi);
      row = bh * g.sq + qi;
      const int v = qi + 1 + (g.sk - g.sq);
      visible = v < 0 ? 0 : (v > g.sk ? g.sk : v);
    }
    const int64_t bi =
        small ? (int64_t)fast_div((uint32_t)bh, g.np_mul, g.np_shift) : bh / g.np;
    const int64_t mr =
        bi * g.mask_b_stride_rows + (g.mask_per_query ? qi : 0);
    mrow = mask + mr * g.sk;
  } else if constexpr (MODE == kModeBias) {
    if (g.batch_inner) {
      // r = (run * nb + batch entry) * 2^group_shift + row within the run
      const int64_t t = r >> g.group_shift;
      const int64_t in_run = r - (t << g.group_shift);
      const int64_t run =
          small ? (int64_t)fast_div((uint32_t)t, g.nb_mul, g.nb_shift) : t / g.nb;
      r = (t - run * g.nb) * g.hq_rows + (run << g.group_shift) + in_run;
      row = r;
    }
    const int64_t bh =
        small ? (int64_t)fast_div((uint32_t)r, g.sq_mul, g.sq_shift) : r / g.sq;
    int qi = (int)(r - bh * g.sq);
    if (g.causal) {
      qi = causal_query(g, qi);
      row = bh * g.sq + qi;
      const int v = qi + 1 + (g.sk - g.sq);
      visible = v < 0 ? 0 : (v > g.sk ? g.sk : v);
    }
    const int64_t bi =
        small ? (int64_t)fast_div((uint32_t)bh, g.np_mul, g.np_shift) : bh / g.np;
    const int64_t hi = bh - bi * g.np;
    // (mask is the additive term's base address here; null in a backward
    //  pass that does not use it)
    mrow = mask + (bi * g.bias_sb + hi * g.bias_sh + qi * g.bias_sq) * g.bias_esize;
  }
}

// One chunk of the additive term, E values of the logits' type T or of float
// (a launch-uniform choice, so one kernel serves both): as loaded (E / 4
// vectors, the first one only for a 16-bit term), then its conversion.
template <typename T, int E, bool ANY>
__device__ __forceinline__ void load_bias_raw(const uint8_t *row, int i0, bool f32, u32x4 *r) {
  if (sizeof(T) == 4 || f32) {
#pragma unroll
    for (int v = 0; v < E / 4; ++v) r[v] = ld16_cached_at<ANY>(row + ((int64_t)i0 + 4 * v) * 4);
  } else {
    r[0] = ld16_cached_at<ANY>(row + (int64_t)i0 * (int64_t)sizeof(T));
  }
}
template <typename T, int E>
__device__ __forceinline__ void unpack_bias_raw(const u32x4 *r, bool f32, float *f) {
  if (sizeof(T) == 4 || f32) {
#pragma unroll
    for (int v = 0; v < E / 4; ++v) io<float>::unpack(r[v], f + 4 * v);
  } else {
    io<T>::unpack(r[0], f);
  }
}

// every term of the chunk absorbs its logit
template <int E>
__device__ __forceinline__ bool bias_all_hidden(const float *f) {
  float m = f[0];
#pragma unroll
  for (int e = 1; e + 1 < E; e += 2) m = fmaxf(fmaxf(m, f[e]), f[e + 1]);  // v_max3_f32
  if constexpr (E % 2 == 0) m = fmaxf(m, f[E - 1]);
  return m <= kBiasHidden;  // (false for NaN)
}

// scalar read of element i of an additive-term row (generic kernels)
template <typename T>
__device__ __forceinline__ float bias_at(const uint8_t *row, int i, bool f32) {
  if (sizeof(T) == 4 || f32) return reinterpret_cast<const float *>(row)[i];
  return io<T>::from_scalar(reinterpret_cast<const T *>(row)[i]);
}

// ---------------------------------------------------------------------------
// Ragged rows (RAG builds; bound: HBM, with dropout VALU): a row length that is
// no multiple of a chunk, or operands off the 16-byte grid.  The chunks are
// counted from the first key of the row and accessed where they lie; the last
// one ends with the row and overlaps the chunk before it, so that every access
// is a whole vector inside the row.  Its first dup_keys() keys are held twice:
// they count once in the sums, and both lanes store the same bits.  One of the
// two chunks may be read and the other not (hidden keys only), so a hidden key
// of these two gets a value that depends on the row alone: zero in the forward
// pass, also in a row of NaN, and hidden_grad() in the backward passes, which
// take its gradient for zero.  (Storing such keys from one of the lanes only, as
// one store for each power of two in their number or merged from the other lane,
// costs 3 to 4 % from 1000 keys on and up to 37 % for short rows.)
// (One wave per row with 2-byte accesses before; bf16 causal [51, 1531, 1531]:
// forward 176 -> 67 us, backward 246 -> 89, with dropout 390 -> 79 and 305 -> 94;
// fp32 1003 keys 94 -> 78 and 126 -> 96 us.)
// ---------------------------------------------------------------------------
template <int E, bool RAG>
__device__ __forceinline__ int chunk_key(int c, int sk) {
  const int i0 = c * E;
  if constexpr (RAG) return i0 < sk - E ? i0 : sk - E;
  return i0;
}
template <int E, bool RAG>
__device__ __forceinline__ int dup_keys(int c, int sk) {
  return RAG ? c * E - chunk_key<E, RAG>(c, sk) : 0;
}

// one of the two chunks that hold the keys of a ragged row held twice
template <int E>
__device__ __forceinline__ bool shares_keys(int c, int sk) { return c * E > sk - 2 * E; }
// input gradient of a hidden key in a row whose sum is s: what scale * y * (g - s)
// comes to for y = 0, g = 0 (a zero, or NaN with the rest of the row)
__device__ __forceinline__ float hidden_grad(float scale, float s) { return scale * (0.f * (0.f - s)); }
// float16 results of a ragged row: the float value converted as it is (in one
// slot of a kernel the product could otherwise be fused into the conversion and
// in another not, which differs on ties)
template <typename T, bool RAG> __device__ __forceinline__ float one_rounding(float v) {
  if constexpr (RAG && __is_same(T, _Float16)) return pinned(v);
  return v;
}

// Dropout of a ragged row: its chunks straddle the groups of eight elements of
// the flattened tensor.  The lanes of the row (`stride` of them, this one is
// number `idx`) draw its groups once, one byte of keep bits each, into LDS
// (kb), as many as reach `keys` keys; a chunk then takes its bits from two
// neighbouring bytes.
template <int E>
__device__ __forceinline__ void draw_row_groups(uint8_t *kb, int64_t row, int sk, int keys,
                                                int idx, int stride, const DropArgs &d) {
  const uint64_t flat = (uint64_t)row * (uint64_t)sk;
  // (all of the last chunk that holds one of the keys)
  const int upto = keys + E - 1 < sk ? keys + E - 1 : sk;
  const int groups = keys > 0 ? ((int)(flat & 7u) + upto + 7) >> 3 : 0;
  for (int t = idx; t < groups; t += stride)
    kb[t] = (uint8_t)dropout_keep_bits((flat >> 3) + (uint64_t)t, d.seed, d.offset, d.threshold);
}
// makes the draws of the row's lanes visible to each other
__device__ __forceinline__ void row_draws_done(int wpr) {
  if (wpr > 1) {
    __syncthreads();
  } else {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}
__device__ __forceinline__ uint32_t row_keep_bits(const uint8_t *kb, int64_t row, int sk, int i0) {
  const uint32_t at = ((uint32_t)((uint64_t)row * (uint64_t)sk) & 7u) + (uint32_t)i0;
  typedef uint16_t u16_any __attribute__((aligned(1)));
  return (uint32_t)*reinterpret_cast<const u16_any *>(kb + (at >> 3)) >> (at & 7u);
}
// -inf where bit e of the hidden keys' bits is set, else v
__device__ __forceinline__ float hide(float v, uint32_t hidden, int e) {
  const uint32_t m = bit_mask(hidden, e);
  return __uint_as_float((m & 0xff800000u) | (~m & __float_as_uint(v)));
}
// s plus the E values of chunk c, without those of the keys held twice.  Only the
// slot of the row's last chunk has such keys (wave-uniform test); one chunk per
// lane of a lane group is that slot in every wave, and the test only costs (term,
// bf16 13 keys 515 -> 499 us, fp32 13 keys 221 -> 211; dropout backward, key mask,
// fp32 13 keys 309 -> 299).
template <int E, bool RAG, bool LAST>
__device__ __forceinline__ float add_chunk(float s, const float *v, int c, int sk) {
  if constexpr (RAG) {
    const int dup = dup_keys<E, RAG>(c, sk);
    // (lanes beyond the row hold nothing that counts)
    if (LAST || __builtin_amdgcn_ballot_w64(dup != 0) != 0) {
#pragma unroll
      for (int e = 0; e < E; ++e) s += e < dup ? 0.f : v[e];
      return s;
    }
  }
#pragma unroll
  for (int e = 0; e < E; ++e) s += v[e];
  return s;
}

// bytes of keep bits per lane group of a row: one for each chunk it can hold,
// one for the group that the row's first key shifts past them, one that is
// read but never used
constexpr int keep_bytes(int lanes, int vpl) { return lanes * vpl + 2; }

// DROP: dropout is applied to the probabilities before they are written
// (oslo/transformers/models/gpt2/modeling_gpt2.py:138-142,
// oslo/transformers/models/bert/modeling_bert.py:306-310) and the row
// statistics {max of the log2-domain logits, 1 / sum} go to stats[row], from
// which the backward pass recomputes the probabilities.  A row without a
// visible key stores {0, -1 / sk}.
//
// LPR lanes hold a row: 64 (a row takes whole waves), or 8 / 16 / 32 for rows
// of at most LPR * VPL chunks, where a wave works on 64 / LPR rows side by side
// (then wpr == 1 and VPL is 1 to 3).
template <typename T, int VPL, int RPW, int MODE, bool DROP, int LPR = kWave,
          bool RAG = false>
__global__ __launch_bounds__(1024) void softmax_fwd_kernel(
    const T *__restrict__ x, const uint8_t *__restrict__ mask,
    T *__restrict__ y, float *__restrict__ stats, SoftmaxGeom g, float scale,
    DropArgs d) {
  d = resolve_drop(d);
  constexpr int E = io<T>::EPV;
  constexpr uint32_t kAll = (1u << E) - 1u;
  static_assert(!RAG || RPW == 1, "ragged rows: one row set per wave");
  __shared__ float red[2][16];
  extern __shared__ uint8_t kbs[];  // ragged rows with dropout: the rows' keep bits
  const int lane = threadIdx.x & 63;
  // the wave index is uniform: keep it (and the row arithmetic) in scalar registers
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rslot = g.wpr == 1 ? wave : wave / g.wpr;  // (uniform: the division is skipped)
  const int first = rslot * g.wpr;
  const int nchunks = RAG ? (g.sk + E - 1) / E : g.sk / E;
  const int cstride = LPR == kWave ? kWave * g.wpr : LPR;
  constexpr int SUB = kWave / LPR;  // rows side by side in a wave
  const int sl = LPR == kWave ? lane : (lane & (LPR - 1));
  const int c0 = (wave - first) * kWave + sl;
  const float ninf = -__builtin_inff();

  // first row of this lane: the wave's first row plus the lane group's index
  const int64_t rbase =
      (work_block<RAG>(g) * g.rpb + rslot) * (RPW * SUB) +
      (LPR == kWave ? 0 : lane / LPR);

  float v[RPW][VPL][E];
  uint32_t mbits[RPW][VPL];  // bit e set: key masked out
  int64_t row[RPW];
  bool rvalid[RPW];
  // additive term: a query that the diagonal leaves without any key (sq > sk)
  // gets zeros (its neighbours in the wave may well see keys, so the
  // wave-uniform shortcuts below do not catch it)
  bool nokey[RPW];
  int vis[RPW];  // keys below the diagonal
  const uint8_t *mrows[RPW];
  bool shared[RPW];  // the row's mask bits are those of the wave's first row
  MaskChunk<E, RAG> mraw[MODE == kModeMasked ? RPW : 1][MODE == kModeMasked ? VPL : 1];
  // additive term (kModeBias): the chunks as loaded, and whether a chunk's
  // logits were left unread
  constexpr bool kBias = MODE == kModeBias;
  u32x4 braw[kBias ? RPW : 1][kBias ? VPL : 1][kBias ? E / 4 : 1];
  RawChunk<T, E> xraw[RPW][VPL];
  bool bhid[kBias ? RPW : 1][kBias ? VPL : 1];
  const bool bias_f32 = g.bias_esize == 4;

#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const int64_t r = rbase + j * SUB;
    rvalid[j] = r < g.rows;
    vis[j] = 0;
    mrows[j] = nullptr;
    row[j] = 0;
    if (rvalid[j]) row_setup<MODE>(g, r, mask, row[j], vis[j], mrows[j]);
    nokey[j] = MODE == kModeBias && rvalid[j] && vis[j] <= 0;
    // consecutive rows of a wave normally share their mask row (a key-padding
    // mask [b, 1, 1, sk]): its bits are then read and unpacked once
    shared[j] = false;
    if constexpr (MODE == kModeMasked && RPW > 1)
      shared[j] = j > 0 && rvalid[j] && rvalid[0] && mrows[j] == mrows[0] && !g.causal;
    if constexpr (MODE == kModeMasked) {
      // (chunks beyond the diagonal do not read their mask bytes)
#pragma unroll
      for (int k = 0; k < VPL; ++k) {
        const int c = c0 + k * cstride;
        const int i0 = chunk_key<E, RAG>(c, g.sk);
        if (!shared[j] && rvalid[j] && c < nchunks && i0 < vis[j]) mraw[j][k].load(mrows[j] + i0);
      }
    }
  }
  if constexpr (MODE == kModeMasked) wait_loads();
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int c = c0 + k * cstride;
      const int i0 = chunk_key<E, RAG>(c, g.sk);
      uint32_t mb = kAll;
      if (rvalid[j] && c < nchunks) {
        mb = beyond_bits<E>(i0, vis[j]);  // (vis == sk without a diagonal)
        if constexpr (MODE == kModeMasked)
          if (mb != kAll) mb |= shared[j] ? mbits[0][k] : mraw[j][k].bits();
      }
      mbits[j][k] = mb;
      if constexpr (MODE == kModeBias) {
        // the additive term of every chunk that has a key below the diagonal
        // (cached loads: its rows are normally shared by many rows of logits)
        bhid[j][k] = false;
        if (mb != kAll) load_bias_raw<T, E, RAG>(mrows[j], i0, bias_f32, braw[j][k]);
      }
    }
  }
  if constexpr (MODE == kModeBias) {
    // a chunk whose terms all absorb their logits takes the terms as its
    // sums: the logits are not read
    if (g.bias_skip) {
      wait_loads();
#pragma unroll
      for (int j = 0; j < RPW; ++j)
#pragma unroll
        for (int k = 0; k < VPL; ++k)
          if (mbits[j][k] != kAll) {
            float bf[E];
            unpack_bias_raw<T, E>(braw[j][k], bias_f32, bf);
            bhid[j][k] = bias_all_hidden<E>(bf);
          }
    }
  }
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const T *xr = x + row[j] * g.sk;
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int c = c0 + k * cstride;
      // (a chunk without a visible key is not loaded; its registers are never
      //  used: every select below takes the masked branch for it)
      bool want = mbits[j][k] != kAll;
      if constexpr (MODE == kModeBias) want = want && !bhid[j][k];
      if (want) xraw[j][k].template load<RAG>(xr + chunk_key<E, RAG>(c, g.sk));
    }
  }
  // (the draws of a ragged row wait in LDS while its loads are in flight)
  uint8_t *kb = nullptr;
  if constexpr (RAG && DROP) {
    kb = kbs + (LPR == kWave ? rslot : wave * SUB + lane / LPR) *
                   keep_bytes(LPR == kWave ? kWave * g.wpr : LPR, VPL);
    if (rvalid[0]) draw_row_groups<E>(kb, row[0], g.sk, vis[0], c0, cstride, d);
  }
  if constexpr (VPL * RPW > 1) wait_loads();

  // Wave-uniform shortcuts: where no lane of the wave sees a key of chunk
  // slot (j, k) the arithmetic is skipped altogether; where every lane sees
  // all its keys the per-element mask selects are skipped.  The logits are
  // kept in the log2 domain, t = x * (scale * log2 e), so exp is one exp2.
  bool none_visible[RPW][VPL], all_visible[RPW][VPL];
  // additive term: no lane of the wave read the logits of the slot (every
  // chunk of it lies beyond the diagonal or under terms that absorb it)
  bool slot_unread[kBias ? RPW : 1][kBias ? VPL : 1];
#pragma unroll
  for (int j = 0; j < RPW; ++j)
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      none_visible[j][k] = __builtin_amdgcn_ballot_w64(mbits[j][k] != kAll) == 0;
      all_visible[j][k] = __builtin_amdgcn_ballot_w64(mbits[j][k] != 0u) == 0;
      if constexpr (kBias)
        slot_unread[j][k] =
            __builtin_amdgcn_ballot_w64(mbits[j][k] != kAll && !bhid[j][k]) == 0;
    }
  const float c2 = scale * kLog2e;

  float mx[RPW];
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    float m = ninf;
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      if (none_visible[j][k]) continue;
      // (the values of a slot are formed first and the hidden ones replaced in a
      //  wave-uniform branch of its own: with the arithmetic in both branches the
      //  compiler evaluates it twice)
      xraw[j][k].unpack(v[j][k]);
      if constexpr (MODE == kModeBias) {
        // the sum scale * x + term as one fused multiply-add, kept in the
        // natural domain: a large negative term (-10000) then costs the logit
        // one rounding, as in a float evaluation of the unfused chain
        // (the terms are converted here, a slot at a time: kept converted next to
        //  the logits they cost a wave per SIMD)
        float bf[E];
        unpack_bias_raw<T, E>(braw[j][k], bias_f32, bf);
        if constexpr (RAG) {
          // (an absorbing term is the sum, whether or not the chunk was read)
          if (g.bias_skip) {
#pragma unroll
            for (int e = 0; e < E; ++e) v[j][k][e] = bf[e] <= kBiasHidden ? 0.f : v[j][k][e];
          }
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const float t = __builtin_fmaf(v[j][k][e], scale, bf[e]);
          v[j][k][e] = bhid[j][k] ? bf[e] : t;  // (a slot that was left unread)
        }
      } else {
        // (rounded product, never fused into the later subtraction: the
        //  backward pass of the dropout variant recomputes it bit for bit)
#pragma unroll
        for (int e = 0; e < E; ++e) v[j][k][e] = mul_rn(v[j][k][e], c2);
      }
      if (!all_visible[j][k]) {
#pragma unroll
        for (int e = 0; e < E; ++e) v[j][k][e] = hide(v[j][k][e], mbits[j][k], e);
      }
#pragma unroll
      for (int e = 0; e < E; ++e) m = fmaxf(m, v[j][k][e]);
    }
    mx[j] = m;
  }
  if constexpr (RPW == 4 && LPR < kWave) {
    group_allreduce4<OpMax, LPR>(mx);
  } else {
#pragma unroll
    for (int j = 0; j < RPW; ++j)
      mx[j] = row_reduce_max<LPR>(mx[j], red[0], wave, first, g.wpr, lane);
  }
  // (one barrier separates the two LDS areas; RPW > 1 implies wpr == 1,
  //  where LDS is not used at all)

  float sm[RPW];
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    float s = 0.f;
    // (with an additive term a row of -inf sums is NaN, as torch.softmax
    //  returns it: the maximum is subtracted as it is)
    const float off = (mx[j] == ninf && !kBias) || nokey[j] ? 0.f : mx[j];
    // (additive term: a slot whose logits were all left unread holds exact
    //  zeros as soon as every row of the wave has another key: no exponentials)
    if constexpr (kBias) {
      const bool hidden_are_zero = __builtin_amdgcn_ballot_w64(!(mx[j] > kBiasHidden)) == 0;
      // (such a slot is written as zeros below, like one that no lane sees:
      //  its registers are not touched again)
#pragma unroll
      for (int k = 0; k < VPL; ++k)
        if (slot_unread[j][k] && hidden_are_zero) none_visible[j][k] = true;
    }
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      if (none_visible[j][k]) continue;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        float d = sub_rn(v[j][k][e], off);
        if constexpr (kBias) d = mul_rn(d, kLog2e);
        v[j][k][e] = __builtin_amdgcn_exp2f(d);  // exp2(-inf) == 0 for masked keys
      }
      s = add_chunk<E, RAG, VPL == 1 && LPR < kWave>(s, v[j][k], c0 + k * cstride, g.sk);
    }
    sm[j] = s;
  }
  if constexpr (RPW == 4 && LPR < kWave) {
    group_allreduce4<OpSum, LPR>(sm);
  } else {
#pragma unroll
    for (int j = 0; j < RPW; ++j)
      sm[j] = row_reduce_sum<LPR>(sm[j], red[1], wave, first, g.wpr, lane);
  }
  if constexpr (RAG && DROP) {
    // a row without a visible key is uniform: all of it is drawn
    if (rvalid[0] && mx[0] == ninf && !kBias)
      draw_row_groups<E>(kb, row[0], g.sk, g.sk, c0, cstride, d);
    row_draws_done(g.wpr);
  }

#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    if (!rvalid[j]) continue;
    // a row without any visible key: uniform distribution, as softmax of a
    // constant fill value gives
    const bool empty = mx[j] == ninf && !kBias;
    float inv = empty || nokey[j] ? 0.f : row_recip(sm[j]);
    float fill = empty ? g.inv_sk : 0.f;
    T *yr = y + row[j] * g.sk;
    // (uniform over the wave: one of its rows is NaN)
    const bool nan_row = __builtin_amdgcn_ballot_w64(sm[j] != sm[j]) != 0;
    if constexpr (DROP) {
      if (c0 == 0) {
        stats[2 * row[j]] = empty || nokey[j] ? 0.f : mx[j];
        stats[2 * row[j] + 1] = empty ? -fill : inv;
      }
      // (the factor of the kept probabilities, once a row)
      inv *= d.scale;
      fill *= d.scale;
    }
    // A 4-element chunk is half a dropout group, and the lanes 2i and 2i + 1
    // hold the two halves: instead of evaluating every group twice, the even
    // lane draws the pair's group of chunk slot 2m, the odd lane that of slot
    // 2m + 1, and one DPP swap hands each lane the other's result.  (Rows of a
    // multiple of 8 keys, so that groups do not straddle rows; the row and the
    // conditions below are uniform over the wave, so all lanes are active.)
    constexpr bool kPairDraw = DROP && !RAG && E == 4 && LPR == kWave && VPL % 2 == 0;
    uint32_t keepk[kPairDraw ? VPL : 1];
    bool paired = false;
    if constexpr (kPairDraw) {
      if ((g.sk & 7) == 0) {
        paired = true;
        const int odd = lane & 1;
#pragma unroll
        for (int m = 0; m < VPL / 2; ++m) {
          keepk[2 * m] = keepk[2 * m + 1] = 0u;
          if (none_visible[j][2 * m] && none_visible[j][2 * m + 1] && !empty) continue;
          const int cpair = (c0 - odd) + (2 * m + odd) * cstride;  // the pair's even chunk
          const uint64_t flat = (uint64_t)row[j] * (uint64_t)g.sk + (uint64_t)cpair * E;
          const uint32_t bits = dropout_keep_bits(flat >> 3, d.seed, d.offset, d.threshold);
          const uint32_t other = (uint32_t)__builtin_amdgcn_update_dpp(
              0, (int)bits, kDppQuadSwap1, 0xF, 0xF, false);
          const uint32_t mine = (bits >> (4 * odd)) & 0xFu;     // slot 2m + odd
          const uint32_t theirs = (other >> (4 * odd)) & 0xFu;  // the other slot
          keepk[2 * m] = odd ? theirs : mine;
          keepk[2 * m + 1] = odd ? mine : theirs;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int c = c0 + k * cstride;
      if (c < nchunks) {
        float o[E];
        // (one store for both sides: two that follow each other are merged by the
        //  compiler without their non-temporal hint, fp32 [.., 40, 40] with a key
        //  mask 102 -> 106 us)
        // (wave-uniform; exact zeros need no draw)
        const bool blank = none_visible[j][k] && !(DROP && empty);
        if (blank) {
#pragma unroll
          for (int e = 0; e < E; ++e) o[e] = fill;
        } else {
          if constexpr (DROP) {
            if (none_visible[j][k]) {  // a row without a visible key: uniform, drawn
#pragma unroll
              for (int e = 0; e < E; ++e) v[j][k][e] = 0.f;
            }
          }
#pragma unroll
          for (int e = 0; e < E; ++e) o[e] = one_rounding<T, RAG && !DROP>(v[j][k][e] * inv + fill);
          if constexpr (RAG) {
            // (with dropout the keep bits of hidden keys are off; a key under an
            //  absorbing term is what a slot that was left unread takes it for)
            if (nan_row && (!DROP || kBias)) {
              const bool skipped = kBias && g.bias_skip;
              const uint32_t hid = sm[j] != sm[j] ? mbits[j][k] : 0u;
#pragma unroll
              for (int e = 0; e < E; ++e)
                o[e] = skipped && v[j][k][e] == 0.f ? 0.f : keep_or_zero(o[e], ~hid, e);
            }
          }
          // (the float value as it is: with a zero fill the product could
          //  otherwise be fused into the conversion to float16 in one build
          //  of the kernel and not in another, which differs on ties)
          if constexpr (kBias) {
#pragma unroll
            for (int e = 0; e < E; ++e) o[e] = pinned(o[e]);
          }
          if constexpr (DROP) {
            if constexpr (kPairDraw || RAG) {
              uint32_t keep;
              if constexpr (RAG)
                keep = row_keep_bits(kb, row[j], g.sk, chunk_key<E, RAG>(c, g.sk)) &
                       ~(empty ? 0u : mbits[j][k]);
              else
                keep = paired ? keepk[k] : chunk_keep_bits<E>(row[j], g.sk, c, d);
#pragma unroll
              for (int e = 0; e < E; ++e) o[e] = keep_or_zero(o[e], keep, e);
            } else {
              const KeepWords<E> keep = chunk_keep_words<E>(row[j], g.sk, c, d);
#pragma unroll
              for (int e = 0; e < E; ++e) o[e] = keep.kept(e) ? o[e] : 0.f;
            }
          }
        }
        store_chunk<T, E, RAG>(yr + chunk_key<E, RAG>(c, g.sk), o);
      }
    }
  }
}

// Backward of softmax + dropout from the saved logits: the probabilities are
// recomputed as exp2(x * scale * log2 e - stats[row][0]) * stats[row][1], the
// keep bits are regenerated from (seed, offset), and
// dx = scale * y * (dp - sum_k dp_k y_k) with dp = keep * dy / (1 - p).
template <typename T, int VPL, int RPW, int MODE, int LPR = kWave, bool RAG = false>
__global__ __launch_bounds__(1024) void softmax_dropout_bwd_kernel(
    const T *__restrict__ dy, const T *__restrict__ x,
    const float *__restrict__ stats, const uint8_t *__restrict__ mask,
    T *__restrict__ dx, SoftmaxGeom g, float scale, DropArgs d) {
  d = resolve_drop(d);
  constexpr int E = io<T>::EPV;
  constexpr uint32_t kAll = (1u << E) - 1u;
  static_assert(!RAG || RPW == 1, "ragged rows: one row set per wave");
  __shared__ float red[16];
  extern __shared__ uint8_t kbs[];  // ragged rows: the rows' keep bits
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rslot = g.wpr == 1 ? wave : wave / g.wpr;  // (uniform: the division is skipped)
  const int first = rslot * g.wpr;
  const int nchunks = RAG ? (g.sk + E - 1) / E : g.sk / E;
  const int cstride = LPR == kWave ? kWave * g.wpr : LPR;
  constexpr int SUB = kWave / LPR;
  const int sl = LPR == kWave ? lane : (lane & (LPR - 1));
  const int c0 = (wave - first) * kWave + sl;
  const int64_t rbase = (work_block<RAG>(g) * g.rpb + rslot) * (RPW * SUB) +
                        (LPR == kWave ? 0 : lane / LPR);
  const float c2 = scale * kLog2e;

  float yv[RPW][VPL][E], gv[RPW][VPL][E];
  uint32_t mbits[RPW][VPL];  // bit e set: key masked out
  int64_t row[RPW];
  bool rvalid[RPW];
  float rmax[RPW], rinv[RPW];
  int vis[RPW];  // keys that count below the diagonal
  const uint8_t *mrows[RPW];
  MaskChunk<E, RAG> mraw[MODE == kModeMasked ? RPW : 1][MODE == kModeMasked ? VPL : 1];
  RawChunk<T, E> xraw[RPW][VPL], graw[RPW][VPL];
  constexpr bool kBias = MODE == kModeBias;
  u32x4 braw[kBias ? RPW : 1][kBias ? VPL : 1][kBias ? E / 4 : 1];
  const bool bias_f32 = g.bias_esize == 4;

#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const int64_t r = rbase + j * SUB;
    rvalid[j] = r < g.rows;
    vis[j] = 0;
    mrows[j] = nullptr;
    row[j] = 0;
    rmax[j] = 0.f;
    rinv[j] = 0.f;
    if (rvalid[j]) {
      row_setup<MODE>(g, r, mask, row[j], vis[j], mrows[j]);
      rmax[j] = stats[2 * row[j]];
      rinv[j] = stats[2 * row[j] + 1];
    }
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int c = c0 + k * cstride;
      const int i0 = chunk_key<E, RAG>(c, g.sk);
      const bool want = rvalid[j] && c < nchunks && i0 < vis[j];
      if constexpr (MODE == kModeMasked) {
        if (want) mraw[j][k].load(mrows[j] + i0);
      }
      if constexpr (kBias) {
        if (want) load_bias_raw<T, E, RAG>(mrows[j], i0, bias_f32, braw[j][k]);
      }
    }
  }
  if constexpr (MODE == kModeMasked) wait_loads();
  if constexpr (kBias)
    if (g.bias_skip) wait_loads();
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    // uniform row: every key counts (with an additive term there is no such
    // convention: the probabilities are what the arithmetic gives)
    const bool empty = rinv[j] < 0.f && !kBias;
    if (empty) vis[j] = g.sk;
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int c = c0 + k * cstride;
      const int i0 = chunk_key<E, RAG>(c, g.sk);
      uint32_t mb = kAll;
      if (rvalid[j] && c < nchunks) {
        mb = beyond_bits<E>(i0, vis[j]);
        if constexpr (MODE == kModeMasked)
          if (mb != kAll && !empty) mb |= mraw[j][k].bits();
      }
      if constexpr (kBias) {
        // A chunk whose terms all absorb their logits has probability 0
        // throughout, unless the row's maximum is such a term itself (a
        // row without any other key): skip it altogether
        if (g.bias_skip && mb != kAll) {
          float bf[E];
          unpack_bias_raw<T, E>(braw[j][k], bias_f32, bf);
          if (rmax[j] > kBiasHidden && bias_all_hidden<E>(bf)) mb = kAll;
          if constexpr (RAG) {
            if (rmax[j] > kBiasHidden && shares_keys<E>(c, g.sk)) {
#pragma unroll
              for (int e = 0; e < E; ++e) mb |= bf[e] <= kBiasHidden ? 1u << e : 0u;
            }
          }
        }
      }
      mbits[j][k] = mb;
    }
  }
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const T *xr = x + row[j] * g.sk;
    const T *gr = dy + row[j] * g.sk;
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int i0 = chunk_key<E, RAG>(c0 + k * cstride, g.sk);
      // (a chunk without a visible key is not loaded: its gradients are zeros
      //  whatever the draw says, its logits are never used)
      graw[j][k].zero();
      if (mbits[j][k] != kAll) {
        xraw[j][k].template load<RAG>(xr + i0);
        graw[j][k].template load<RAG>(gr + i0);
      }
    }
  }
  // (the draws of a ragged row are made while its loads are in flight)
  uint8_t *kb = nullptr;
  if constexpr (RAG) {
    kb = kbs + (LPR == kWave ? rslot : wave * SUB + lane / LPR) *
                   keep_bytes(LPR == kWave ? kWave * g.wpr : LPR, VPL);
    if (rvalid[0]) draw_row_groups<E>(kb, row[0], g.sk, vis[0], c0, cstride, d);
    row_draws_done(g.wpr);
  }
  if constexpr (VPL * RPW > 1) wait_loads();
  bool none_loaded[RPW][VPL];
#pragma unroll
  for (int j = 0; j < RPW; ++j)
#pragma unroll
    for (int k = 0; k < VPL; ++k)
      none_loaded[j][k] = __builtin_amdgcn_ballot_w64(mbits[j][k] != kAll) == 0;

  float s[RPW];
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    float a = 0.f;
    const bool empty = rinv[j] < 0.f && !kBias;
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      if (none_loaded[j][k]) continue;
      const int c = c0 + k * cstride;
      KeepWords<E> keep;
      uint32_t keep_bits = 0;
      if constexpr (RAG) {
        // (hidden keys take their gradient for zero)
        keep_bits = row_keep_bits(kb, row[j], g.sk, chunk_key<E, RAG>(c, g.sk)) & ~mbits[j][k];
      } else {
        keep = chunk_keep_words<E>(row[j], g.sk, c, d);
      }
      float bf[kBias ? E : 1];
      float pd[E];
      if constexpr (kBias) unpack_bias_raw<T, E>(braw[j][k], bias_f32, bf);
      xraw[j][k].unpack(yv[j][k]);
      graw[j][k].unpack(gv[j][k]);
      // (the selects below stay per element: a wave-uniform branch around
      //  them for slots in which every lane sees all its keys measured 12 %
      //  slower at [256, 2048, 2048], 690 -> 772 us)
#pragma unroll
      for (int e = 0; e < E; ++e) {
        // the product is rounded before the subtraction, exactly as the
        // forward pass formed its exponent (no fused multiply-add here)
        float p;
        if constexpr (kBias) {
          // (the forward pass takes a term that absorbs its logit for the sum
          //  without reading the logit; the fused multiply-add returns that
          //  same term)
          const float u = __builtin_fmaf(yv[j][k][e], scale, bf[e]);
          p = __builtin_amdgcn_exp2f(mul_rn(sub_rn(u, rmax[j]), kLog2e)) * rinv[j];
        } else {
          p = __builtin_amdgcn_exp2f(sub_rn(mul_rn(yv[j][k][e], c2), rmax[j])) * rinv[j];
        }
        if (empty) p = -rinv[j];
        p = keep_or_zero(p, ~mbits[j][k], e);
        float dp;
        if constexpr (RAG)
          dp = keep_or_zero(mul_rn(gv[j][k][e], d.scale), keep_bits, e);
        else
          dp = keep.kept(e) ? mul_rn(gv[j][k][e], d.scale) : 0.f;
        yv[j][k][e] = p;
        gv[j][k][e] = dp;
        if constexpr (RAG)
          pd[e] = p * dp;
        else
          a += p * dp;
      }
      if constexpr (RAG) a = add_chunk<E, RAG, VPL == 1 && LPR < kWave>(a, pd, c, g.sk);
    }
    s[j] = a;
  }
#pragma unroll
  for (int j = 0; j < RPW; ++j)
    s[j] = row_reduce_sum<LPR>(s[j], red, wave, first, g.wpr, lane);

#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    if (!rvalid[j]) continue;
    T *dxr = dx + row[j] * g.sk;
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int c = c0 + k * cstride;
      if (c < nchunks) {
        float o[E];
        if (none_loaded[j][k]) {
#pragma unroll
          for (int e = 0; e < E; ++e) o[e] = RAG ? hidden_grad(scale, s[j]) : 0.f;
        } else {
#pragma unroll
          for (int e = 0; e < E; ++e)
            o[e] = one_rounding<T, RAG>(scale * (yv[j][k][e] * (gv[j][k][e] - s[j])));
        }
        store_chunk<T, E, RAG>(dxr + chunk_key<E, RAG>(c, g.sk), o);
      }
    }
  }
}

template <typename T, int VPL, int RPW, int MODE, int LPR = kWave, bool RAG = false>
__global__ __launch_bounds__(1024) void softmax_bwd_kernel(
    const T *__restrict__ dy, const T *__restrict__ y,
    const uint8_t *__restrict__ mask, T *__restrict__ dx, SoftmaxGeom g,
    float scale) {
  constexpr int E = io<T>::EPV;
  constexpr uint32_t kAll = (1u << E) - 1u;
  __shared__ float red[2][16];
  const int lane = threadIdx.x & 63;
  // the wave index is uniform: keep it (and the row arithmetic) in scalar registers
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rslot = g.wpr == 1 ? wave : wave / g.wpr;  // (uniform: the division is skipped)
  const int first = rslot * g.wpr;
  const int nchunks = RAG ? (g.sk + E - 1) / E : g.sk / E;
  const int cstride = LPR == kWave ? kWave * g.wpr : LPR;
  constexpr int SUB = kWave / LPR;
  const int sl = LPR == kWave ? lane : (lane & (LPR - 1));
  const int c0 = (wave - first) * kWave + sl;

  const int64_t rbase = (work_block<RAG>(g) * g.rpb + rslot) * (RPW * SUB) +
                        (LPR == kWave ? 0 : lane / LPR);

  float yv[RPW][VPL][E], gv[RPW][VPL][E];
  bool skip[RPW][VPL];
  int64_t row[RPW];
  bool rvalid[RPW];
  constexpr bool kBias = MODE == kModeBias;
  MaskChunk<E, RAG> mraw[MODE == kModeMasked ? VPL : 1];
  u32x4 braw[kBias ? VPL : 1][kBias ? E / 4 : 1];
  RawChunk<T, E> yraw[RPW][VPL], graw[RPW][VPL];
  constexpr bool kHides = RAG && MODE != kModeDense;
  uint32_t hid[kHides ? VPL : 1];  // hidden keys of the chunks that share keys

#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const int64_t r = rbase + j * SUB;
    rvalid[j] = r < g.rows;
    int visible = 0;
    const uint8_t *mrow = nullptr;
    row[j] = 0;
    if (rvalid[j]) row_setup<MODE>(g, r, mask, row[j], visible, mrow);
    float anyvis = 0.f;
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int c = c0 + k * cstride;
      const int i0 = chunk_key<E, RAG>(c, g.sk);
      const bool want = rvalid[j] && c < nchunks && (MODE == kModeDense || i0 < visible);
      skip[j][k] = !want;
      if constexpr (MODE == kModeMasked) {
        if (want) mraw[k].load(mrow + i0);
      }
      if constexpr (kBias) {
        if (want) load_bias_raw<T, E, RAG>(mrow, i0, g.bias_esize == 4, braw[k]);
      }
    }
    if constexpr (MODE == kModeMasked || kBias) wait_loads();
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int c = c0 + k * cstride;
      const bool shares = kHides && shares_keys<E>(c, g.sk);
      if constexpr (kHides) hid[k] = 0;
      if constexpr (MODE == kModeMasked) {
        const int i0 = chunk_key<E, RAG>(c, g.sk);
        if (!skip[j][k]) {
          const uint32_t bits = mraw[k].bits() | beyond_bits<E>(i0, visible);
          skip[j][k] = bits == kAll;
          if constexpr (kHides) hid[k] = shares && !skip[j][k] ? bits : 0u;
        }
      } else if constexpr (kHides) {
        if (shares && !skip[j][k]) hid[k] = beyond_bits<E>(chunk_key<E, RAG>(c, g.sk), visible);
      }
      if constexpr (kBias) {
        // every additive term of the chunk absorbs its logit: the
        // probabilities are zeros (unless the whole row is like that, which
        // the test below catches)
        if (!skip[j][k]) {
          float bf[E];
          unpack_bias_raw<T, E>(braw[k], g.bias_esize == 4, bf);
          skip[j][k] = bias_all_hidden<E>(bf);
          if (shares) {
#pragma unroll
            for (int e = 0; e < E; ++e) hid[kHides ? k : 0] |= bf[e] <= kBiasHidden ? 1u << e : 0u;
          }
          if (kHides && skip[j][k]) hid[kHides ? k : 0] = 0;
        }
      }
      if (!skip[j][k]) anyvis = 1.f;
    }
    if constexpr (MODE != kModeDense) {
      // a row with no visible key holds the uniform distribution: read it all
      if constexpr (MODE == kModeCausal) {
        anyvis = visible > 0 ? 1.f : 0.f;  // (known without a look at the row)
      } else {
        anyvis = row_reduce_max<LPR>(anyvis, red[0], wave, first, g.wpr, lane);
        if (g.wpr > 1) __syncthreads();
      }
      if (anyvis == 0.f) {
#pragma unroll
        for (int k = 0; k < VPL; ++k) {
          skip[j][k] = !(rvalid[j] && c0 + k * cstride < nchunks);
          if constexpr (kHides) hid[k] = 0;
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const T *yr = y + row[j] * g.sk;
    const T *gr = dy + row[j] * g.sk;
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int i0 = chunk_key<E, RAG>(c0 + k * cstride, g.sk);
      yraw[j][k].zero();
      graw[j][k].zero();
      if (!skip[j][k]) {
        yraw[j][k].template load<RAG>(yr + i0);
        graw[j][k].template load<RAG>(gr + i0);
      }
    }
  }
  if constexpr (VPL * RPW > 1) wait_loads();
  // wave-uniform: no lane of the wave loaded chunk slot (j, k) -> no arithmetic
  bool none_loaded[RPW][VPL];
#pragma unroll
  for (int j = 0; j < RPW; ++j)
#pragma unroll
    for (int k = 0; k < VPL; ++k)
      none_loaded[j][k] = __builtin_amdgcn_ballot_w64(!skip[j][k]) == 0;

  float s[RPW];
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    float a = 0.f;
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      if (none_loaded[j][k]) continue;
      yraw[j][k].unpack(yv[j][k]);
      graw[j][k].unpack(gv[j][k]);
      if constexpr (kHides) {
        if (__builtin_amdgcn_ballot_w64(hid[k] != 0u) != 0) {
#pragma unroll
          for (int e = 0; e < E; ++e) {
            yv[j][k][e] = keep_or_zero(yv[j][k][e], ~hid[k], e);
            gv[j][k][e] = keep_or_zero(gv[j][k][e], ~hid[k], e);
          }
        }
      }
      if constexpr (RAG) {
        float yg[E];
#pragma unroll
        for (int e = 0; e < E; ++e) yg[e] = yv[j][k][e] * gv[j][k][e];
        a = add_chunk<E, RAG, VPL == 1 && LPR < kWave>(a, yg, c0 + k * cstride, g.sk);
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e) a += yv[j][k][e] * gv[j][k][e];
      }
    }
    s[j] = a;
  }
#pragma unroll
  for (int j = 0; j < RPW; ++j)
    s[j] = row_reduce_sum<LPR>(s[j], red[1], wave, first, g.wpr, lane);

#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    if (!rvalid[j]) continue;
    T *dxr = dx + row[j] * g.sk;
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int c = c0 + k * cstride;
      if (c < nchunks) {
        float o[E];
        if (none_loaded[j][k]) {
#pragma unroll
          for (int e = 0; e < E; ++e) o[e] = RAG ? hidden_grad(scale, s[j]) : 0.f;
        } else {
#pragma unroll
          for (int e = 0; e < E; ++e)
            o[e] = one_rounding<T, RAG>(scale * (yv[j][k][e] * (gv[j][k][e] - s[j])));
        }
        store_chunk<T, E, RAG>(dxr + chunk_key<E, RAG>(c, g.sk), o);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// generic kernels: rows beyond sixteen waves; one 256-thread workgroup per row,
// three passes over the (L2-resident) row.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float block_reduce_256(float v, float *sh, bool is_max) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = is_max ? wave_max(v) : wave_sum(v);
  __syncthreads();
  if (lane == 0) sh[wave] = v;
  __syncthreads();
  return is_max ? fmaxf(fmaxf(sh[0], sh[1]), fmaxf(sh[2], sh[3]))
                : (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

template <typename T, int MODE, bool DROP>
__global__ __launch_bounds__(256) void softmax_fwd_generic_kernel(
    const T *__restrict__ x, const uint8_t *__restrict__ mask,
    T *__restrict__ y, float *__restrict__ stats, SoftmaxGeom g, float scale,
    DropArgs d) {
  d = resolve_drop(d);
  __shared__ float sh[4];
  const float ninf = -__builtin_inff();
  // log2-domain logits t = x * (scale * log2 e), the same rounded products
  // and differences as in the register kernel
  const float c2 = scale * kLog2e;
  for (int64_t r = blockIdx.x; r < g.rows; r += gridDim.x) {
    int64_t row;
    int visible;
    const uint8_t *mrow;
    row_setup<MODE>(g, r, mask, row, visible, mrow);
    const T *xr = x + row * g.sk;
    T *yr = y + row * g.sk;
    constexpr bool kBias = MODE == kModeBias;
    const bool bias_f32 = g.bias_esize == 4;
    auto is_hidden = [&](int i) {
      if constexpr (MODE == kModeMasked) return mrow[i] != 0 || i >= visible;
      return i >= visible;
    };
    // the logit of key i, and its exponent relative to the row maximum m
    auto logit = [&](int i) {
      if constexpr (kBias)
        return __builtin_fmaf(io<T>::from_scalar(xr[i]), scale, bias_at<T>(mrow, i, bias_f32));
      return mul_rn(io<T>::from_scalar(xr[i]), c2);
    };
    auto expo = [&](int i, float m) {
      const float d = sub_rn(logit(i), m);
      return kBias ? mul_rn(d, kLog2e) : d;
    };
    float m = ninf;
    for (int i = threadIdx.x; i < g.sk; i += 256)
      if (!is_hidden(i)) m = fmaxf(m, logit(i));
    m = block_reduce_256(m, sh, true);
    const bool empty = m == ninf && !kBias;
    float s = 0.f;
    for (int i = threadIdx.x; i < g.sk; i += 256)
      if (!is_hidden(i)) s += __builtin_amdgcn_exp2f(expo(i, m));
    s = block_reduce_256(s, sh, false);
    const float inv = empty ? 0.f : row_recip(s);
    const float fill = empty ? g.inv_sk : 0.f;
    const float factor = DROP ? inv * d.scale : inv, rest = DROP ? fill * d.scale : fill;
    for (int i = threadIdx.x; i < g.sk; i += 256) {
      float p = 0.f;
      if (!is_hidden(i)) p = __builtin_amdgcn_exp2f(expo(i, m));
      float o = p * factor + rest;
      // (a key beyond the diagonal is an exact zero in a NaN row, too)
      if (kBias && is_hidden(i)) o = 0.f;
      if constexpr (kBias) o = pinned(o);
      if constexpr (DROP)
        o = keep_element(row * g.sk + i, d) ? o : 0.f;
      yr[i] = io<T>::to_scalar(o);
    }
    if constexpr (DROP) {
      if (threadIdx.x == 0) {
        // (a query that the diagonal leaves without any key: zeros above, and
        //  finite statistics for the backward pass)
        const bool nokey = kBias && visible <= 0;
        stats[2 * row] = empty || nokey ? 0.f : m;
        stats[2 * row + 1] = empty ? -fill : (nokey ? 0.f : inv);
      }
    }
  }
}

template <typename T, int MODE>
__global__ __launch_bounds__(256) void softmax_dropout_bwd_generic_kernel(
    const T *__restrict__ dy, const T *__restrict__ x,
    const float *__restrict__ stats, const uint8_t *__restrict__ mask,
    T *__restrict__ dx, SoftmaxGeom g, float scale, DropArgs d) {
  d = resolve_drop(d);
  __shared__ float sh[4];
  const float c2 = scale * kLog2e;
  for (int64_t r = blockIdx.x; r < g.rows; r += gridDim.x) {
    int64_t row;
    int visible;
    const uint8_t *mrow;
    row_setup<MODE>(g, r, mask, row, visible, mrow);
    const T *xr = x + row * g.sk;
    const T *gr = dy + row * g.sk;
    T *dxr = dx + row * g.sk;
    const float m = stats[2 * row], inv = stats[2 * row + 1];
    constexpr bool kBias = MODE == kModeBias;
    const bool bias_f32 = g.bias_esize == 4;
    const bool empty = inv < 0.f && !kBias;
    auto prob = [&](int i) {
      if (empty) return -inv;
      bool hidden = i >= visible;
      if constexpr (MODE == kModeMasked) hidden = hidden || mrow[i] != 0;
      if (hidden) return 0.f;
      if constexpr (kBias) {
        const float u =
            __builtin_fmaf(io<T>::from_scalar(xr[i]), scale, bias_at<T>(mrow, i, bias_f32));
        return __builtin_amdgcn_exp2f(mul_rn(sub_rn(u, m), kLog2e)) * inv;
      }
      return __builtin_amdgcn_exp2f(
                 sub_rn(mul_rn(io<T>::from_scalar(xr[i]), c2), m)) *
             inv;
    };
    auto dprob = [&](int i) {
      return keep_element(row * g.sk + i, d)
                 ? mul_rn(io<T>::from_scalar(gr[i]), d.scale)
                 : 0.f;
    };
    float s = 0.f;
    for (int i = threadIdx.x; i < g.sk; i += 256) s += prob(i) * dprob(i);
    s = block_reduce_256(s, sh, false);
    for (int i = threadIdx.x; i < g.sk; i += 256)
      dxr[i] = io<T>::to_scalar(scale * (prob(i) * (dprob(i) - s)));
  }
}

template <typename T>
__global__ __launch_bounds__(256) void softmax_bwd_generic_kernel(
    const T *__restrict__ dy, const T *__restrict__ y, T *__restrict__ dx,
    int64_t rows, int sk, float scale) {
  __shared__ float sh[4];
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    const T *yr = y + r * sk;
    const T *gr = dy + r * sk;
    T *dxr = dx + r * sk;
    float s = 0.f;
    for (int i = threadIdx.x; i < sk; i += 256)
      s += io<T>::from_scalar(yr[i]) * io<T>::from_scalar(gr[i]);
    s = block_reduce_256(s, sh, false);
    for (int i = threadIdx.x; i < sk; i += 256) {
      const float yy = io<T>::from_scalar(yr[i]);
      dxr[i] = io<T>::to_scalar(scale * (yy * (io<T>::from_scalar(gr[i]) - s)));
    }
  }
}

// ---------------------------------------------------------------------------
// rows of fewer keys than a chunk (below 8 in a 16-bit type, below 4 in fp32):
// eight lanes hold a row, one key each.  The arithmetic is that of the kernels
// above, term for term.
// ---------------------------------------------------------------------------
constexpr int kTinyLanes = 8;
constexpr int kTinyRows = 256 / kTinyLanes;  // rows of a workgroup

template <typename T, int MODE, bool DROP>
__global__ __launch_bounds__(256) void softmax_fwd_tiny_kernel(
    const T *__restrict__ x, const uint8_t *__restrict__ mask,
    T *__restrict__ y, float *__restrict__ stats, SoftmaxGeom g, float scale,
    DropArgs d) {
  d = resolve_drop(d);
  const int i = threadIdx.x % kTinyLanes;  // key of this lane
  const float ninf = -__builtin_inff();
  constexpr bool kBias = MODE == kModeBias;
  for (int64_t r0 = (int64_t)blockIdx.x * kTinyRows; r0 < g.rows;
       r0 += (int64_t)gridDim.x * kTinyRows) {
    const int64_t r = r0 + threadIdx.x / kTinyLanes;
    int64_t row = 0;
    int visible = 0;
    const uint8_t *mrow = nullptr;
    if (r < g.rows) row_setup<MODE>(g, r, mask, row, visible, mrow);
    const bool in_row = r < g.rows && i < g.sk;
    bool hidden = !in_row || i >= visible;
    if constexpr (MODE == kModeMasked)
      if (!hidden) hidden = mrow[i] != 0;
    float v = ninf;
    if (!hidden) {
      const float t = io<T>::from_scalar(x[row * g.sk + i]);
      if constexpr (kBias)
        v = __builtin_fmaf(t, scale, bias_at<T>(mrow, i, g.bias_esize == 4));
      else
        v = mul_rn(t, scale * kLog2e);
    }
    const float m = group_allreduce<OpMax, kTinyLanes>(v);
    const bool empty = m == ninf && !kBias;
    float dd = sub_rn(v, empty ? 0.f : m);
    if constexpr (kBias) dd = mul_rn(dd, kLog2e);
    // (0 for hidden keys; a lane beyond the row counts nothing even where the
    //  row's maximum is -inf or NaN)
    const float p = in_row ? __builtin_amdgcn_exp2f(dd) : 0.f;
    const float s = group_allreduce<OpSum, kTinyLanes>(p);
    if (!in_row) continue;
    const float inv = empty ? 0.f : row_recip(s);
    const float fill = empty ? g.inv_sk : 0.f;
    float o = DROP ? p * (inv * d.scale) + fill * d.scale : p * inv + fill;
    // (a key beyond the diagonal is an exact zero in a NaN row, too)
    if (kBias && i >= visible) o = 0.f;
    if constexpr (kBias) o = pinned(o);
    if constexpr (DROP) o = keep_element(row * g.sk + i, d) ? o : 0.f;
    y[row * g.sk + i] = io<T>::to_scalar(o);
    if constexpr (DROP) {
      if (i == 0) {
        // (a query that the diagonal leaves without any key: zeros above, and
        //  finite statistics for the backward pass)
        const bool nokey = kBias && visible <= 0;
        stats[2 * row] = empty || nokey ? 0.f : m;
        stats[2 * row + 1] = empty ? -fill : (nokey ? 0.f : inv);
      }
    }
  }
}

template <typename T, int MODE>
__global__ __launch_bounds__(256) void softmax_dropout_bwd_tiny_kernel(
    const T *__restrict__ dy, const T *__restrict__ x,
    const float *__restrict__ stats, const uint8_t *__restrict__ mask,
    T *__restrict__ dx, SoftmaxGeom g, float scale, DropArgs d) {
  d = resolve_drop(d);
  const int i = threadIdx.x % kTinyLanes;
  constexpr bool kBias = MODE == kModeBias;
  for (int64_t r0 = (int64_t)blockIdx.x * kTinyRows; r0 < g.rows;
       r0 += (int64_t)gridDim.x * kTinyRows) {
    const int64_t r = r0 + threadIdx.x / kTinyLanes;
    int64_t row = 0;
    int visible = 0;
    const uint8_t *mrow = nullptr;
    if (r < g.rows) row_setup<MODE>(g, r, mask, row, visible, mrow);
    const bool in_row = r < g.rows && i < g.sk;
    float p = 0.f, dp = 0.f;
    if (in_row) {
      const float m = stats[2 * row], inv = stats[2 * row + 1];
      const bool empty = inv < 0.f && !kBias;
      bool hidden = i >= visible;
      if constexpr (MODE == kModeMasked)
        if (!hidden) hidden = mrow[i] != 0;
      if (empty) {
        p = -inv;
      } else if (!hidden) {
        const float t = io<T>::from_scalar(x[row * g.sk + i]);
        if constexpr (kBias) {
          const float u = __builtin_fmaf(t, scale, bias_at<T>(mrow, i, g.bias_esize == 4));
          p = __builtin_amdgcn_exp2f(mul_rn(sub_rn(u, m), kLog2e)) * inv;
        } else {
          p = __builtin_amdgcn_exp2f(sub_rn(mul_rn(t, scale * kLog2e), m)) * inv;
        }
      }
      // (a rounded product: fused into the subtraction below it would leave the
      //  product's rounding error where an exact zero belongs; keys beyond the
      //  diagonal contribute nothing)
      if ((empty || i < visible) && keep_element(row * g.sk + i, d))
        dp = mul_rn(io<T>::from_scalar(dy[row * g.sk + i]), d.scale);
    }
    const float s = group_allreduce<OpSum, kTinyLanes>(p * dp);
    if (in_row) dx[row * g.sk + i] = io<T>::to_scalar(scale * (p * (dp - s)));
  }
}

template <typename T>
__global__ __launch_bounds__(256) void softmax_bwd_tiny_kernel(
    const T *__restrict__ dy, const T *__restrict__ y, T *__restrict__ dx,
    int64_t rows, int sk, float scale) {
  const int i = threadIdx.x % kTinyLanes;
  for (int64_t r0 = (int64_t)blockIdx.x * kTinyRows; r0 < rows;
       r0 += (int64_t)gridDim.x * kTinyRows) {
    const int64_t row = r0 + threadIdx.x / kTinyLanes;
    const bool in_row = row < rows && i < sk;
    const float yv = in_row ? io<T>::from_scalar(y[row * sk + i]) : 0.f;
    const float gv = in_row ? io<T>::from_scalar(dy[row * sk + i]) : 0.f;
    const float s = group_allreduce<OpSum, kTinyLanes>(yv * gv);
    if (in_row) dx[row * sk + i] = io<T>::to_scalar(scale * (yv * (gv - s)));
  }
}

static inline dim3 tiny_grid(int64_t rows) {
  const int64_t want = ceil_div(rows, kTinyRows), cap = max_workgroups(256);
  return dim3((unsigned)(want < cap ? want : cap));
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct SoftmaxPlan {
  int vpl, rpw, wpr, rpb;
  int lpr;  // lanes that hold a row: 64, or 8 / 16 / 32 for short rows
  bool ok;
};

// Rows that do not fill two chunks per lane of 8, 16 or 32 lanes and take them
// all the same: the most chunks for each, the fewest altogether, and the row sets
// of a wave then.
struct TwoChunks {
  int most8, most16, most32, from, rpw;
};

// max_elems: elements of one operand a lane may hold (register budget).
static SoftmaxPlan plan_softmax(int64_t sk, int E, int max_elems,
                                int default_rpw, int one_chunk_rpw,
                                const TwoChunks *two = nullptr) {
  SoftmaxPlan p{0, 1, 1, 1, kWave, false};
  if (sk % E != 0) return p;
  const int64_t nchunks = sk / E;
  const int maxvpl = max_elems / E;  // 8 or 4 for 16-bit types, 16 or 8 for fp32
  int64_t wpr = ceil_div(nchunks, (int64_t)kWave * (maxvpl > 8 ? 8 : maxvpl));
  if (wpr > 16) return p;
  const int64_t need = ceil_div(nchunks, kWave * wpr);
  int vpl = need <= 1 ? 1 : need <= 2 ? 2 : need <= 4 ? 4 : 8;
  int rpw = 1;
  // short rows: several rows side by side in a wave instead of idle lanes
  if (nchunks <= 32 && g_tune.softmax_lanes_per_row != kWave) {
    p.lpr = nchunks <= 8 ? 8 : nchunks <= 16 ? 16 : 32;
    if (g_tune.softmax_lanes_per_row == 8 || g_tune.softmax_lanes_per_row == 16 ||
        g_tune.softmax_lanes_per_row == 32)
      if (g_tune.softmax_lanes_per_row >= p.lpr) p.lpr = g_tune.softmax_lanes_per_row;
  }
  // rows of exactly 3 x 8 / 16 / 32 / 64 chunks (192, 384, 768, 1536 16-bit
  // keys): three chunks per lane, no idle lane
  if (nchunks % 3 == 0 && g_tune.softmax_lanes_per_row != kWave && 3 * E <= max_elems) {
    const int64_t q = nchunks / 3;
    if (q == 8 || q == 16 || q == 32 || q == 64) {
      p.vpl = 3;
      p.rpw = 1;
      p.wpr = 1;
      p.rpb = g_tune.softmax_rows_per_block > 0 ? g_tune.softmax_rows_per_block : 4;
      p.lpr = (int)q;
      p.ok = true;
      return p;
    }
  }
  // forward: rows of exactly 2 x 8 / 16 / 32 chunks (128, 256, 512 16-bit
  // keys) as two chunks per lane in a lane group, and rows that leave nearly
  // half of the lanes without keys otherwise, or half of the second chunks then
  if (two != nullptr && g_tune.softmax_lanes_per_row != kWave &&
      g_tune.softmax_lanes_per_row != 1) {
    const int64_t q = nchunks <= 8 ? 0 : nchunks <= 16 ? 8 : nchunks <= 32 ? 16 : nchunks <= 64 ? 32 : 0;
    const bool part = g_tune.softmax_lanes_per_row == 0 && nchunks >= two->from &&
                      nchunks <= (q == 8 ? two->most8 : q == 16 ? two->most16 : two->most32);
    if (q != 0 && (nchunks == 2 * q || part)) {
      // one row set per wave without a mask tensor, two with one (measured)
      int want = g_tune.softmax_rows_per_wave > 0 ? g_tune.softmax_rows_per_wave
                                                  : (part ? two->rpw : default_rpw);
      p.vpl = 2;
      p.rpw = want >= 2 && 2 * 2 * E <= max_elems ? 2 : 1;
      p.wpr = 1;
      // (one wave per workgroup: 6 % faster at sequence length 128)
      p.rpb = g_tune.softmax_rows_per_block > 0 ? g_tune.softmax_rows_per_block : 1;
      p.lpr = (int)q;
      p.ok = true;
      return p;
    }
  }
  if (wpr == 1) {
    // row sets a wave handles at once; measured best on MI355X: one, or two
    // for the forward with a mask tensor (its loads wait for the mask bytes);
    // a forward that holds one chunk per lane (rows of up to 512 16-bit
    // keys) wants four, which hides its two dependent reductions
    int want = g_tune.softmax_rows_per_wave > 0
                   ? g_tune.softmax_rows_per_wave
                   : (vpl == 1 ? one_chunk_rpw : default_rpw);
    rpw = want >= 4 ? 4 : (want >= 2 ? 2 : 1);
    while (rpw > 1 && (rpw * vpl * E > max_elems || rpw * vpl > 8)) rpw >>= 1;
  }
  p.vpl = vpl;
  p.rpw = rpw;
  p.wpr = (int)wpr;
  // one row (set) per workgroup: workgroups of a single wave measure 3-6 %
  // faster on MI355X than four waves that each own a row (bf16 [256,2048,2048]
  // causal forward 570 -> 537 us, backward 744 -> 707 us)
  p.rpb = wpr == 1 || wpr >= 4 ? 1 : (int)(4 / wpr);
  if (g_tune.softmax_rows_per_block > 0) p.rpb = g_tune.softmax_rows_per_block;
  while (p.rpb * p.wpr > 16) --p.rpb;
  p.ok = true;
  return p;
}

// Ragged rows: at least one chunk, at most 64 bytes of an operand per lane and
// sixteen waves.  Rows of up to 96 chunks are held by 8, 16 or 32 lanes with one
// to three chunks each.  More chunks in fewer lanes share the reductions, the
// cut of the row's ends and, with dropout, the Philox rounds among more rows of a
// wave; against it stand the pieces that a row is read in, of 128, 256 or 512
// bytes at odd addresses (one line more per piece than aligned), and lanes
// without keys.  us at 300 MB: forward with dropout, plain forward, backward with
// dropout, under the diagonal unless said; first as the line below it would hold
// the rows (one chunk per lane, or what is named):
//   two of 8 lanes    bf16 67 keys 257, 167, 267 / 149, 120, 175; 95: 179, 123, 193
//                     / 126, 117, 172; 125, one chunk: 146, 100, 159 / 135, 142,
//                     176; fp32 33: 215, 144, 218 / 129, 116, 161; 47, one chunk:
//                     151, 108, 164 / 128, 126, 159; a term shared by the batch,
//                     bf16 79, one chunk: 228, 175, 262 / 237, 206, 300
//   two of 16 lanes   bf16 201 keys 172, 121, 184 / 107, 100, 136; 253: 140, 99, 153
//                     / 98, 97, 135; fp32 111: 131, 97, 142 / 102, 94, 129; 127, one
//                     chunk: 117, 90, 130 / 102, 101, 128, with a term 125: 133,
//                     103, 150 / 118, 114, 164; a term shared by the batch, bf16 223,
//                     one chunk: 11 % faster, 12 and 15 % slower than two
//   ... from three of 8, bf16 133 keys 162, 126, 184 / 135, 101, 153; fp32 79: 166,
//                     121, 161 / 103, 99, 137; but 16 bits, three of 8: key mask 157
//                     keys 160, 157, 206 / 179, 130, 202, term 133: 179, 159, 248 /
//                     213, 146, 253
//   three of 16       bf16 261 keys against two of 32: 108, 98, 137 / 131, 97, 148;
//                     fp32 131: 109, 96, 132 / 114, 90, 134; 171, two of 32: 97, 94,
//                     127 / 95, 86, 121; key mask 173: 111, 108, 146 / 119, 104, 140
//   two of 32         bf16 389 keys 167, 121, 176 / 109, 86, 125; 507: 130, 98, 143
//                     / 89, 84, 115; fp32 195: 154, 109, 146 / 89, 85, 117; 253:
//                     121, 91, 118 / 86, 84, 111
//   three of 32       bf16 517 keys against two of a wave: 90, 91, 120 / 128, 95, 140
// Plain and dropout forward of a row hold it alike, so that they add in one order.
// The plain backward has neither Philox rounds nor a row to cut twice, and takes
// two chunks only where one leaves nearly half of the lanes idle: bf16 133 keys
// 161 -> 140, 261: 161 -> 121, 341: 127 -> 118, but 181: 131 -> 140, 443: 110 -> 116
// (without a diagonal, whose rows need all their chunks, 129: 180 -> 193, 143: 175 ->
// 182, 341: 160 -> 165, but 317: 168 -> 162);
// fp32 67: 146 -> 139, 131: 146 -> 120, 171: 121 -> 116, but 189: 114 -> 116.
// Two rows (of waves or sets of lane groups) to a workgroup: the line that two
// rows share is then written through one L2 (bf16 1003 keys: causal backward
// 102 -> 88 us, dense 156 -> 130 us; four measure the same, and slower beyond
// 2048 keys).
enum RaggedPass { kRaggedFwd, kRaggedDropBwd, kRaggedBwd };
template <typename T, int MODE>
static SoftmaxPlan plan_softmax_ragged(int64_t sk, RaggedPass pass, bool shared_term = false) {
  constexpr int E = io<T>::EPV;
  constexpr bool k16 = sizeof(T) == 2;
  constexpr bool term = MODE == kModeBias, masked = MODE == kModeMasked;
  const bool fwd = pass == kRaggedFwd, plain = pass == kRaggedBwd;
  SoftmaxPlan p{0, 1, 1, 1, kWave, false};
  if (sk < E) return p;
  const int64_t nchunks = ceil_div(sk, E);
  const int64_t wpr = ceil_div(nchunks, kWave * 4);
  if (wpr > 16) return p;
  p.ok = true;
  p.wpr = (int)wpr;
  const auto group = [&](int chunks, int lanes) {
    p.vpl = chunks;
    p.lpr = lanes;
  };
  // (16-bit rows behind a mask or with a term: up to where three of 8 lanes
  //  remain the better)
  const bool shared = term && shared_term;
  // (16-bit plain backward of rows that are not cut off by a diagonal)
  constexpr bool whole16 = k16 && MODE == kModeDense;
  const int three8 = !k16 || plain ? 0 : fwd ? (term || masked ? 20 : 0) : (term ? 18 : 0);
  if (nchunks <= 8) {
    group(1, 8);
  } else if (nchunks <= (shared ? (k16 ? 9 : 8) : k16 ? 12 : 10) && !plain) {
    group(2, 8);
  } else if (nchunks <= 16) {
    group(1, 16);
  } else if (nchunks <= three8) {
    group(3, 8);
  } else if (nchunks <= (plain ? (whole16 ? 16 : 18) : shared ? 24 : k16 ? 32 : 28)) {
    group(2, 16);
  } else if (nchunks <= 32) {
    group(1, 32);
  } else if (nchunks <= (k16 || masked ? 48 : 40) && !plain) {
    group(3, 16);
  } else if (nchunks <= (plain ? (whole16 ? 42 : 44) : 64)) {
    group(2, 32);
  } else if (nchunks > 64 && nchunks <= 96 && !plain) {
    group(3, 32);
  } else {
    group((int)ceil_div(nchunks, kWave * wpr), kWave);
  }
  p.rpb = g_tune.softmax_rows_per_block > 0 ? g_tune.softmax_rows_per_block : 2;
  while (p.rpb * p.wpr > 16) --p.rpb;
  return p;
}
// The blocks of ragged rows that are dealt out by die (work_block): all groups of
// 64.  Not those of rows of whole waves that add a term shared by the batch: the
// blocks of the same rows of its entries are 16 apart there and meet on one die in
// launch order, whose L2 serves the term to all but the first (fp32 forward at
// 300 MB, by die / in launch order: 1111 keys 106 / 87 us, 1777: 183 / 148, bf16
// 1777: 130 / 118).  In lane groups the rows of one run fill two to four blocks and
// the die makes up for it (fp32 97 keys 147 / 158).
template <int MODE> static int64_t ragged_die_end(const SoftmaxGeom &g, const SoftmaxPlan &pl, int64_t nblocks) {
  return MODE == kModeBias && g.batch_inner && pl.lpr == kWave ? 0 : nblocks & ~(int64_t)63;
}

// ... and the builds that it can come out with
template <typename T, int MODE>
constexpr bool ragged_plan_reaches(int vpl, int lpr, RaggedPass pass) {
  constexpr bool k16 = sizeof(T) == 2, term = MODE == kModeBias, masked = MODE == kModeMasked;
  const bool plain = pass == kRaggedBwd;
  if (lpr == kWave) return vpl > 1 || plain;
  if (vpl == 3 && lpr == 8) return k16 && (term || (masked && pass == kRaggedFwd)) && !plain;
  if (vpl == 3) return !plain;
  if (vpl == 2) return !plain || (lpr != 8 && !(lpr == 16 && k16 && MODE == kModeDense));
  return lpr != 32 || plain || !k16 || term;
}
#define OSLO_SM_RAGGED_CASES(LAUNCH)       \
  if (pl.lpr == 8 && pl.vpl == 1) {        \
    LAUNCH(1, 8);                          \
  } else if (pl.lpr == 16 && pl.vpl == 1) { \
    LAUNCH(1, 16);                         \
  } else if (pl.lpr == 32 && pl.vpl == 1) { \
    LAUNCH(1, 32);                         \
  } else if (pl.lpr == 8 && pl.vpl == 2) { \
    LAUNCH(2, 8);                          \
  } else if (pl.lpr == 16 && pl.vpl == 2) { \
    LAUNCH(2, 16);                         \
  } else if (pl.lpr == 32 && pl.vpl == 2) { \
    LAUNCH(2, 32);                         \
  } else if (pl.lpr == 8) {                \
    LAUNCH(3, 8);                          \
  } else if (pl.lpr == 16) {               \
    LAUNCH(3, 16);                         \
  } else if (pl.lpr == 32) {               \
    LAUNCH(3, 32);                         \
  } else if (pl.vpl == 1) {                \
    LAUNCH(1, kWave);                      \
  } else if (pl.vpl == 2) {                \
    LAUNCH(2, kWave);                      \
  } else if (pl.vpl == 3) {                \
    LAUNCH(3, kWave);                      \
  } else {                                 \
    LAUNCH(4, kWave);                      \
  }
// LDS of a ragged launch with dropout: the keep bits of the workgroup's rows
static inline unsigned ragged_keep_lds(const SoftmaxPlan &pl) {
  const int lanes = pl.lpr == kWave ? kWave * pl.wpr : pl.lpr;
  return (unsigned)(pl.rpb * (kWave / pl.lpr) * keep_bytes(lanes, pl.vpl));
}

// Waves of a launch to keep on a CU, 0 for as many as fit.  A wave requests its
// whole row at once, so the waves on a CU decide how much of the operands is
// requested at a time, and the memory serves a launch fastest when that is some
// 64 KB per CU (forward) or 96 KB (backward): less leaves it idle, more widens
// the window of addresses that is open at once.  Measured at 1 GB tensors, waves
// that fit -> waves kept: bf16 causal 2048 keys forward 252 -> 241 us (16),
// backward 328 -> 307 (12); 1024 keys backward 318 -> 308 (24); fp32 1024 keys
// 253 -> 235 (14) and 338 -> 309 (12); [256, 2048, 2048] forward 547 -> 508,
// backward 694 -> 655.
// Launches that spend the time on arithmetic (dropout on 16-bit rows), on mask
// bytes, or on the barrier between the waves of a row want more waves: with
// dropout 160 KB in the backward (20 waves of 2048 keys: 317 us, 12: 343) and no
// limit in the 16-bit forward, causal with a key mask 160 KB (314 against 342 us),
// rows of several waves 160 and 96 KB (4096 keys backward 322 against 348 us),
// ragged rows, two to a workgroup, 128 KB.
// All of these are of rows that fill the lanes that hold them.  A wave with idle
// lanes requests less, so more of them are kept: 16 waves of rows that fill five
// lanes of eight, or half of them, is 20 to 30 % slower than no limit (additive
// term, fp32 80 keys forward 178 -> 142 us; causal fp16 8 keys 768 -> 627, 72 keys
// 198 -> 163, 288 keys 203 -> 165; key mask, fp32 608 keys backward 189 -> 172).
// So it is in the forward of ragged rows in lane groups, where a limit pays for
// groups that are nearly full: three chunks with dropout under the diagonal (20
// waves of full groups, 24 of 32 lanes in 16 bits: bf16 379 keys 108 -> 94 us, 765:
// 91 -> 87, fp32 383: 88 -> 82), two without it (24, of 8 lanes 18: bf16 95 keys
// 132 -> 117, 253: 99 -> 96, fp32 111: 99 -> 94; not behind a key mask, 95 keys 133
// -> 144).  Behind a key mask three chunks in 8 or 16 lanes take 24 to 28 waves
// (bf16 133 keys 160 -> 146, with dropout 167 -> 152; 305: 124 -> 111, fp32 173: 112
// -> 108), but not 16 lanes in 16 bits with dropout (373 keys: 111, with 24 waves
// 118), nor fp32 under the diagonal while a third of the chunks is empty (131 keys:
// 107, with 28 waves 108).  A term that the batch shares is served by the L2s if
// fewer rows are under way: 16 waves with dropout (bf16 133 keys 278 -> 249, 345: 191
// -> 179, fp32 153: 179 -> 156), in 16 bits of full groups of 16 lanes (261 keys: 194
// without a limit, 205 with 16, 186 with 23).
// Additive terms with several rows to a wave, which waits for both operands: 96 KB
// (bf16 392 keys 373 -> 327 us, fp16 352 keys 387 -> 362 at 900 MB), in fp32 lane
// groups 72 KB (140 keys 122 -> 114, 172: 114 -> 107).
template <typename T, int MODE>
static int softmax_waves_per_cu(const SoftmaxPlan &pl, int sk, bool backward, bool drop,
                                bool causal, bool ragged, bool shared_term = false) {
  constexpr bool k16 = sizeof(T) == 2;
  int kb;
  if (backward) {
    kb = MODE == kModeDense || MODE == kModeBias ? 112 : 96;
    if (ragged) kb = 128;
    if (drop) kb = k16 ? 160 : 112;
    if (pl.wpr > 1 || (MODE == kModeMasked && causal)) kb = 160;
  } else {
    kb = MODE == kModeMasked ? 112 : 64;
    if (MODE == kModeBias && pl.rpw > 1) kb = 96;
    if (MODE == kModeBias && !k16 && !drop && pl.rpw == 2 && pl.vpl == 2 && pl.lpr < kWave) return 18;
    if (drop) kb = 96;
    if (pl.wpr > 1 && kb < 96) kb = 96;
    if (ragged && pl.vpl == 3 && pl.lpr < kWave && drop && MODE == kModeCausal)
      return (int)((k16 && pl.lpr == 32 ? 24 : 20) * (int64_t)pl.vpl * pl.lpr /
                   ceil_div(sk, io<T>::EPV));
    if (ragged && pl.vpl == 3 && pl.lpr < 32) {
      const int nchunks = (int)ceil_div(sk, io<T>::EPV);
      if (MODE == kModeMasked && !k16 && causal && !drop && nchunks <= 38) return 0;
      if (MODE == kModeMasked && !drop) return k16 && !causal ? 24 : 28;
      if (MODE == kModeMasked && (!k16 || pl.lpr == 8)) return k16 && !causal ? 24 : 28;
      if (MODE == kModeBias && drop && shared_term)
        return k16 && pl.lpr == 16 ? 16 * 48 / nchunks : 16;
    }
    if (ragged && pl.vpl == 2 && pl.lpr < kWave && !drop && MODE != kModeMasked)
      return (int)((pl.lpr == 8 ? 18 : 24) * (int64_t)pl.vpl * pl.lpr / ceil_div(sk, io<T>::EPV));
    if (drop && k16) return 0;
  }
  int waves = kb / (pl.vpl * pl.rpw * (backward ? 2 : 1));  // (1 KB per chunk slot and operand)
  // forward rows that would leave room for more than 28 waves: 3-5 % faster
  // with 28, but for 16-bit causal rows of whole waves (1024 keys: 3 % slower)
  // and ragged rows (197 keys: 5 % slower)
  if (!backward && !drop && !ragged && waves > 28 &&
      !(MODE == kModeCausal && k16 && pl.lpr == kWave))
    waves = 28;
  if (ragged) return waves;  // (measured as they are)
  const int64_t slots = (int64_t)pl.vpl * (pl.lpr == kWave ? kWave * pl.wpr : pl.lpr);
  return (int)(waves * slots / ceil_div(sk, io<T>::EPV));
}

// LDS that a launch of `nblocks` workgroups reserves in order to keep at most
// `waves` of its waves on a CU.  (Not for workgroups of a third of the CU and
// more, and not for launches of a few rounds, whose tail would grow.)
static inline unsigned occupancy_lds(int waves, int threads, int64_t nblocks) {
  const bool asked = g_tune.softmax_waves_per_cu > 0;
  if (asked) waves = g_tune.softmax_waves_per_cu;
  const int blocks = waves * kWave / threads;
  if (waves <= 0 || waves >= 32 || blocks < 3) return 0;
  if (!asked && nblocks < (int64_t)device_cu_count() * blocks * 4) return 0;
  return (unsigned)(160 * 1024 / blocks - 512);
}

constexpr int kFwdMaxElems = 64;  // one operand resident
constexpr int kBwdMaxElems = 32;  // two operands resident

#define OSLO_SM_CASES_LPR(LAUNCH, LPR_)    \
  if (pl.rpw == 1) {                       \
    LAUNCH(1, 1, LPR_);                    \
  } else if (pl.rpw == 2) {                \
    LAUNCH(1, 2, LPR_);                    \
  } else {                                 \
    LAUNCH(1, 4, LPR_);                    \
  }
#define OSLO_SM_CASES(LAUNCH)              \
  if (pl.vpl == 3 && pl.lpr == 8) {        \
    LAUNCH(3, 1, 8);                       \
  } else if (pl.vpl == 3 && pl.lpr == 16) { \
    LAUNCH(3, 1, 16);                      \
  } else if (pl.vpl == 3 && pl.lpr == 32) { \
    LAUNCH(3, 1, 32);                      \
  } else if (pl.vpl == 3) {                \
    LAUNCH(3, 1, kWave);                   \
  } else if (pl.vpl == 2 && pl.lpr == 8 && pl.rpw == 1) {  \
    LAUNCH(2, 1, 8);                       \
  } else if (pl.vpl == 2 && pl.lpr == 8) { \
    LAUNCH(2, 2, 8);                       \
  } else if (pl.vpl == 2 && pl.lpr == 16 && pl.rpw == 1) { \
    LAUNCH(2, 1, 16);                      \
  } else if (pl.vpl == 2 && pl.lpr == 16) { \
    LAUNCH(2, 2, 16);                      \
  } else if (pl.vpl == 2 && pl.lpr == 32 && pl.rpw == 1) { \
    LAUNCH(2, 1, 32);                      \
  } else if (pl.vpl == 2 && pl.lpr == 32) { \
    LAUNCH(2, 2, 32);                      \
  } else if (pl.lpr == 8) {                \
    OSLO_SM_CASES_LPR(LAUNCH, 8)           \
  } else if (pl.lpr == 16) {               \
    OSLO_SM_CASES_LPR(LAUNCH, 16)          \
  } else if (pl.lpr == 32) {               \
    OSLO_SM_CASES_LPR(LAUNCH, 32)          \
  } else if (pl.vpl == 1 && pl.rpw == 1) { \
    LAUNCH(1, 1, kWave);                   \
  } else if (pl.vpl == 1 && pl.rpw == 2) { \
    LAUNCH(1, 2, kWave);                   \
  } else if (pl.vpl == 1 && pl.rpw == 4) { \
    LAUNCH(1, 4, kWave);                   \
  } else if (pl.vpl == 2 && pl.rpw == 1) { \
    LAUNCH(2, 1, kWave);                   \
  } else if (pl.vpl == 2 && pl.rpw == 2) { \
    LAUNCH(2, 2, kWave);                   \
  } else if (pl.vpl == 2 && pl.rpw == 4) { \
    LAUNCH(2, 4, kWave);                   \
  } else if (pl.vpl == 4 && pl.rpw == 1) { \
    LAUNCH(4, 1, kWave);                   \
  } else if (pl.vpl == 4 && pl.rpw == 2) { \
    LAUNCH(4, 2, kWave);                   \
  } else {                                 \
    LAUNCH(8, 1, kWave);                   \
  }

// The (chunks per lane, row sets per wave, lanes per row) triples that the
// plan of a backward pass can come out with: at most 32 resident elements of
// each operand per lane in a 16-bit type and 16 in fp32 (32 only for rows that
// need eight chunks per lane, which take one row set), and two chunks per lane
// in a lane group only in the forward pass.  Other triples are not built.
template <typename T>
constexpr bool bwd_plan_reaches(int vpl, int rpw, int lpr) {
  constexpr int E = io<T>::EPV;
  if (vpl == 2 && lpr < kWave) return false;
  if (sizeof(T) == 4) return vpl * rpw * E <= 16 || (vpl == 8 && rpw == 1);
  return vpl * rpw * E <= kBwdMaxElems;
}

// The register kernels read the additive term in 16-byte vectors: its base
// address and the byte offsets of its rows must be multiples of 16.
static inline bool bias_vec_ok(const SoftmaxGeom &g, const uint8_t *bias) {
  if (bias == nullptr) return true;
  const int64_t es = g.bias_esize;
  return aligned16(bias) && (g.bias_sb * es) % 16 == 0 && (g.bias_sh * es) % 16 == 0 &&
         (g.bias_sq * es) % 16 == 0;
}

// elements of one operand per lane the kernels with an additive term hold at
// most (the term's chunks stay resident next to the logits)
constexpr int kBiasMaxElems = 32;

// stats != nullptr selects the dropout variant (d is ignored otherwise).
template <typename T, int MODE>
int launch_softmax_fwd(const void *x, const uint8_t *mask, void *y,
                              float *stats, DropArgs d, SoftmaxGeom g,
                              float scale, hipStream_t st) {
  constexpr int E = io<T>::EPV;
  set_fast_div(g);
  const bool drop = stats != nullptr;
  // 64 bytes of the operand per lane (32 16-bit or 16 fp32 elements) measure
  // 10-25 % faster than twice that (rows of 4096 and more 16-bit keys then
  // take two or more waves); 64 elements only where a row would otherwise not
  // fit one workgroup
  const int cap = g_tune.softmax_fwd_elems > 0 ? g_tune.softmax_fwd_elems
                                               : (sizeof(T) == 4 ? 16 : 32);
  // (two row sets per wave where the loads of the logits wait for mask bytes;
  //  with an additive term one measures faster, 186 against 232 us at
  //  [16,16,1024,1024] fp16, whether or not the loads wait for the term)
  const int default_rpw = MODE == kModeMasked ? 2 : 1;
  // (two chunks per lane against one in twice the lanes, us at 300 MB, forward with
  //  dropout and plain forward.  16 bits, 72 keys: causal 167, 114 / 120, 109, key mask
  //  166, 117 / 121, 117, term 185, 136 / 161, 129, but 80: 134, 98 / 116, 116; 136:
  //  167, 112 / 110, 100, 180, 128 / 113, 110, 199, 145 / 167, 120; 160: 139, 101 / 99,
  //  93, 156, 114 / 106, 101, but 176: 128, 100 / 98, 99, 145, 104 / 111, 111; 264: 153,
  //  102 / 113, 95, 179, 131 / 115, 100, 189, 139 / 174, 124; 352: 120, 97 / 94, 81, 137,
  //  101 / 104, 92, but 392: 107, 96 / 92, 94, 124, 96 / 104, 103.  fp32 68: 143, 94 / 104,
  //  95, 148, 102 / 112, 112; 132: 127, 91 / 103, 94; 144: 115, 89 / 96, 85, 141, 99 / 98,
  //  93; 176: 98, 83 / 83, 82.  Longer rows gain behind a key mask with the diagonal,
  //  504 bf16 keys 106, 86 / 88, 83, but add in the order of the key mask alone)
  constexpr bool k16 = sizeof(T) == 2;
  // (with a term, fp32 takes two row sets then: in one the two chunks wait for each
  //  other, 140 keys 117 us by one chunk, 128 / 114 with one / two sets, 164: 105, 119
  //  / 106, with dropout 163, 130 / 123)
  const TwoChunks two = {k16 ? 9 : 8, k16 ? 20 : 16, 44, k16 ? 9 : 34,
                         MODE == kModeBias && !k16 ? 2 : default_rpw};
  SoftmaxPlan pl = plan_softmax(g.sk, E, cap, default_rpw, 4, &two);
  if (!pl.ok && cap < kFwdMaxElems && MODE != kModeBias)
    pl = plan_softmax(g.sk, E, kFwdMaxElems, default_rpw, 4);
  if (MODE == kModeBias && pl.ok && pl.vpl * pl.rpw * E > kBiasMaxElems) pl.ok = false;
  const bool vec_ok = pl.ok && aligned16(x) && aligned16(y) &&
                      (MODE != kModeMasked ||
                       (reinterpret_cast<uintptr_t>(mask) % E) == 0) &&
                      (MODE != kModeBias || bias_vec_ok(g, mask));
  const bool ragged = !vec_ok;
  if (ragged) pl = plan_softmax_ragged<T, MODE>(g.sk, kRaggedFwd, g.batch_inner != 0);
  if (ragged && g.sk < E) {
    const dim3 grid = tiny_grid(g.rows);
    if (drop)
      softmax_fwd_tiny_kernel<T, MODE, true><<<grid, 256, 0, st>>>((const T *)x, mask, (T *)y,
                                                                   stats, g, scale, d);
    else
      softmax_fwd_tiny_kernel<T, MODE, false><<<grid, 256, 0, st>>>((const T *)x, mask, (T *)y,
                                                                    nullptr, g, scale, d);
    return check_launch("softmax_fwd_tiny_kernel");
  }
  if (!pl.ok) {
    const int64_t grid = g.rows < (int64_t)device_cu_count() * 32
                             ? g.rows
                             : (int64_t)device_cu_count() * 32;
    if (drop)
      softmax_fwd_generic_kernel<T, MODE, true>
          <<<dim3((unsigned)grid), 256, 0, st>>>((const T *)x, mask, (T *)y,
                                                 stats, g, scale, d);
    else
      softmax_fwd_generic_kernel<T, MODE, false>
          <<<dim3((unsigned)grid), 256, 0, st>>>((const T *)x, mask, (T *)y,
                                                 nullptr, g, scale, d);
    return check_launch("softmax_fwd_generic_kernel");
  }
  g.wpr = pl.wpr;
  // (rows of several waves run faster in stored order: sequence 4096, 3-12 %)
  if (g_tune.softmax_causal_order == 0 && pl.wpr > 1) g.causal_order = 1;
  g.rpb = pl.rpb;
  const int threads = kWave * pl.wpr * pl.rpb;
  const unsigned keep_lds = ragged_keep_lds(pl);
  const int64_t nblocks =
      ceil_div(g.rows, (int64_t)pl.rpb * pl.rpw * (kWave / pl.lpr));
  const unsigned occ = occupancy_lds(
      softmax_waves_per_cu<T, MODE>(pl, g.sk, false, drop, g.causal, ragged, g.batch_inner != 0),
      threads, nblocks);
  const int64_t per_launch = max_workgroups(threads);
  if (ragged) g.die_end = ragged_die_end<MODE>(g, pl, nblocks);
#define OSLO_SM_FWD(VPL, RPW, LPR_)                                  \
  if constexpr (VPL * RPW * E <= (MODE == kModeBias ? kBiasMaxElems : kFwdMaxElems)) { \
    if (drop)                                                        \
      softmax_fwd_kernel<T, VPL, RPW, MODE, true, LPR_>              \
          <<<dim3((unsigned)grid), threads, occ, st>>>(                \
              (const T *)x, mask, (T *)y, stats, g, scale, d);       \
    else                                                             \
      softmax_fwd_kernel<T, VPL, RPW, MODE, false, LPR_>             \
          <<<dim3((unsigned)grid), threads, occ, st>>>(                \
              (const T *)x, mask, (T *)y, nullptr, g, scale, d);     \
  } else                                                             \
    return fail(OSLO_ERR_UNSUPPORTED, "softmax fwd: no kernel for %d x %d chunks per lane", VPL, RPW)
#define OSLO_SM_FWD_RAGGED(VPL, LPR_)                                \
  if constexpr (ragged_plan_reaches<T, MODE>(VPL, LPR_, kRaggedFwd)) {    \
    if (drop)                                                        \
      softmax_fwd_kernel<T, VPL, 1, MODE, true, LPR_, true>          \
          <<<dim3((unsigned)grid), threads, keep_lds > occ ? keep_lds : occ, st>>>( \
              (const T *)x, mask, (T *)y, stats, g, scale, d);       \
    else                                                             \
      softmax_fwd_kernel<T, VPL, 1, MODE, false, LPR_, true>         \
          <<<dim3((unsigned)grid), threads, occ, st>>>(                \
              (const T *)x, mask, (T *)y, nullptr, g, scale, d);     \
  } else                                                             \
    return fail(OSLO_ERR_UNSUPPORTED, "softmax fwd: no kernel for %d chunks in %d lanes", VPL, LPR_)
  // (rows of a term shared by the batch: one die per run of consecutive blocks)
  int64_t launch_blocks = nblocks;
  if (MODE == kModeBias && g.batch_inner && g_tune.softmax_bias_order == 3 &&
      nblocks >= 64 && nblocks + 8 <= per_launch) {
    g.xcd_wpx = ceil_div(nblocks, 8);
    launch_blocks = 8 * g.xcd_wpx;
  }
  for (g.blk0 = 0; g.blk0 < launch_blocks; g.blk0 += per_launch) {
    const int64_t grid = launch_blocks - g.blk0 < per_launch ? launch_blocks - g.blk0 : per_launch;
    if (ragged) {
      OSLO_SM_RAGGED_CASES(OSLO_SM_FWD_RAGGED)
    } else {
      OSLO_SM_CASES(OSLO_SM_FWD)
    }
    const int rc = check_launch("softmax_fwd_kernel");
    if (rc != OSLO_OK) return rc;
  }
#undef OSLO_SM_FWD
#undef OSLO_SM_FWD_RAGGED
  return OSLO_OK;
}

// Whether the plain backward of ragged rows looks at the mask.  It only saves
// loads of keys whose probability is zero, and short rows wait for it longer
// than those take.  400 MB tensors, a quarter of the keys hidden, us with and
// without it, bf16: key mask 66 keys 282 / 220, 270: 272 / 226, 381: 227 / 205,
// 508: 196 / 204, 653: 189 / 203; under the diagonal (without it the whole row is
// read, since a row without a visible key is uniform) 134: 278 / 218, 381:
// 208 / 205, 508: 166 / 204; fp32 187 keys 211 / 209 and 190 / 209.  Additive term
// (-10000, which hides nothing; -inf): 381 keys 253, 242 / 206, 1077: 227, 204 / 205,
// 1531: 210, 184 / 192; fp32 187: 224, 211 / 212, 509: 201, 188 / 201.
template <typename T, int MODE> static bool ragged_bwd_reads_mask(int sk, bool causal) {
  const int64_t nchunks = ceil_div(sk, io<T>::EPV);
  if (MODE == kModeBias) return nchunks > (sizeof(T) == 2 ? 128 : 64);
  return nchunks > 48 || (causal && sizeof(T) == 4);
}

// ... and the builds that are then left (one wave holds up to 64 VPL chunks)
template <typename T, int MODE> constexpr bool ragged_bwd_plan_reaches(int vpl, int lpr) {
  if (MODE == kModeBias) return lpr == kWave && vpl > (sizeof(T) == 2 ? 2 : 1);
  return MODE != kModeMasked || lpr == kWave || sizeof(T) == 4;
}

template <typename T, int MODE>
int launch_softmax_bwd(const void *dy, const void *y,
                              const uint8_t *mask, void *dx, SoftmaxGeom g,
                              float scale, hipStream_t st) {
  constexpr int E = io<T>::EPV;
  set_fast_div(g);
  // (fp32: 16 elements of each operand per lane, as in the forward)
  SoftmaxPlan pl = plan_softmax(g.sk, E, sizeof(T) == 4 ? 16 : kBwdMaxElems, 1, 1);
  if (!pl.ok && sizeof(T) == 4) pl = plan_softmax(g.sk, E, kBwdMaxElems, 1, 1);
  const bool vec_ok = pl.ok && aligned16(dy) && aligned16(y) &&
                      aligned16(dx) &&
                      (MODE != kModeMasked ||
                       (reinterpret_cast<uintptr_t>(mask) % E) == 0) &&
                      (MODE != kModeBias || bias_vec_ok(g, mask));
  const bool ragged = !vec_ok;
  if constexpr (MODE == kModeMasked || MODE == kModeBias) {
    if (ragged && !ragged_bwd_reads_mask<T, MODE>(g.sk, g.causal)) {
      if (MODE == kModeBias && g.causal)
        return launch_softmax_bwd<T, kModeCausal>(
            dy, y, nullptr, dx, SoftmaxGeom{g.rows, g.sq, g.sk, 1, 0, 0, 1, 1}, scale, st);
      return launch_softmax_bwd<T, kModeDense>(dy, y, nullptr, dx, g, scale, st);
    }
  }
  if (ragged) pl = plan_softmax_ragged<T, MODE>(g.sk, kRaggedBwd);
  if (ragged && g.sk < E) {
    softmax_bwd_tiny_kernel<T><<<tiny_grid(g.rows), 256, 0, st>>>(
        (const T *)dy, (const T *)y, (T *)dx, g.rows, g.sk, scale);
    return check_launch("softmax_bwd_tiny_kernel");
  }
  if (!pl.ok) {
    const int64_t grid = g.rows < (int64_t)device_cu_count() * 32
                             ? g.rows
                             : (int64_t)device_cu_count() * 32;
    softmax_bwd_generic_kernel<T><<<dim3((unsigned)grid), 256, 0, st>>>(
        (const T *)dy, (const T *)y, (T *)dx, g.rows, g.sk, scale);
    return check_launch("softmax_bwd_generic_kernel");
  }
  g.wpr = pl.wpr;
  // (rows of several waves run faster in stored order: sequence 4096, 3-12 %)
  if (g_tune.softmax_causal_order == 0 && pl.wpr > 1) g.causal_order = 1;
  g.rpb = pl.rpb;
  const int threads = kWave * pl.wpr * pl.rpb;
  const int64_t nblocks =
      ceil_div(g.rows, (int64_t)pl.rpb * pl.rpw * (kWave / pl.lpr));
  const unsigned occ = occupancy_lds(
      softmax_waves_per_cu<T, MODE>(pl, g.sk, true, false, g.causal, ragged), threads, nblocks);
  const int64_t per_launch = max_workgroups(threads);
  if (ragged) g.die_end = ragged_die_end<MODE>(g, pl, nblocks);
#define OSLO_SM_BWD(VPL, RPW, LPR_)                        \
  if constexpr (bwd_plan_reaches<T>(VPL, RPW, LPR_))       \
    softmax_bwd_kernel<T, VPL, RPW, MODE, LPR_>            \
        <<<dim3((unsigned)grid), threads, occ, st>>>(        \
            (const T *)dy, (const T *)y, mask, (T *)dx, g, scale); \
  else                                                     \
    return fail(OSLO_ERR_UNSUPPORTED, "softmax bwd: no kernel for %d x %d chunks per lane", VPL, RPW)
#define OSLO_SM_BWD_RAGGED(VPL, LPR_)                      \
  if constexpr (ragged_plan_reaches<T, MODE>(VPL, LPR_, kRaggedBwd) && \
                ragged_bwd_plan_reaches<T, MODE>(VPL, LPR_)) \
    softmax_bwd_kernel<T, VPL, 1, MODE, LPR_, true>        \
        <<<dim3((unsigned)grid), threads, occ, st>>>(        \
            (const T *)dy, (const T *)y, mask, (T *)dx, g, scale); \
  else                                                     \
    return fail(OSLO_ERR_UNSUPPORTED, "softmax bwd: no kernel for %d chunks in %d lanes", VPL, LPR_)
  for (g.blk0 = 0; g.blk0 < nblocks; g.blk0 += per_launch) {
    const int64_t grid = nblocks - g.blk0 < per_launch ? nblocks - g.blk0 : per_launch;
    if (ragged) {
      OSLO_SM_RAGGED_CASES(OSLO_SM_BWD_RAGGED)
    } else {
      OSLO_SM_CASES(OSLO_SM_BWD)
    }
    const int rc = check_launch("softmax_bwd_kernel");
    if (rc != OSLO_OK) return rc;
  }
#undef OSLO_SM_BWD
#undef OSLO_SM_BWD_RAGGED
  return OSLO_OK;
}

template <typename T, int MODE>
int launch_softmax_dropout_bwd(const void *dy, const void *x,
                                      const float *stats, const uint8_t *mask,
                                      void *dx, DropArgs d, SoftmaxGeom g,
                                      float scale, hipStream_t st) {
  constexpr int E = io<T>::EPV;
  set_fast_div(g);
  // (fp32: 16 elements of each operand per lane, as in the forward)
  SoftmaxPlan pl = plan_softmax(g.sk, E, sizeof(T) == 4 ? 16 : kBwdMaxElems, 1, 1);
  if (!pl.ok && sizeof(T) == 4) pl = plan_softmax(g.sk, E, kBwdMaxElems, 1, 1);
  // (with an additive term resident next to the two operands, four row sets
  //  per wave no longer fit the register budget)
  if (MODE == kModeBias && pl.rpw > 2) pl.rpw = 2;
  const bool vec_ok = pl.ok && aligned16(dy) && aligned16(x) && aligned16(dx) &&
                      (MODE != kModeMasked ||
                       (reinterpret_cast<uintptr_t>(mask) % E) == 0) &&
                      (MODE != kModeBias || bias_vec_ok(g, mask));
  const bool ragged = !vec_ok;
  if (ragged) pl = plan_softmax_ragged<T, MODE>(g.sk, kRaggedDropBwd, g.batch_inner != 0);
  if (ragged && g.sk < E) {
    softmax_dropout_bwd_tiny_kernel<T, MODE><<<tiny_grid(g.rows), 256, 0, st>>>(
        (const T *)dy, (const T *)x, stats, mask, (T *)dx, g, scale, d);
    return check_launch("softmax_dropout_bwd_tiny_kernel");
  }
  if (!pl.ok) {
    const int64_t grid = g.rows < (int64_t)device_cu_count() * 32
                             ? g.rows
                             : (int64_t)device_cu_count() * 32;
    softmax_dropout_bwd_generic_kernel<T, MODE>
        <<<dim3((unsigned)grid), 256, 0, st>>>((const T *)dy, (const T *)x,
                                               stats, mask, (T *)dx, g, scale,
                                               d);
    return check_launch("softmax_dropout_bwd_generic_kernel");
  }
  g.wpr = pl.wpr;
  // (rows of several waves run faster in stored order: sequence 4096, 3-12 %)
  if (g_tune.softmax_causal_order == 0 && pl.wpr > 1) g.causal_order = 1;
  g.rpb = pl.rpb;
  const int threads = kWave * pl.wpr * pl.rpb;
  const unsigned keep_lds = ragged_keep_lds(pl);
  const int64_t nblocks =
      ceil_div(g.rows, (int64_t)pl.rpb * pl.rpw * (kWave / pl.lpr));
  const unsigned occ = occupancy_lds(
      softmax_waves_per_cu<T, MODE>(pl, g.sk, true, true, g.causal, ragged), threads, nblocks);
  const int64_t per_launch = max_workgroups(threads);
  if (ragged) g.die_end = ragged_die_end<MODE>(g, pl, nblocks);
#define OSLO_SM_DBWD(VPL, RPW, LPR_)                                \
  if constexpr (bwd_plan_reaches<T>(VPL, RPW, LPR_) && (MODE != kModeBias || RPW <= 2)) \
    softmax_dropout_bwd_kernel<T, VPL, RPW, MODE, LPR_>             \
        <<<dim3((unsigned)grid), threads, occ, st>>>(                 \
            (const T *)dy, (const T *)x, stats, mask, (T *)dx, g,   \
            scale, d);                                              \
  else                                                              \
    return fail(OSLO_ERR_UNSUPPORTED, "softmax dropout bwd: no kernel for %d x %d chunks per lane", VPL, RPW)
#define OSLO_SM_DBWD_RAGGED(VPL, LPR_)                              \
  if constexpr (ragged_plan_reaches<T, MODE>(VPL, LPR_, kRaggedDropBwd))     \
    softmax_dropout_bwd_kernel<T, VPL, 1, MODE, LPR_, true>         \
        <<<dim3((unsigned)grid), threads, keep_lds > occ ? keep_lds : occ, st>>>( \
            (const T *)dy, (const T *)x, stats, mask, (T *)dx, g, scale, d); \
  else                                                              \
    return fail(OSLO_ERR_UNSUPPORTED, "softmax dropout bwd: no kernel for %d chunks in %d lanes", VPL, LPR_)
  // (rows of a term shared by the batch: one die per run of consecutive blocks)
  int64_t launch_blocks = nblocks;
  if (MODE == kModeBias && g.batch_inner && g_tune.softmax_bias_order == 3 &&
      nblocks >= 64 && nblocks + 8 <= per_launch) {
    g.xcd_wpx = ceil_div(nblocks, 8);
    launch_blocks = 8 * g.xcd_wpx;
  }
  for (g.blk0 = 0; g.blk0 < launch_blocks; g.blk0 += per_launch) {
    const int64_t grid = launch_blocks - g.blk0 < per_launch ? launch_blocks - g.blk0 : per_launch;
    if (ragged) {
      OSLO_SM_RAGGED_CASES(OSLO_SM_DBWD_RAGGED)
    } else {
      OSLO_SM_CASES(OSLO_SM_DBWD)
    }
    const int rc = check_launch("softmax_dropout_bwd_kernel");
    if (rc != OSLO_OK) return rc;
  }
#undef OSLO_SM_DBWD
#undef OSLO_SM_DBWD_RAGGED
  return OSLO_OK;
}

// Every (type, mode) pair of the three launchers, as explicit instantiations:
// softmax_inst.hip defines them, one type and one direction per translation
// unit (so that the units build in parallel), softmax.hip declares them extern.
#define OSLO_SM_FWD_INSTANCES(PREFIX, T)                                                   \
  PREFIX template int launch_softmax_fwd<T, kModeCausal>(const void *, const uint8_t *, void *, \
      float *, DropArgs, SoftmaxGeom, float, hipStream_t);                                 \
  PREFIX template int launch_softmax_fwd<T, kModeMasked>(const void *, const uint8_t *, void *, \
      float *, DropArgs, SoftmaxGeom, float, hipStream_t);                                 \
  PREFIX template int launch_softmax_fwd<T, kModeBias>(const void *, const uint8_t *, void *, \
      float *, DropArgs, SoftmaxGeom, float, hipStream_t);
#define OSLO_SM_BWD_ONE(PREFIX, T, MODE)                                                   \
  PREFIX template int launch_softmax_bwd<T, MODE>(const void *, const void *, const uint8_t *, \
      void *, SoftmaxGeom, float, hipStream_t);
#define OSLO_SM_DBWD_ONE(PREFIX, T, MODE)                                                  \
  PREFIX template int launch_softmax_dropout_bwd<T, MODE>(const void *, const void *,      \
      const float *, const uint8_t *, void *, DropArgs, SoftmaxGeom, float, hipStream_t);
#define OSLO_SM_BWD_INSTANCES(PREFIX, T)   \
  OSLO_SM_BWD_ONE(PREFIX, T, kModeCausal)  \
  OSLO_SM_BWD_ONE(PREFIX, T, kModeMasked)  \
  OSLO_SM_BWD_ONE(PREFIX, T, kModeDense)   \
  OSLO_SM_BWD_ONE(PREFIX, T, kModeBias)    \
  OSLO_SM_DBWD_ONE(PREFIX, T, kModeCausal) \
  OSLO_SM_DBWD_ONE(PREFIX, T, kModeMasked) \
  OSLO_SM_DBWD_ONE(PREFIX, T, kModeBias)

}  // namespace oslo
