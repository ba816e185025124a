// Device building blocks shared by the LM-head kernels (lm_head.hip,
// lm_head_ring.hip): launch arguments, MFMA wrappers, rounding, the final
// RMSNorm arithmetic, the scoring of logits and the cross-block reduce.
#pragma once
#include "nvjsel_device.h"
#include "nvjsel_host.h"

static constexpr int kLmNt = 1;  // non-temporal (streaming) loads of W

namespace nvjsel {

template <typename T>
__device__ __forceinline__ T stream_load(const T* p) {
  if constexpr (kLmNt) return __builtin_nontemporal_load(p);
  else return *p;
}

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef u32x4_t u32x4_any_t __attribute__((aligned(2)));  // a 16-byte load from any element address

// The eight 16-bit elements of w moved down by s places (0 <= s <= 7).
__device__ __forceinline__ u32x4_t shift_down8(u32x4_t w, int s) {
  const uint64_t lo = ((uint64_t)w.y << 32) | w.x, hi = ((uint64_t)w.w << 32) | w.z;
  const int b = 16 * (s & 3);
  const uint64_t l1 = s & 4 ? hi : lo, h1 = s & 4 ? 0ull : hi;
  const uint64_t l2 = b ? (l1 >> b) | (h1 << (64 - b)) : l1, h2 = h1 >> b;
  return u32x4_t{(uint32_t)l2, (uint32_t)(l2 >> 32), (uint32_t)h2, (uint32_t)(h2 >> 32)};
}

// GREEDY: argmax id per row; SAMPLE: Gumbel-max id per row; LOGITS: the
// (REDUCE_CAST-rounded) logits themselves, written to out_logits.
enum { MODE_GREEDY = 0, MODE_SAMPLE = 1, MODE_LOGITS = 2 };

struct LmArgs {
  const void* W;
  const void* hidden;
  int hidden_dtype;    // element type of `hidden` as stored
  // final RMSNorm prologue (prenorm != 0): the kernel multiplies against
  // act(in(rms_norm(hidden) * (1 + norm_w))) instead of `hidden`
  int prenorm;
  const void* norm_w;
  int norm_dtype;
  float eps;
  int act_dtype;
  int weight_dtype;
  int layout;
  int B;  // rows handled by this launch
  int H;
  int V;
  int reduce_cast;
  const float* temperature;  // MODE_SAMPLE, offset to this launch's first row
  const uint32_t* keys;      // MODE_SAMPLE, [B,2]
  unsigned long long* row_keys;
  unsigned int* counter;
  int32_t* out_ids;
  float* out_best;
  void* out_logits;      // MODE_LOGITS: [B, out_stride] of out_dtype, offset to this launch's first row
  int out_dtype;         // DT_F32, DT_BF16 or DT_F16
  long long out_stride;  // elements between output rows
};

// MODE_LOGITS store of logit (b, v): f32 as is, bf16 / f16 rounded to nearest even.
__device__ __forceinline__ void store_logit(const LmArgs& a, int b, int v, float val) {
  const size_t i = (size_t)b * (size_t)a.out_stride + (size_t)v;
  if (a.out_dtype == DT_F32) ((float*)a.out_logits)[i] = val;
  else if (a.out_dtype == DT_BF16) ((__bf16*)a.out_logits)[i] = (__bf16)val;
  else ((_Float16*)a.out_logits)[i] = (_Float16)val;
}

template <int WT>
__device__ __forceinline__ f32x4_t mfma16x16x32(u32x4_t a, u32x4_t b, f32x4_t c) {
  if constexpr (WT == DT_BF16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  }
}

typedef float f32x16_t __attribute__((ext_vector_type(16)));

// v_mfma_f32_32x32x16_bf16 / _f16: lane l holds A row (l & 31) and B column (l & 31)
// at k = 8 (l >> 5) .. +7; D element e of lane l is row 8 (e >> 2) +
// 4 (l >> 5) + (e & 3), column l & 31.  Twice the work of a 16x16x32 in
// about the same issue time on gfx950 (measured ~2.2 vs ~1.25 PFLOP/s).
template <int WT>
__device__ __forceinline__ f32x16_t mfma32x32x16(u32x4_t a, u32x4_t b, f32x16_t c) {
  if constexpr (WT == DT_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0,
                                                  0, 0);
}

__device__ __forceinline__ float apply_cast(float v, int rc) {
  if (rc == 1) return round_bf16(v);
  if (rc == 2) return round_f16(v);
  return v;
}

__device__ __forceinline__ uint32_t bf16_bits_rne(float v) {
  uint32_t u = __float_as_uint(v);
  if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (u >> 16) | 0x40u;
  return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

// rounds v to element type dt (f32: unchanged)
__device__ __forceinline__ float round_to_dtype(float v, int dt) {
  return apply_cast(v, dt == DT_BF16 ? 1 : dt == DT_F16 ? 2 : 0);
}

// Final RMSNorm of the LM-head prologue, as layers.py:22-29 followed by the
// activation cast of model.py:758-760: with ss = sum of x^2 over the row (fp32),
//   y = x * (1 / sqrt(ss / H + eps)) * (1 + w), rounded to the hidden's own type
// (rms_norm's output.astype(input_dtype)) and then to the activation type.
__device__ __forceinline__ float prenorm_inv(const LmArgs& a, float ss) {
  return 1.0f / sqrtf(ss / (float)a.H + a.eps);
}
__device__ __forceinline__ float prenorm_apply_w(const LmArgs& a, float x, float inv, float w) {
  const float y = (x * inv) * (1.0f + w);
  return round_to_dtype(round_to_dtype(y, a.hidden_dtype), a.act_dtype);
}
__device__ __forceinline__ float prenorm_apply(const LmArgs& a, float x, float inv, int k) {
  return prenorm_apply_w(a, x, inv, load_as_f32(a.norm_w, a.norm_dtype, (size_t)k));
}

__device__ __forceinline__ uint32_t f16_bits(float v) {
  _Float16 h = (_Float16)v;
  uint16_t b;
  __builtin_memcpy(&b, &h, 2);
  return b;
}

// Block-wide max of per-(wave, row) keys held in LDS, then one atomic per row.
// Each thread waits for its atomics to be performed (their returned values
// feed an opaque use) before the block barrier, so the ticket taken after the
// barrier is ordered after every max of the block -- no release fence, which
// on gfx950 writes back and invalidates the XCD's L2.
template <int WAVES, int BP>
__device__ __forceinline__ void block_commit(unsigned long long* red, int B,
                                             unsigned long long* row_keys) {
  __syncthreads();
  for (int b = threadIdx.x; b < B; b += blockDim.x) {
    unsigned long long m = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) m = max_u64(m, red[w * BP + b]);
    if (m) (void)after(atomicMax(&row_keys[b], m));
  }
}

// Last block to arrive converts the per-row keys into ids and re-zeroes the
// accumulators and the ticket counter for the next call.  `flag`: a word of
// LDS that no thread uses between the two barriers here.
__device__ __forceinline__ void finish_rows(unsigned long long* row_keys, unsigned int* counter,
                                            int B, int32_t* out_ids, float* out_best, int* flag) {
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned int t = ticket_add(counter);
    *flag = (t == gridDim.x - 1);
  }
  __syncthreads();
  if (!*flag) return;
  for (int b = threadIdx.x; b < B; b += blockDim.x) {
    unsigned long long k =
        __hip_atomic_load(&row_keys[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    out_ids[b] = (int32_t)(~(uint32_t)k);
    if (out_best) out_best[b] = unord_f32((uint32_t)(k >> 32));
    __hip_atomic_store(&row_keys[b], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (threadIdx.x == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void finish_rows(unsigned long long* row_keys, unsigned int* counter,
                                            int B, int32_t* out_ids, float* out_best) {
  __shared__ int s_last;
  finish_rows(row_keys, counter, B, out_ids, out_best, &s_last);
}

// Scores N consecutive vocabulary entries v0.. of one batch row (raw fp32
// dots).  Greedy: folds argmax keys into `best`.  Sample: computes the fast
// approximate scores for all N in one straight-line block (N interleaved
// Threefry chains) and marks in q[] (logit xq[], approximate score aq[]) every
// entry that can still be the row's exact maximum.  The approximate score
// multiplies with rtp = 1 / tp (the exact rescoring divides; a division per
// draw cost ~10% of the draws' time).  |approx - exact| <= d(s) = 1e-4 + 4.8e-7
// |s| + 1.8e-7 |x|, |x| <= |s| + 16 (hardware log error ~1e-6 on the draw, one
// ulp of the sum, three roundings of the product), so the exact maximum j has
// approx_j >= approx_k - d(s_j) - d(s_k) for every k and is queued when it
// arrives, whatever set of approximate scores `amax` is the maximum of
// (score_slack: the two together).  Magnitudes are clamped so -inf stays -inf;
// a NaN scaled logit scores +inf.
__device__ __forceinline__ float score_slack(float ap, float am) {
  return 2.2e-4f + 6.8e-7f * (fminf(fabsf(ap), 1e30f) + fminf(fabsf(am), 1e30f));
}

template <int MODE, int N>
__device__ __forceinline__ void score_run(const float (&raw)[N], int v0, int V, int reduce_cast, bool greedy_row,
                                          float rtp, float tp, const TfKey& key, float& amax,
                                          unsigned long long& best, bool (&q)[N], float (&xq)[N], float (&aq)[N]) {
  // one branch per run, not per element: the cast and the bounds are uniform
  float val[N];
  if (reduce_cast == 1) {
#pragma unroll
    for (int e = 0; e < N; ++e) val[e] = round_bf16(raw[e]);
  } else if (reduce_cast == 2) {
#pragma unroll
    for (int e = 0; e < N; ++e) val[e] = round_f16(raw[e]);
  } else {
#pragma unroll
    for (int e = 0; e < N; ++e) val[e] = raw[e];
  }
  if (MODE == MODE_SAMPLE && !greedy_row) {
    float xv[N], ap[N];
    uint32_t bits[N];
#pragma unroll
    for (int e = 0; e < N; ++e) xv[e] = val[e] * rtp;
    float mag = fabsf(xv[0]);
#pragma unroll
    for (int e = 1; e < N; ++e) mag = fmaxf(mag, fabsf(xv[e]));
    if (!(mag < 1e30f)) {  // infinities and the edge of the float range: divide
#pragma unroll
      for (int e = 0; e < N; ++e) xv[e] = val[e] / tp;
    }
    uint32_t idx[N];
#pragma unroll
    for (int e = 0; e < N; ++e) idx[e] = (uint32_t)(v0 + e);
    random_bits32_n<N>(key, idx, bits);
    // NaN only from a NaN logit (the draw is finite); selecting on the sum
    // keeps the draws unconditional, so the N chains stay one straight block
#pragma unroll
    for (int e = 0; e < N; ++e) {
      const float t = xv[e] + gumbel_fast_from_bits(bits[e]);
      ap[e] = (t != t) ? INFINITY : t;
    }
    // every draw feeds an unconditional select, so none is sunk into a branch.
    // One threshold per run instead of the per-entry slack: an entry that
    // passes ap + score_slack(ap, am) >= am has |ap| <= |am| + slack, so slack
    // <= 2.21e-4 + 1.37e-6 |am| and ap >= am - that bound: the queued set only
    // grows (the filter before exact rescoring applies the per-entry test).
    // am = -inf queues every entry, am = +inf only +inf.
    const float am = amax;
    const float thr = am - (2.21e-4f + 1.37e-6f * fminf(fabsf(am), 1e30f));
    const bool all_in = v0 + N <= V;  // uniform per run except in the last tile
#pragma unroll
    for (int e = 0; e < N; ++e) {
      const bool ok = all_in || v0 + e < V;
      q[e] = ok && ap[e] >= thr;
      xq[e] = val[e];
      aq[e] = ap[e];
      amax = fmaxf(amax, ok ? ap[e] : -INFINITY);
    }
  } else {
#pragma unroll
    for (int e = 0; e < N; ++e)
      if (v0 + e < V) best = max_u64(best, argmax_key(val[e], (uint32_t)(v0 + e)));
  }
}

// Packs eight values into NS bf16 B-fragment words per term: NS = 1 rounds
// each value to bf16 (exact for bf16 activations); NS = 3 splits an fp32 value
// exactly into three bf16 terms (hi + mid + lo = v: 8 + 8 + 8 significand bits),
// so that three bf16 x bf16 products, each exact in fp32, give an fp32-accurate dot.
template <int NS, int KPW>
__device__ __forceinline__ void split_terms(const float (&v)[8], u32x4_t (&hb)[NS][KPW], int kk) {
  float r[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = v[e];
#pragma unroll
  for (int t = 0; t < NS; ++t) {
    uint32_t bits[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      bits[e] = bf16_bits_rne(r[e]);
      r[e] = r[e] - __uint_as_float(bits[e] << 16);
    }
    hb[t][kk] = u32x4_t{bits[0] | (bits[1] << 16), bits[2] | (bits[3] << 16), bits[4] | (bits[5] << 16),
                        bits[6] | (bits[7] << 16)};
  }
}

// NaN logits of f32 hidden in three bf16 terms, summed again from the f32
// values.  The split holds for finite operands: an infinite value (or one that
// rounds to bf16's infinity) leaves NaN remainders, and an infinite weight
// meets lower terms that are zero or of the other sign, where the fp32
// products have an infinity, or a finite sum.  Rows that hold a NaN keep it.
// d: the wave's 32 x 32 tiles; at(tv, e, b, v): batch and vocabulary row of
// element e of tile (tv, TBI) of this lane, whether it is a live one; ROWLANE: a lane's elements all belong to one batch row.  The whole
// wave sums each such logit (V = 248,320, H = 1024, 64 [V, H] / 24 [H, V] rows,
// one of them holding an infinity: 2.5 ms in place of 117 / 198 us; a NaN:
// 137 / 213 us); finite operands pay the callers' test for a NaN, out of a
// maximum over the tile's values (within the runs' noise).
__device__ __forceinline__ bool row_has_nan(const LmArgs& a, int b, int lane) {
  const float* x = (const float*)a.hidden + (size_t)b * a.H;
  bool nan = false;
  for (int k = lane; k < a.H; k += 64) nan |= x[k] != x[k];
  return __any(nan);
}
__device__ __forceinline__ float wave_dot_f32(const LmArgs& a, int b, int v, int lane) {
  const float* x = (const float*)a.hidden + (size_t)b * a.H;
  const uint16_t* w = (const uint16_t*)a.W + (a.layout == NVJSEL_W_VH ? (size_t)v * a.H : (size_t)v);
  const size_t step = a.layout == NVJSEL_W_VH ? 1 : (size_t)a.V;
  float s = 0.0f;
  for (int k = lane; k < a.H; k += 64) s = fmaf(x[k], __uint_as_float((uint32_t)w[k * step] << 16), s);
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
  return s;
}
template <int TBI, bool ROWLANE, int TV, int TB, typename At>
__device__ __forceinline__ void redo_nan_logits(const LmArgs& a, f32x16_t (&d)[TV][TB], int lane, At at) {
  unsigned long long keep = 0;  // lanes whose row holds a NaN
#pragma unroll
  for (int tv = 0; tv < TV; ++tv) {
    const f32x16_t& t = d[tv][TBI];
    bool nan = false;
#pragma unroll
    for (int e = 0; e < 16; ++e) nan |= t[e] != t[e];
    if (!__any(nan)) continue;
#pragma unroll 1
    for (int e = 0; e < 16; ++e) {  // wave-uniform: indexed registers
      const float x = d[tv][TBI][e];
      int b, v;
      const bool live = at(tv, e, b, v);
      unsigned long long todo = __ballot(live && x != x) & ~keep;
      while (todo) {  // wave-uniform
        const int row = __builtin_amdgcn_readlane(b, __builtin_ctzll(todo));
        unsigned long long same = __ballot(b == row) & todo;
        todo &= ~same;
        if (row_has_nan(a, row, lane)) {
          if (ROWLANE) keep |= __ballot(b == row);
          continue;
        }
        for (; same; same &= same - 1) {
          const int l = __builtin_ctzll(same);
          const float s = wave_dot_f32(a, row, __builtin_amdgcn_readlane(v, l), lane);
          d[tv][TBI][e] = lane == l ? s : d[tv][TBI][e];
        }
      }
    }
  }
}
// The maximum of column TBI of the wave's tiles; NaN if one of them is.
template <int TBI, int TV, int TB>
__device__ __forceinline__ float tile_max(const f32x16_t (&d)[TV][TB]) {
  float m = d[0][TBI][0];
#pragma unroll
  for (int i = 1; i < TV * 16 - 1; i += 2)
    m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, d[i / 16][TBI][i % 16]),
                                      d[(i + 1) / 16][TBI][(i + 1) % 16]);
  return __builtin_elementwise_maximum(m, d[TV - 1][TBI][15]);
}

// lm_head_ring.hip: one pass over W for up to kRingRows batch rows (sampling:
// kRingSampleRows); 16-bit weight [V, H] and hidden of the same type, or bf16
// weight and f32 hidden (kRingF32Rows), 16-byte aligned, H % 64 == 0
// (sampling: V < 2^25).
static constexpr int kRingRows = 256, kRingSampleRows = 128, kRingF32Rows = 64;
int launch_ring(int mode, const LmArgs& a, hipStream_t stream);

// lm_head_gemm.hip: one pass over W for up to kGemmBB rows; hv: [H, V] weights
// (16-bit hidden of the same type -- f16 at most 64 rows -- or f32 on bf16),
// else on bf16 [V, H] bf16 sampling or f32 hidden; H % (2 kGemmKC) == 0.
static constexpr int kGemmBB = 256, kGemmKC = 32;
int launch_gemm(int mode, bool hv, const LmArgs& a, hipStream_t stream);

}  // namespace nvjsel
