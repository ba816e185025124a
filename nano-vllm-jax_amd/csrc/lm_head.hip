// LM-head projection fused with greedy top-1 or Gumbel-max sampling (gfx950).
//
// Replaces nanovllm_jax/kernels/lm_head_triton.py:22-186 (two-stage Triton
// top-1) and the dense dot + argmax / categorical of nanovllm_jax/model.py:
// 806-830, 894, 901-938.  Logits are never written to memory.
//
// Hot path (weight [V,H] bf16, hidden bf16 or f32): one pass over W.
//   * Matrix cores: v_mfma_f32_16x16x32_bf16 with M = 16 vocabulary rows,
//     N = 16 batch rows, K = 32.  Lane l loads 16 contiguous bytes of vocab row
//     (l % 16) straight from HBM into its A operand (group g = l / 16 takes
//     k = 8g..8g+7 of each 32-wide step), so W is read once with 128-bit loads
//     and never staged.  B operands (hidden) are staged once per block in LDS
//     in fragment order, so each lane's ds_read_b128 is contiguous across the
//     16 lanes that share a k group.
//   * An f32 hidden is split exactly into three bf16 terms (hi + mid + lo =
//     h); bf16 x bf16 products are exact in fp32, so the three MFMAs give an
//     fp32-accurate dot while W stays bf16 and is still read once.
//   * Epilogue per 16x16 tile: optional bf16/f16 rounding of the logit
//     (REDUCE_CAST), optional temperature division + Threefry Gumbel noise at
//     the vocabulary index, then a running max of 64-bit (value, ~index) keys.
//   * Cross-block reduce: one 64-bit atomicMax per (block, row) into the
//     workspace, then the last block to finish (ticket counter) writes the ids
//     and re-zeroes the workspace -- a single launch per call.
// Any other dtype/layout/shape goes through a generic VALU kernel with the same
// reduction and epilogue.
#include <mutex>
#include <type_traits>

#include "lm_head_common.h"
#include "route_rules.h"

// Launch shapes (chosen by measurement on MI355X).
static constexpr int kLmWaves = 8;  // waves per block
static constexpr int kLmMt1 = 4;  // 16-row vocab tiles per wave when B <= 16
static constexpr int kLmMtn = 2;  // ... when B > 16
static constexpr int kLmKu = 4;  // 32-wide k-steps per prefetch chunk
static constexpr int kLmDepth = 3;  // k-chunks of W in flight per wave
static constexpr int kLmBpc = 0;  // blocks per CU (0 = as many as occupancy allows)

static constexpr int kGemvWaves = 4;  // waves per block of the streaming GEMV
static constexpr int kGemvDepth = 2;  // row groups in flight per wave (measured on the dot2 path: 2 > 3 > 4)
static constexpr int kGemvBpc = 1;  // blocks per CU for the streaming GEMV (0 = occupancy)
static constexpr int kTileQcap = 768;  // queue entries per epilogue wave (sample mode)
static constexpr int kGemvR = 4;  // rows per wave step of the streaming GEMV
static constexpr bool kGemvDot = true;  // bf16 hidden without prologue: v_dot2c_f32_bf16

namespace nvjsel {

// ------------------------------------------------------------------ MFMA kernel
// WT: weight element type (DT_BF16 / DT_F16).  NSPLIT: hidden terms (1, or 3
// for an exact f32 hidden on bf16 weights).  NB: 16-row batch tiles.  MT:
// 16-row vocab tiles per wave.  KU: k-steps (32 each) per prefetch chunk.
template <int WT, int NSPLIT, int NB, int MT, int WAVES, int KU, int DEPTH, int MODE>
__global__ void __launch_bounds__(WAVES * 64)
lm_head_mfma_kernel(LmArgs a) {
  constexpr int BP = NB * 16;
  extern __shared__ u32x4_t lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int g = lane >> 4;
  const int r = lane & 15;
  const int H = a.H, V = a.V, B = a.B;
  const int KQ = H >> 3;  // 8-element groups per row

  // ---- stage hidden [B, H] into LDS fragments: lds[(kq * NSPLIT + s) * BP + n]
  for (int f = tid; f < KQ * BP; f += WAVES * 64) {
    const int n = f % BP;
    const int kq = f / BP;
    float v[8];
    load8_as_f32(a.hidden, a.hidden_dtype, (size_t)(n < B ? n : 0) * H + kq * 8, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = n < B ? v[j] : 0.0f;
#pragma unroll
    for (int s = 0; s < NSPLIT; ++s) {
      uint32_t bits[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if constexpr (WT == DT_BF16) {
          bits[j] = bf16_bits_rne(v[j]);
          v[j] = v[j] - __uint_as_float(bits[j] << 16);
        } else {
          bits[j] = f16_bits(v[j]);
        }
      }
      u32x4_t p;
      p.x = bits[0] | (bits[1] << 16);
      p.y = bits[2] | (bits[3] << 16);
      p.z = bits[4] | (bits[5] << 16);
      p.w = bits[6] | (bits[7] << 16);
      lds[(kq * NSPLIT + s) * BP + n] = p;
    }
  }
  __syncthreads();

  float tp[NB];
  bool greedy_row[NB];
  TfKey key[NB];
  if constexpr (MODE == MODE_SAMPLE) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int b = nb * 16 + r;
      float t = (b < B) ? a.temperature[b] : 0.0f;
      greedy_row[nb] = (t <= 0.0f);
      tp[nb] = temp_floor(t);
      key[nb] = (b < B) ? tf_key(a.keys[2 * b], a.keys[2 * b + 1]) : tf_key(0u, 0u);
    }
  }

  unsigned long long best[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) best[nb] = 0;

  const int ksteps = H >> 5;
  const int nch = ksteps / KU;  // the host guarantees KU divides ksteps
  constexpr int ROWS = 16 * MT;
  const int ntiles = (V + ROWS - 1) / ROWS;
  const uint16_t* W = (const uint16_t*)a.W;

  // Each wave walks its tiles (grid-stride) as one sequence of k-chunks q and
  // keeps DEPTH-1 chunks of W requested ahead of the chunk it multiplies, across
  // tile boundaries.
  const int nwaves = gridDim.x * WAVES;
  const int gw = blockIdx.x * WAVES + wave;
  const int n_my_tiles = gw < ntiles ? (ntiles - gw + nwaves - 1) / nwaves : 0;
  const int nq = n_my_tiles * nch;
  auto load_q = [&](u32x4_t(&A)[KU][MT], int q) NVJSEL_INLINE {
    const int tile = gw + (q / nch) * nwaves;
    const int c = q % nch;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      int row = tile * ROWS + t * 16 + r;
      row = row < V ? row : V - 1;
      const u32x4_t* p = (const u32x4_t*)(W + (size_t)row * H) + g + c * KU * 4;
#pragma unroll
      for (int u = 0; u < KU; ++u) A[u][t] = stream_load(p + u * 4);
    }
    __builtin_amdgcn_sched_barrier(0);  // the whole chunk is requested before any use
  };
  f32x4_t acc[MT][NB];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[t][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  u32x4_t ring[DEPTH][KU][MT];
#pragma unroll
  for (int d = 0; d < DEPTH - 1; ++d)
    if (d < nq) load_q(ring[d], d);
  for (int q = 0; q < nq; ++q) {
    if (q + DEPTH - 1 < nq) load_q(ring[DEPTH - 1], q + DEPTH - 1);
    const int c = q % nch;
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const int kb = c * KU + u;
#pragma unroll
      for (int s = 0; s < NSPLIT; ++s)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const u32x4_t bfr = lds[((kb * 4 + g) * NSPLIT + s) * BP + nb * 16 + r];
#pragma unroll
          for (int t = 0; t < MT; ++t) acc[t][nb] = mfma16x16x32<WT>(ring[0][u][t], bfr, acc[t][nb]);
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
#pragma unroll
      for (int u = 0; u < KU; ++u)
#pragma unroll
        for (int t = 0; t < MT; ++t) ring[d][u][t] = ring[d + 1][u][t];
    if (c != nch - 1) continue;

    // ---- epilogue: D[row = 4g + i][col = r] of each 16x16 tile
    const int v0 = (gw + (q / nch) * nwaves) * ROWS;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int b = nb * 16 + r;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int v = v0 + t * 16 + g * 4 + i;
          if (v < V && b < B) {
            float val = apply_cast(acc[t][nb][i], a.reduce_cast);
            if constexpr (MODE == MODE_LOGITS) {
              store_logit(a, b, v, val);
            } else {
              if constexpr (MODE == MODE_SAMPLE) {
                if (!greedy_row[nb]) val = val / tp[nb] + gumbel_at(key[nb], (uint32_t)v);
              }
              best[nb] = max_u64(best[nb], argmax_key(val, (uint32_t)v));
            }
          }
        }
        acc[t][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
  }

  if constexpr (MODE == MODE_LOGITS) return;
  // ---- reduce the four k-groups, then the waves, then across blocks
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    best[nb] = max_u64(best[nb], shfl_xor_u64(best[nb], 16));
    best[nb] = max_u64(best[nb], shfl_xor_u64(best[nb], 32));
  }
  __syncthreads();  // hidden fragments are dead from here on
  unsigned long long* red = (unsigned long long*)lds;
  if (g == 0) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) red[wave * BP + nb * 16 + r] = best[nb];
  }
  block_commit<WAVES, BP>(red, B, a.row_keys);
  finish_rows(a.row_keys, a.counter, B, a.out_ids, a.out_best);
}

// ------------------------------------------------------------------ streaming GEMV kernel
// Small batch (B <= 4), weight [V,H] bf16 with H = KJ * 512.  Every load
// instruction of a wave reads 1 KB of W contiguous (64 lanes x 16 B), the
// pattern that streams HBM at full rate: lane l holds k = 512 j + 8 l .. +7 of
// each row.  A wave takes R consecutive rows per step (R * 2H bytes
// contiguous), forms per-lane partial dots against the hidden held in
// registers, then a butterfly transpose-reduction leaves each group of 64/R
// lanes with the full dot of one row (log2(64) shuffle rounds, halving the
// values carried at each of the first log2(R) rounds).
template <int NB, int R, int KJ, int MODE, bool DOT>
__global__ void __launch_bounds__(kGemvWaves * 64) lm_head_gemv_kernel(LmArgs a) {
  // DOT (bf16 activations): the hidden is held as bf16 pairs (k, k+1) --
  // the pairs of each 32-bit word of W too -- so one v_dot2c_f32_bf16
  // (exact products, fp32 sums) replaces two convert-and-FMA steps.  Without
  // the prologue the pairs are the hidden's own words; with it they are
  // packed from the normalised rows (already rounded to bf16)
  constexpr int WAVES = kGemvWaves;
  __shared__ unsigned long long red[WAVES * NB];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int H = KJ * 512, V = a.V, B = a.B;
  float hv[NB][KJ][8];
  uint32_t hp[NB][KJ][DOT ? 4 : 1];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      if (DOT && !a.prenorm) {
        const u32x4_t v = b < B ? *((const u32x4_t*)((const uint16_t*)a.hidden + (size_t)b * H + j * 512) + lane)
                                : u32x4_t{0u, 0u, 0u, 0u};
        hp[b][j][0] = v.x; hp[b][j][1] = v.y; hp[b][j][2] = v.z; hp[b][j][3] = v.w;
      } else {
        load8_as_f32(a.hidden, a.hidden_dtype, (size_t)(b < B ? b : 0) * H + j * 512 + lane * 8, hv[b][j]);
#pragma unroll
        for (int e = 0; e < 8; ++e) hv[b][j][e] = b < B ? hv[b][j][e] : 0.0f;
      }
    }
  // RMSNorm prologue: its operands are requested with the hidden, and it runs
  // once the first weight groups are in flight (finish_prenorm below)
  float nwv[KJ][8] = {};
  if (a.prenorm) {
#pragma unroll
    for (int j = 0; j < KJ; ++j) load8_as_f32(a.norm_w, a.norm_dtype, (size_t)(j * 512 + lane * 8), nwv[j]);
  }
  auto finish_prenorm = [&]() NVJSEL_INLINE {
    {
      if (!a.prenorm) return;
      // the wave holds whole rows: per-lane sum of squares, then the butterfly
      // leaves the same total in every lane (and every wave)
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < KJ; ++j)
#pragma unroll
          for (int e = 0; e < 8; ++e) ss = fmaf(hv[b][j][e], hv[b][j][e], ss);
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) ss += __shfl_xor(ss, m, 64);
        const float inv = prenorm_inv(a, ss);
#pragma unroll
        for (int j = 0; j < KJ; ++j)
#pragma unroll
          for (int e = 0; e < 8; ++e) hv[b][j][e] = prenorm_apply_w(a, hv[b][j][e], inv, nwv[j][e]);
        if constexpr (DOT) {
#pragma unroll
          for (int j = 0; j < KJ; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              hp[b][j][e] = (__float_as_uint(hv[b][j][2 * e]) >> 16) | (__float_as_uint(hv[b][j][2 * e + 1]) & 0xFFFF0000u);
        }
      }
    }
  };

  float tp[NB];
  bool greedy_row[NB];
  TfKey key[NB];
  if constexpr (MODE == MODE_SAMPLE) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const float t = (b < B) ? a.temperature[b] : 0.0f;
      greedy_row[b] = (t <= 0.0f);
      tp[b] = temp_floor(t);
      key[b] = (b < B) ? tf_key(a.keys[2 * b], a.keys[2 * b + 1]) : tf_key(0u, 0u);
    }
  }
  unsigned long long best[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) best[b] = 0;

  const uint16_t* W = (const uint16_t*)a.W;
  const int ngroups = (V + R - 1) / R;
  const int nwaves = gridDim.x * WAVES;
  const int gw = blockIdx.x * WAVES + wave;
  // round-robin groups: wave gw takes gw, gw + nwaves, ...  (measured faster
  // than contiguous slices per wave or per block)
  const int g_begin = gw, g_end = ngroups, g_step = nwaves;

  auto load_grp = [&](u32x4_t(&w)[R][KJ], int grp) NVJSEL_INLINE {
    const int v0 = grp * R;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int row = (v0 + r < V) ? v0 + r : V - 1;
#pragma unroll
      for (int j = 0; j < KJ; ++j)
        w[r][j] = stream_load((const u32x4_t*)(W + (size_t)row * H + j * 512) + lane);
    }
    // keep every load of the step ahead of the first use: R*KJ KB in flight per wave
    __builtin_amdgcn_sched_barrier(0);
  };

  auto proc_grp = [&](const u32x4_t(&w)[R][KJ], int grp) NVJSEL_INLINE {
    const int v0 = grp * R;
    float p[NB][R];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j < KJ; ++j) {
          const uint32_t q[4] = {w[r][j].x, w[r][j].y, w[r][j].z, w[r][j].w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (DOT) {
              acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, q[e]),
                                                    __builtin_bit_cast(bf16x2_t, hp[b][j][e]), acc, false);
            } else {
              acc = fmaf(__uint_as_float(q[e] << 16), hv[b][j][2 * e], acc);
              acc = fmaf(__uint_as_float(q[e] & 0xFFFF0000u), hv[b][j][2 * e + 1], acc);
            }
          }
        }
        p[b][r] = acc;
      }
    // transpose-reduce: after the halving rounds lane holds row `sel` only.
    // Rounds across lane halves and 16-lane rows are register permutes
    // (v_permlane32/16_swap), the sums within a row DPP rotations: no LDS.
    int sel = 0;
    int mask = 32;
#pragma unroll
    for (int cnt = R; cnt > 1; cnt >>= 1, mask >>= 1) {
      const int half = cnt >> 1;
      const bool upper = (lane & mask) != 0;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < half; ++i) {
          if (mask == 32) {
            p[b][i] = xpose_add32(p[b][i], p[b][i + half]);
          } else if (mask == 16) {
            p[b][i] = xpose_add16(p[b][i], p[b][i + half]);
          } else {
            const float keep = upper ? p[b][i + half] : p[b][i];
            const float send = upper ? p[b][i] : p[b][i + half];
            p[b][i] = keep + __shfl_xor(send, mask, 64);
          }
        }
      if (upper) sel += half;
    }
#pragma unroll
    for (; mask >= 1; mask >>= 1)
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        if (mask == 8) p[b][0] = row_ror_add<8>(p[b][0]);
        else if (mask == 4) p[b][0] = row_ror_add<4>(p[b][0]);
        else if (mask == 2) p[b][0] = row_ror_add<2>(p[b][0]);
        else if (mask == 1) p[b][0] = row_ror_add<1>(p[b][0]);
        else p[b][0] += __shfl_xor(p[b][0], mask, 64);
      }
    const int v = v0 + sel;
    if (v < V) {
      // every lane of a row group (64 / R lanes) holds the same totals; in
      // sample and logits mode lane j of the group handles batch row j
      const int gl = lane & (64 / R - 1);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        if (b >= B) continue;
        float val = apply_cast(p[b][0], a.reduce_cast);
        if constexpr (MODE == MODE_LOGITS) {
          if (gl == b) store_logit(a, b, v, val);
          continue;
        }
        if constexpr (MODE == MODE_SAMPLE) {
          if (gl != b) continue;
          if (!greedy_row[b]) val = val / tp[b] + gumbel_at(key[b], (uint32_t)v);
        }
        best[b] = max_u64(best[b], argmax_key(val, (uint32_t)v));
      }
    }
  };

  // ring of DEPTH row groups in flight: group i+DEPTH-1 is requested before i is reduced
  // ring of DEPTH * R * KJ 16-byte loads per lane
  constexpr int DEPTH = MODE == MODE_SAMPLE ? (KJ >= 4 || NB > 2 ? 2 : 3) : (NB > 2 ? 2 : kGemvDepth);
  const int n_mine = g_end > g_begin ? (g_end - g_begin + g_step - 1) / g_step : 0;
  auto gid = [&](int i) { return g_begin + i * g_step; };
  u32x4_t ring[DEPTH][R][KJ];
  if constexpr (MODE == MODE_SAMPLE) {
    ring_pipeline<DEPTH>(
        n_mine, [&](auto S, int j) NVJSEL_INLINE { load_grp(ring[decltype(S)::value], gid(j)); },
        [&](auto S, int i) NVJSEL_INLINE { proc_grp(ring[decltype(S)::value], gid(i)); }, finish_prenorm);
  } else {
    // Greedy streams fastest (measured) with the shifting ring: the register
    // copies wait for every outstanding load at the top of each step, so one
    // group is in flight while the previous one is reduced.
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
      if (d < n_mine) load_grp(ring[d], gid(d));
    finish_prenorm();
    for (int i = 0; i < n_mine; ++i) {
      if (i + DEPTH - 1 < n_mine) load_grp(ring[DEPTH - 1], gid(i + DEPTH - 1));
      proc_grp(ring[0], gid(i));
#pragma unroll
      for (int d = 0; d < DEPTH - 1; ++d)
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int j = 0; j < KJ; ++j) ring[d][r][j] = ring[d + 1][r][j];
    }
  }
  if constexpr (MODE == MODE_LOGITS) return;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    best[b] = wave_max_u64(best[b]);
    if (lane == 0) red[wave * NB + b] = best[b];
  }
  block_commit<WAVES, NB>(red, B, a.row_keys);
  finish_rows(a.row_keys, a.counter, B, a.out_ids, a.out_best);
}

// ------------------------------------------------------------------ [H, V] streaming kernel
// Weight stored [H, V] bf16 or f16 (WT), vocabulary contiguous: the reference's
// materialised lm_head operand (nanovllm_jax/load_weights.py:256-258; the
// layout lm_head_triton.py:51-55 reads), B <= 8, activations of any dtype
// (fp32 activations multiply exactly: every product and sum is fp32).
// A block owns a 512-column vocabulary strip; wave w of WAVES takes the
// k-slice [w * H / WAVES, (w + 1) * H / WAVES).  Lane l loads 16 bytes
// (columns 8 l .. 8 l + 7) of every W row of its slice, so each load
// instruction of a wave reads 1 KB of one row, contiguous, and (DEPTH - 1) *
// KU rows are in flight per wave; acc[b][c] += h[b][k] * W[k][col + c] in
// fp32, with h broadcast from LDS.  The slices' partial sums meet in LDS,
// summed in slice order, and each thread then scores two columns of every row.
// VEC8: rows of whole, aligned 16-byte groups (V % 8 == 0).  Else any V >= 8:
// rows start at any element, so the loads are 16 bytes from any element
// address (one instruction; V = 50,257, H = 768, B = 4 sampled 1700 -> 23 us
// against one thread per column).  A group that ends past its row reads on into
// the next one (those columns are never scored); in the last row it is loaded
// from V - 8 and moved down.  One body for both cost the aligned rows up to 50%
// (V = 32,000, H = 1024, f32 B = 1 / 8 38.9 / 72.8 us against 29.1 / 63.8; V =
// 98,304, bf16 B = 8 46.7 against 42.9).
template <int WT, int NB, int WAVES, int MODE, bool DOTP, bool VEC8>
__global__ void __launch_bounds__(WAVES * 64) lm_head_hv_kernel(LmArgs a) {
  // DOT (bf16 hidden, a k-slice of even length): the hidden sits in LDS as
  // bf16 pairs (k, k+1) and each pair of W rows is packed per column with
  // v_perm, so one v_dot2c_f32_bf16 does two multiply-adds (products exact,
  // fp32 sums): half the VALU work per weight element
  constexpr bool DOT = DOTP;
  constexpr int KU = 4;
  constexpr int DEPTH = NB <= 2 ? 6 : 4;
  constexpr int STRIP = 512;
  extern __shared__ float lds_f[];  // hidden [H][NB], then partial sums [WAVES][NB][STRIP]
  __shared__ unsigned long long red[WAVES * NB];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int H = a.H, V = a.V, B = a.B;
  const int vb = blockIdx.x * STRIP;
  // groups wholly past the row end: any columns (VEC8: the last group)
  const int col = VEC8 ? min(vb + lane * 8, V - 8) : vb + lane * 8 < V ? vb + lane * 8 : V - 8;
  const int over = VEC8 ? 0 : max(col - (V - 8), 0);  // elements of the group past the row end
  if constexpr (DOT) {
    uint32_t* lds_p = (uint32_t*)lds_f;  // [H / 2][NB] bf16 pairs
    const uint16_t* hs = (const uint16_t*)a.hidden;
    for (int i = threadIdx.x; i < (H / 2) * NB; i += WAVES * 64) {
      const int kp = i / NB, b = i - kp * NB;
      lds_p[i] = b < B ? ((uint32_t)hs[(size_t)b * H + 2 * kp] | ((uint32_t)hs[(size_t)b * H + 2 * kp + 1] << 16)) : 0u;
    }
  } else {
    for (int i = threadIdx.x; i < H * NB; i += WAVES * 64) {
      const int k = i / NB, b = i - k * NB;
      lds_f[i] = b < B ? load_as_f32(a.hidden, a.hidden_dtype, (size_t)b * H + k) : 0.0f;
    }
  }
  float tp[NB];
  bool greedy_row[NB];
  TfKey key[NB];
  if constexpr (MODE == MODE_SAMPLE) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const float t = (b < B) ? a.temperature[b] : 0.0f;
      greedy_row[b] = (t <= 0.0f);
      tp[b] = temp_floor(t);
      key[b] = (b < B) ? tf_key(a.keys[2 * b], a.keys[2 * b + 1]) : tf_key(0u, 0u);
    }
  }
  __syncthreads();
  const int kper = (H + WAVES - 1) / WAVES;
  const int k0 = min(H, wave * kper), k1 = min(H, k0 + kper);
  const int nsteps = (k1 - k0 + KU - 1) / KU;
  const uint16_t* W = (const uint16_t*)a.W;
  float acc[NB][8];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[b][c] = 0.0f;
  u32x4_t ring[DEPTH][KU];
  ring_pipeline<DEPTH>(
      nsteps,
      [&](auto S, int j) NVJSEL_INLINE {
#pragma unroll
        for (int u = 0; u < KU; ++u) {
          const int k = min(k0 + j * KU + u, k1 - 1);
          if constexpr (VEC8) {
            ring[decltype(S)::value][u] = stream_load((const u32x4_t*)(W + (size_t)k * V + col));
          } else {
            const int c = k == H - 1 ? col - over : col;
            ring[decltype(S)::value][u] = __builtin_nontemporal_load((const u32x4_any_t*)(W + (size_t)k * V + c));
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      },
      [&](auto S, int i) NVJSEL_INLINE {
        if constexpr (DOT) {
#pragma unroll
          for (int u = 0; u < KU; u += 2) {
            const int k = k0 + i * KU + u;
            if (k >= k1) continue;  // wave-uniform; the slice length is even
            u32x4_t w0 = ring[decltype(S)::value][u], w1 = ring[decltype(S)::value][u + 1];
            if (!VEC8 && k + 1 == H - 1) w1 = shift_down8(w1, over);  // (H is even)
            const uint32_t q0[4] = {w0.x, w0.y, w0.z, w0.w}, q1[4] = {w1.x, w1.y, w1.z, w1.w};
            uint32_t wp[8];  // column c: (W[k][c], W[k+1][c]) as a bf16 pair
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              wp[2 * e] = __builtin_amdgcn_perm(q1[e], q0[e], 0x05040100u);
              wp[2 * e + 1] = __builtin_amdgcn_perm(q1[e], q0[e], 0x07060302u);
            }
            const uint32_t* hk = (const uint32_t*)lds_f + (k >> 1) * NB;
#pragma unroll
            for (int b = 0; b < NB; ++b) {
              const bf16x2_t h = __builtin_bit_cast(bf16x2_t, hk[b]);
#pragma unroll
              for (int c = 0; c < 8; ++c)
                acc[b][c] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, wp[c]), h, acc[b][c], false);
            }
          }
          return;
        }
#pragma unroll
        for (int u = 0; u < KU; ++u) {
          const int k = k0 + i * KU + u;
          if (k >= k1) continue;  // wave-uniform (last step of the slice)
          u32x4_t w = ring[decltype(S)::value][u];
          if (!VEC8 && k == H - 1) w = shift_down8(w, over);
          const uint32_t q[4] = {w.x, w.y, w.z, w.w};
          float wf[8];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            wf[2 * e] = WT == DT_BF16 ? __uint_as_float(q[e] << 16) : f16_to_f32((uint16_t)(q[e] & 0xFFFFu));
            wf[2 * e + 1] = WT == DT_BF16 ? __uint_as_float(q[e] & 0xFFFF0000u) : f16_to_f32((uint16_t)(q[e] >> 16));
          }
          const float* hk = lds_f + k * NB;
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            const float h = hk[b];
#pragma unroll
            for (int c = 0; c < 8; ++c) acc[b][c] = fmaf(h, wf[c], acc[b][c]);
          }
        }
      });
  __syncthreads();  // the hidden is dead: the LDS takes the partial sums
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int c = 0; c < 8; ++c) lds_f[(wave * NB + b) * STRIP + lane * 8 + c] = acc[b][c];
  __syncthreads();
  unsigned long long best[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) best[b] = 0;
  for (int cc = threadIdx.x; cc < STRIP; cc += WAVES * 64) {
    const int v = vb + cc;
    if (v >= V) continue;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (b >= B) continue;
      float sum = lds_f[b * STRIP + cc];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) sum += lds_f[(w * NB + b) * STRIP + cc];
      float val = apply_cast(sum, a.reduce_cast);
      if constexpr (MODE == MODE_LOGITS) {
        store_logit(a, b, v, val);
        continue;
      }
      if constexpr (MODE == MODE_SAMPLE) {
        if (!greedy_row[b]) val = val / tp[b] + gumbel_at(key[b], (uint32_t)v);
      }
      best[b] = max_u64(best[b], argmax_key(val, (uint32_t)v));
    }
  }
  if constexpr (MODE == MODE_LOGITS) return;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    best[b] = wave_max_u64(best[b]);
    if (lane == 0) red[wave * NB + b] = best[b];
  }
  block_commit<WAVES, NB>(red, B, a.row_keys);
  finish_rows(a.row_keys, a.counter, B, a.out_ids, a.out_best);
}

// ------------------------------------------------------------------ LDS-staged MFMA tile kernel
// bf16 hidden x bf16 W [V, 1024], 3 <= B <= 64.  A block holds GW "GEMM" waves
// and NB "epilogue" waves.
//  * GEMM waves load each 16-row W tile (32 KB, contiguous) with 16-byte loads
//    covering 4 KB per block instruction -- the streaming pattern -- keeping
//    DEPTH-1 tiles in flight in a register ring, and store it to LDS in
//    A-fragment order (row XOR-swizzled so both the stores and the 16-lane
//    fragment reads are conflict-free).  Hidden fragments stay in registers:
//    GEMM wave w owns batch tile w % NB and k-steps [(w / NB) * KPW, +KPW), and
//    leaves its k-split partial sums of tile i in an LDS ring.
//  * Epilogue waves meanwhile sum, cast and score tile i-1.  Epilogue lane L
//    (of NB * 64) owns batch row L % (NB * 16) and vocabulary rows
//    4 * (L / (NB * 16)) .. +3 of every tile.  Sample mode scores with the
//    hardware log and rescores exactly (fp64 logs), a wave at a time, only the
//    entries that can still be a row's maximum.
// One barrier per tile orders both rings, so a tile costs max(GEMM, epilogue)
// rather than their sum, and the epilogue's VALU work (Threefry + logs) runs
// beside the GEMM waves' LDS, MFMA and memory waits on the same SIMDs.
// PN: the final RMSNorm prologue is compiled in (a.prenorm set); kept out of
// the plain kernel so its registers do not constrain the main loops.
template <int NB, int GW, int MODE, int DEPTH, int EPM, bool PN, int NS>
__global__ void __launch_bounds__((GW + NB * EPM) * 64) lm_head_tile_kernel(LmArgs a) {
  constexpr int EW = NB * EPM;     // epilogue waves
  constexpr int EPL = 4 / EPM;     // vocabulary rows per epilogue lane per tile
  static_assert(EPM == 1 || EPM == 2, "one or two epilogue waves per batch tile");
  constexpr int NT = (GW + EW) * 64;
  constexpr int NTG = GW * 64;
  constexpr int KSPLIT = GW / NB;
  static_assert(KSPLIT >= 1 && GW % NB == 0, "GEMM waves split k evenly");
  constexpr int KS = 32;  // 32-wide k-steps of H = 1024
  constexpr int KPW = KS / KSPLIT;
  static_assert(KS % KSPLIT == 0, "k-steps split evenly");
  constexpr int LPT = 2048 / NTG;  // 16-byte loads per GEMM thread per 32 KB tile
  static_assert(2048 % NTG == 0, "tile loads split evenly");
  constexpr int ROWS = NB * 16;    // batch rows of the block
  // per-epilogue-wave queue of entries that may be their row's maximum; it is
  // filtered against the rows' current approximate maxima when it fills and
  // at the end, and only the survivors are rescored exactly
  constexpr int QCAP = kTileQcap * 4 / (EW > 4 ? EW : 4);  // LDS: 12 B per entry
  static_assert(QCAP >= 2 * 64 * EPL, "room for a filtered queue plus one tile");
  __shared__ u32x4_t wt[2][16 * 128];
  __shared__ f32x4_t part[2][KSPLIT * NB * 64];
  __shared__ float qx[MODE == MODE_SAMPLE ? EW : 1][QCAP];
  __shared__ uint32_t qv[MODE == MODE_SAMPLE ? EW : 1][QCAP];
  __shared__ float qa[MODE == MODE_SAMPLE ? EW : 1][QCAP];
  __shared__ unsigned long long qbest[MODE == MODE_SAMPLE ? EW : 1][64];
  __shared__ unsigned long long red[EW * 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool gemm = wave < GW;
  const int B = a.B, V = a.V;
  const uint16_t* W = (const uint16_t*)a.W;
  const int ntiles = (V + 15) >> 4;
  const int grid = gridDim.x;
  const int my_tiles = blockIdx.x < ntiles ? (ntiles - blockIdx.x + grid - 1) / grid : 0;

  // ---- GEMM-wave state
  const int g = lane >> 4, r = lane & 15;
  const int nb = wave % NB, ks = wave / NB;  // meaningful for GEMM waves
  u32x4_t hb[NS][KPW];  // hidden fragments: NS bf16 terms (3 split an fp32 value exactly)
  u32x4_t ring[DEPTH][LPT];
  // ---- epilogue-wave state
  const int ew = wave - GW;                      // epilogue wave index
  const int el = (ew < 0 ? 0 : ew) * 64 + lane;  // epilogue lane id
  const int erow = el % ROWS, evq = el / ROWS;   // batch row, vocab run (EPL rows)
  float tp = 1.0f, rtp = 1.0f;
  bool greedy_row = true;
  TfKey key = tf_key(0u, 0u);
  unsigned long long best = 0;
  float amax = -INFINITY;
  uint32_t qcount = 0;  // wave-uniform: entries in this epilogue wave's queue

  auto load_tile = [&](u32x4_t(&dst)[LPT], int i) NVJSEL_INLINE {
    const int tile = blockIdx.x + i * grid;
#pragma unroll
    for (int u = 0; u < LPT; ++u) {
      const int c = tid + NTG * u;
      int row = tile * 16 + (c >> 7);
      row = row < V ? row : V - 1;
      dst[u] = stream_load((const u32x4_t*)(W + (size_t)row * 1024) + (c & 127));
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // exact scores of the queued elements, a full wave at a time; an entry holds
  // the logit and (vocab << 6 | lane that found it); results fold into qbest[lane]
  auto flush = [&]() {
    if constexpr (MODE == MODE_SAMPLE) {
      const uint32_t n = qcount;
      for (uint32_t e0 = 0; e0 < n; e0 += 64) {  // wave-uniform trip count
        const uint32_t e = e0 + lane;
        const bool live = e < n;
        const uint32_t pv = live ? qv[ew][e] : 0u;
        const uint32_t v = pv >> 6, src = pv & 63u;
        // the shuffles run with the whole wave active
        const TfKey k2{(uint32_t)__shfl((int)key.k0, (int)src, 64), (uint32_t)__shfl((int)key.k1, (int)src, 64),
                       (uint32_t)__shfl((int)key.k2, (int)src, 64)};
        const float t2 = __shfl(tp, (int)src, 64);
        if (live) atomicMax(&qbest[ew][src], argmax_key(qx[ew][e] / t2 + gumbel_at(k2, v), v));
      }
      qcount = 0;
    }
  };
  // drops the queued entries that can no longer be their row's maximum: an
  // entry (approximate score a) survives while a + slack(a, m) >= m for the
  // current maximum m of the lane that queued it -- the test it passed when
  // it was queued, against a maximum that has only grown since.  Compaction
  // in place: a wave reads each 64-entry group before writing survivors at or
  // below it.
  auto compact = [&]() {
    if constexpr (MODE == MODE_SAMPLE) {
      uint32_t nk = 0;
      for (uint32_t e0 = 0; e0 < qcount; e0 += 64) {  // wave-uniform trip count
        const uint32_t e = e0 + lane;
        const bool live = e < qcount;
        const float x = live ? qx[ew][e] : 0.0f;
        const float ap = live ? qa[ew][e] : -INFINITY;
        const uint32_t pv = live ? qv[ew][e] : 0u;
        const float am = __shfl(amax, (int)(pv & 63u), 64);
        const bool keep = live && !(ap + score_slack(ap, am) < am);
        const unsigned long long m = __ballot(keep);
        if (keep) {
          const uint32_t slot = nk + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
          qx[ew][slot] = x;
          qa[ew][slot] = ap;
          qv[ew][slot] = pv;
        }
        nk += (uint32_t)__popcll(m);
      }
      qcount = nk;
    }
  };

  __shared__ float pre_ss[KSPLIT][ROWS];
  // prologue with a 16-byte-aligned bf16 pre-norm hidden (block-uniform)
  const bool raw16 = PN && a.hidden_dtype == DT_BF16 && (((uintptr_t)a.hidden) & 15) == 0;
  if (gemm) {
    const int brow = nb * 16 + r;
    if constexpr (!PN && NS == 1) {
      const uint16_t* hp = (const uint16_t*)a.hidden + (size_t)(brow < B ? brow : 0) * 1024;
#pragma unroll
      for (int kk = 0; kk < KPW; ++kk) {
        const int kb = ks * KPW + kk;
        hb[0][kk] = brow < B ? *(const u32x4_t*)(hp + kb * 32 + g * 8) : u32x4_t{0u, 0u, 0u, 0u};
      }
    } else if constexpr (!PN) {
      static_for<KPW>([&](auto KK) NVJSEL_INLINE {
        constexpr int kk = decltype(KK)::value;
        float v[8];
        load8_as_f32(a.hidden, a.hidden_dtype, (size_t)(brow < B ? brow : 0) * 1024 + (ks * KPW + kk) * 32 + g * 8, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = brow < B ? v[e] : 0.0f;
        split_terms<NS>(v, hb, kk);
      });
    } else {
      // RMSNorm prologue, pass 1: this lane's sum of squares; the four lanes
      // of a row combine by butterfly, the k-split waves through LDS
      float ss = 0.0f;
      const size_t rb = (size_t)(brow < B ? brow : 0) * 1024;  // rows past B: any row, unused
      if (raw16) {
        // bf16 hidden: the raw fragments go straight into hb (all loads in
        // flight at once); pass 2 normalises them in place
#pragma unroll
        for (int kk = 0; kk < KPW; ++kk)
          hb[0][kk] = *(const u32x4_t*)((const uint16_t*)a.hidden + rb + (ks * KPW + kk) * 32 + g * 8);
#pragma unroll
        for (int kk = 0; kk < KPW; ++kk)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float lo = __uint_as_float(hb[0][kk][e] << 16), hi = __uint_as_float(hb[0][kk][e] & 0xFFFF0000u);
            ss = fmaf(lo, lo, ss);
            ss = fmaf(hi, hi, ss);
          }
      } else {
#pragma unroll 4
        for (int kk = 0; kk < KPW; ++kk) {
          float x[8];
          load8_as_f32(a.hidden, a.hidden_dtype, rb + (ks * KPW + kk) * 32 + g * 8, x);
#pragma unroll
          for (int e = 0; e < 8; ++e) ss = fmaf(x[e], x[e], ss);
        }
      }
      if (brow >= B) ss = 0.0f;
      ss += __shfl_xor(ss, 16, 64);
      ss += __shfl_xor(ss, 32, 64);
      if (g == 0) pre_ss[ks][brow] = ss;
    }
  } else {
    if constexpr (MODE == MODE_SAMPLE) {
      const float t = erow < B ? a.temperature[erow] : 0.0f;
      greedy_row = (t <= 0.0f);
      tp = temp_floor(t);
      rtp = 1.0f / tp;
      if (erow < B) key = tf_key(a.keys[2 * erow], a.keys[2 * erow + 1]);
      qbest[ew][lane] = 0;
    }
  }

  // The two roles run separate loops with one barrier per iteration each
  // (my_tiles + 1 of them), so neither keeps the other's registers live.  The
  // barrier orders: W(i) stores before its fragment reads; partials of tile i-1
  // before the epilogue reads them; every read of a slot before it is rewritten.
  // pass 2 of the RMSNorm prologue (GEMM waves), run once the first W tiles
  // are in flight; its barrier pairs with the epilogue waves' first one
  auto finish_prenorm = [&]() NVJSEL_INLINE {
    if constexpr (!PN) return;
    __syncthreads();  // the row sums are in LDS
    // pass 2: normalise, round, pack this lane's fragments
    const int brow = nb * 16 + r;
    float tot = 0.0f;
#pragma unroll
    for (int s2 = 0; s2 < KSPLIT; ++s2) tot += pre_ss[s2][brow];
    const float inv = prenorm_inv(a, tot);
    // compile-time k-steps (a plain loop was left partly rolled, which put
    // the fragment array in scratch memory for the whole tile loop)
    static_for<KPW>([&](auto KK) NVJSEL_INLINE {
      constexpr int kk = decltype(KK)::value;
      const int k0 = (ks * KPW + kk) * 32 + g * 8;
      float v[8], w[8];
      if (raw16) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[2 * e] = __uint_as_float(hb[0][kk][e] << 16);
          v[2 * e + 1] = __uint_as_float(hb[0][kk][e] & 0xFFFF0000u);
        }
      } else {
        load8_as_f32(a.hidden, a.hidden_dtype, (size_t)(brow < B ? brow : 0) * 1024 + k0, v);
      }
      load8_as_f32(a.norm_w, a.norm_dtype, (size_t)k0, w);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = brow < B ? prenorm_apply_w(a, v[e], inv, w[e]) : 0.0f;
      split_terms<NS>(v, hb, kk);
    });
  };

  if (gemm) {
    ring_pipeline<DEPTH>(my_tiles, [&](auto S, int j) NVJSEL_INLINE { load_tile(ring[decltype(S)::value], j); },
                         [&](auto S, int i) NVJSEL_INLINE {
      u32x4_t* buf = wt[i & 1];
#pragma unroll
      for (int u = 0; u < LPT; ++u) {
        const int c = tid + NTG * u;
        const int row = c >> 7, q = c & 127;
        buf[q * 16 + (row ^ (q & 15))] = ring[decltype(S)::value][u];
      }
      __syncthreads();
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KPW; ++kk) {
        const int q = (ks * KPW + kk) * 4 + g;
        const u32x4_t af = buf[q * 16 + (r ^ (q & 15))];
#pragma unroll
        for (int t = 0; t < NS; ++t) acc = mfma16x16x32<DT_BF16>(af, hb[t][kk], acc);
      }
      part[i & 1][(ks * NB + nb) * 64 + lane] = acc;
    }, finish_prenorm);
    __syncthreads();  // the epilogue waves' last iteration
  } else {
    if constexpr (PN) __syncthreads();  // pairs with the GEMM waves' prologue barrier
    for (int i = 0; i <= my_tiles; ++i) {
      __syncthreads();
      if (i == 0) continue;
      // tile i-1: sum the k-split partials of (row erow, vocab rows EPL evq + e);
      // GEMM lane (g, r) holds vocab rows 4 g .. 4 g + 3 of batch row r
      const int vr = EPL * evq;
      const int pnb = erow >> 4, pl = (vr >> 2) * 16 + (erow & 15), c0 = vr & 3;
      f32x4_t s = part[(i - 1) & 1][pnb * 64 + pl];
#pragma unroll
      for (int s2 = 1; s2 < KSPLIT; ++s2) {
        const f32x4_t p = part[(i - 1) & 1][(s2 * NB + pnb) * 64 + pl];
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += p[e];
      }
      const int v0 = (blockIdx.x + (i - 1) * grid) * 16 + vr;
      if constexpr (MODE == MODE_SAMPLE) {
        if constexpr (ROWS < 64) {
          // lanes holding the same batch row share their approximate maximum
#pragma unroll
          for (int m = ROWS; m < 64; m <<= 1) amax = fmaxf(amax, __shfl_xor(amax, m, 64));
        }
        if (qcount > (uint32_t)(QCAP - 64 * EPL)) {  // room for this tile
          compact();
          if (qcount > (uint32_t)(QCAP - 64 * EPL)) flush();
        }
      }
      bool q[EPL];
      float xq[EPL], aq[EPL];
#pragma unroll
      for (int e = 0; e < EPL; ++e) q[e] = false;
      if (erow < B) {
        float raw[EPL];
#pragma unroll
        for (int e = 0; e < EPL; ++e) raw[e] = EPL == 4 ? s[e] : (c0 == 0 ? s[e] : s[e + 2]);
        if constexpr (MODE == MODE_LOGITS) {
#pragma unroll
          for (int e = 0; e < EPL; ++e)
            if (v0 + e < V) store_logit(a, erow, v0 + e, apply_cast(raw[e], a.reduce_cast));
        } else {
          score_run<MODE, EPL>(raw, v0, V, a.reduce_cast, greedy_row, rtp, tp, key, amax, best, q, xq, aq);
        }
      }
      if constexpr (MODE == MODE_SAMPLE) {
        // queue the marked entries with the whole wave active: slots from a
        // ballot, no LDS counter
        bool anyq = false;
#pragma unroll
        for (int e = 0; e < EPL; ++e) anyq |= q[e];
        if (__any(anyq)) {
#pragma unroll
          for (int e = 0; e < EPL; ++e) {
            const unsigned long long m = __ballot(q[e]);
            if (q[e]) {
              const uint32_t slot = qcount + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                       __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
              qx[ew][slot] = xq[e];
              qa[ew][slot] = aq[e];
              qv[ew][slot] = ((uint32_t)(v0 + e) << 6) | (uint32_t)lane;
            }
            qcount += (uint32_t)__popcll(m);
          }
        }
      }
    }
  }
  if constexpr (MODE == MODE_LOGITS) return;
  if (!gemm) {
    if constexpr (MODE == MODE_SAMPLE) {
      compact();
      flush();
      if (!greedy_row) best = max_u64(best, qbest[ew][lane]);
    }
    red[el] = best;
  }
  __syncthreads();
  for (int b = tid; b < B && b < ROWS; b += NT) {
    unsigned long long m = 0;
#pragma unroll
    for (int q = 0; q < 4 * EPM; ++q) m = max_u64(m, red[q * ROWS + b]);
    if (m) (void)after(atomicMax(&a.row_keys[b], m));
  }
  finish_rows(a.row_keys, a.counter, B, a.out_ids, a.out_best);
}

static constexpr int kTileDepth = 2;  // W tiles in flight per block (registers)
static constexpr int kTileW1 = 4;  // waves per block by batch tiles: 1, 2, 4
static constexpr int kTileW2 = 8;
static constexpr int kTileW4 = 8;
static constexpr int kTileBpc = 1;  // blocks per CU of the tile kernel

template <int NB, int GW, int MODE, int NS>
static int launch_tile(const LmArgs& a, hipStream_t stream) {
  // a second epilogue wave per batch tile (sample mode; measured B=32 91 ->
  // 81 us, B=64 125 -> 118 us): two waves per SIMD issue the draws
  constexpr int EPM = (MODE == MODE_SAMPLE && NB >= 2) ? 2 : 1;
  // (the fused prologue of bf16 activations: up to kTilePrenormRows rows)
  constexpr bool kFused = MODE != MODE_LOGITS && (NS == 3 || NB <= 2);
  auto kern = lm_head_tile_kernel<NB, GW, MODE, kTileDepth, EPM, false, NS>;
  if (a.prenorm) {
    if constexpr (kFused) kern = lm_head_tile_kernel<NB, GW, MODE, kTileDepth, EPM, true, NS>;
    else return fail(NVJSEL_EINVAL, "launch_tile: no such variant");
  }
  int grid = kTileBpc * device_cu_count();
  const int ntiles = (a.V + 15) / 16;
  if (grid > ntiles) grid = ntiles;
  hipLaunchKernelGGL(kern, dim3(grid), dim3((GW + NB * EPM) * 64), 0, stream, a);
  NVJSEL_CHECK_LAUNCH("lm_head_tile_kernel");
  return NVJSEL_OK;
}

// Activations other than bf16 (a.act_dtype f32 / f16) take three bf16 terms
// per value, in launches of at most 16 rows (the terms' registers: 32 rows
// per block would spill).
template <int MODE>
static int dispatch_tile(const LmArgs& a, hipStream_t s) {
  if (a.act_dtype != DT_BF16) return launch_tile<1, kTileW1, MODE, 3>(a, s);
  if (a.B <= 16) return launch_tile<1, kTileW1, MODE, 1>(a, s);
  if (a.B <= 32) return launch_tile<2, kTileW2, MODE, 1>(a, s);
  return launch_tile<4, kTileW4, MODE, 1>(a, s);
}

// ------------------------------------------------------------------ generic kernel
// One vocabulary entry per thread, every batch row, any dtype/layout.
template <int MODE>
__global__ void __launch_bounds__(256) lm_head_generic_kernel(LmArgs a) {
  __shared__ unsigned long long red[4 * 64];
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  auto logit = [&](int b) {
    float acc = 0.0f;
    for (int kk = 0; kk < a.H; ++kk) {
      size_t wi = (a.layout == NVJSEL_W_VH) ? (size_t)v * a.H + kk : (size_t)kk * a.V + v;
      acc = fmaf(load_as_f32(a.hidden, a.hidden_dtype, (size_t)b * a.H + kk), load_as_f32(a.W, a.weight_dtype, wi),
                 acc);
    }
    return apply_cast(acc, a.reduce_cast);
  };
  if constexpr (MODE == MODE_LOGITS) {
    if (v < a.V)
      for (int b = 0; b < a.B; ++b) store_logit(a, b, v, logit(b));
    return;
  }
  for (int b0 = 0; b0 < a.B; b0 += 64) {
    const int nb = min(64, a.B - b0);
    for (int bb = 0; bb < nb; ++bb) {
      const int b = b0 + bb;
      unsigned long long k = 0;
      if (v < a.V) {
        float val = logit(b);
        if constexpr (MODE == MODE_SAMPLE) {
          float t = a.temperature[b];
          if (!(t <= 0.0f))
            val = val / temp_floor(t) + gumbel_at(tf_key(a.keys[2 * b], a.keys[2 * b + 1]), (uint32_t)v);
        }
        k = argmax_key(val, (uint32_t)v);
      }
      k = wave_max_u64(k);
      if (lane == 0) red[wave * 64 + bb] = k;
    }
    __syncthreads();
    for (int bb = threadIdx.x; bb < nb; bb += blockDim.x) {
      unsigned long long m = 0;
      for (int w = 0; w < 4; ++w) m = max_u64(m, red[w * 64 + bb]);
      if (m) (void)after(atomicMax(&a.row_keys[b0 + bb], m));
    }
    __syncthreads();
  }
  finish_rows(a.row_keys, a.counter, a.B, a.out_ids, a.out_best);
}

// ------------------------------------------------------------------ RMSNorm prologue kernel
// For the paths without a fused prologue: one block per row writes the
// activation-typed normalised hidden (same arithmetic as prenorm_apply) into
// the workspace, and the LM-head kernel reads it as its hidden.
__global__ void __launch_bounds__(256) lm_prenorm_kernel(LmArgs a, void* out) {
  __shared__ float wsum[4];
  const int b = blockIdx.x, H = a.H;
  float ss = 0.0f;
  for (int k = threadIdx.x; k < H; k += 256) {
    const float x = load_as_f32(a.hidden, a.hidden_dtype, (size_t)b * H + k);
    ss = fmaf(x, x, ss);
  }
  for (int m = 32; m >= 1; m >>= 1) ss += __shfl_xor(ss, m, 64);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float inv = prenorm_inv(a, (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]));
  for (int k = threadIdx.x; k < H; k += 256) {
    const float y = prenorm_apply(a, load_as_f32(a.hidden, a.hidden_dtype, (size_t)b * H + k), inv, k);
    const size_t i = (size_t)b * H + k;
    if (a.act_dtype == DT_F32) ((float*)out)[i] = y;
    else if (a.act_dtype == DT_BF16) ((uint16_t*)out)[i] = (uint16_t)bf16_bits_rne(y);
    else ((uint16_t*)out)[i] = (uint16_t)f16_bits(y);
  }
}

// Re-zeroes n 32-bit words (the prologue rows in the workspace), keeping the
// workspace zero at rest for the next call whatever its shape.
__global__ void __launch_bounds__(256) lm_zero_kernel(uint32_t* p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = 0u;
}

// ------------------------------------------------------------------ host side
static constexpr int kWaves = kLmWaves;
// LDS reserved for the kernel's static shared variables (finish_rows flag).
static constexpr size_t kStaticLdsSlack = 256;

template <int WT, int NSPLIT, int NB, int KU, int MODE>
static int launch_mfma_ku(const LmArgs& a, hipStream_t stream) {
  constexpr int MT = (NB == 1) ? kLmMt1 : kLmMtn;
  auto kern = lm_head_mfma_kernel<WT, NSPLIT, NB, MT, kWaves, KU, kLmDepth, MODE>;
  size_t lds = (size_t)a.H * NSPLIT * NB * 16 * 2;
  size_t red = (size_t)kWaves * NB * 16 * 8;
  if (lds < red) lds = red;
  if (lds > 64 * 1024) {
    NVJSEL_CHECK_HIP(hipFuncSetAttribute((const void*)kern,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  }
  int per_cu = 0;
  NVJSEL_CHECK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kWaves * 64, lds));
  if (per_cu < 1) per_cu = 1;
  if (kLmBpc > 0 && per_cu > kLmBpc) per_cu = kLmBpc;
  const int rows = 16 * MT * kWaves;
  const int need = (a.V + rows - 1) / rows;
  int grid = per_cu * device_cu_count();
  if (grid > need) grid = need;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(kWaves * 64), lds, stream, a);
  NVJSEL_CHECK_LAUNCH("lm_head_mfma_kernel");
  return NVJSEL_OK;
}

// KU must divide the number of 32-wide k-steps; odd hidden sizes use KU = 1.
template <int WT, int NSPLIT, int NB, int MODE>
static int launch_mfma(const LmArgs& a, hipStream_t stream) {
  if (((a.H >> 5) % kLmKu) == 0) return launch_mfma_ku<WT, NSPLIT, NB, kLmKu, MODE>(a, stream);
  return launch_mfma_ku<WT, NSPLIT, NB, 1, MODE>(a, stream);
}

template <int NB, int KJ, int MODE>
static int launch_gemv(const LmArgs& a, hipStream_t stream) {
  constexpr int R = kGemvR;
  const bool dot = kGemvDot && (a.prenorm ? a.act_dtype == DT_BF16
                                           : a.hidden_dtype == DT_BF16 && (((uintptr_t)a.hidden) & 15) == 0);
  auto kern = dot ? lm_head_gemv_kernel<NB, R, KJ, MODE, true> : lm_head_gemv_kernel<NB, R, KJ, MODE, false>;
  int per_cu = 0;
  constexpr int WAVES = kGemvWaves;
  NVJSEL_CHECK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, WAVES * 64, 0));
  if (per_cu < 1) per_cu = 1;
  if (kGemvBpc > 0 && per_cu > kGemvBpc) per_cu = kGemvBpc;
  const int need = (a.V + R * WAVES - 1) / (R * WAVES);
  int grid = per_cu * device_cu_count();
  if (grid < 1) grid = 1;
  if (grid > need) grid = need;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(WAVES * 64), 0, stream, a);
  NVJSEL_CHECK_LAUNCH("lm_head_gemv_kernel");
  return NVJSEL_OK;
}

template <int MODE>
static int dispatch_gemv(const LmArgs& a, hipStream_t s) {
  const int kj = a.H / 512;
  if (a.B == 1) {
    if (kj == 1) return launch_gemv<1, 1, MODE>(a, s);
    if (kj == 2) return launch_gemv<1, 2, MODE>(a, s);
    return launch_gemv<1, 4, MODE>(a, s);
  }
  if (MODE == MODE_SAMPLE || a.B <= 2) {
    if (kj == 1) return launch_gemv<2, 1, MODE>(a, s);
    if (kj == 2) return launch_gemv<2, 2, MODE>(a, s);
    return launch_gemv<2, 4, MODE>(a, s);
  }
  if constexpr (MODE != MODE_SAMPLE) {  // 3-4 rows: greedy / logits only
    if (kj == 1) return launch_gemv<4, 1, MODE>(a, s);
    if (kj == 2) return launch_gemv<4, 2, MODE>(a, s);
    return launch_gemv<4, 4, MODE>(a, s);
  }
  return NVJSEL_EINVAL;
}

template <int WT, int NSPLIT, int MODE>
static int dispatch_nb(const LmArgs& a, hipStream_t s) {
  const int nb = (a.B + 15) / 16;
  switch (nb) {
    case 1: return launch_mfma<WT, NSPLIT, 1, MODE>(a, s);
    case 2: return launch_mfma<WT, NSPLIT, 2, MODE>(a, s);
    case 3: return launch_mfma<WT, NSPLIT, 3, MODE>(a, s);
    default: return launch_mfma<WT, NSPLIT, 4, MODE>(a, s);
  }
}


static size_t lm_ws_keys_bytes(int batch) { return align_up((size_t)batch * 8, 256); }

// The workspace of every greedy/sample path: per-row keys and the ticket line.
static size_t lm_ws_small_bytes(int batch) {
  return batch <= 0 ? 0 : lm_ws_keys_bytes(batch) + 256;
}
// [V, H] bf16 sampling in the blocked GEMM: above 192 rows, and 129-160 (one
// box, H = 1024: B = 144 / 160 264 / 270 us in the GEMM against 270-279 /
// 280-285 in three tile passes, B = 176 / 192 296-298 / 300 against 318 / 323)
static constexpr int kGemmMinBatchTileSample = 192;
static constexpr int kGemmBandSample = 160;
static constexpr int kTilePrenormRows = 32;  // bf16 activations: the fused prologue of the tile kernel up to here
// [H, V] weights of many strips (hv_gemm_min): the GEMM above 8 rows for bf16 activations (V = 248k, up
// to 64 rows in the narrow layout: ~94-98 us greedy, ~113-143 us sampled,
// against 8-row streaming passes of ~88-100 us each) and for fp32 above 8
// (~168-180 / ~185-218 us against passes of ~97 / ~111 us: B = 12 sampled
// 185 vs 206 us in two passes)
static constexpr int kRing3MaxRows = 192;  // f32 activations on [V, H]: the blocked GEMM above
static constexpr int kMix3MaxBatch = 128;  // f32 activations, 64-row narrow passes up to here
static constexpr int kGemmHvMinBatch = 8, kGemmHvMinBatchSample = 8, kGemm3HvMinBatch = 8, kGemm3HvMinBatchSample = 8;


// Final-RMSNorm prologue request (norm_w == nullptr: hidden is already normed).
struct Prenorm {
  const void* norm_w = nullptr;
  int norm_dtype = DT_F32;
  float eps = 0.0f;
  int act_dtype = DT_F32;
};

static size_t lm_prenorm_bytes(int batch, int H) { return align_up((size_t)batch * H * 4, 256); }

static constexpr bool kHvDot = true;  // bf16 hidden: the v_dot2c_f32_bf16 path

// Dynamic LDS of lm_head_hv_kernel with NB rows: the hidden [H][NB] f32, then
// the partial sums [WAVES][NB][512] f32 (the same bytes, reused).
static size_t hv_lds_bytes(int nb, int H) {
  const int p2 = nb <= 1 ? 1 : nb <= 2 ? 2 : nb <= 4 ? 4 : 8;
  const size_t waves = 4;
  const size_t a = (size_t)H * p2, b = waves * p2 * 512;
  return (a > b ? a : b) * 4;
}

// MODE_LOGITS destination.
struct LogitsOut {
  void* ptr = nullptr;
  int dtype = DT_F32;
  long long stride = 0;
};

template <int WT, int NB, int MODE>
static int launch_hv(const LmArgs& a, hipStream_t stream) {
  constexpr int WAVES = 4;  // measured: 4 waves per block beat 8 and 16 at B = 1 and 8
  auto kern = lm_head_hv_kernel<WT, NB, WAVES, MODE, false, false>;
  if constexpr (WT == DT_BF16) {
    const bool vec8 = (a.V % 8) == 0 && (((uintptr_t)a.W) & 15) == 0;
    if (kHvDot && a.hidden_dtype == DT_BF16 && (a.H % (2 * WAVES)) == 0)
      kern = vec8 ? lm_head_hv_kernel<WT, NB, WAVES, MODE, true, true> : lm_head_hv_kernel<WT, NB, WAVES, MODE, true, false>;
    else if (vec8)
      kern = lm_head_hv_kernel<WT, NB, WAVES, MODE, false, true>;
  }
  const size_t lds = hv_lds_bytes(NB, a.H);
  if (lds > 48 * 1024)
    NVJSEL_CHECK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(kern, dim3((a.V + 511) / 512), dim3(WAVES * 64), lds, stream, a);
  NVJSEL_CHECK_LAUNCH("lm_head_hv_kernel");
  return NVJSEL_OK;
}

template <int WT, int MODE>
static int dispatch_hv_type(const LmArgs& a, hipStream_t s) {
  if (a.B == 1) return launch_hv<WT, 1, MODE>(a, s);
  if (a.B == 2) return launch_hv<WT, 2, MODE>(a, s);
  if (a.B <= 4) return launch_hv<WT, 4, MODE>(a, s);
  return launch_hv<WT, 8, MODE>(a, s);
}

template <int MODE>
static int dispatch_hv(const LmArgs& a, hipStream_t s) {
  return a.weight_dtype == DT_BF16 ? dispatch_hv_type<DT_BF16, MODE>(a, s) : dispatch_hv_type<DT_F16, MODE>(a, s);
}

static int lm_head_entry(int mode, const void* hidden, int hidden_dtype, const void* weight,
                         int weight_dtype, int layout, int batch, int H, int V, int reduce_cast,
                         const float* temperature, const uint32_t* keys, int32_t* out_ids,
                         float* out_best, void* workspace, size_t ws_bytes, void* stream,
                         const Prenorm& pn = Prenorm(), const LogitsOut& lo = LogitsOut()) {
  clear_error();
  const bool prenorm = pn.norm_w != nullptr;
  const char* who = mode == MODE_LOGITS ? "lm_head_logits"
                    : mode == MODE_GREEDY ? (prenorm ? "lm_head_top1_prenorm" : "lm_head_top1")
                                          : (prenorm ? "lm_head_sample_prenorm" : "lm_head_sample");
  if (!hidden || !weight || (mode != MODE_LOGITS && !out_ids) || (mode == MODE_LOGITS && !lo.ptr)) {
    set_error("%s: null hidden/weight/output", who);
    return NVJSEL_EINVAL;
  }
  if (batch <= 0 || H <= 0 || V <= 0) {
    set_error("%s requires non-empty dimensions (batch=%d hidden=%d vocab=%d)", who, batch, H, V);
    return NVJSEL_EINVAL;
  }
  if (V >= 0x7FFFFFFF) { set_error("%s: vocab too large", who); return NVJSEL_EINVAL; }
  if (!valid_dtype(hidden_dtype) || !valid_dtype(weight_dtype)) {
    set_error("%s: unsupported dtype (hidden=%d weight=%d)", who, hidden_dtype, weight_dtype);
    return NVJSEL_EINVAL;
  }
  if (layout != NVJSEL_W_VH && layout != NVJSEL_W_HV) { set_error("%s: bad weight layout %d", who, layout); return NVJSEL_EINVAL; }
  if (reduce_cast < 0 || reduce_cast > 2) { set_error("%s: reduce_cast must be 0, 1 or 2", who); return NVJSEL_EINVAL; }
  if (mode == MODE_SAMPLE && (!temperature || !keys)) { set_error("%s: null temperature/keys", who); return NVJSEL_EINVAL; }
  if (mode == MODE_LOGITS) {
    if (!valid_dtype(lo.dtype)) { set_error("%s: out dtype must be f32, bf16 or f16", who); return NVJSEL_EINVAL; }
    if (lo.stride < V) { set_error("%s: out row stride < vocab", who); return NVJSEL_EINVAL; }
  }
  if (prenorm) {
    if (!valid_dtype(pn.norm_dtype) || !valid_dtype(pn.act_dtype)) {
      set_error("%s: unsupported dtype (norm=%d act=%d)", who, pn.norm_dtype, pn.act_dtype);
      return NVJSEL_EINVAL;
    }
    if (!(pn.eps >= 0.0f)) { set_error("%s: eps must be >= 0", who); return NVJSEL_EINVAL; }
  }
  const size_t need = mode == MODE_LOGITS ? 0 : lm_ws_small_bytes(batch) + (prenorm ? lm_prenorm_bytes(batch, H) : 0);
  if (need && (!workspace || ws_bytes < need)) {
    set_error("%s: workspace %zu bytes < required %zu", who, ws_bytes, need);
    return NVJSEL_EWORKSPACE;
  }
  hipStream_t s = (hipStream_t)stream;
  unsigned long long* row_keys = (unsigned long long*)workspace;
  unsigned int* counter = need ? (unsigned int*)((char*)workspace + lm_ws_keys_bytes(batch)) : nullptr;

  // Paths with a fused prologue: the streaming GEMV and the bf16 tile kernel.
  // Elsewhere the prologue kernel writes the normalised hidden into the
  // workspace first and the LM head reads it.
  const int eff_dtype = prenorm ? pn.act_dtype : hidden_dtype;
  const bool aligned = (((uintptr_t)weight) & 15) == 0;
  const bool bf16_mfma = layout == NVJSEL_W_VH && weight_dtype == NVJSEL_BF16 && (H % 32) == 0 && aligned;
  const bool f16_mfma = layout == NVJSEL_W_VH && weight_dtype == NVJSEL_F16 &&
                        eff_dtype == NVJSEL_F16 && (H % 32) == 0 && aligned;
  const int nsplit = (bf16_mfma && eff_dtype != NVJSEL_BF16) ? 3 : 1;
  // streaming GEMV ([V, H] bf16, any activation; fp32 products on the VALU):
  // greedy / logits up to 2 rows, 4 for activations other than bf16 (fp32 B
  // = 3 / 4 ~76 / ~78-80 us against ~84 in a tile pass; bf16 at 3-4 rows
  // ~92-96 against ~77); sampling where the tile kernel cannot take the call,
  // and for one row of non-bf16 activations (fp32 B = 1 ~82 vs ~84 us; bf16
  // B = 1 / 2 77.5 / 77 us in a tile pass against 80 / 98.5 here, fp32 B = 2
  // 83 vs 113)
  const bool gemv_shape = layout == NVJSEL_W_VH && weight_dtype == NVJSEL_BF16 && aligned &&
                          (H == 512 || H == 1024 || H == 2048);
  const bool tile_shape = bf16_mfma && H == 1024 && (prenorm || (((uintptr_t)hidden) & 15) == 0);
  const bool gemv = gemv_shape && (mode == MODE_SAMPLE
                                       ? batch <= 2 && (!tile_shape || (batch == 1 && eff_dtype != NVJSEL_BF16))
                                       : batch <= 2 || (batch <= 4 && eff_dtype != NVJSEL_BF16));
  // [H, V] 16-bit streaming kernel, up to 8 rows per launch, any V >= 8
  const bool hv = layout == NVJSEL_W_HV && weight_dtype != NVJSEL_F32 && (((uintptr_t)weight) & 1) == 0 && V >= 8 &&
                  hv_lds_bytes(batch < 8 ? batch : 8, H) + kStaticLdsSlack <= device_max_lds_per_block();
  // rows per launch: LDS holds H * nsplit * rows bf16 values
  int chunk = 0;
  if ((bf16_mfma || f16_mfma) && (size_t)H * nsplit * 16 * 2 + kStaticLdsSlack <= device_max_lds_per_block()) {
    size_t per16 = (size_t)H * nsplit * 16 * 2;
    size_t max_lds = device_max_lds_per_block();
    max_lds = max_lds > kStaticLdsSlack ? max_lds - kStaticLdsSlack : 0;
    int tiles = (int)(max_lds / per16);
    if (tiles > 4) tiles = 4;
    if (nsplit == 3 && tiles > 1) tiles = 1;
    chunk = tiles * 16;
  }
  // Staged GEMM on direct LDS loads (lm_head_ring.hip; 16-bit weight and
  // activations of one type).  Greedy and logits above the GEMV's rows: H =
  // 1024, V = 248k, B = 16 / 64 / 100 / 256 76 / 78 / 84 / 131 us against 77 /
  // 78 / 157 / 189 in 64-row tile passes and the blocked GEMM; logits B = 64 /
  // 80 / 256 97 / 110 / 179 against 148 / 246 / 289; H = 2560, V = 152k, B =
  // 16 / 64 120 / 134 against 259 / 1010 in the straight-to-registers kernel.
  // Where the tile kernel takes the shape too, up to 64 rows by the share of W
  // per block (ring_takes_small).  With the norm in the call (a prologue and a
  // zeroing launch, ~11 us) the tile kernel's fused prologue stays up to 32
  // rows (85-88 us; 64 rows 100 against 89).  Sampling: wherever the tile
  // kernel does not take the shape, up to 128 rows per pass; where it does at
  // 65-128 rows by the share (ring_takes_sample; B = 64 117-123 us against
  // 103-106) -- above 128 rows the blocked GEMM's single pass is faster (B =
  // 144 / 256 264 / 340 against 278 / 377), but for the band it leaves.
  const bool ring_ok = layout == NVJSEL_W_VH && aligned && weight_dtype != NVJSEL_F32 && eff_dtype == weight_dtype &&
                       (H % 64) == 0 && (prenorm || (((uintptr_t)hidden) & 15) == 0) &&
                       (mode != MODE_SAMPLE || V < (1 << 25));
  const bool ring1 = !gemv && ring_ok &&
                    (mode == MODE_SAMPLE
                         ? (tile_shape ? batch > 64 && batch <= kRingSampleRows &&
                                             ring_takes_sample(batch, V, device_cu_count())
                                       : batch <= kRingSampleRows || weight_dtype == NVJSEL_F16)
                         : !tile_shape || batch > 64 ||
                               (!(prenorm && batch <= kTilePrenormRows) &&
                                ring_takes_small(mode == MODE_LOGITS, batch, V, device_cu_count())));
  // f32 activations on bf16 [V, H] weights: the same kernel on three bf16
  // terms per value, 64 rows per pass (H = 1024, V = 248k, one box: greedy B =
  // 32 / 64 / 80 / 128 87 / 121 / 203 / 238 us, where 16-row tile passes and
  // 64-row passes of the blocked GEMM took 171 / 183 / 260 / 362; sampled 109 /
  // 172 / 267 / 337 against 177 / 229 / 318 / 447; H = 2048, V = 124k, B = 16
  // 110 us against 17 ms in the generic kernel).  Up to 16 rows at H = 1024 the
  // tile kernel (85 us; sampled 90 against 98-109), and the GEMV for a rest of
  // two; more than 192 rows take the blocked GEMM's 256 per pass (461 us, 616
  // sampled, against 477 / 677)
  const bool ring3 = !gemv && layout == NVJSEL_W_VH && weight_dtype == NVJSEL_BF16 && aligned && (H % 64) == 0 &&
                     eff_dtype == NVJSEL_F32 && (prenorm || (((uintptr_t)hidden) & 15) == 0) &&
                     (mode != MODE_SAMPLE || V < (1 << 25)) && !(tile_shape && batch <= 16);
  const bool ring = ring1 || ring3;
  const bool tile = !gemv && !ring && tile_shape;
  // blocked GEMM: sampling bf16 activations on [V, H] above 128 rows (H =
  // 1024: at 129-160 and above 192), one pass over W per 256 rows (sample
  // mode packs vocabulary ids into 25 bits of its queue entries); [H, V]
  // weights (transposing LDS reads) every mode, above the rows of the [H, V]
  // streaming kernel, which takes 8 per pass over W (hv_gemm_min)
  const bool hv_gemm_ok = layout == NVJSEL_W_HV && V >= 8 && (((uintptr_t)weight) & 1) == 0 &&
                          (weight_dtype == NVJSEL_BF16 || (weight_dtype == NVJSEL_F16 && eff_dtype == NVJSEL_F16));
  const bool gemm_ok = (bf16_mfma || hv_gemm_ok) && (H % (2 * kGemmKC)) == 0 &&
                       (prenorm || (((uintptr_t)hidden) & 15) == 0) && (mode != MODE_SAMPLE || V < (1 << 25));
  // Its 512-column strips leave CUs idle on a small vocabulary (V = 50,257, H
  // = 768, 99 blocks: sampled B = 1 / 4 / 8 30 / 36 / 46 us; the GEMM's 197
  // tiles ~28 at 1-16 rows), and f16 weights have no two-product dot there
  // (V = 128,256, H = 2048, B = 1 / 8 84 / 142 us against 94).  Whole aligned
  // groups of short weights stream faster: greedy / logits of one row at H < 1024
  // (V = 32,000, H = 512 15.9 us against 16.5; H = 1024 26.4 against 23.4),
  // sampled of one row at H < 2048 (H = 1024 / 2048 27.5 / 46 against 30.3 / 44),
  // two at H < 1024 (H = 768 / 1024, B = 2 23.8 / 30.3 against 26.4 / 30.3), four
  // at H < 768 (H = 512, B = 4 / 5 22.4 / 28.3 against 23.7 / 23.6; H = 768, B = 3
  // 27.8 against 26.6)
  const bool hv_vec8 = weight_dtype == NVJSEL_BF16 && aligned && (V % 8) == 0;
  const int hv_small_min = !hv_vec8              ? 0
                           : mode != MODE_SAMPLE ? (H < 1024 ? 1 : 0)
                                                 : (H < 768 ? 4 : H < 1024 ? 2 : H < 2048 ? 1 : 0);
  const int hv_gemm_min = (V + 511) / 512 <= device_cu_count() / 2 ? hv_small_min
                          : weight_dtype == NVJSEL_F16             ? 2
                          : mode == MODE_SAMPLE                    ? kGemmHvMinBatchSample
                                                                   : kGemmHvMinBatch;
  const bool gemm = gemm_ok && !ring && eff_dtype == weight_dtype &&
                    (hv_gemm_ok ? batch > hv_gemm_min
                                : mode == MODE_SAMPLE && batch > kRingSampleRows &&
                                      (!tile || batch > kGemmMinBatchTileSample || batch <= kGemmBandSample));
  // [H, V], f32 activations: the same one-pass GEMM on three bf16 terms per
  // value, from 9 rows; at 65-128 rows passes of 64 rows through its narrow
  // layout while more than 8 rows are left, then a streaming pass (greedy B =
  // 65 / 72 / 96-128 ~262 / ~278 / ~350 us, sampled ~302 / ~333 / ~409-434 us,
  // against ~376-396 / ~494-504 us in the 256-row kernel); where the streaming
  // kernel's LDS does not fit (8 rows from H = 5120) the 256-row kernel takes
  // the whole call
  const bool mix3 = gemm_ok && hv_gemm_ok && hv && eff_dtype == NVJSEL_F32 && batch > 64 && batch <= kMix3MaxBatch;
  const int mix_rest = mode == MODE_SAMPLE ? kGemm3HvMinBatchSample : kGemm3HvMinBatch;
  const bool gemm3 = !mix3 && gemm_ok && hv_gemm_ok && eff_dtype == NVJSEL_F32 && batch > mix_rest;
  const bool fused_prenorm = prenorm && !gemm && !gemm3 && !mix3 &&
                             (gemv || (tile && (eff_dtype != NVJSEL_BF16 || batch <= kTilePrenormRows)));
  if (prenorm && !fused_prenorm) {
    LmArgs p{};
    p.hidden = hidden;
    p.hidden_dtype = hidden_dtype;
    p.H = H;
    p.norm_w = pn.norm_w;
    p.norm_dtype = pn.norm_dtype;
    p.eps = pn.eps;
    p.act_dtype = pn.act_dtype;
    void* normed = (char*)workspace + lm_ws_small_bytes(batch);
    hipLaunchKernelGGL(lm_prenorm_kernel, dim3(batch), dim3(256), 0, s, p, normed);
    NVJSEL_CHECK_LAUNCH("lm_prenorm_kernel");
    hidden = normed;
    hidden_dtype = pn.act_dtype;
  }
  if (tile) chunk = eff_dtype == NVJSEL_BF16 ? 64 : 16;
  if (gemv) chunk = 0;
  if (hv) chunk = 8;
  if (gemm || gemm3) chunk = gemm && weight_dtype == NVJSEL_F16 ? 64 : kGemmBB;
  if (ring1) chunk = mode == MODE_SAMPLE ? kRingSampleRows : kRingRows;
  auto by_mode = [&](auto fn) -> int {
    if (mode == MODE_GREEDY) return fn(std::integral_constant<int, MODE_GREEDY>{});
    if (mode == MODE_SAMPLE) return fn(std::integral_constant<int, MODE_SAMPLE>{});
    return fn(std::integral_constant<int, MODE_LOGITS>{});
  };
  for (int b0 = 0, nb = 0; b0 < batch; b0 += nb) {
    LmArgs a{};
    const int left = batch - b0;
    const bool gv = gemv || (ring3 && left <= 2 && gemv_shape && mode != MODE_SAMPLE);
    const bool t16 = !gv && ring3 && left <= 16 && tile_shape;
    const bool g3 = gemm3 || (mix3 && (b0 == 0 || left > mix_rest)) || (ring3 && left > kRing3MaxRows);
    const int step = ring3  ? (g3 ? kGemmBB : t16 ? 16 : kRingF32Rows)
                     : mix3 ? (g3 ? 64 : chunk)
                            : (chunk > 0 ? chunk : batch);
    nb = left < step ? left : step;
    if (nb <= 0) return fail(NVJSEL_EINVAL, "lm_head: a pass of no rows");  // (every pass above takes some)
    a.W = weight;
    a.hidden = (const char*)hidden + (size_t)b0 * H * dtype_size(hidden_dtype);
    a.hidden_dtype = hidden_dtype;
    a.prenorm = fused_prenorm ? 1 : 0;
    a.norm_w = pn.norm_w;
    a.norm_dtype = pn.norm_dtype;
    a.eps = pn.eps;
    a.act_dtype = fused_prenorm ? pn.act_dtype : hidden_dtype;
    a.weight_dtype = weight_dtype;
    a.layout = layout;
    a.B = nb;
    a.H = H;
    a.V = V;
    a.reduce_cast = reduce_cast;
    a.temperature = temperature ? temperature + b0 : nullptr;
    a.keys = keys ? keys + 2 * (size_t)b0 : nullptr;
    a.row_keys = row_keys ? row_keys + b0 : nullptr;
    a.counter = counter;
    a.out_ids = out_ids ? out_ids + b0 : nullptr;
    a.out_best = out_best ? out_best + b0 : nullptr;
    a.out_logits = lo.ptr ? (char*)lo.ptr + (size_t)b0 * (size_t)lo.stride * (lo.dtype == DT_F32 ? 4 : 2) : nullptr;
    a.out_dtype = lo.dtype;
    a.out_stride = lo.stride;
    int rc;
    if (gemm || g3) {
      rc = launch_gemm(mode, hv_gemm_ok, a, s);
    } else if (ring && !gv && !t16) {
      rc = launch_ring(mode, a, s);
    } else if (gv) {
      rc = by_mode([&](auto M) { return dispatch_gemv<decltype(M)::value>(a, s); });
    } else if (hv) {
      rc = by_mode([&](auto M) { return dispatch_hv<decltype(M)::value>(a, s); });
    } else if (tile || t16) {
      rc = by_mode([&](auto M) { return dispatch_tile<decltype(M)::value>(a, s); });
    } else if (chunk > 0) {
      if (f16_mfma)
        rc = by_mode([&](auto M) { return dispatch_nb<DT_F16, 1, decltype(M)::value>(a, s); });
      else if (nsplit == 1)
        rc = by_mode([&](auto M) { return dispatch_nb<DT_BF16, 1, decltype(M)::value>(a, s); });
      else
        rc = by_mode([&](auto M) { return launch_mfma<DT_BF16, 3, 1, decltype(M)::value>(a, s); });
    } else {
      const int grid = (V + 255) / 256;
      rc = by_mode([&](auto M) -> int {
        hipLaunchKernelGGL(lm_head_generic_kernel<decltype(M)::value>, dim3(grid), dim3(256), 0, s, a);
        NVJSEL_CHECK_LAUNCH("lm_head_generic_kernel");
        return (int)NVJSEL_OK;
      });
    }
    if (rc != NVJSEL_OK) return rc;
  }
  if (prenorm && !fused_prenorm) {
    const size_t words = lm_prenorm_bytes(batch, H) / 4;
    const unsigned grid = (unsigned)((words + 255) / 256 < 1024 ? (words + 255) / 256 : 1024);
    hipLaunchKernelGGL(lm_zero_kernel, dim3(grid), dim3(256), 0, s,
                       (uint32_t*)((char*)workspace + lm_ws_small_bytes(batch)), words);
    NVJSEL_CHECK_LAUNCH("lm_zero_kernel");
  }
  return NVJSEL_OK;
}

// ------------------------------------------------------------------ fixed scratch (no allocation)
// For callers that cannot allocate (code under graph capture, tight serving
// loops): the workspace of nvjsel_lm_head_top1 -- per-row argmax keys and the
// last-block ticket -- lives in a file-scope device array.  Each device holds
// its own copy for the life of the process; host code reaches it only through
// the address hipGetSymbolAddress returns for that device.  It is zeroed once
// per device at set-up and every successful call leaves it zeroed again.
static constexpr int kNoAllocMaxBatch = 4096;
static constexpr size_t kNoAllocScratchBytes = (size_t)kNoAllocMaxBatch * 8 + 256;  // keys + ticket line
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

static std::mutex g_scratch_mu;
static void* g_scratch_ptr[64] = {};

// The current device's scratch address, set up (address lookup + one zero
// fill on `stream`) on the first call on that device.
static int noalloc_scratch(hipStream_t stream, void** out) {
  int dev = 0;
  NVJSEL_CHECK_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) return fail(NVJSEL_EUNSUPPORTED, "lm_head_top1_noalloc: device id >= 64");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    NVJSEL_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return fail(NVJSEL_EHIP, "lm_head_top1_noalloc: no device address for the scratch array");
    // No fill: the array has static storage duration without an initializer,
    // so the code object's loader zero-fills it on every device, and every
    // call leaves it zero again.  (A fill launched here would, on a first call
    // made under graph capture, only be recorded into the graph.)
    (void)stream;
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return NVJSEL_OK;
}

}  // namespace nvjsel

using namespace nvjsel;

extern "C" int nvjsel_lm_head_top1_noalloc(const void* hidden, int hidden_dtype, const void* weight,
                                           int weight_dtype, int weight_layout, int batch, int hidden_dim,
                                           int vocab, int reduce_cast, int32_t* out_ids, float* out_best,
                                           void* stream) {
  clear_error();
  if (batch > kNoAllocMaxBatch) {
    set_error("lm_head_top1_noalloc: batch %d exceeds the fixed scratch's maximum of %d rows", batch,
              kNoAllocMaxBatch);
    return NVJSEL_EUNSUPPORTED;
  }
  if (batch <= 0) {
    set_error("lm_head_top1_noalloc requires non-empty dimensions (batch=%d)", batch);
    return NVJSEL_EINVAL;
  }
  void* ws = nullptr;
  const int rc = noalloc_scratch((hipStream_t)stream, &ws);
  if (rc != NVJSEL_OK) return rc;
  return lm_head_entry(MODE_GREEDY, hidden, hidden_dtype, weight, weight_dtype, weight_layout, batch, hidden_dim,
                       vocab, reduce_cast, nullptr, nullptr, out_ids, out_best, ws, kNoAllocScratchBytes, stream);
}

extern "C" size_t nvjsel_lm_head_workspace_size(int batch) {
  return lm_ws_small_bytes(batch);
}

extern "C" int nvjsel_lm_head_top1(const void* hidden, int hidden_dtype, const void* weight,
                                   int weight_dtype, int weight_layout, int batch, int hidden_dim,
                                   int vocab, int reduce_cast, int32_t* out_ids, float* out_best,
                                   void* workspace, size_t workspace_bytes, void* stream) {
  return lm_head_entry(MODE_GREEDY, hidden, hidden_dtype, weight, weight_dtype, weight_layout, batch,
                       hidden_dim, vocab, reduce_cast, nullptr, nullptr, out_ids, out_best, workspace,
                       workspace_bytes, stream);
}

extern "C" int nvjsel_lm_head_logits(const void* hidden, int hidden_dtype, const void* weight, int weight_dtype,
                                     int weight_layout, int batch, int hidden_dim, int vocab, int reduce_cast,
                                     void* out_logits, int out_dtype, int64_t out_row_stride, void* stream) {
  LogitsOut lo;
  lo.ptr = out_logits;
  lo.dtype = out_dtype;
  lo.stride = out_row_stride;
  return lm_head_entry(MODE_LOGITS, hidden, hidden_dtype, weight, weight_dtype, weight_layout, batch, hidden_dim,
                       vocab, reduce_cast, nullptr, nullptr, nullptr, nullptr, nullptr, 0, stream, Prenorm(), lo);
}

extern "C" size_t nvjsel_lm_head_prenorm_workspace_size(int batch, int hidden_dim) {
  if (batch <= 0 || hidden_dim <= 0) return 0;
  return nvjsel_lm_head_workspace_size(batch) + lm_prenorm_bytes(batch, hidden_dim);
}

extern "C" int nvjsel_rms_norm(const void* hidden, int hidden_dtype, const void* norm_weight, int norm_dtype,
                               float eps, int act_dtype, int batch, int hidden_dim, void* out, void* stream) {
  clear_error();
  if (!hidden || !norm_weight || !out) return fail(NVJSEL_EINVAL, "rms_norm: null pointer");
  if (batch <= 0 || hidden_dim <= 0) return fail(NVJSEL_EINVAL, "rms_norm: empty dimensions");
  if (!valid_dtype(hidden_dtype) || !valid_dtype(norm_dtype) || !valid_dtype(act_dtype))
    return fail(NVJSEL_EINVAL, "rms_norm: unsupported dtype");
  if (!(eps >= 0.0f)) return fail(NVJSEL_EINVAL, "rms_norm: eps must be >= 0");
  LmArgs p{};
  p.hidden = hidden;
  p.hidden_dtype = hidden_dtype;
  p.H = hidden_dim;
  p.norm_w = norm_weight;
  p.norm_dtype = norm_dtype;
  p.eps = eps;
  p.act_dtype = act_dtype;
  hipLaunchKernelGGL(lm_prenorm_kernel, dim3(batch), dim3(256), 0, (hipStream_t)stream, p, out);
  NVJSEL_CHECK_LAUNCH("lm_prenorm_kernel");
  return NVJSEL_OK;
}

extern "C" int nvjsel_lm_head_top1_prenorm(const void* hidden, int hidden_dtype, const void* norm_weight,
                                           int norm_dtype, float eps, int act_dtype, const void* weight,
                                           int weight_dtype, int weight_layout, int batch, int hidden_dim,
                                           int vocab, int reduce_cast, int32_t* out_ids, float* out_best,
                                           void* workspace, size_t workspace_bytes, void* stream) {
  if (!norm_weight) { clear_error(); set_error("lm_head_top1_prenorm: null norm_weight"); return NVJSEL_EINVAL; }
  Prenorm pn;
  pn.norm_w = norm_weight;
  pn.norm_dtype = norm_dtype;
  pn.eps = eps;
  pn.act_dtype = act_dtype;
  return lm_head_entry(MODE_GREEDY, hidden, hidden_dtype, weight, weight_dtype, weight_layout, batch,
                       hidden_dim, vocab, reduce_cast, nullptr, nullptr, out_ids, out_best, workspace,
                       workspace_bytes, stream, pn);
}

extern "C" int nvjsel_lm_head_sample_prenorm(const void* hidden, int hidden_dtype, const void* norm_weight,
                                             int norm_dtype, float eps, int act_dtype, const void* weight,
                                             int weight_dtype, int weight_layout, int batch, int hidden_dim,
                                             int vocab, int reduce_cast, const float* temperature,
                                             const uint32_t* keys, int32_t* out_ids, void* workspace,
                                             size_t workspace_bytes, void* stream) {
  if (!norm_weight) { clear_error(); set_error("lm_head_sample_prenorm: null norm_weight"); return NVJSEL_EINVAL; }
  Prenorm pn;
  pn.norm_w = norm_weight;
  pn.norm_dtype = norm_dtype;
  pn.eps = eps;
  pn.act_dtype = act_dtype;
  return lm_head_entry(MODE_SAMPLE, hidden, hidden_dtype, weight, weight_dtype, weight_layout, batch,
                       hidden_dim, vocab, reduce_cast, temperature, keys, out_ids, nullptr, workspace,
                       workspace_bytes, stream, pn);
}

extern "C" int nvjsel_lm_head_sample(const void* hidden, int hidden_dtype, const void* weight,
                                     int weight_dtype, int weight_layout, int batch, int hidden_dim,
                                     int vocab, int reduce_cast, const float* temperature,
                                     const uint32_t* keys, int32_t* out_ids, void* workspace,
                                     size_t workspace_bytes, void* stream) {
  return lm_head_entry(MODE_SAMPLE, hidden, hidden_dtype, weight, weight_dtype, weight_layout, batch,
                       hidden_dim, vocab, reduce_cast, temperature, keys, out_ids, nullptr, workspace,
                       workspace_bytes, stream);
}
