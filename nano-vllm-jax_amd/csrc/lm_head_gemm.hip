// LM head as a blocked GEMM staged through registers into the LDS (gfx950):
// [H, V] weights, every mode, above the streaming kernel's rows (8; 16-bit
// activations fewer on f16 weights and on vocabularies up to 512 columns for
// half of the CUs, from the first row); on [V, H] bf16 sampling above 128 rows
// and f32 activations above 192.
#include "lm_head_common.h"

namespace nvjsel {

// ------------------------------------------------------------------ blocked GEMM, 1 <= B <= 256
// 16-bit W [V, H] or [H, V], hidden of the same type or f32 on bf16, H % 64 ==
// 0, up to 256 rows in ONE pass over W (f16: 64).  The hidden of 256 rows (512
// KB at H = 1024) is a CU's whole register file, so unlike the tile kernel
// nothing is held for the whole call: a block tile is 256 vocabulary rows x all
// 256 batch rows (NARROW, 64 rows and fewer: below), and K is streamed in
// stages of 32 -- the W stage (256 x 32, 16 KB, from HBM) and the hidden
// stage (256 x 32, 16 KB, L2-resident) staged through a two-buffer LDS ring.
// Each thread loads 4 x 16 B per stage into registers; two register sets
// keep the stages s+2 and s+3 in flight while stage s is multiplied, so every
// load has two compute phases to land, and the pipeline runs on across the
// block's vocabulary tiles (round robin) without draining.  One barrier per
// stage.  Each wave computes a 128 x 64 sub-tile (vocab part, batch quarter)
// as 4 x 2 v_mfma_f32_32x32x16_bf16 tiles (128 accumulators per lane),
// reading 4 A and 2 B fragments per 16-wide k-step.
// LDS layout: 16-byte column q of row `row` at q * ROWS + (row ^ 2q): the 32
// lanes of a fragment read hit 32 distinct slots of one 512 B window, and the
// 8 lanes (2 rows x 4 columns) of a store phase hit 8 distinct bank groups.
// Blocks keep, per batch row, a running best key, fold it into the row's
// maximum with one atomicMax per row, and the last block to finish writes the
// ids (finish_rows; a reduce kernel over stored per-block keys cost ~7 us
// more).  MODE_LOGITS stores the rounded logits instead; MODE_SAMPLE scores
// every tile with the fast Gumbel draws after its K loop and rescores the
// near-maximal entries exactly (the sample epilogue in the kernel).
static constexpr int kGemmQcap = 768;  // queue entries per wave (sample mode; LDS: 12 B each)

// Epilogue of one block tile of the blocked GEMM for the wave's 128 x 64
// sub-tile: D[vocab 8 (e >> 2) + 4 h + (e & 3)][batch c32] of 32 x 32 tile
// (tv, tb), vocabulary rows from v0.  Greedy: per (tile, lane) the maximum of
// the 16 raw values (v_maximum3: NaN propagates), rounded; only where that
// beats the lane's running best (bo, bi) is the first element rounding to it
// looked up.  Rounding is monotone, so max(round(x)) = round(max(x)), and ties
// keep the lowest vocabulary row (rows ascend with e and with the tiles).
// Rows past V hold other data ([V, H]: row V - 1; [H, V]: the last or the next row's
// group) and are masked in the last tile.
template <int MODE, int TV>
__device__ __forceinline__ void gemm_epilogue(const LmArgs& a, const f32x16_t (&acc)[TV][2], int v0, int bj, int h,
                                              int c32, uint32_t (&bo)[2], uint32_t (&bi)[2]) {
#pragma unroll
  for (int tv = 0; tv < TV; ++tv)
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      const f32x16_t& d = acc[tv][tb];
      if constexpr (MODE == MODE_LOGITS) {
        const int b = bj * 64 + tb * 32 + c32;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int v = v0 + tv * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
          if (v < a.V && b < a.B) store_logit(a, b, v, apply_cast(d[e], a.reduce_cast));
        }
      } else {
        f32x16_t dm = d;
        if (v0 + tv * 32 + 32 > a.V) {  // the last tile: rows past V hold re-read data
#pragma unroll
          for (int e = 0; e < 16; ++e)
            if (v0 + tv * 32 + 8 * (e >> 2) + 4 * h + (e & 3) >= a.V) dm[e] = -INFINITY;
        }
        float m = dm[0];
#pragma unroll
        for (int e = 1; e < 15; e += 2)
          m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, dm[e]), dm[e + 1]);
        m = __builtin_elementwise_maximum(m, dm[15]);
        const float rm = apply_cast(m, a.reduce_cast);
        const uint32_t om = ord_f32(rm);
        const bool up = om > bo[tb];
        if (__builtin_amdgcn_ballot_w64(up)) {
          int first = 15;
          const bool nan = rm != rm;
#pragma unroll
          for (int e = 14; e >= 0; --e) {
            const float x = apply_cast(dm[e], a.reduce_cast);
            if (nan ? x != x : x == rm) first = e;
          }
          if (up) {
            bo[tb] = om;
            bi[tb] = (uint32_t)(v0 + tv * 32 + 8 * (first >> 2) + 4 * h + (first & 3));
          }
        }
      }
    }
}

// The blocks' final step: the lanes' best keys of each batch column, reduced
// over the two lane halves and the vocabulary parts, folded into the rows'
// running maxima (one atomicMax per block and row); the last block to finish
// writes the ids and re-zeroes the keys (finish_rows).
template <int VH, int NT, int KBR>
__device__ __forceinline__ void gemm_finish_rows(const LmArgs& a, unsigned long long (&best)[2], int vi, int bj,
                                                 int h, int c32, unsigned long long (*kred)[KBR]) {
#pragma unroll
  for (int tb = 0; tb < 2; ++tb) {
    best[tb] = max_u64(best[tb], shfl_xor_u64(best[tb], 32));
    if (h == 0) kred[vi][bj * 64 + tb * 32 + c32] = best[tb];
  }
  __syncthreads();
  for (int b = threadIdx.x; b < a.B; b += NT) {
    unsigned long long m = kred[0][b];
#pragma unroll
    for (int q = 1; q < VH; ++q) m = max_u64(m, kred[q][b]);
    if (m) (void)after(atomicMax(&a.row_keys[b], m));
  }
  finish_rows(a.row_keys, a.counter, a.B, a.out_ids, a.out_best);
}


// NS = 1: bf16 hidden.  NS = 3: f32 hidden, each value split exactly into
// three bf16 terms as it is staged into LDS (split_terms), and three MFMAs
// per fragment pair (fp32 products and sums, as the tile kernel's NS = 3).
// KC: K per stage (32; 16 for f32 hidden in sample mode above 64 rows, whose
// three-term 256-row stages and candidate queues would not fit the LDS at 32;
// the narrow layout's 64-row stages do, ~144 KB).
// HV: weight stored [H, V] (vocabulary contiguous).  A W stage is then KC
// k-rows of BV columns (512-byte rows, read whole), kept row-major in LDS
// (rows padded by 16 bytes), and the A fragments -- 8 consecutive k of one
// vocabulary column per lane -- come from two transposing LDS reads
// (ds_read_b64_tr_b16: in each 16-lane group, lane j receives element j & 3
// of the 8-byte chunks addressed by lanes (j >> 2) + 4m, m = 0..3; group lane
// r addresses k = kb + (r >> 2), columns c0 + 4 (r & 3) .. + 3, so lane j gets
// k = kb .. kb + 3 of column c0 + j).
// PART: B <= 192, some 64-row batch quarter holds only repeats of row B - 1.
// NARROW: B <= 64; each wave owns 32 vocabulary rows x the 64 batch rows
// (instead of 128 x 64 of one batch quarter), so all 8 waves multiply and,
// in sample mode, draw.
// WT: weight (and NS = 1: hidden) element type.  VEC8: [H, V] rows of whole,
// aligned 16-byte groups (V % 8 == 0); groups past the row end re-read the last
// one.  Else rows start at any element (V >= 8): 16-byte loads from element
// addresses; a group that ends past its row reads on into the next one (columns
// masked where they could win), in the last row it is loaded from V - 8 and
// moved down as it is stored: 2-6% more time on aligned rows (V = 32,000, H =
// 1024, f32 hidden B = 32 48.8 us against 47.6, bf16 B = 256 46.7 against 44.4),
// but for 16-bit hidden in the narrow layout (B = 32 23.2 against 24.1 with VEC8).
template <int WT, int MODE, int BV, int NS, int KC, bool HV, bool VEC8, bool PART, bool NARROW>
__global__ void __launch_bounds__(BV * 2, 256 / BV) lm_head_gemm_kernel(LmArgs a) {
  constexpr int Q = KC / 8;  // 8-element columns per row and stage
  static_assert(!(PART && NARROW), "one batch layout");
  constexpr int TV = NARROW ? 1 : 4;  // 32-row vocabulary tiles per wave
  constexpr int VH = BV / (32 * TV);  // vocabulary parts
  constexpr int NBQ = NARROW ? 1 : 4;  // 64-row batch quarters
  constexpr int NT = VH * NBQ * 64;  // threads
  constexpr int KBR = NARROW ? 64 : kGemmBB;  // batch rows of the block's row reduction
  // hidden rows staged per stage (NARROW with f32 hidden: only the 64 the
  // waves multiply, loaded by the first Q * 64 threads -- whole waves; 291 ->
  // ~180 us greedy at B = 40-64; with bf16 hidden it measured ~7 us slower)
  constexpr int XB = (NARROW && NS == 3) ? 64 : kGemmBB;
  constexpr int XT = Q * XB < NT ? Q * XB : NT;  // threads loading hidden pieces
  constexpr int PA = Q * BV / NT, PB = Q * XB / XT;  // 8-element load pieces per loading thread (W, hidden)
  constexpr int HB = NS == 1 ? 1 : 2;  // 16-byte loads per hidden piece
  static_assert(PA >= 1 && PA * NT == Q * BV && PB * XT == Q * XB && XT % 64 == 0, "whole load pieces per thread");
  static_assert(NS == 1 || NS == 3, "bf16 or three-term f32 hidden");
  constexpr int ROWV = BV + 8;  // HV: LDS row length in elements (16-byte pad)
  constexpr int AW = HV ? KC * ROWV / 8 : Q * BV;  // 16-byte slots of a W stage
  __shared__ u32x4_t As[2][AW];
  __shared__ u32x4_t Bs[2][NS][Q * XB];
  __shared__ unsigned long long kred[VH][KBR];
  // sample mode: per-wave queue of entries that may be their row's maximum
  // (logit, approximate score, vocab << 7 | tb << 6 | lane) and the
  // exact best key of each (lane, tb) row slot
  constexpr bool SMP = MODE == MODE_SAMPLE;
  constexpr int NW = NT / 64;
  constexpr int QC = SMP ? kGemmQcap : 1;
  __shared__ float gqx[SMP ? NW : 1][QC];
  __shared__ float gqa[SMP ? NW : 1][QC];
  __shared__ uint32_t gqv[SMP ? NW : 1][QC];
  __shared__ unsigned long long gqbest[SMP ? NW : 1][SMP ? 128 : 1];
  // the wave index in a scalar register and the lane from mbcnt: nothing
  // derived from threadIdx.x has to stay live (or spill) across the loops
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)__lane_id();
  const int tid = wave * 64 + lane;
  const int vi = wave % VH, bj = wave / VH;
  const int B = a.B, V = a.V, H = a.H;
  const uint16_t* W = (const uint16_t*)a.W;
  const int ntiles = (V + BV - 1) / BV;
  const int nkc = H / KC;
  const int my_tiles = blockIdx.x < ntiles ? (ntiles - 1 - blockIdx.x) / gridDim.x + 1 : 0;
  const int S = my_tiles * nkc;  // stages of this block
  // load piece p: row p >> 2, 16-byte column p & 3, LDS slot q * ROWS + (row ^ 2q)
  int arow[PA], aq[PA], aslot[PA], bslot[PB];
  const u32x4_t* xp[PB];
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    const unsigned p = (unsigned)(tid + NT * i);  // (unsigned: / Q and % Q are a shift and a mask)
    if constexpr (HV) {  // k-row p / (BV / 8), 8-column group p % (BV / 8)
      arow[i] = (int)(p / (BV / 8));
      aq[i] = (int)(p % (BV / 8));
      aslot[i] = (arow[i] * ROWV + aq[i] * 8) / 8;
    } else {
      arow[i] = (int)(p / Q);
      aq[i] = (int)(p % Q);
      aslot[i] = aq[i] * BV + (arow[i] ^ (aq[i] << 1));
    }
  }
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    const unsigned p = (unsigned)(tid + XT * i);
    const int row = (int)(p / Q), q = (int)(p % Q);
    bslot[i] = q * XB + (row ^ (q << 1));
    // rows >= B repeat row B - 1: a fixed count of loads in flight and no
    // select on the loaded data (which would make the compiler wait for it
    // early); their batch columns are never read
    xp[i] = NS == 1 ? (const u32x4_t*)((const uint16_t*)a.hidden + (size_t)min(row, B - 1) * H) + q
                    : (const u32x4_t*)((const float*)a.hidden + (size_t)min(row, B - 1) * H) + 2 * q;
  }
  // Two register sets: stages s+2 and s+3 (W and hidden) are in flight while
  // stage s is multiplied.  Loads past the last stage re-read it, so every
  // path has the same loads in flight and each LDS store waits for exactly
  // its own stage.
  u32x4_t RA[2][PA], RB[2][PB][HB];
  int over[2][PA] = {};  // HV: places each piece moves down
  auto stage_of = [&](int st, int& v0, int& kc) NVJSEL_INLINE {
    st = st < S ? st : S - 1;
    const int t = st / nkc;
    kc = st - t * nkc;
    v0 = (blockIdx.x + t * gridDim.x) * BV;
  };
  auto gload_a = [&](auto set, int st) NVJSEL_INLINE {
    constexpr int e = decltype(set)::value;
    int v0, kc;
    stage_of(st, v0, kc);
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      if constexpr (HV && VEC8) {
        const int v = min(v0 + aq[i] * 8, V - 8);
        RA[e][i] = *(const u32x4_t*)(W + (size_t)(kc * KC + arow[i]) * V + v);
      } else if constexpr (HV) {
        const int k = kc * KC + arow[i];
        const int v = v0 + aq[i] * 8 < V ? v0 + aq[i] * 8 : V - 8;
        over[e][i] = k == H - 1 ? max(v - (V - 8), 0) : 0;
        RA[e][i] = *(const u32x4_any_t*)(W + (size_t)k * V + (v - over[e][i]));
      } else {
        const int v = min(v0 + arow[i], V - 1);
        RA[e][i] = *((const u32x4_t*)(W + (size_t)v * H + kc * KC) + aq[i]);
      }
    }
  };
  auto gload_b = [&](auto set, int st) NVJSEL_INLINE {
    constexpr int e = decltype(set)::value;
    int v0, kc;
    stage_of(st, v0, kc);
    if (XT < NT && tid >= XT) return;  // (wave-uniform)
#pragma unroll
    for (int i = 0; i < PB; ++i)
#pragma unroll
      for (int j = 0; j < HB; ++j) RB[e][i][j] = xp[i][kc * Q * HB + j];
  };
  auto lstore = [&](auto set, auto buf) NVJSEL_INLINE {
    constexpr int e = decltype(set)::value, f = decltype(buf)::value;
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      if constexpr (HV && !VEC8) {
        if (__any(over[e][i])) RA[e][i] = shift_down8(RA[e][i], over[e][i]);
      }
      As[f][aslot[i]] = RA[e][i];
    }
    if (XT < NT && tid >= XT) return;  // (wave-uniform)
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      if constexpr (NS == 1) {
        Bs[f][0][bslot[i]] = RB[e][i][0];
      } else {
        float v[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[j] = __uint_as_float(RB[e][i][0][j]);
          v[4 + j] = __uint_as_float(RB[e][i][1][j]);
        }
        u32x4_t t3[NS][1];
        split_terms<NS>(v, t3, 0);
#pragma unroll
        for (int t = 0; t < NS; ++t) Bs[f][t][bslot[i]] = t3[t][0];
      }
    }
  };
  // 32 x 32 tiles: 4 (vocab) x 2 (batch) per wave
  const int h = lane >> 5, c32 = lane & 31;
  // HV: this lane's transposing-read position in a stage (k-row, column)
  const int trk = 8 * (lane >> 5) + ((lane & 15) >> 2), trc = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  f32x16_t acc[TV][2];
  auto zero_acc = [&]() NVJSEL_INLINE {
#pragma unroll
    for (int tv = 0; tv < TV; ++tv)
#pragma unroll
      for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[tv][tb][e] = 0.f;
  };
  auto compute = [&](auto buf) NVJSEL_INLINE {
    constexpr int f = decltype(buf)::value;
#pragma unroll
    for (int ks = 0; ks < KC / 16; ++ks) {
      const int q = ks * 2 + h, sw = q << 1;
      u32x4_t bf[NS][2];
#pragma unroll
      for (int t = 0; t < NS; ++t)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) bf[t][tb] = Bs[f][t][q * XB + ((bj * 64 + tb * 32 + c32) ^ sw)];
#pragma unroll
      for (int tv = 0; tv < TV; ++tv) {
        u32x4_t af;
        if constexpr (HV) {
          typedef __bf16 bf16x4_lds __attribute__((ext_vector_type(4)));
          typedef __attribute__((address_space(3))) bf16x4_lds lds_bf16x4;
          const int off = (ks * 16 + trk) * ROWV + vi * 32 * TV + tv * 32 + trc;
          auto* base = (__attribute__((address_space(3))) uint16_t*)(uint16_t*)As[f];
          const bf16x4_lds lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(base + off));
          const bf16x4_lds hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(base + off + 4 * ROWV));
          uint32_t w[4];
          __builtin_memcpy(w, &lo, 8);
          __builtin_memcpy(w + 2, &hi, 8);
          af = u32x4_t{w[0], w[1], w[2], w[3]};
        } else {
          af = As[f][q * BV + ((vi * 32 * TV + tv * 32 + c32) ^ sw)];
        }
#pragma unroll
        for (int t = 0; t < NS; ++t)
#pragma unroll
          for (int tb = 0; tb < 2; ++tb) acc[tv][tb] = mfma32x32x16<WT>(af, bf[t][tb], acc[tv][tb]);
      }
    }
  };
  uint32_t bo[2] = {0u, 0u}, bi[2] = {0u, 0u};  // running best: ordered value, row
  // sample mode: the lane's two batch rows bj * 64 + tb * 32 + c32
  float tp[2] = {1.0f, 1.0f}, rtp[2] = {1.0f, 1.0f}, amax[2] = {-INFINITY, -INFINITY};
  bool greedy_row[2] = {true, true};
  TfKey key[2] = {tf_key(0u, 0u), tf_key(0u, 0u)};
  unsigned long long sbest[2] = {0ull, 0ull};
  uint32_t qcount = 0;  // wave-uniform
  if constexpr (SMP) {
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      const int b = bj * 64 + tb * 32 + c32;
      const float t = b < B ? a.temperature[b] : 0.0f;
      greedy_row[tb] = (t <= 0.0f);
      tp[tb] = temp_floor(t);
      rtp[tb] = 1.0f / tp[tb];
      if (b < B) key[tb] = tf_key(a.keys[2 * b], a.keys[2 * b + 1]);
      gqbest[wave][tb * 64 + lane] = 0ull;
    }
  }
  // drops queued entries that can no longer be their row's maximum (the test
  // each passed when queued, against the row slot's maximum, which has only
  // grown since); compaction in place, a 64-entry group read before any
  // survivor is written at or below it
  auto gcompact = [&]() NVJSEL_INLINE {
    uint32_t nk = 0;
    for (uint32_t e0 = 0; e0 < qcount; e0 += 64) {  // wave-uniform trip count
      const uint32_t e = e0 + lane;
      const bool live = e < qcount;
      const float x = live ? gqx[wave][e] : 0.0f;
      const float ap = live ? gqa[wave][e] : -INFINITY;
      const uint32_t pv = live ? gqv[wave][e] : 0u;
      const int sl = (int)(pv & 63u);
      const float a0 = __shfl(amax[0], sl, 64), a1 = __shfl(amax[1], sl, 64);
      const float am = (pv & 64u) ? a1 : a0;
      const bool keep = live && !(ap + score_slack(ap, am) < am);
      const unsigned long long m = __ballot(keep);
      if (keep) {
        const uint32_t slot = nk + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                             __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        gqx[wave][slot] = x;
        gqa[wave][slot] = ap;
        gqv[wave][slot] = pv;
      }
      nk += (uint32_t)__popcll(m);
    }
    qcount = nk;
  };
  // exact scores (fp64 logs) of the queued entries, a full wave at a time,
  // folded into the row slots' exact best keys
  auto gflush = [&]() NVJSEL_INLINE {
    for (uint32_t e0 = 0; e0 < qcount; e0 += 64) {  // wave-uniform trip count
      const uint32_t e = e0 + lane;
      const bool live = e < qcount;
      const uint32_t pv = live ? gqv[wave][e] : 0u;
      const int sl = (int)(pv & 63u);
      const bool t1 = (pv & 64u) != 0u;
      // the shuffles run with the whole wave active
      uint32_t kw[2][3];
#pragma unroll
      for (int tb = 0; tb < 2; ++tb) {
        kw[tb][0] = (uint32_t)__shfl((int)key[tb].k0, sl, 64);
        kw[tb][1] = (uint32_t)__shfl((int)key[tb].k1, sl, 64);
        kw[tb][2] = (uint32_t)__shfl((int)key[tb].k2, sl, 64);
      }
      const TfKey k2{t1 ? kw[1][0] : kw[0][0], t1 ? kw[1][1] : kw[0][1], t1 ? kw[1][2] : kw[0][2]};
      const uint32_t v = pv >> 7;
      const float u0 = __shfl(tp[0], sl, 64), u1 = __shfl(tp[1], sl, 64);
      if (live) atomicMax(&gqbest[wave][pv & 127u], argmax_key(gqx[wave][e] / (t1 ? u1 : u0) + gumbel_at(k2, v), v));
    }
    qcount = 0;
  };
  // one tile of the sample epilogue: runs of 2 consecutive vocabulary rows
  // (D elements 2 qq, 2 qq + 1: rows v0 + tv * 32 + 8 (qq >> 1) + 4 h +
  // 2 (qq & 1) + j) scored with the hardware log; entries that can still be
  // the row's maximum queue.  Two Threefry chains per run and a runtime loop
  // over the four vocabulary sub-tiles (acc[0] is scored, then the tiles
  // shift down) keep the 128 accumulators, the loads in flight and the
  // draws within the register file, and the loop body within the
  // instruction cache.
  auto sample_epilogue = [&](int v0) NVJSEL_INLINE {
    // the two lane halves hold the same batch rows: share their maxima
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) amax[tb] = xor32_max(amax[tb]);
#pragma unroll 1
    for (int tv = 0; tv < TV; ++tv) {
#pragma unroll
      for (int qq = 0; qq < 8; ++qq)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
          if (qcount > (uint32_t)(QC - 128)) {  // room for one run of the wave
            gcompact();
            if (qcount > (uint32_t)(QC - 128)) gflush();
          }
          const int b = bj * 64 + tb * 32 + c32;
          const int vs = v0 + tv * 32 + 8 * (qq >> 1) + 4 * h + 2 * (qq & 1);
          bool q[2] = {false, false};
          float xq[2], aq[2];
          if (b < B) {
            const float raw[2] = {acc[0][tb][2 * qq], acc[0][tb][2 * qq + 1]};
            score_run<MODE_SAMPLE, 2>(raw, vs, V, a.reduce_cast, greedy_row[tb], rtp[tb], tp[tb], key[tb],
                                      amax[tb], sbest[tb], q, xq, aq);
          }
          // queue the marked entries with the whole wave active: slots from a ballot
          if (__any(q[0] | q[1])) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              const unsigned long long m = __ballot(q[j]);
              if (q[j]) {
                const uint32_t slot = qcount + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                         __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                gqx[wave][slot] = xq[j];
                gqa[wave][slot] = aq[j];
                gqv[wave][slot] = ((uint32_t)(vs + j) << 7) | ((uint32_t)tb << 6) | (uint32_t)lane;
              }
              qcount += (uint32_t)__popcll(m);
            }
          }
        }
#pragma unroll
      for (int t = 0; t < TV - 1; ++t)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) acc[t][tb] = acc[t + 1][tb];
    }
  };
  auto epilogue = [&](int t) NVJSEL_INLINE {
    const int v0 = (blockIdx.x + t * gridDim.x) * BV + vi * 32 * TV;
    if constexpr (NS == 3) {
      auto redo = [&](auto TBI) NVJSEL_INLINE {
        constexpr int tb = decltype(TBI)::value;
        const float m = tile_max<tb>(acc);
        if (__builtin_amdgcn_ballot_w64(m != m))
          redo_nan_logits<tb, true>(a, acc, lane, [&](int tv, int e, int& b, int& v) NVJSEL_INLINE {
            b = bj * 64 + tb * 32 + c32;
            v = v0 + tv * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
            return b < B && v < V;
          });
      };
      redo(std::integral_constant<int, 0>{});
      redo(std::integral_constant<int, 1>{});
    }
    if constexpr (SMP)
      sample_epilogue(v0);
    else
      gemm_epilogue<MODE, TV>(a, acc, v0, bj, h, c32, bo, bi);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  if (S > 0) {  // S is even: nkc = H / KC with H % (2 KC) == 0
    // prologue: stage 0 in LDS buffer 0, stages 1 and 2 in sets 1 and 0 --
    // issued in the order the loop's back edge leaves them in flight, so the
    // wait counts agree at the loop head and no store waits for more than
    // its own stage
    gload_b(I0{}, 0);
    gload_a(I0{}, 0);
    lstore(I0{}, I0{});
    gload_b(I1{}, 1);
    gload_a(I1{}, 1);
    gload_b(I0{}, 2);
    gload_a(I0{}, 2);
    __syncthreads();
    // stage s: store stage s+1 (set (s+1)&1) to buffer (s+1)&1, load stage
    // s+3 into that set, multiply buffer s&1
    auto step = [&](int st, auto cur, auto live) NVJSEL_INLINE {
      constexpr int c = decltype(cur)::value;
      using N = std::integral_constant<int, 1 - c>;
      lstore(N{}, N{});
      gload_b(N{}, st + 3);
      gload_a(N{}, st + 3);
      if constexpr (decltype(live)::value) compute(cur);
      __syncthreads();
    };
    // the accumulators are zeroed and read outside the stage loop, so they
    // stay in place across it.  PART: a wave whose 64 batch rows all lie past
    // B (repeats of row B - 1) runs the stages without fragment reads or
    // products (B = 64 leaves 2 of the 8 waves multiplying); the full-batch
    // kernel has one loop and no test
    auto tiles = [&](auto live) NVJSEL_INLINE {
      for (int t = 0; t < my_tiles; ++t) {
        zero_acc();
        for (int kc = 0; kc < nkc; kc += 2) {
          step(t * nkc + kc, I0{}, live);
          step(t * nkc + kc + 1, I1{}, live);
        }
        epilogue(t);
      }
    };
    if constexpr (PART) {
      if (bj * 64 < B)  // wave-uniform
        tiles(std::true_type{});
      else
        tiles(std::false_type{});
    } else {
      tiles(std::true_type{});
    }
  }
  if constexpr (MODE == MODE_LOGITS) return;
  unsigned long long best[2];
  if constexpr (SMP) {
    gcompact();
    gflush();
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) best[tb] = greedy_row[tb] ? sbest[tb] : max_u64(sbest[tb], gqbest[wave][tb * 64 + lane]);
  } else {
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) best[tb] = ((unsigned long long)bo[tb] << 32) | (unsigned long long)(~bi[tb]);
  }
  gemm_finish_rows<VH, NT, KBR>(a, best, vi, bj, h, c32, kred);
}


// vocabulary rows per block tile: 256 (8 waves, one block per CU; measured
// 185 us at B = 256, V = 248320) or 128 (4 waves, two blocks per CU: 195 us)
static constexpr int kGemmBV = 256;
static constexpr int kGemmBpc = 256 / kGemmBV;  // blocks per CU of the blocked GEMM
template <int WT, int MODE, int NS, bool HV, bool VEC8>
static int launch_gemm_shape(const LmArgs& a, hipStream_t stream) {
  const int ntiles = (a.V + kGemmBV - 1) / kGemmBV;
  int grid = kGemmBpc * device_cu_count();
  if (grid > ntiles) grid = ntiles;
  constexpr int KC = (NS == 3 && MODE == MODE_SAMPLE) ? kGemmKC / 2 : kGemmKC;
  // ([V, H] calls of <= 64 rows take other kernels; the narrow layout's 64-row
  // f32 stages leave room for K stages of 32 in sample mode)
  constexpr bool kNarrow = HV;
  if constexpr (kNarrow) {
    if (a.B <= 64) {
      hipLaunchKernelGGL((lm_head_gemm_kernel<WT, MODE, kGemmBV, NS, kGemmKC, HV, VEC8 && NS == 3, false, true>), dim3(grid), dim3(kGemmBV * 2), 0, stream, a);
      NVJSEL_CHECK_LAUNCH("lm_head_gemm_kernel");
      return NVJSEL_OK;
    }
  }
  if constexpr (WT == DT_F16) {
    return fail(NVJSEL_EINVAL, "launch_gemm: f16 weights take at most 64 rows");
  } else {
    if constexpr (HV || NS == 1) {  // ([V, H] f32 passes of <= 192 rows take the staged GEMM)
      if (a.B <= kGemmBB - 64) {
        hipLaunchKernelGGL((lm_head_gemm_kernel<WT, MODE, kGemmBV, NS, KC, HV, VEC8, true, false>), dim3(grid), dim3(kGemmBV * 2), 0, stream, a);
        NVJSEL_CHECK_LAUNCH("lm_head_gemm_kernel");
        return NVJSEL_OK;
      }
    }
    hipLaunchKernelGGL((lm_head_gemm_kernel<WT, MODE, kGemmBV, NS, KC, HV, VEC8, false, false>), dim3(grid), dim3(kGemmBV * 2), 0, stream, a);
  }
  NVJSEL_CHECK_LAUNCH("lm_head_gemm_kernel");
  return NVJSEL_OK;
}

int launch_gemm(int mode, bool hv, const LmArgs& a, hipStream_t stream) {
  auto by_mode = [&](auto fn) -> int {
    if (mode == MODE_GREEDY) return fn(std::integral_constant<int, MODE_GREEDY>{});
    if (mode == MODE_SAMPLE) return fn(std::integral_constant<int, MODE_SAMPLE>{});
    return fn(std::integral_constant<int, MODE_LOGITS>{});
  };
  if (!hv && a.hidden_dtype == DT_F32)
    return by_mode([&](auto M) { return launch_gemm_shape<DT_BF16, decltype(M)::value, 3, false, false>(a, stream); });
  if (!hv) {
    if (mode != MODE_SAMPLE || a.hidden_dtype != DT_BF16)
      return fail(NVJSEL_EINVAL, "launch_gemm: [V, H] weights take the staged GEMM");
    return launch_gemm_shape<DT_BF16, MODE_SAMPLE, 1, false, false>(a, stream);
  }
  // (f16 weights take the any-element loads: their rows were never faster)
  if (a.weight_dtype == DT_F16)
    return by_mode([&](auto M) { return launch_gemm_shape<DT_F16, decltype(M)::value, 1, true, false>(a, stream); });
  const bool vec8 = (a.V % 8) == 0 && (((uintptr_t)a.W) & 15) == 0;
  if (a.hidden_dtype == DT_F32)
    return by_mode([&](auto M) {
      return vec8 ? launch_gemm_shape<DT_BF16, decltype(M)::value, 3, true, true>(a, stream)
                  : launch_gemm_shape<DT_BF16, decltype(M)::value, 3, true, false>(a, stream);
    });
  return by_mode([&](auto M) {
    return vec8 ? launch_gemm_shape<DT_BF16, decltype(M)::value, 1, true, true>(a, stream)
                : launch_gemm_shape<DT_BF16, decltype(M)::value, 1, true, false>(a, stream);
  });
}

}  // namespace nvjsel
