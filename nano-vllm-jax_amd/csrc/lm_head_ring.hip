// LM head as a staged GEMM whose operands reach the LDS by direct loads (gfx950).
//
// 16-bit weight [V, H] x hidden of the same type, H % 64 == 0, up to 256 batch
// rows per pass over W (sampling: 128), or bf16 weight x f32 hidden, up to 64:
// greedy top-1, dense logits, Gumbel-max.
//
// One block of 8 waves per CU takes an equal, contiguous share of the
// vocabulary in tiles of 256 rows x all batch rows; K streams in stages of 64.
//  * What bounds it: up to ~128 rows the stream of W, above that matrix and
//    LDS work together.  A read-only probe of this access pattern takes 79-82
//    us for 508 MB in 128-byte pieces, non-temporal (64-byte pieces 90 us,
//    the pieces of a 32-wide stage; 128-byte pieces without the hint 92).
//  * global_load_lds writes 16 bytes per lane straight into the LDS, so no
//    registers hold stages in flight; the slots are swizzled through the
//    lane's global address (16-byte column q of row r at q ^ (r >> 1) % 8, the
//    same cache line), which leaves fragment reads without bank conflicts.
//    The compiler does not count these loads: each stage waits for its own
//    with vmcnt and leaves the newer ones in flight (stage_barrier).
//  * W runs RW - 1 stages ahead, the hidden (L2) RX - 1.
//  * Fragments are read one k-step ahead of the products, across the barrier
//    (B = 256 158 -> 155 us).
//  * Greedy epilogue: one maximum per lane and batch row over the tile, and
//    the index looked up by comparing raw values with the smallest float that
//    rounds to that maximum (a lookup per 32 x 32 tile with rounded values:
//    B = 128 / 256 106 / 162 us against 93 / 147).
//  * Logits: operands swapped, so that 32 lanes hold 64 contiguous bytes of
//    one row, and quads of lanes transposed for 8-byte stores (B = 80 / 256
//    2-byte stores 118 / 206 us, 8-byte 114 / 184; 32-byte runs 240 / 273).
//  * Sampling: a finished tile's logits stay in registers and are scored in
//    small units beside the next tile's stages (B = 64 136 -> 117-123 us, B =
//    128 224 -> 183); the waves share the rows' maxima through the LDS, so few
//    entries queue for exact scores.
//  * f32 hidden (NS = 3): a stage arrives as f32 beside the ring and is split
//    into three bf16 terms in the middle of the stage before its own (once per
//    block; through registers, whose waits drained the W stage in flight too,
//    B = 16 took 99 us against 87).  Fragment reads bound it at 64 rows: 64 x
//    32 per wave instead of 32 x 64 reads 160 KB per stage instead of 224 (B =
//    64 126 -> 121 us).
//  * A share that ends in part of a tile pays the whole one's requests and
//    products (V = 66,000, two tiles for 264 rows, B = 16 31 us where the tile
//    kernel takes 24): bf16 calls at H = 1024 that the tile kernel takes too go by
//    the share (route_rules.h).
// H = 1024, V = 248,320, greedy B = 16 / 64 / 128 / 256: 76 / 78 / 90 / 136 us
// (6.6 / 6.5 / 5.7 / 3.7 TB/s; 956 TFLOP/s at 256) where 64-row passes of the
// tile kernel and the blocked GEMM took 78 / 81 / 160 / 177.
#include <limits.h>

#include "lm_head_common.h"
#include "route_rules.h"

namespace nvjsel {

static constexpr int kRingKC = 64;  // K per stage: 128-byte pieces of W rows, whole cache lines

// NBR: batch rows of the block (rows past B repeat row B - 1).  NS: terms per
// hidden value (3: f32 hidden, each value split exactly into three bf16 terms
// as it is staged, three products per fragment pair).
template <int MODE, int NBR, int NS>
struct RingShape {
  static_assert(NS == 1 || (NS == 3 && NBR <= 64), "the terms' slots fit the LDS");
  static constexpr bool SMP = MODE == MODE_SAMPLE;
  static constexpr int NW = 8;                        // waves; one block per CU
  static constexpr int BV = 256;                      // vocabulary rows of a block tile
  static constexpr int TB = NBR <= 32 || NS == 3 ? 1 : 2;  // 32-row batch tiles per wave
  static constexpr int WB = NBR / (32 * TB);          // waves along the batch
  static constexpr int WV = NW / WB;                  // waves along the vocabulary
  static constexpr int TV = BV / (32 * WV);           // 32-row vocabulary tiles per wave
  // ring slots: W stages come from HBM, hidden stages from L2
  static constexpr int RW = NS == 3 ? (SMP && NBR == 64 ? 2 : 3) : SMP ? (NBR <= 64 ? 3 : 2) : NBR <= 32 ? 4 : 3;
  static constexpr int RX = NS == 3 || SMP ? 2 : NBR <= 32 ? 4 : NBR <= 128 ? 3 : 2;
  static constexpr int LDS_RAW = NS == 3 ? NBR * kRingKC * 4 : 0;  // one stage of f32 values
  static constexpr int LDS_RING = (RW * BV + RX * NS * NBR) * kRingKC * 2 + LDS_RAW;
  // sample mode: rows scored at a time, queue entries per wave (12 B each), and
  // per batch row the block's largest approximate score and best exact key
  static constexpr int RUN = 4;
  static constexpr int QC = NS == 3 ? 320 : NBR == 64 ? 480 : 512;
  static constexpr int LDS_QUEUE = SMP ? NW * QC * 12 + NBR * 12 : 0;
  static_assert(QC >= 64 * RUN, "room for one unit");
  static_assert(LDS_RING + LDS_QUEUE <= 160 * 1024, "fits the LDS");
};

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // M0 is written for the load right behind it
// One 16-byte direct load per lane from `base` + voff (bytes) to LDS byte
// address lds + 16 * lane.  Outstanding loads are counted by the kernel itself
// (wait_stage); M0 holds the LDS address.
__device__ __forceinline__ void dma16(const void* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base)
               : "memory", "m0");
}
__device__ __forceinline__ void dma16_nt(const void* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds), "v"(voff), "s"(base)
               : "memory", "m0");
}

#pragma clang diagnostic pop

// This wave's direct loads but the newest N have landed and its LDS reads are
// done; then the block barrier: the stage about to be multiplied is whole, and
// nobody reads the one about to be overwritten.
template <int N>
__device__ __forceinline__ void stage_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// The smallest float that rounds (to nearest even) to the bf16 value r, not NaN.
__device__ __forceinline__ float bf16_round_low(float r) {
  uint32_t u = __float_as_uint(r);
  if (u == 0xFF800000u) return r;   // -inf
  if (u == 0u) u = 0x80000000u;     // -0.0 == +0.0: what rounds to -0.0 counts
  const uint32_t half = 0x8000u - ((u >> 16) & 1u);  // ties go to the even neighbour
  return __uint_as_float((u & 0x80000000u) ? u + half : u - half);
}

// The next of the three bf16 terms of four f32 values (round to nearest even),
// which leave the remainders: hi + mid + lo = v exactly (8 + 8 + 8 bits).
__device__ __forceinline__ uint2 next_term(float (&v)[4]) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  uint32_t o[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    o[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{v[2 * j], v[2 * j + 1]}), bf16x2_t));
    v[2 * j] = v[2 * j] - __uint_as_float(o[j] << 16);
    v[2 * j + 1] = v[2 * j + 1] - __uint_as_float(o[j] & 0xFFFF0000u);
  }
  return uint2{o[0], o[1]};
}

// This wave's direct loads but the newest N have landed.
template <int N>
__device__ __forceinline__ void wave_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// x[j]: this lane's value of row j, its column the lane's place in its quad.
// Lane j of the quad gets row j's four columns as 16-bit values (bf16 or f16,
// round to nearest even).
__device__ __forceinline__ uint2 quad_transpose16(const float (&x)[4], int dtype, int lane) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  uint32_t r02, r13;  // rows 0 | 2 << 16 and 1 | 3 << 16 of this column
  if (dtype == DT_BF16) {
    r02 = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x[0], x[2]}), bf16x2_t));
    r13 = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x[1], x[3]}), bf16x2_t));
  } else {
    r02 = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x[0], x[2]}), f16x2));
    r13 = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x[1], x[3]}), f16x2));
  }
  const bool odd = lane & 1, high = lane & 2;
  // with lane ^ 1: an even lane keeps rows 0 and 2, an odd one rows 1 and 3
  const uint32_t got = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(odd ? r02 : r13), 0xB1, 0xF, 0xF, false);
  const uint32_t own = odd ? r13 : r02, lo = odd ? got : own, hi = odd ? own : got;
  const uint32_t p = __builtin_amdgcn_perm(hi, lo, 0x05040100u);  // row (odd): this column pair
  const uint32_t q = __builtin_amdgcn_perm(hi, lo, 0x07060302u);  // row 2 + (odd)
  // with lane ^ 2: the low pair keeps rows 0 and 1, the high pair rows 2 and 3
  const uint32_t g2 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(high ? p : q), 0x4E, 0xF, 0xF, false);
  return high ? uint2{g2, q} : uint2{p, g2};
}

// rows: vocabulary rows per block (a multiple of 8).
template <int WT, int MODE, int NBR, int NS>
__global__ void __launch_bounds__(512) lm_head_ring_kernel(LmArgs a, int rows) {
  using S = RingShape<MODE, NBR, NS>;
  constexpr int TV = S::TV, TB = S::TB, WV = S::WV, RW = S::RW, RX = S::RX, NW = S::NW, QC = S::QC, RUN = S::RUN;
  constexpr int BV = S::BV;
  constexpr int WBYTES = BV * kRingKC * 2, XBYTES = NS * NBR * kRingKC * 2;
  constexpr int WL = WBYTES / (NW * 1024);                              // W loads per wave and stage
  constexpr int XL = XBYTES >= NW * 1024 ? XBYTES / (NW * 1024) : 1;     // hidden loads per wave and stage
  constexpr int XLANES = XBYTES >= NW * 1024 ? 64 : XBYTES / (NW * 16);  // lanes of each
  // loads a wave may leave in flight when stage s starts: those issued after
  // X(s) and W(s) (each stage issues X(s + RX - 1), then W(s + RW - 1))
  // (NS = 3: X(s) is split already; W(s + 1) is in flight where RW = 3)
  constexpr int LIVE = NS == 3 ? (RW - 2) * WL : (RX - 2) * (WL + XL) + (RW > RX ? WL : 0);
  static_assert(RW >= RX && RX >= 2, "W runs at least as far ahead as the hidden");
  constexpr int XRING = RW * WBYTES;  // LDS offset of the hidden's slots
  __shared__ __attribute__((aligned(1024))) char ring[S::LDS_RING + S::LDS_QUEUE];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)__lane_id();
  const int wv = wave % WV, wb = wave / WV;
  // this block's vocabulary rows r0 .. r1 - 1 in tiles of BV
  const int B = a.B;
  const uint32_t rowb = (uint32_t)a.H * 2u;
  const char* hidden = (const char*)a.hidden;
  const int nkc = a.H / kRingKC;
  const int r0 = (int)blockIdx.x * rows, r1 = min(r0 + rows, a.V);
  const int my_tiles = r0 < r1 ? (r1 - r0 + BV - 1) / BV : 0;
  auto tile_row = [&](int t) NVJSEL_INLINE { return r0 + t * BV; };
  const uint32_t ring0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)ring;

  // ---- load cursors: the next W stage to request (K offset lko of tile lt,
  // lleft stages left in it) and hidden stage (K offset xko), with their slots
  int lt = 0, lleft = nkc, lw = 0, lx = 0;
  uint32_t lko = 0, lstep = kRingKC * 2, xko = 0;
  uint32_t woff[WL], xoff[XL];
  const char* wtile = (const char*)a.W;
  auto load_tile_start = [&]() NVJSEL_INLINE {  // row offsets of tile lt (rows past its end repeat its last row)
    const int v0 = tile_row(lt), last = min(tile_row(lt + 1), r1) - v0 - 1;
    wtile = (const char*)a.W + (size_t)v0 * rowb;
#pragma unroll
    for (int i = 0; i < WL; ++i) {
      const int row = (i * NW + wave) * 8 + (lane >> 3);
      const int q = (lane & 7) ^ ((row >> 1) & 7);
      woff[i] = (uint32_t)min(row, last) * rowb + (uint32_t)(q * 16);
    }
  };
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int p = (i * NW + wave) * XLANES + lane;  // (XL > 1: XLANES = 64)
    const int row = p >> 3;
    const int q = (p & 7) ^ ((row >> 1) & 7);
    xoff[i] = (uint32_t)min(row, B - 1) * rowb + (uint32_t)(q * 16);
  }
  auto issue_x = [&]() NVJSEL_INLINE {
    const uint32_t dst = ring0 + (uint32_t)(XRING + lx * XBYTES);
    const char* src = hidden + xko;
    if (XLANES == 64 || lane < XLANES) {
#pragma unroll
      for (int i = 0; i < XL; ++i) dma16(src, xoff[i], dst + (uint32_t)((i * NW + wave) * XLANES * 16));
    }
    lx = lx + 1 == RX ? 0 : lx + 1;
    xko = xko + kRingKC * 2 == rowb ? 0u : xko + kRingKC * 2;
  };
  // NS = 3: the next hidden stage arrives as f32 in `raw`, each thread's 16-byte
  // pieces (four values) where it reads them back itself, and is split into
  // the other slot in the middle of a stage
  constexpr int RL = S::LDS_RAW / (NW * 1024);  // raw loads per wave and stage
  constexpr int RAW = XRING + RX * XBYTES;
  auto issue_raw = [&]() NVJSEL_INLINE {
    const char* src = hidden + 2 * xko;
#pragma unroll
    for (int i = 0; i < RL; ++i) {
      const int p = (i * NW + wave) * 64 + lane;  // row p >> 4, values 4 (p & 15) .. + 3
      dma16(src, (uint32_t)min(p >> 4, B - 1) * (2 * rowb) + (uint32_t)(p & 15) * 16u,
            ring0 + (uint32_t)(RAW + (i * NW + wave) * 1024));
    }
    xko = xko + kRingKC * 2 == rowb ? 0u : xko + kRingKC * 2;
  };
  auto split_raw = [&]() NVJSEL_INLINE {  // (this wave's raw loads have landed)
    char* dst = ring + XRING + lx * XBYTES;
    lx ^= 1;
#pragma unroll
    for (int i = 0; i < RL; ++i) {
      const int p = (i * NW + wave) * 64 + lane, row = p >> 4, q = (p & 15) >> 1;
      const u32x4_t r = *(const u32x4_t*)(ring + RAW + p * 16);
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = __uint_as_float(r[j]);
      char* at = dst + row * (kRingKC * 2) + ((q ^ ((row >> 1) & 7)) * 16) + (p & 1) * 8;
#pragma unroll
      for (int t = 0; t < 3; ++t) *(uint2*)(at + t * (NBR * kRingKC * 2)) = next_term(v);
    }
  };
  auto issue_w = [&]() NVJSEL_INLINE {
    const uint32_t dst = ring0 + (uint32_t)(lw * WBYTES);
    const char* src = wtile + lko;
#pragma unroll
    for (int i = 0; i < WL; ++i) dma16_nt(src, woff[i], dst + (uint32_t)((i * NW + wave) * 1024));
    lw = lw + 1 == RW ? 0 : lw + 1;
    lko += lstep;
    if (--lleft == 0) {
      lko = 0;
      lleft = nkc;
      if (++lt < my_tiles) {
        load_tile_start();
      } else {
        // past the end: every further load of W reads its first 16 bytes (the
        // number of loads in flight stays the same for the waits)
        wtile = (const char*)a.W;
        lstep = 0;
        lleft = INT_MAX;
#pragma unroll
        for (int i = 0; i < WL; ++i) woff[i] = 0u;
      }
    }
  };
  f32x16_t acc[TV][TB];
  const int h = lane >> 5, c32 = lane & 31, sw = (c32 >> 1) & 7;
  // Fragments are read one 16-wide k-step ahead of the products, across the
  // stage barrier too: two register sets, the scheduling barriers keep the
  // reads of the next step ahead of this step's products.
  int cw = 0, cx = 0;  // ring slots of the stage being multiplied
  u32x4_t fa[2][TV], fb[2][NS][TB];
  auto read_step = [&](auto set, auto KS) NVJSEL_INLINE {
    constexpr int f = decltype(set)::value, ks = decltype(KS)::value;
    const int col = ((ks * 2 + h) ^ sw) * 16 + c32 * (kRingKC * 2);
    const char* wbuf = ring + cw * WBYTES + wv * TV * 32 * (kRingKC * 2) + col;
    const char* xbuf = ring + XRING + cx * XBYTES + wb * 32 * TB * (kRingKC * 2) + col;
#pragma unroll
    for (int t = 0; t < NS; ++t)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) fb[f][t][tb] = *(const u32x4_t*)(xbuf + (t * NBR + tb * 32) * (kRingKC * 2));
#pragma unroll
    for (int tv = 0; tv < TV; ++tv) fa[f][tv] = *(const u32x4_t*)(wbuf + tv * 32 * (kRingKC * 2));
    __builtin_amdgcn_sched_barrier(0);
  };
  auto multiply = [&](auto set) NVJSEL_INLINE {
    constexpr int f = decltype(set)::value;
#pragma unroll
    for (int tv = 0; tv < TV; ++tv)
#pragma unroll
      for (int t = 0; t < NS; ++t)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
          acc[tv][tb] = MODE == MODE_LOGITS ? mfma32x32x16<WT>(fb[f][t][tb], fa[f][tv], acc[tv][tb])
                                            : mfma32x32x16<WT>(fa[f][tv], fb[f][t][tb], acc[tv][tb]);
    __builtin_amdgcn_sched_barrier(0);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  // one stage; `rest`: the previous stage of the tile left its last step's products
  auto stage = [&](auto rest) NVJSEL_INLINE {
    stage_barrier<LIVE>();
    if constexpr (NS == 3)
      issue_raw();
    else
      issue_x();
    issue_w();
    read_step(I0{}, I0{});
    if constexpr (decltype(rest)::value) multiply(I1{});
    read_step(I1{}, I1{});
    multiply(I0{});
    if constexpr (NS == 3) {
      wave_wait<WL>();  // the W stage requested behind the raw values stays in flight
      split_raw();
    }
    read_step(I0{}, I2{});
    multiply(I1{});
    read_step(I1{}, I3{});
    multiply(I0{});
    cw = cw + 1 == RW ? 0 : cw + 1;
    cx = cx + 1 == RX ? 0 : cx + 1;
  };
  uint32_t bo[TB], bi[TB];
#pragma unroll
  for (int tb = 0; tb < TB; ++tb) bo[tb] = bi[tb] = 0u;
  // ---- sample mode: per wave a queue of the entries that may be their row's
  // maximum (logit, approximate score, vocab << 7 | tb << 6 | lane); shared by
  // the waves, each row's best exact key and largest approximate score (ord_f32)
  float* const qx = (float*)(ring + S::LDS_RING) + wave * QC;
  float* const qa = (float*)(ring + S::LDS_RING) + (NW + wave) * QC;
  uint32_t* const qv = (uint32_t*)(ring + S::LDS_RING) + (2 * NW + wave) * QC;
  unsigned long long* const rowbest = (unsigned long long*)(ring + S::LDS_RING + NW * QC * 12);  // [NBR]
  uint32_t* const rowmax = (uint32_t*)(rowbest + NBR) + wb * 32 * TB + c32;
  float tp[TB], rtp[TB], amax[TB];
  bool greedy_row[TB];
  TfKey key[TB];
  unsigned long long sbest[TB];
  uint32_t qcount = 0;  // wave-uniform
  if constexpr (S::SMP) {
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
      const int b = wb * 32 * TB + tb * 32 + c32;
      const float t = b < B ? a.temperature[b] : 0.0f;
      greedy_row[tb] = (t <= 0.0f);
      tp[tb] = temp_floor(t);
      rtp[tb] = 1.0f / tp[tb];
      key[tb] = b < B ? tf_key(a.keys[2 * b], a.keys[2 * b + 1]) : tf_key(0u, 0u);
      amax[tb] = -INFINITY;
      sbest[tb] = 0ull;
      rowbest[wb * 32 * TB + tb * 32 + c32] = 0ull;  // (ordered before their first use by the stages' barriers)
      rowmax[tb * 32] = 0u;
    }
  }
  // drops queued entries that can no longer be their row's maximum (the test
  // each passed when queued, against a maximum that has only grown since);
  // compaction in place, a 64-entry group read before any survivor is written
  // at or below it
  auto compact = [&]() NVJSEL_INLINE {
    uint32_t nk = 0;
    for (uint32_t e0 = 0; e0 < qcount; e0 += 64) {  // wave-uniform trip count
      const uint32_t e = e0 + lane;
      const bool live = e < qcount;
      const float x = live ? qx[e] : 0.0f;
      const float ap = live ? qa[e] : -INFINITY;
      const uint32_t pv = live ? qv[e] : 0u;
      const int sl = (int)(pv & 63u);
      float am = __shfl(amax[0], sl, 64);
      if constexpr (TB == 2) {
        const float a1 = __shfl(amax[1], sl, 64);
        if (pv & 64u) am = a1;
      }
      const bool keep = live && !(ap + score_slack(ap, am) < am);
      const unsigned long long m = __ballot(keep);
      if (keep) {
        const uint32_t slot = nk + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                             __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        qx[slot] = x;
        qa[slot] = ap;
        qv[slot] = pv;
      }
      nk += (uint32_t)__popcll(m);
    }
    qcount = nk;
  };
  // exact scores (correctly rounded division, fp64 logs) of the queued entries,
  // a full wave at a time, folded into the rows' best keys
  auto flush = [&]() NVJSEL_INLINE {
    for (uint32_t e0 = 0; e0 < qcount; e0 += 64) {  // wave-uniform trip count
      const uint32_t e = e0 + lane;
      const bool live = e < qcount;
      const uint32_t pv = live ? qv[e] : 0u;
      const int sl = (int)(pv & 63u);
      const bool t1 = TB == 2 && (pv & 64u) != 0u;
      // the shuffles run with the whole wave active
      uint32_t kw[TB][2];
      float tw[TB];
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) {
        kw[tb][0] = (uint32_t)__shfl((int)key[tb].k0, sl, 64);
        kw[tb][1] = (uint32_t)__shfl((int)key[tb].k1, sl, 64);
        tw[tb] = __shfl(tp[tb], sl, 64);
      }
      const TfKey k2 = tf_key(t1 ? kw[TB - 1][0] : kw[0][0], t1 ? kw[TB - 1][1] : kw[0][1]);
      const uint32_t v = pv >> 7;
      if (live) atomicMax(&rowbest[wb * 32 * TB + (t1 ? 32 : 0) + (sl & 31)],
                          argmax_key(qx[e] / (t1 ? tw[TB - 1] : tw[0]) + gumbel_at(k2, v), v));
    }
    qcount = 0;
  };
  // A finished tile's logits wait in `pend` and are scored in units -- RUN
  // consecutive vocabulary rows of one of the lane's batch rows (D element e:
  // row pv0 + tv * 32 + 8 (e >> 2) + 4 h + (e & 3)) -- spread over the next
  // tile's stages, so that the draws run while W streams; the two waves of a
  // SIMD are half a period apart.  After a unit the row's elements shift
  // down: the indices stay compile-time constants.
  constexpr int NUNIT = S::SMP ? TV * (16 / RUN) * TB : 0;
  f32x16_t pend[S::SMP ? TV : 1][TB];
  int pv0 = 0, pvend = 0, punit = NUNIT, credit = 0;
  auto pending = [&]() NVJSEL_INLINE {  // (false: all scored, or only repeats of the tile's last row left)
    return punit < NUNIT && pv0 + (punit / TB * RUN >> 2) * 8 < pvend;
  };
  auto score_row = [&](auto TBI) NVJSEL_INLINE {
    constexpr int tb = decltype(TBI)::value;
    const int e0 = punit / TB * RUN, vs = pv0 + (e0 >> 2) * 8 + 4 * h + (e0 & 3);
    {
      if (qcount > (uint32_t)(QC - 64 * RUN)) {  // room for one unit of the wave
        compact();
        if (qcount > (uint32_t)(QC - 64 * RUN)) flush();
      }
      bool q[RUN], any = false;
      float val[RUN], ap[RUN];
#pragma unroll
      for (int j = 0; j < RUN; ++j) q[j] = false;
#pragma unroll
      for (int j = 0; j < RUN; ++j) val[j] = pend[0][tb][j];
      if (a.reduce_cast == 1) {
#pragma unroll
        for (int j = 0; j < RUN; ++j) val[j] = round_bf16(val[j]);
      } else if (a.reduce_cast == 2) {
#pragma unroll
        for (int j = 0; j < RUN; ++j) val[j] = round_f16(val[j]);
      }
      const bool row = wb * 32 * TB + tb * 32 + c32 < B;
      if (row && greedy_row[tb]) {
#pragma unroll
        for (int j = 0; j < RUN; ++j)
          if (vs + j < pvend) sbest[tb] = max_u64(sbest[tb], argmax_key(val[j], (uint32_t)(vs + j)));
      }
      if (row && !greedy_row[tb]) {
        float x[RUN];
        uint32_t idx[RUN], bits[RUN];
        bool big = false;
#pragma unroll
        for (int j = 0; j < RUN; ++j) {
          x[j] = val[j] * rtp[tb];
          big |= !(fabsf(x[j]) < 1e30f);  // NaN, infinities and the edge of the range: divide
          idx[j] = (uint32_t)(vs + j);
        }
        if (big) {
#pragma unroll
          for (int j = 0; j < RUN; ++j) x[j] = val[j] / tp[tb];
        }
        random_bits32_n<RUN>(key[tb], idx, bits);
        const float am = fmaxf(amax[tb], unord_f32(rowmax[tb * 32]));
        const float thr = am - (2.21e-4f + 1.37e-6f * fminf(fabsf(am), 1e30f));
        float top = -INFINITY;
#pragma unroll
        for (int j = 0; j < RUN; ++j) {
          const float t = x[j] + gumbel_fast_from_bits(bits[j]);
          ap[j] = (t != t) ? INFINITY : t;  // NaN only from a NaN logit or temperature
          const bool ok = vs + j < pvend;
          q[j] = ok && ap[j] >= thr;
          top = fmaxf(top, ok ? ap[j] : -INFINITY);
        }
        if (top > am) atomicMax(&rowmax[tb * 32], ord_f32(top));
        amax[tb] = fmaxf(am, top);
      }
      // queue the marked entries with the whole wave active: slots from a ballot
      #pragma unroll
      for (int j = 0; j < RUN; ++j) any |= q[j];
      if (__any(any)) {
#pragma unroll
        for (int j = 0; j < RUN; ++j) {
          const unsigned long long m = __ballot(q[j]);
          if (q[j]) {
            const uint32_t slot = qcount + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                     __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            qx[slot] = val[j];
            qa[slot] = ap[j];
            qv[slot] = ((uint32_t)(vs + j) << 7) | ((uint32_t)tb << 6) | (uint32_t)lane;
          }
          qcount += (uint32_t)__popcll(m);
        }
      }
      // shift the row's elements down
#pragma unroll
      for (int e = 0; e < (S::SMP ? TV : 1) * 16 - RUN; ++e)
        pend[e / 16][tb][e % 16] = pend[(e + RUN) / 16][tb][(e + RUN) % 16];
    }
    ++punit;
  };
  auto score_unit = [&]() NVJSEL_INLINE {
    if (TB == 1 || (punit & 1) == 0)
      score_row(std::integral_constant<int, 0>{});
    else
      score_row(std::integral_constant<int, TB - 1>{});
  };
  auto epilogue = [&](int t) NVJSEL_INLINE {
    const int t0 = tile_row(t);
    const int vend = min(tile_row(t + 1), r1);
    const int v0 = t0 + wv * TV * 32;
    if constexpr (NS == 3) {
      const float m = tile_max<0>(acc);
      if (__builtin_amdgcn_ballot_w64(m != m))
        redo_nan_logits<0, MODE != MODE_LOGITS>(a, acc, lane, [&](int tv, int e, int& b, int& v) NVJSEL_INLINE {
          const int row = 8 * (e >> 2) + 4 * h + (e & 3);  // of D (logits: the batch row)
          b = wb * 32 + (MODE == MODE_LOGITS ? row : c32);
          v = v0 + tv * 32 + (MODE == MODE_LOGITS ? c32 : row);
          return b < B && v < vend;
        });
    }
    if constexpr (MODE == MODE_LOGITS) {
      // operands swapped: D[batch 8 (e >> 2) + 4 h + (e & 3)][vocab c32], so
      // 32 lanes hold 32 consecutive logits of one row.  16-bit logits are
      // transposed in quads of lanes (four rows x four columns) and stored 8
      // bytes per lane, at any element address (V = 50,257, H = 512, B = 129 /
      // 256 28 / 34 us, as 2-byte stores 42 / 52); the vocabulary's last quad may be partial.
      typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
      typedef u32x2_t u32x2_any_t __attribute__((aligned(2)));
      const bool quads = a.out_dtype != DT_F32;
#pragma unroll
      for (int tv = 0; tv < TV; ++tv) {
        const int v = v0 + tv * 32 + c32;
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int b = wb * 32 * TB + tb * 32 + 8 * i + 4 * h;
            float x[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = apply_cast(acc[tv][tb][4 * i + j], a.reduce_cast);
            if (quads) {
              const uint2 q = quad_transpose16(x, a.out_dtype, lane);
              const int left = vend - (v & ~3);  // columns of this quad
              if (left > 0 && b + (lane & 3) < B) {
                uint16_t* out = (uint16_t*)a.out_logits + (size_t)(b + (lane & 3)) * (size_t)a.out_stride + (v & ~3);
                if (left >= 4) {
                  *(u32x2_any_t*)out = u32x2_t{q.x, q.y};
                } else {
                  out[0] = (uint16_t)q.x;
                  if (left > 1) out[1] = (uint16_t)(q.x >> 16);
                  if (left > 2) out[2] = (uint16_t)q.y;
                }
              }
            } else {
#pragma unroll
              for (int j = 0; j < 4; ++j)
                if (v < vend && b + j < B) store_logit(a, b + j, v, x[j]);
            }
          }
      }
    } else if constexpr (S::SMP) {
#pragma unroll
      for (int tv = 0; tv < TV; ++tv)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) pend[tv][tb] = acc[tv][tb];
      pv0 = v0;
      pvend = vend;
      punit = 0;
      credit = wave >= NW / 2 ? nkc / 2 : 0;
    } else {
      if (v0 + TV * 32 > vend) {  // rows past the tile's end repeat its last row
#pragma unroll
        for (int tv = 0; tv < TV; ++tv)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            if (v0 + tv * 32 + 8 * (e >> 2) + 4 * h + (e & 3) >= vend) {
#pragma unroll
              for (int tb = 0; tb < TB; ++tb) acc[tv][tb][e] = -INFINITY;
            }
      }
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) {
        float m = acc[0][tb][0];
#pragma unroll
        for (int i = 1; i < TV * 16 - 1; i += 2)
          m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, acc[i / 16][tb][i % 16]),
                                            acc[(i + 1) / 16][tb][(i + 1) % 16]);
        m = __builtin_elementwise_maximum(m, acc[TV - 1][tb][15]);
        const float rm = apply_cast(m, a.reduce_cast);
        const uint32_t om = ord_f32(rm);
        const bool up = om > bo[tb];
        if (__builtin_amdgcn_ballot_w64(up)) {
          // the first element that rounds to the maximum: rounding is monotone,
          // so these are the elements at or above a bound (a NaN maximum and
          // f16 rounding are compared value by value)
          int first = 0;
          if (a.reduce_cast == 2 || __builtin_amdgcn_ballot_w64(rm != rm)) {
            const bool nan = rm != rm;
#pragma unroll
            for (int i = TV * 16 - 1; i >= 0; --i) {
              const float x = apply_cast(acc[i / 16][tb][i % 16], a.reduce_cast);
              if (nan ? x != x : x == rm) first = (i / 16) * 32 + 8 * ((i % 16) >> 2) + (i & 3);
            }
          } else {
            const float lo = a.reduce_cast == 1 ? bf16_round_low(rm) : m;
#pragma unroll
            for (int i = TV * 16 - 1; i >= 0; --i)
              if (acc[i / 16][tb][i % 16] >= lo) first = (i / 16) * 32 + 8 * ((i % 16) >> 2) + (i & 3);
          }
          if (up) {
            bo[tb] = om;
            bi[tb] = (uint32_t)(v0 + first + 4 * h);
          }
        }
      }
    }
  };
  // the pending tile's share of units of one stage
  auto score_share = [&]() NVJSEL_INLINE {
    for (credit += NUNIT; credit >= nkc; credit -= nkc)
      if (pending()) score_unit();
  };
  if (my_tiles > 0) {
    load_tile_start();
    // as the loop would have left them: X(0) .. X(RX - 2), each W stage RW - RX
    // ahead of the hidden stage issued with it
    if constexpr (NS == 3) {
      issue_raw();
      wave_wait<0>();
      split_raw();
      for (int s = 0; s < RW - 1; ++s) issue_w();
    } else {
      for (int s = 0; s < RW - RX; ++s) issue_w();
      for (int s = 0; s < RX - 1; ++s) {
        issue_x();
        issue_w();
      }
    }
    for (int t = 0; t < my_tiles; ++t) {
#pragma unroll
      for (int tv = 0; tv < TV; ++tv)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[tv][tb][e] = 0.f;
      stage(std::false_type{});
      for (int kc = 1; kc < nkc; ++kc) {
        if constexpr (S::SMP) score_share();
        stage(std::true_type{});
      }
      if constexpr (S::SMP) score_share();
      multiply(I1{});
      epilogue(t);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still write the LDS when it is given back
  }
  if constexpr (MODE == MODE_LOGITS) return;
  unsigned long long (*kred)[NBR] = (unsigned long long (*)[NBR])ring;  // [WV][NBR]
  unsigned long long best[TB];
  if constexpr (S::SMP) {
    while (pending()) score_unit();  // the last tile
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) amax[tb] = fmaxf(amax[tb], unord_f32(rowmax[tb * 32]));
    compact();
    flush();
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) best[tb] = sbest[tb];  // (sampled rows: rowbest)
  } else {
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) best[tb] = bo[tb] ? ((unsigned long long)bo[tb] << 32) | (unsigned long long)(~bi[tb]) : 0ull;
  }
  __syncthreads();  // every wave has left the ring
#pragma unroll
  for (int tb = 0; tb < TB; ++tb) {
    best[tb] = max_u64(best[tb], shfl_xor_u64(best[tb], 32));
    if (h == 0) kred[wv][wb * 32 * TB + tb * 32 + c32] = best[tb];
  }
  __syncthreads();
  for (int b = (int)threadIdx.x; b < B; b += NW * 64) {
    unsigned long long m = kred[0][b];
#pragma unroll
    for (int q = 1; q < WV; ++q) m = max_u64(m, kred[q][b]);
    if constexpr (S::SMP) m = max_u64(m, rowbest[b]);
    if (m) (void)after(atomicMax(&a.row_keys[b], m));
  }
  __syncthreads();
  finish_rows(a.row_keys, a.counter, a.B, a.out_ids, a.out_best, (int*)ring);
}

template <int WT, int MODE, int NBR, int NS>
static int launch_ring_rows(const LmArgs& a, hipStream_t stream) {
  using S = RingShape<MODE, NBR, NS>;
  const int rows = ring_share(a.V, device_cu_count());  // every block reads the same share of W, contiguous
  hipLaunchKernelGGL((lm_head_ring_kernel<WT, MODE, NBR, NS>), dim3((a.V + rows - 1) / rows), dim3(S::NW * 64), 0, stream,
                     a, rows);
  NVJSEL_CHECK_LAUNCH("lm_head_ring_kernel");
  return NVJSEL_OK;
}

template <int WT, int MODE>
static int launch_ring_mode(const LmArgs& a, hipStream_t stream) {
  if (a.B <= 32) return launch_ring_rows<WT, MODE, 32, 1>(a, stream);
  if (a.B <= 64) return launch_ring_rows<WT, MODE, 64, 1>(a, stream);
  if (a.B <= 128) return launch_ring_rows<WT, MODE, 128, 1>(a, stream);
  if constexpr (MODE != MODE_SAMPLE) return launch_ring_rows<WT, MODE, 256, 1>(a, stream);
  return fail(NVJSEL_EINVAL, "launch_ring: at most 128 sampled rows per pass");
}

template <int MODE>
static int launch_ring_f32(const LmArgs& a, hipStream_t stream) {
  if (a.B <= 32) return launch_ring_rows<DT_BF16, MODE, 32, 3>(a, stream);
  if (a.B <= 64) return launch_ring_rows<DT_BF16, MODE, 64, 3>(a, stream);
  return fail(NVJSEL_EINVAL, "launch_ring: at most 64 rows of f32 activations per pass");
}

int launch_ring(int mode, const LmArgs& a, hipStream_t stream) {
  auto by_mode = [&](auto fn) -> int {
    if (mode == MODE_GREEDY) return fn(std::integral_constant<int, MODE_GREEDY>{});
    if (mode == MODE_SAMPLE) return fn(std::integral_constant<int, MODE_SAMPLE>{});
    return fn(std::integral_constant<int, MODE_LOGITS>{});
  };
  if (a.hidden_dtype == DT_F32) return by_mode([&](auto M) { return launch_ring_f32<decltype(M)::value>(a, stream); });
  if (a.weight_dtype == DT_F16) return by_mode([&](auto M) { return launch_ring_mode<DT_F16, decltype(M)::value>(a, stream); });
  return by_mode([&](auto M) { return launch_ring_mode<DT_BF16, decltype(M)::value>(a, stream); });
}

}  // namespace nvjsel
