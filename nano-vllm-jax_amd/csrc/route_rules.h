// Rules that choose between paths by sizes alone, in plain C++ (constexpr:
// usable in host and device code, and compiled by the CPU tests).
#pragma once

namespace nvjsel {

// ---- top-k rows of the sampler (k <= 256) on `nc` scan chunks of four waves,
// the last one `fill` eighths full (1-8).  Each wave publishes its four largest
// lane maximums and each chunk lists its elements down to tier A (at least 32
// of them); a row is settled from the lists if the row floor -- the larger of
// the k-th of the 16 nc published values and the largest chunk floor -- reaches
// every chunk's tier A, and takes a whole-row descent if not (64 f32 rows at 10
// chunks 380 us against 25).  k <= 32 rows always settle (a chunk's own floor
// does); the others want twice the published values until 16 nc = 7/5 k (one
// more load: no measured cost), and below 16 nc = k tier B, the lists down to
// the chunk's own floor (k = 128-160 rows 31 us with it where they settle
// without, 26), as long as its floors come out high enough:
//  * from the published values, once 32 nc (counting the last chunk's fill)
//    reaches 0.88 k, 1.16 k above 160 (k = 160 at 4.25 / 5 chunks 187 / 51 us
//    with, 172 / 196 without; k = 200 at 6.25 / 9 253 / 37 and 240 / 441), and
//  * from a single chunk's, while the survivors stay below 512: k = 128 at 2 /
//    2.25 / 2.6 chunks 40 / 93 / 127 us with, 97 / 106 / 118 without; k = 160 at
//    1.25 / 1.6 chunks 43 / 94 and 75 / 87.
// Above k = 200 the lists hold tier B only just before nothing needs it (k =
// 256 at 12 chunks of 16 bits 52 us with, 230 without; at 11 434 and 430).
constexpr bool topk_more_tops(int nc, int k) { return k > 32 && k <= 256 && 80 * nc < 7 * k; }
constexpr bool topk_tier_b(int nc, int k, int fill) {
  if (k <= 32 || 16 * nc >= k) return false;
  const int e = 8 * (nc - 1) + fill;  // the row in eighths of a chunk
  if (k <= 160) return 50 * e >= 11 * k || e * k <= (k <= 128 ? 2400 : 1600);
  if (k <= 200) return 100 * e >= 29 * k;
  return 200 * e >= 73 * k && 1600 * nc <= 82 * k;
}

}  // namespace nvjsel
