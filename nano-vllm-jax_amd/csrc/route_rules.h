// Rules that choose between paths by sizes alone, in plain C++ (constexpr:
// usable in host and device code, and compiled by the CPU tests).
#pragma once

namespace nvjsel {

// ---- top-k rows of the sampler (k <= 256) on `nc` scan chunks of four waves.
// Each wave publishes its four largest lane maximums and each chunk lists its
// elements down to tier A (at least 32 of them); a row is settled from the
// lists if the row floor -- the larger of the k-th of the 16 nc published
// values and the largest chunk floor -- reaches every chunk's tier A, and
// takes a whole-row descent if not.  That holds for k <= 32 (a chunk's own
// floor does) and from 16 nc = 9/8 k on: those rows want nothing more, and
// publishing or listing more for them only costs (k = 256 at 31 chunks 37 us
// against 58 with tier B).  Below, eight maximums per wave settle the row
// where 32 nc >= 7/5 k (the last chunk may hold little); tier B (the lists down
// to the chunk's own floor) where 32 nc >= 6/5 k, or few chunks hold the row,
// and the lists stay within their 512 entries.  Elsewhere (k = 256 below 12
// chunks, k = 160 at two, 200 at one) most rows would still miss, and their
// descent is not delayed by it
// (k = 256 at one chunk 55 us against 71 with tier B).
// V = 50,257 / 98,304, k = 100, 64 rows: 270 / 413 -> 51 / 31 us.
constexpr bool topk_floor_low(int nc, int k) { return k > 32 && 128 * nc < 9 * k; }
constexpr bool topk_tier_b(int nc, int k) {
  return topk_floor_low(nc, k) && 64 * nc < 3 * k && (160 * nc >= 6 * k ? k <= 200 : k <= 160 && nc * k <= 300);
}
constexpr bool topk_more_tops(int nc, int k) {
  return topk_floor_low(nc, k) && (160 * nc >= 7 * k || topk_tier_b(nc, k));
}

}  // namespace nvjsel
