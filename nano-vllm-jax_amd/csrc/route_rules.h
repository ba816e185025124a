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
// does); the others take the next four of each wave too until 16 nc = 7/5 k (they
// come in the same words), and below 16 nc = k tier B, the lists down to
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

// ---- the staged GEMM (lm_head_ring.hip) against the tile kernel: 16-bit
// weights [V, 1024] and bf16 activations, which both take.

// Vocabulary rows per block of the staged GEMM, and the tiles of 256 they are
// cut into: a remainder costs a whole tile's requests and products.
constexpr int ring_share(int V, int cus) { return ((V + cus - 1) / cus + 7) / 8 * 8; }
constexpr int ring_tiles(int share) { return (share + 255) / 256; }

// Whether the staged GEMM takes a greedy / logits call of up to 64 rows.
// Greedy: both stream W; the tile kernel (tiles of 16 rows, round robin) is
// 2-30% faster on most vocabularies (V = 66,000 / 151,936 / 200,064, B = 16 24 /
// 49 / 62 us against 31 / 52 / 68), equal on long shares that fill their tiles
// (V = 248,320 / 311,296 76-77 / 95 both ways; not at whole MBs of W, 80 against
// 84 at V = 262,144), and 3-12% slower from 49 rows on one well filled tile (V
// = 57,344, B = 64 28.0 against 25.1).  Logits: the tile kernel stores a row's
// logits 32 bytes at a time, so the staged GEMM is ahead from fewer full tiles
// the more rows there are (V = 98,304, B = 8 / 16 / 24 / 64 34 / 36 / 40 / 59 us
// in the tile kernel against 35 / 35 / 36 / 42).
constexpr bool ring_takes_small(bool logits, int batch, int V, int cus) {
  const int share = ring_share(V, cus), tiles = ring_tiles(share), full = 256 * tiles;
  const bool longer = tiles >= 4 && 18 * share >= 17 * full && share % 1024 != 0;
  if (!logits) return longer || (batch > 48 && tiles == 1 && 4 * share >= 3 * full);
  if (batch <= 8) return longer;
  if (batch <= 16) return 32 * share >= (batch <= 12 ? 28 : 25) * full && share != 256;
  if (batch <= 24) return 4 * share >= 3 * full;
  if (tiles == 1) return 8 * share >= 3 * full;
  return batch > 32 || 8 * share >= 5 * full;
}

// Whether it takes a sampled call of 65-128 rows: it costs about 21 + 33 t, 13 +
// 40 t, 13 + 41 t or 16 + 49 t us for t tiles (a remainder of a few rows half a
// tile) at 65-68, 69-80, 81-96 or more rows, the tile kernel's two passes 22 +
// 0.17 r, 24 + 0.18 r, 28 + 0.16 r or 30 + 0.18 r for a share of r rows (V =
// 40,960 / 98,304 / 248,320, each call after a pause: B = 80 56 / 92 / 183 us in the
// tile kernel against 53 / 92 / 162; B = 96 56 / 89 / 182 against 54 / 92 / 166; B =
// 128 63 / 101 / 197 against 63 / 109 / 194).
constexpr bool ring_takes_sample(int batch, int V, int cus) {
  const int share = ring_share(V, cus), rem = share % 256;
  const int t8 = share / 256 * 8 + (rem == 0 ? 0 : rem <= 16 ? 4 : rem <= 32 ? 5 : 8);  // eighths of tiles
  if (batch <= 68) return 8 * share >= 230 * t8 - 600;
  if (batch <= 80) return 8 * share >= 225 * t8 - 528;
  if (batch <= 96) return 8 * share >= 255 * t8 - 768;
  return 8 * share >= 268 * t8 - 784;
}

}  // namespace nvjsel
