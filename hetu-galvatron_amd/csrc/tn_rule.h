// Which kernel a 16-bit dW launch (TN) takes: 128x128 tiles (gmm.hip), 256x256 ones (gmm_dtl.hip), or 128x256 ones with two
// workgroups per CU (gmm_tn.hip).  Only the host asks.
#pragma once
#include <cstdint>

namespace gmoe {

enum TnKernel { TN_SMALL, TN_LARGE, TN_SHORT };

// dW results from here on are written past the caches (gmm_common.h).
inline bool tn_streams(int64_t E, int64_t K, int64_t M) { return E * K * M * 2 >= (256ll << 20); }

// The 128x128 kernel runs at about 0.4 of the large one's rate per FLOP, so the large tiles win as soon as the small
// ones need a second round of their 512 slots (one expert, 176 large tiles: 0.29 -> 0.22 ms)
inline bool tn_large_tiles(int64_t E, int64_t K, int64_t M) {
  return K >= 512 && M >= 256 && E * ((K + 255) / 256) * ((M + 255) / 256) >= 129;
}

// dW of 16-bit operands with a short reduction (gmm_tn.hip: 128x256 tiles, two workgroups per CU) against the
// 256x256 LDS-DMA kernel, or 128x128 tiles where that one does not apply; n = rows per expert, us of that kernel /
// of this one.  From one round of 256x256 tiles on that kernel, whose tiles run into each other, is the faster one
// (n 128 402 / 484, n 383 784 / 879, n 1024 1671 / 1875, 8 experts of 4096 x 28672) except for few rows: n 24, 8
// experts of 6144 x 16384 291 / 266, n 48 291 / 297, n 96 299 / 368; in whole steps n 8 717 / 707, n 32 1662 / 1649,
// n 45 1693 / 1692, n 56 834 / 846, n 75 1752 / 1824, n 100 1128 / 1182 us. A result under 256 MB has the ordinary
// stores there and nontemporal ones here, which moves the line: 1024 x 5632, 16 n 24 44 / 41, n 64 45 / 44, n 96 49
// / 47; 1024 x 1024, 64 n 64 33 / 34, n 96 37 / 36; 2048 x 1184, 32 n 64 40 / 40, n 96 42 / 43.  With less than a
// round of 256x256 tiles, and where its rows would be padding (K under 512), the smaller tiles spread better: 128
// tiles of 256x256 14.0 / 11.1 (n 256, 1024 x 1024, 8), 240 17.8 / 15.4 (n 300, 640 x 1280, 16), n 384 of 384 x
// 4096 over 64 159 / 117.  That holds beyond the 768 rows up to which it is used (n 1024 of 1024 x 1024 29.4 /
// 22.5).  Fewer than three quarters of a tile per CU stay with 128x128 ones (128 tiles of 1024 x 512, 8: 10.1 /
// 9.9).
constexpr int64_t kTnFewRows = 112, kTnFewRowsStreamed = 48;
inline bool tn_short_pays(int64_t E, int64_t N, int64_t K, int64_t M, int64_t cus) {
  const int64_t n = N / E, col_tiles = (M + 255) / 256;
  if (K < 128 || M < 256 || E * ((K + 127) / 128) * col_tiles * 4 < cus * 3) return false;
  const bool few = n < (tn_streams(E, K, M) ? kTnFewRowsStreamed : kTnFewRows);
  if (!few && K >= 512 && E * ((K + 255) / 256) * col_tiles >= cus) return false;
  return n <= 768;
}

// dW outside those two rules (narrow results: K under 512, M under 256, or fewer than 129 tiles of 256x256): the
// kernel with the least estimated time, us, of n rows per expert in `rounds` rounds of its tiles.  Two workgroups of
// the smaller tiles share a CU, and a last round of at most half their slots takes `half` of one.  Fitted to 5600
// launches of 1 to 64 experts, 1 to 9000 rows each, even and uneven loads, K and M of 128 to 16000; an estimate
// has to be 8 % better to leave the 128x128 tiles.  Over those launches it costs 1.1 % against the best kernel of each, the
// 128x128 tiles throughout 8.6 %; 38 % of the launches are more than 3 % faster than in those, 2 % are more than 3 %
// slower: uneven loads, of which the host knows nothing and where the heaviest expert's tiles decide.  us on 128x128 /
// 256x256 / 128x256 tiles: 1619 rows, 64 experts, 256 x 7680 613 / 402 / 516; 22 rows, 16 experts, 704 x 128 6.2 / 8.1 /
// 5.4; 1975 rows, 32 experts, 384 x 896, the heaviest 12114 129 / 219 / 189.
struct TnCosts {
  int rows, cols, per_cu;
  double launch, round, per_row, half;
};
constexpr TnCosts kTnSmall = {128, 128, 2, 3.0, 6.91, 0.0174, 0.489}, kTnLarge = {256, 256, 1, 3.69, 4.87, 0.0235, 0.82},
                  kTnShort = {128, 256, 2, 1.56, 5.0, 0.0292, 0.618};
inline double tn_estimate(const TnCosts& c, int64_t E, int64_t N, int64_t K, int64_t M, int64_t cus) {
  const int64_t tiles = E * ((K + c.rows - 1) / c.rows) * ((M + c.cols - 1) / c.cols);
  const int64_t slots = c.per_cu * cus, rest = tiles % slots;
  const double rounds = (double)(tiles / slots) + (rest == 0 ? 0.0 : rest * 2 <= slots ? c.half : 1.0);
  return c.launch + rounds * (c.round + c.per_row * (double)(N / E));
}

// `narrow`: whether the estimate is asked (32-bit results, the gate's, were not part of the fit).
inline TnKernel tn_kernel(int64_t E, int64_t N, int64_t K, int64_t M, int64_t cus, bool narrow) {
  if (E < 1) E = 1;
  if (tn_short_pays(E, N, K, M, cus)) return TN_SHORT;
  if (tn_large_tiles(E, K, M)) return TN_LARGE;
  if (!narrow || K < 128 || M < 128) return TN_SMALL;
  const double large = tn_estimate(kTnLarge, E, N, K, M, cus), both = tn_estimate(kTnShort, E, N, K, M, cus);
  if ((large < both ? large : both) >= 0.92 * tn_estimate(kTnSmall, E, N, K, M, cus)) return TN_SMALL;
  return large < both ? TN_LARGE : TN_SHORT;
}

}  // namespace gmoe
