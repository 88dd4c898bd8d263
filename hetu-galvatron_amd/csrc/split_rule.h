// Into how many pieces the reduction of a 128x128-tile launch is cut.  The host asks to choose a launch and
// its workspace, and both kernels of a split launch ask for themselves: the first writes partial tiles where
// the second expects them only if all come to the same count.  Hence integers, in nanoseconds: a comparison
// of floats may be rounded differently where two compilations contract its products differently.
#pragma once
#include <cstdint>

namespace gmoe {

constexpr int kMaxSplit = 8;
// workgroups a split launch may spread over, i.e. the 128x128 partial tiles its workspace holds
constexpr int kSplitSlots = 512;

// Time of a K tile (64 elements) of a tile that has its CU to itself, of the second kernel, and of the 128 KiB
// of partial sums that a piece writes and reads again.
constexpr int64_t kSplitNsPerKTile = 420, kSplitReduceNs = 6000, kSplitNsPerPiece = 26;

// Time in which the weights stream from memory, at 6.5 TB/s.
__host__ __device__ constexpr int64_t weight_stream_ns(int64_t E, int64_t K, int64_t M, int elem_bytes) {
  return E * K * M * elem_bytes / 6500;
}

// Pieces for every tile, 1 for an unsplit launch.  A split launch cannot end before the weights have been
// streamed (`stream_ns`).  Measured on both sides of the line: 128 tiles of 44 K tiles 27 unsplit against
// 32 us in four pieces, 64 tiles of 16 K tiles 13 against 21, 96 tiles of 64 K tiles 45 against 32;
// 256 tiles of 224 K tiles (940 MB of weights) 159 against 193.
__host__ __device__ inline int split_pieces(int64_t k_tiles, int64_t tiles, int64_t slots, int64_t stream_ns) {
  if (tiles <= 0) return 1;
  int64_t most = slots / tiles;
  if (most > kMaxSplit) most = kMaxSplit;
  if (most > k_tiles) most = k_tiles;
  if (most < 2) return 1;
  const int64_t whole = kSplitNsPerKTile * k_tiles, per_piece = kSplitNsPerPiece * tiles;
  // sqrt(whole / per_piece), where whole / s + per_piece * s is smallest, rounded to the nearest
  int64_t s = most;
  while (s > 2 && (2 * s - 1) * (2 * s - 1) * per_piece > 4 * whole) --s;
  const int64_t split = whole / s > stream_ns ? whole / s : stream_ns;
  return whole - split > kSplitReduceNs + per_piece * s ? (int)s : 1;
}

// Pieces of the reduction of an fp32 NN / NT launch (gmm_f32.hip), each a result of its own in the workspace; only
// the host asks.  Times in ns per stage of 32 reduction elements, measured: 2600 for two 128-row tiles of a CU,
// 2000 for a lone one, 1700 and 1300 for 64-row tiles, 5000 around a tile, 4000 and the traffic for the sums.
// A round of 512 tiles ends with its slowest, so three pieces of 144 tiles beat two and four (us in 1, 2, 3, 4, 6
// pieces, 4096 x 2048 x 512 over 8 experts: 110, 93, 73, 88, 84; 2000 x 5632 x 1024: 269, 214, 170, 204, 187;
// 130 x 3584 x 896 over 4, in 1, 4, 8, 16: 153, 48, 30, 24).  A launch with a full round stays whole (4096 x
// 512 x 2048: 81, in two pieces 87).
constexpr int kF32MaxPieces = 16;

inline int gmm_f32_pieces(int64_t E, int64_t N, int64_t K, int64_t M) {
  if (N < 1) return 1;
  const int64_t cols = (M + 127) / 128, busy = N < E ? N : E, stages = (K + 31) / 32;
  // the last tile of an expert is half full on average
  int64_t tiles128 = (N + 127) / 128 + E / 2, tiles64 = (N + 63) / 64 + E / 2;
  if (tiles128 < busy) tiles128 = busy;
  if (tiles64 < busy) tiles64 = busy;
  const int64_t stream_ns = weight_stream_ns(E, K, M, 4);
  int best = 1;
  int64_t best_ns = 0;
  for (int s = 1; s <= kF32MaxPieces && s <= stages; ++s) {
    if (s > 1 && s * N * M > (int64_t)kSplitSlots * 128 * 128) break;
    const bool small = tiles128 * cols * s <= kSplitSlots / 2;  // the kernel's own rule
    int64_t tiles = (small ? tiles64 : tiles128) * cols * s;
    tiles += tiles / 16;  // loads are uneven
    const int64_t rounds = tiles / kSplitSlots, rest = tiles % kSplitSlots, per_piece = (stages + s - 1) / s;
    const int64_t pair = per_piece * (small || tiles64 == tiles128 ? 1700 : 2600) + 5000;
    const int64_t lone = per_piece * (small || tiles64 == tiles128 ? 1300 : 2000) + 5000;
    int64_t ns = rounds * pair + (rest == 0 ? 0 : (rest <= kSplitSlots / 2 ? lone : pair));
    if (ns < stream_ns) ns = stream_ns;
    if (s > 1) ns += 4000 + (s + 1) * N * M / 1000;  // 4 bytes at 4 TB/s
    if (s == 1 || ns < best_ns) {
      best = s;
      best_ns = ns;
    }
  }
  return best;
}

}  // namespace gmoe
