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

// Time of a K tile of 128 bytes of a tile that has its CU to itself, of the second kernel, and of the 128 KiB
// of partial sums that a piece writes and reads again.
__host__ __device__ constexpr int64_t split_ns_per_k_tile(int elem_bytes) { return elem_bytes == 2 ? 420 : 2100; }
constexpr int64_t kSplitReduceNs = 6000, kSplitNsPerPiece = 26;

// Time in which the weights stream from memory, at 6.5 TB/s.
__host__ __device__ constexpr int64_t weight_stream_ns(int64_t E, int64_t K, int64_t M, int elem_bytes) {
  return E * K * M * elem_bytes / 6500;
}

// Pieces for every tile, 1 for an unsplit launch.  A split launch cannot end before the weights have been
// streamed (`stream_ns`).  Measured on both sides of the line: 128 tiles of 44 K tiles 27 unsplit against
// 32 us in four pieces, 64 tiles of 16 K tiles 13 against 21, 96 tiles of 64 K tiles 45 against 32, fp32
// 4 tiles of 16 K tiles 36 against 14; 256 tiles of 224 K tiles (940 MB of weights) 159 against 193.
__host__ __device__ inline int split_pieces(int64_t ns_per_k_tile, int64_t k_tiles, int64_t tiles, int64_t slots,
                                            int64_t stream_ns) {
  if (tiles <= 0) return 1;
  int64_t most = slots / tiles;
  if (most > kMaxSplit) most = kMaxSplit;
  if (most > k_tiles) most = k_tiles;
  if (most < 2) return 1;
  const int64_t whole = ns_per_k_tile * k_tiles, per_piece = kSplitNsPerPiece * tiles;
  // sqrt(whole / per_piece), where whole / s + per_piece * s is smallest, rounded to the nearest
  int64_t s = most;
  while (s > 2 && (2 * s - 1) * (2 * s - 1) * per_piece > 4 * whole) --s;
  const int64_t split = whole / s > stream_ns ? whole / s : stream_ns;
  return whole - split > kSplitReduceNs + per_piece * s ? (int)s : 1;
}

}  // namespace gmoe
