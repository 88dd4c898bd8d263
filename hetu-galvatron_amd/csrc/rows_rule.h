// Whether a 16-bit NN / NT launch goes to the row-adaptive tiles (gmm_rows.hip): what it takes there against what
// it takes on the 256x256 tiles, or on 128x128 ones where those are too few (only the
// host asks); and into which chunks the kernel cuts an expert's rows.
//
// Both sides were measured for 3400 shapes (E 1-64, 72-2040 rows per expert, K 256-28672, M 128-28672, 3e8 to 4e12
// operations, weights from HBM, loads that differ by 7 %), and the constants are fitted to them.  us of the other
// tiles / of these, with the choice (rows per expert, K x M, experts):
//   * forward with activation: 382, 4096 x 28672, 8 1004 / 724 these; 139, 2048 x 2816, 64 238 / 188 these; 640,
//     1024 x 5632, 16 162 / 168 others; 1024, 7168 x 4096, 32 1657 / 1624 these.
//   * NN: 382, 14336 x 4096, 8 537 / 330 these; 1024, 1408 x 2048, 64 374 / 370 these; 267, 576 x 832, 64 34 / 41
//     others; 921, 1536 x 128, 64 39 / 55 others.
//   * NT: 382, 28672 x 4096, 8 1074 / 737 these; 640, 5632 x 1024, 16 158 / 137 these; 740, 14336 x 4096, 8 644 / 729
//     others (here two operands come in 64-byte pieces of a row, there in 128-byte ones); 1000, 640 x 128, 64 29 / 38
//     others.
//   * activation backward: 382, 4096 x 14336, 8 525 / 455 these; 640, 1024 x 2816, 16 128 / 119 these; 1000, 4096 x
//     14336, 8 886 / 945 others; 192, 1024 x 1024, 48 55 / 60 others.
// It knows the average load only, and where that is close to whole rounds it can be wrong: 376, 576 x 1376, 16 24.5 /
// 26.6 these; 402, 896 x 1408, 24 with activation 50 / 57 these; 937, 4896 x 1728, 4 77 / 71 others.  In all, the
// choice costs 1.2 % against the better side of every shape; a limit on each size cost 1.9 %, and these tiles only
// from 1024 reduction elements and three quarters of a round on 2.7 %.
#pragma once
#include "split_rule.h"

namespace gmoe {

// Rows of a chunk, in units of 64: the size, of 4, 3 and 2, that ends first.  v[0]: units of all experts, v[2..4]:
// their chunks of up to so many units.  A stage of a tile of u units takes as long as its operands stream, 16 + 4 u
// KiB at 42 GB/s; prologue and epilogue take as long as 250 KiB.  Where the largest chunks leave a round part
// empty, smaller ones fill it (us with chunks of up to 256 rows / with these, rows per expert: NT 640, 5632 x 1024,
// 16 experts 146 / 137; NN 640, 2816 x 1024, 16 75 / 69; with the activation 817, 6432 x 4832, 8 468 / 428).  Asked
// by the kernel.
constexpr int kRowsMaxUnits = 4;
__host__ __device__ inline int rows_chunk_units(const int (&v)[kRowsMaxUnits + 1], int col_tiles, int grid, int64_t K) {
  const float fixed = 16.f + 250.f / (float)((K + 31) / 32);
  int best = kRowsMaxUnits;
  float least = 0.f;
#pragma unroll
  for (int u = kRowsMaxUnits; u >= 2; --u) {
    const int rounds = (int)(((long long)v[u] * col_tiles + grid - 1) / grid);
    const float cost = (float)rounds * (fixed + 4.f * (float)v[0] / (float)(v[u] > 0 ? v[u] : 1));
    if (u == kRowsMaxUnits || cost < 0.95f * least) {
      best = u;
      least = cost;
    }
  }
  return best;
}

enum RowsKind { ROWS_NN, ROWS_NN_GLU, ROWS_NT, ROWS_NT_GLU_BWD };

// Times in ns, rates in bytes or operations per ns.
struct RowsCosts {
  // row-adaptive: around a tile, around each 64 rows of it, a stage of 32 reduction elements, share of a tile's
  // time that a round saves as its tiles get fewer, around the launch, operations
  double tile, unit, stage, lone_gain, launch, ops;
  // 256x256 tiles: around one, 64 reduction elements, operations
  double large_tile, large_step, large_ops;
  // 128x128 tiles: around one, 64 reduction elements with two tiles on a CU and with one, around the split's sums
  double small_tile, small_pair, small_lone, sums;
  // around either launch; the weights' stream
  double other_launch, weights;
};
constexpr RowsCosts kRowsCosts[] = {
    {5320, 795, 721, 0.44, 6650, 1.14e6, 8000, 1410, 1.0e6, 3540, 1250, 563, 8890, 5550, 4470},
    {2610, 1850, 814, 0.52, 7170, 1.6e6, 8610, 1500, 1.06e6, 4900, 1250, 753, 0, 1120, 4840},
    {4310, 918, 778, 0.05, 6170, 1.6e6, 6170, 1360, 1.37e6, 831, 1420, 365, 0, 8230, 5380},
    {0, 5240, 848, 0.11, 8970, 1.03e6, 22600, 1410, 1.57e6, 1360, 1580, 387, 4680, 15000, 4120}};
constexpr double kRowsWeights = 6000;

// Rows per expert from which short last row tiles have a launch of their own beside the 256x256 ones.
constexpr int64_t kNnRemainderRows = 2048;

// 256x256 tiles for NN / NT: an expert's share of rows can fill them and there are enough for every CU.
inline bool nn_large_tiles(int64_t E, int64_t N, int64_t M) {
  return N / E >= 512 && M >= 256 && (N + 255) / 256 * ((M + 255) / 256) >= 256;
}

// Pieces of a 128x128-tile launch's reduction (16-bit), from the host-side sizes: an expert has at least one row
// tile, and its last one is half full on average.
inline int nn_split_pieces(int64_t E, int64_t N, int64_t K, int64_t M) {
  const int64_t least = N < E ? N : E, average = (N + 127) / 128 + E / 2;
  const int64_t tiles = (average > least ? average : least) * ((M + 127) / 128);
  return split_pieces((K * 2 + 127) / 128, tiles, kSplitSlots, weight_stream_ns(E, K, M, 2));
}

// Five times the mean of f(rows of an expert), for loads that differ by up to 14 %.
template <typename F>
inline int64_t over_loads(int64_t E, int64_t n, F f) {
  if (E == 1) return 5 * f(n);
  int64_t sum = 0;
  for (int q = -2; q <= 2; ++q) sum += f(n * (100 + 7 * q) / 100);
  return sum;
}

// K, M as in the product (with the activation M = 2F); cus: workgroups of a persistent grid, one per CU.
inline bool rows_pays(RowsKind kind, int64_t E, int64_t N, int64_t K, int64_t M, int64_t cus) {
  const int64_t n = N / (E > 0 ? E : 1);
  // fewer rows: an expert is one tile either way, and its weights bound the launch; shorter reductions:
  // prologue and epilogue weigh as much; many rows: the 256x256 tiles have their remainder launches
  if (n < 96 || n >= kNnRemainderRows || K <= 512) return false;
  const RowsCosts& c = kRowsCosts[kind];
  const bool glu = kind == ROWS_NN_GLU, large = nn_large_tiles(E, N, M);
  const double weights = (double)E * K * M * 2, ops = 2.0 * N * K * M;
  auto cdiv = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  auto most = [](double a, double b) { return a > b ? a : b; };

  // the chunk size that ends first, as the kernel chooses it
  const int64_t cols = glu ? cdiv(M / 2, 128) : cdiv(M, 256);
  const int64_t units = over_loads(E, n, [&](int64_t r) { return cdiv(r, 64); });
  double rows = 0;
  for (int u = 4; u >= 2; --u) {
    const int64_t chunks = over_loads(E, n, [&](int64_t r) { return cdiv(cdiv(r, 64), u); });
    const int64_t tiles = cdiv(E * chunks * cols, 5), rounds = cdiv(tiles, cus), last = tiles - (rounds - 1) * cus;
    const double tile = c.tile + c.unit * units / chunks + c.stage * cdiv(K, 32);
    const double t = tile * (rounds - c.lone_gain * (1 - (double)last / cus));
    if (u == 4 || t < rows) rows = t;
  }
  rows = most(most(rows, weights / kRowsWeights), ops / c.ops) + c.launch;

  const int64_t edge = large ? 256 : 128, steps = cdiv(K, 64);
  const int64_t tiles = cdiv(E * over_loads(E, n, [&](int64_t r) { return cdiv(r, edge); }) * cdiv(M, edge), 5);
  const int pieces = large || glu || kind == ROWS_NT_GLU_BWD ? 1 : nn_split_pieces(E, N, K, M);
  double other;
  if (large) {
    other = most(cdiv(tiles, cus) * (c.large_tile + c.large_step * steps), ops / c.large_ops);
  } else if (pieces > 1) {
    other = (tiles * pieces > cus ? c.small_pair : c.small_lone) * steps / pieces + c.sums +
            (double)kSplitNsPerPiece * tiles * pieces;
  } else {
    const int64_t rounds = tiles / (2 * cus), rest = tiles % (2 * cus);
    const double pair = c.small_tile + c.small_pair * steps, lone = c.small_tile + c.small_lone * steps;
    other = rounds * pair;
    if (rest > 0) other += rest <= cus ? lone : lone + (pair - lone) * (rest - cus) / cus;
  }
  other = most(other, weights / c.weights) + c.other_launch;
  // the activation as a launch of its own
  if (glu && !large) other += 3000 + (double)N * M * 3 / 4000;
  return rows < other;
}

}  // namespace gmoe
