// Which 16-bit NN / NT launches go to the row-adaptive tiles (gmm_rows_kernel.h), and into which chunks the kernel cuts an
// expert's rows.
#pragma once
#include "split_rule.h"

namespace gmoe {

// What a tile costs besides 4 KiB of rows per unit (of 64) and stage (of 32 reduction elements), as KiB of operand
// stream: per stage, around the tile, around each unit of it; and by which factor chunks of more than four units cost more.
struct ChunkCosts {
  float stage, tile, unit, tall;
};
constexpr ChunkCosts kChunkCosts{16.f, 250.f, 0.f, 1.f};
// The activation backward reads fc1 and writes d(fc1) around a tile, four times the bytes of a plain result, with every
// compute unit at it at once: taller chunks save little and leave a part empty last round longer.  us in chunks of up to
// 128 / 192 / 256 / 320 / 384 rows (K x F): 16 experts of 640, 1024 x 2816 115 / 108 / 122 / 122 / 122; 8 of 366 to 402,
// 4096 x 14336 477 / 489 / 454 / 447 / 474; 60 of 386, 6272 x 2688 1070 / 1009 / 953 / 957 / 943; 8 of 1000, 4096 x 14336
// 1017 / 992 / 867 / 871 / 975.  Over 1059 launches (E 1-64, 40-6000 rows per expert, even and uneven loads, K and F
// 128-16384) the costs above lose 0.9 % against the best size of each (p95 6 %), these 0.3 % (2 %).
constexpr ChunkCosts kChunkCostsGluBwd{8.f, 120.f, 650.f, 1.04f};

// Rows of a chunk, in units of 64: of the sizes SIZES - 1 to 2 the one that ends first.  v[0]: units of all experts,
// v[u]: their chunks of up to u units.  Smaller chunks are taken where they cost less than `ahead` of the
// best larger ones.  The kernel asks with ahead 1: over 8600 launches of 96 rows per expert and more that costs 1.1 %
// against the best size of each, 0.95 costs 2.0 % (us in chunks of up to 128 / 192 / 256 / 320 / 384 rows, rows per
// expert: with activation 383, 4096 x 28672, 8 experts 890 / 776 / 739 / 745 / 686; 640, 1024 x 5632, 16 172 / 152 /
// 150 / 147 / 135; NN 640, 2816 x 1024, 16 86 / 60 / 67 / 73 / 81; NT 383, 28672 x 4096, 8 817 / 935 / 691 / 700 / 926).
constexpr int kRowsMaxUnits = 4;
constexpr int kTallMaxUnits = 6;
template <int SIZES>
__host__ __device__ inline int rows_chunk_units(const int (&v)[SIZES], int col_tiles, int grid, int64_t K,
                                                float ahead = 0.95f, ChunkCosts c = kChunkCosts) {
  const float stages = (float)((K + 31) / 32), fixed = c.stage + c.tile / stages, unit = 4.f + c.unit / stages;
  int best = SIZES - 1;
  float least = 0.f;
#pragma unroll
  for (int u = SIZES - 1; u >= 2; --u) {
    const int rounds = (int)(((long long)v[u] * col_tiles + grid - 1) / grid);
    const float cost = (float)rounds * (fixed + unit * (float)v[0] / (float)(v[u] > 0 ? v[u] : 1)) * (u > 4 ? c.tall : 1.f);
    if (u == SIZES - 1 || cost < ahead * least) {
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

// Rows per expert from which rows_pays is not asked (gmm.hip).
constexpr int64_t kRowsManyRows = 2048;

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

// The line for chunks of up to 256 rows, with constants fitted to 3400 shapes measured both ways (E 1-64, 72-2040 rows
// per expert, K 256-28672, M 128-28672) when the kernel had no larger ones and streamed its rows in half cache lines: a
// launch that paid then pays more now, and tall_pays adds those that pay only now.
// K, M as in the product (with the activation M = 2F); cus: workgroups of a persistent grid, one per CU.
inline bool rows_pays(RowsKind kind, int64_t E, int64_t N, int64_t K, int64_t M, int64_t cus) {
  const int64_t n = N / (E > 0 ? E : 1);
  // fewer rows: an expert is one tile either way, and its weights bound the launch; shorter reductions:
  // prologue and epilogue weigh as much
  if (n < 96 || n >= kRowsManyRows || K <= 512) return false;
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

// Times in ns as above: row-adaptive tiles with chunks of up to 384 rows (a stage is stage + unit_stage per 64 rows),
// then 128x128 tiles.
struct TallCosts {
  double tile, unit, stage, unit_stage, lone_gain, launch, weights, ops;
  double small_tile, small_pair, small_lone, sums, small_launch, small_weights, small_ops, act;
};
constexpr TallCosts kTallCosts[] = {
    {4620, 960, 217, 141, 0.31, 4200, 4830, 1.48e6, 3760, 1260, 520, 8700, 6300, 4320, 1e6, 0},
    {3130, 1900, 386, 109, 0.38, 5100, 5700, 1.487e6, 2170, 1180, 500, 22300, 6200, 5540, 0.783e6, 3500},
    {3840, 1140, 223, 144, 0.30, 4100, 4390, 1.41e6, 2860, 1240, 530, 7400, 6900, 4080, 1e6, 0},
    {690, 5880, 294, 127, 0.36, 5200, 4080, 1.487e6, 9950, 1350, 560, 0, 3800, 3640, 1e6, 0}};

// Whether a launch that has too few rows or tiles for 256x256 ones is faster in row-adaptive tiles than in 128x128
// ones.  Fitted to 15000 launches measured both ways (E 1-64, 2-8192 rows per expert, K 128-28672, M 128-28672, 2e8 to
// 6e12 operations, operands from HBM, loads that differ by 6 or 30 %).  From 96 rows per expert on it costs 0.9 to 2.4
// % against the better side of each, all of them in 128x128 tiles 6 to 27 %, rows_pays alone 2 to 22 %.  Below 96 rows
// an expert's weights bound the launch on either side; there only the launch with the activation may come here, which
// is two on the other tiles (1.9 % against the better side, the other tiles 5.4 %, without the host's time for the
// second launch), and only where those are not split, which spreads the weights' stream evenly over the CUs.  us in
// 128x128 tiles / in these (rows per expert, K x M, experts): NN 137, 2560 x 10240, 24 389 / 264; 656, 1280 x 1280, 2
// 18.0 / 24.6; with activation 389, 512 x 14336, 64 924 / 562; 121, 7168 x 256, 8 72 / 101; 3, 4096 x 28672, 8 317 /
// 346; 3, 4096 x 14336, 8 176 / 172; NT 938, 12544 x 2112, 4 280 / 217; 866, 19968 x 1536, 1 97 / 260; activation
// backward 386, 6272 x 2688, 60 1210 / 956; 599, 304 x 544, 6 15.8 / 26.4.
inline bool tall_pays(RowsKind kind, int64_t E, int64_t N, int64_t K, int64_t M, int64_t cus) {
  const int64_t n = N / (E > 0 ? E : 1);
  const bool glu = kind == ROWS_NN_GLU;
  if (n < (glu ? 1 : 96)) return false;
  const TallCosts& c = kTallCosts[kind];
  const double weights = (double)E * K * M * 2, ops = 2.0 * N * K * M;
  auto cdiv = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  auto most = [](double a, double b) { return a > b ? a : b; };

  const int64_t cols = glu ? cdiv(M / 2, 128) : cdiv(M, 256), stages = 2 * cdiv(K, 64);
  const int64_t units = over_loads(E, n, [&](int64_t r) { return cdiv(r, 64); });
  double tall = 0, idle = 0;
  for (int u = kTallMaxUnits; u >= 2; --u) {
    const int64_t chunks = over_loads(E, n, [&](int64_t r) { return cdiv(cdiv(r, 64), u); });
    const int64_t tiles = cdiv(E * chunks * cols, 5), rounds = cdiv(tiles, cus), last = tiles - (rounds - 1) * cus;
    const double average = (double)units / chunks;
    const double tile = c.tile + c.unit * average + (c.stage + c.unit_stage * average) * stages;
    const double t = tile * (rounds - c.lone_gain * (1 - (double)last / cus));
    if (u == kTallMaxUnits || t < tall) {
      tall = t;
      idle = rounds > 0 ? (1 - (double)last / cus) / rounds : 0;
    }
  }
  // a last round that is part empty does not stream the weights at the whole chip's rate
  tall = most(most(tall, weights / c.weights * (1 + 0.6 * idle)), ops / c.ops) + c.launch;

  const int64_t steps = cdiv(K, 64), tiles = cdiv(E * over_loads(E, n, [&](int64_t r) { return cdiv(r, 128); }) * cdiv(M, 128), 5);
  const int pieces = kind == ROWS_NT_GLU_BWD ? 1 : nn_split_pieces(E, N, K, M);
  if (n < 96 && pieces > 1) return false;
  double small;
  if (pieces > 1) {
    small = (tiles * pieces > cus ? c.small_pair : c.small_lone) * steps / pieces + c.sums +
            (double)kSplitNsPerPiece * tiles * pieces;
  } else {
    const int64_t rounds = tiles / (2 * cus), rest = tiles % (2 * cus);
    const double pair = c.small_tile + c.small_pair * steps, lone = c.small_tile + c.small_lone * steps;
    small = rounds * pair;
    if (rest > 0) small += rest <= cus ? lone : lone + (pair - lone) * (rest - cus) / cus;
  }
  small = most(most(small, weights / c.small_weights), ops / c.small_ops) + c.small_launch;
  if (glu) small += c.act + (double)N * M * 3 / 4000;  // the activation as a launch of its own
  return tall < (glu ? 1.0 : 0.97) * small;
}

}  // namespace gmoe
