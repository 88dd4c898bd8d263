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
// 1017 / 992 / 867 / 871 / 975; 8 of 358, 61, 931, 83, 155, 6, 730 and 738, 4096 x 14336 471 / 454 / 426 / 470 / 488.
// Over 1059 launches (E 1-64, 40-6000 rows per expert, even and uneven loads, K and F 128-16384) the costs above lose
// 0.9 % against the best size of each (p95 6 %), these 0.3 % (2 %).  With more than 1024 rows per expert the costs above
// stay: there are many rounds, little is lost (1 %), and what a part empty one leaves idle is used by what runs beside (8192
// tokens of 2048, 64 experts of 1408, top 8, the shared experts on their own stream: the step 5085 us, with these 5115).
constexpr ChunkCosts kChunkCostsGluBwd{7.3f, 390.f, 866.f, 1.07f};
// units: of all E experts
__host__ __device__ inline ChunkCosts chunk_costs(bool glu_bwd, int units, int E) {
  return glu_bwd && units <= 16 * E ? kChunkCostsGluBwd : kChunkCosts;
}

// Rows of a chunk, in units of 64: of the sizes kTallMaxUnits to 2 the one that ends first.  v[0]: units of all experts,
// v[u]: their chunks of up to u units.  Over 8600 launches of 96 rows per expert and more it costs 1.1 % against the best
// size of each (us in chunks of up to 128 / 192 / 256 / 320 / 384 rows, rows per expert: with activation 383, 4096 x
// 28672, 8 experts 890 / 776 / 739 / 745 / 686; 640, 1024 x 5632, 16 172 / 152 / 150 / 147 / 135; NN 640, 2816 x 1024, 16
// 86 / 60 / 67 / 73 / 81; NT 383, 28672 x 4096, 8 817 / 935 / 691 / 700 / 926).
constexpr int kTallMaxUnits = 6;
__host__ __device__ inline int rows_chunk_units(const int (&v)[kTallMaxUnits + 1], int col_tiles, int grid, int64_t K,
                                                ChunkCosts c) {
  const float stages = (float)((K + 31) / 32), fixed = c.stage + c.tile / stages, unit = 4.f + c.unit / stages;
  int best = kTallMaxUnits;
  float least = 0.f;
#pragma unroll
  for (int u = kTallMaxUnits; u >= 2; --u) {
    const int rounds = (int)(((long long)v[u] * col_tiles + grid - 1) / grid);
    const float cost = (float)rounds * (fixed + unit * (float)v[0] / (float)(v[u] > 0 ? v[u] : 1)) * (u > 4 ? c.tall : 1.f);
    if (u == kTallMaxUnits || cost < least) {
      best = u;
      least = cost;
    }
  }
  return best;
}

enum RowsKind { ROWS_NN, ROWS_NN_GLU, ROWS_NT, ROWS_NT_GLU_BWD };

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

// Times in ns, rates in bytes or operations per ns.
struct RowsCosts {
  // row-adaptive tiles: around a tile and each 64 rows of it, a stage of 32 reduction elements of it and of each 64
  // rows, share of a tile's time that a round saves as its tiles get fewer, around the launch, traffic, operations
  double tile, unit, stage, unit_stage, lone_gain, launch, bytes, ops;
  // 128x128 tiles: around one, 64 reduction elements with two tiles on a CU and with one, around the launch, traffic,
  // operations; around a split's sums; the activation's launch
  double small_tile, small_pair, small_lone, small_launch, small_bytes, small_ops, sums, act;
  // 256x256 tiles (plain NT): around one, 64 reduction elements, operations
  double large_tile, large_step, large_ops;
};
constexpr RowsCosts kRowsCosts[] = {
    {2840, 741, 275, 69.3, 0.0819, 9590, 7840, 0.991e6, 2730, 1250, 628, 2260, 4810, 0.563e6, 1990, 0, 0, 0, 0},
    {3820, 2080, 343, 111, 0.0366, 1890, 6840, 1.49e6, 1110, 1310, 417, 3670, 5580, 0.484e6, 0, 2070, 0, 0, 0},
    {2990, 1340, 176, 159, 0.14, 4650, 6800, 1.62e6, 2320, 1270, 614, 2730, 4720, 0.551e6, 4720, 0, 6670, 1630, 1.16e6},
    {6890, 6480, 123, 102, 0.0491, 1020, 6580, 1.0e6, 10600, 1430, 422, 2500, 5630, 1.0e6, 0, 0, 0, 0, 0}};

// What a launch reads and writes once.
inline double rows_bytes(RowsKind kind, int64_t E, int64_t N, int64_t K, int64_t M) {
  return 2.0 * E * K * M + 2.0 * N * K + (double)N * M * (kind == ROWS_NN_GLU ? 3 : kind == ROWS_NT_GLU_BWD ? 8 : 2);
}

// Time of a launch in the other tiles (with the activation of two), ns, from one row per expert on.
inline double others_ns(RowsKind kind, int64_t E, int64_t N, int64_t K, int64_t M, int64_t cus) {
  const RowsCosts& c = kRowsCosts[kind];
  const int64_t n = N / E;
  const bool glu = kind == ROWS_NN_GLU, bwd = kind == ROWS_NT_GLU_BWD, large = kind == ROWS_NT && nn_large_tiles(E, N, M);
  const double ops = 2.0 * N * K * M, bytes = rows_bytes(kind, E, N, K, M);
  auto cdiv = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  auto most = [](double a, double b) { return a > b ? a : b; };
  const int64_t edge = large ? 256 : 128, steps = cdiv(K, 64);
  const int64_t tiles = cdiv(E * over_loads(E, n, [&](int64_t r) { return cdiv(r, edge); }) * cdiv(M, edge), 5);
  // the launches with an activation have no workspace for a split
  const int pieces = large || glu || bwd ? 1 : nn_split_pieces(E, N, K, M);
  double other;
  if (large) {
    other = most(cdiv(tiles, cus) * (c.large_tile + c.large_step * steps), ops / c.large_ops);
  } else {
    if (pieces > 1) {
      other = (tiles * pieces > cus ? c.small_pair : c.small_lone) * steps / pieces + c.sums +
              (double)kSplitNsPerPiece * tiles * pieces;
    } else {
      const int64_t rounds = tiles / (2 * cus), rest = tiles % (2 * cus);
      const double pair = c.small_tile + c.small_pair * steps, lone = c.small_tile + c.small_lone * steps;
      other = rounds * pair;
      if (rest > 0) other += rest <= cus ? lone : lone + (pair - lone) * (rest - cus) / cus;
    }
    other = most(most(other, bytes / c.small_bytes), ops / c.small_ops);
  }
  other += c.small_launch;
  if (glu) other += c.act + (double)N * M * 3 / 4000;
  return other;
}

// Whether a 16-bit NN / NT launch is faster in row-adaptive tiles than in the others: 128x128 ones, for plain NT that
// could fill them 256x256 ones (only the host asks).  K, M as in the product (with the activation M = 2F); cus:
// workgroups of a persistent grid, one per CU.
//
// Fitted to 6600 launches measured both ways, half of them of layers as they are trained, half spread over E 1-64, 1-9000
// rows per expert, K and M 128-16384 (operands from HBM, loads that differ by 2 to 80 %), a third of them under 30 us.
// Over them it costs 0.5 % (NN), 0.8 % (with activation), 0.8 % (NT) and 1.1 % (activation backward) against the better
// side of each; the others throughout 11, 12, 6 and 7 %, these throughout 19, 8, 20 and 12 %.  The 3 % that these have to
// be ahead by cost nothing and keep launches at the line where they were.
//
// Fewer than 96 rows per expert: an expert is one row tile and its weights bound the launch on either side.  Only the launch
// with the activation, which is two on the other tiles, may come here, and only where its tiles fill their rounds: a
// workgroup per CU streams the weights at the chip's rate only while all of them have a tile (rows per expert, K x M,
// experts; 3, 4096 x 28672, 8, 3.5 rounds 319 / 350 others; 16, 2048 x 2816, 64, 2.75 rounds 142 / 131 these; 16, 1024 x
// 5632, 16, 1.4 rounds 43 / 46 others).  Under 4 rows per expert the host cannot tell how many experts have any.  Over 3500
// such launches 1.9 % are lost against the better side, in the other tiles throughout 2.3 %, here 9.8 %.
//
// us in the other tiles / in these (rows per expert, K x M, experts):
//   * NN: 382, 14336 x 4096, 8 437 / 337 these; 363, 512 x 5120, 8 32 / 32; 267, 576 x 832, 64 45 / 36 these; 941, 768 x
//     128, 32 18 / 24 others; 656, 1280 x 1280, 2 14 / 23 others; 1701, 10848 x 160, 4 79 / 133 others.
//   * With activation: 382, 4096 x 28672, 8 976 / 650 these; 640, 1024 x 5632, 16 189 / 138 these; 208, 128 x 512, 32 12
//     / 13 others; 103, 768 x 1024, 4 13 / 18 others; 121, 7168 x 256, 8 65 / 95 others.
//   * NT: 382, 28672 x 4096, 8 860 / 628 these; 600, 2056 x 4104, 8 116 / 112 these; 1111, 5632 x 2048, 1 49 / 77 others;
//     1769, 1408 x 512, 4 16 / 24 others; 1000, 28672 x 4096, 8 1439 / 1413 these.
//     Short reductions of fewer than 768 rows per expert that fill 256x256 tiles stay there: of 36 such launches a third is
//     slower here, by up to 7 %.
//   * Activation backward: 382, 4096 x 14336, 8 470 / 382 these; 1024, 7168 x 2048, 32 1119 / 835 these; 640, 1024 x 2816,
//     16 103 / 111 others; 599, 304 x 544, 6 15 / 29 others; 322, 4992 x 1024, 4 53 / 73 others.
// It knows the average load only, and where that is close to whole rounds it can be wrong.
inline bool rows_pays(RowsKind kind, int64_t E, int64_t N, int64_t K, int64_t M, int64_t cus) {
  if (E < 1) E = 1;
  const int64_t n = N / E;
  const bool glu = kind == ROWS_NN_GLU;
  auto cdiv = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  auto most = [](double a, double b) { return a > b ? a : b; };
  const int64_t cols = glu ? cdiv(M / 2, 128) : cdiv(M, 256);
  if (n < 96) {
    const int64_t tiles = E * cols;
    return glu && n >= 4 && 10 * tiles >= 9 * cus * cdiv(tiles, cus);
  }
  if (kind == ROWS_NT && n < 768 && K <= 2560 && nn_large_tiles(E, N, M)) return false;
  const RowsCosts& c = kRowsCosts[kind];
  const double ops = 2.0 * N * K * M, bytes = rows_bytes(kind, E, N, K, M);
  const int64_t stages = 2 * cdiv(K, 64);
  const int64_t units = over_loads(E, n, [&](int64_t r) { return cdiv(r, 64); });
  double rows = 0, idle = 0;
  for (int u = kTallMaxUnits; u >= 2; --u) {
    const int64_t chunks = over_loads(E, n, [&](int64_t r) { return cdiv(cdiv(r, 64), u); });
    const int64_t tiles = cdiv(E * chunks * cols, 5), rounds = cdiv(tiles, cus), last = tiles - (rounds - 1) * cus;
    const double average = (double)units / chunks, part = 1 - (double)last / cus;
    const double tile = c.tile + c.unit * average + (c.stage + c.unit_stage * average) * stages;
    const double t = tile * (rounds - c.lone_gain * part);
    if (u == kTallMaxUnits || t < rows) {
      rows = t;
      idle = part / rounds;
    }
  }
  // a last round that is part empty does not stream at the whole chip's rate
  rows = most(most(rows, bytes / c.bytes * (1 + 0.6 * idle)), ops / c.ops) + c.launch;

  return rows < 0.97 * others_ns(kind, E, N, K, M, cus);
}

// Whether fc1 and its activation are so short that one launch is better than two for the host's sake, although these tiles
// take longer for it: programs of such launches wait for the host, which a launch costs 3 to 4 us.  us in one launch / in
// two, and of the whole step called eagerly: 128 rows, 4 experts, 128 x 512 9.4 / 8.2 and 272 / 277; 128 rows, 8 experts,
// forward, 512 x 1024 68.4 / 71.1.  Of 3500 launches of few rows these are 850; they take 1.3 us longer than two would.
// Not asked while a graph is captured, whose replay takes the host no time.
inline bool rows_one_launch_pays(int64_t E, int64_t N, int64_t K, int64_t M, int64_t cus) {
  if (E < 1) E = 1;
  return N >= 1 && others_ns(ROWS_NN_GLU, E, N, K, M, cus) < 12000;
}

}  // namespace gmoe
