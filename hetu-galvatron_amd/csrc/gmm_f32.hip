// Grouped GEMM of fp32 operands on the bf16 matrix cores of gfx950, without loss of precision: NN, NT and
// TN of gmm.hip's contract, with the activation backward as an epilogue of NT.
//
//   * An fp32 value is the sum of three bf16 values: the value rounded to bf16, what is left rounded to bf16,
//     and the rest.  A product is the sum of the six largest of the nine partial products; the dropped ones
//     are below 2^-24 of it.  Six bf16 MFMAs do what takes sixteen times as long per product on the fp32 one.
//   * Sums: per 32 reduction elements the five small partial products are accumulated first and the two MFMAs
//     of the large one last, in accumulators that start at zero; the block is then added to the running sum
//     in fp32.  (One accumulator for everything would be rounded 12 times per block inside the MFMA.)
//     Error against float64, 2-norm, normal operands, this kernel and the fp32 MFMA kernel it replaces:
//     K 512 0.9e-7 / 4.1e-7, K 2048 1.6e-7 / 8.1e-7, K 4096 2.2e-7 / 11e-7, K 4 3.2e-8 / 4.4e-8.
//   * Three planes hold an fp32 value exactly from 2^-110 on: its last bit is then no smaller than the smallest
//     bf16 number (the matrix cores take subnormal ones as they are).  An infinity (also a value that bf16
//     rounds to one) leaves NaN as its remainder, so every result that depends on an infinity or NaN is NaN.
//     A tile that met a smaller operand, other than zero, or that holds a NaN is computed again on the fp32
//     MFMA.  The look at the operands costs 1-2 % of a launch, 2-4 % on 64-row tiles: a minimum over the stage,
//     and only where that finds a zero or a small value, the exact look (operands with a seventh of zero rows:
//     1-5 % more; always exact: 8 % of a launch).  A launch computed again as a whole takes 2 to 6 times as
//     long.
//   * Buffer resources are made uniform by hand: the rows' addresses come from the offset table, and the
//     compiler repeated every load of the K loop for each value a lane might hold (4146 x 2048 x 512 over 8
//     experts NN 111 -> 100 us, NT 103 -> 97; 8192 x 2048 x 2048 over 8 NN 398 -> 388, NT 392 -> 384).
//   * Tiles of RF*64 rows (RF = 1, 2: an expert's rows are shared out in 64-row units) x 128 columns, 2x2
//     wavefronts of (RF*32) x 64, two workgroups per CU: one splits operands while the other multiplies.  With
//     at most one tile per CU the tiles are cut to 64 rows (4096 x 1024 x 512 over 8 experts 75 -> 62 us).
//   * NN / NT launches that leave CUs idle cut their reduction into pieces (gmm_f32_pieces in split_rule.h).  A
//     piece's results go to the workspace as a matrix of their own, and a second launch adds the matrices, bound by
//     that traffic: dX of 4096 x 2048 x 512 over 8 experts 102 -> 70 us, 2000 x 5632 x 1024 267 -> 163, 130 x
//     3584 x 896 over 4 44 -> 24 (there against the fp32 MFMA in pieces).
//     Error against float64, whole and in pieces: 1.6e-7 / 1.1e-7, 2.6e-7 / 1.7e-7 and 2.1e-7 / 1.2e-7.
//   * Operands go through registers (the split) into one LDS stage of 32 reduction elements:
//     [operand][plane][octet of k][row][8], so that the fragment reads of 32 rows are contiguous; octets lie
//     32 bytes off a multiple of 128, which takes the bank conflicts out of the writes of 4 octets x 2 rows
//     (64 bytes off: 4 cycles more per write, launches 3-6 % slower).
//   * Bound by: the matrix cores are busy for half the time at 1.9 GHz; a stage is a chain of writes, barrier,
//     reads, MFMAs, additions that two workgroups overlap in part.  Splitting the next stage's operands
//     between the MFMAs of this one: a lone workgroup 10 % faster, two 2-5 % slower; requesting them a
//     stage earlier as well: no further gain, and scratch.
//   * 16384 x 1024 x 4096 over 8 experts 1243 -> 810 us (170 TFLOP/s; the fp32 MFMA peaks at 157), 4096 x 512 x
//     2048 over 8 114 -> 88, 64 x 4096 x 4096 over 16 494 -> 270 (weights: 1.07 GB).
#include "gmm_common.h"

namespace gmoe {

namespace f32s {

constexpr int BN = 128;
constexpr int BKT = 32;       // reduction elements per stage
constexpr int kUnit = 64;     // rows per unit
constexpr int kMaxUnits = 2;  // units per tile
constexpr int OCTET = 128 * 16 + 32;
constexpr int PLANE = (BKT / 8) * OCTET;
constexpr int OPERAND = 3 * PLANE;
constexpr int LDS_BYTES = 2 * OPERAND;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, int64_t bytes) {
  // the same in every lane, which the compiler cannot see: it would repeat each load for every distinct value
  const uint64_t p = (uint64_t)(uintptr_t)base;
  const uint64_t u = (uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(p >> 32)) << 32 |
                     (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)p);
  const uint32_t n = bytes <= 0 ? 0u : (bytes > 0x7fffffffll ? 0x7fffffffu : (uint32_t)bytes);
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(u), 0, __builtin_amdgcn_readfirstlane((int)n),
                                           0x00020000);
}

// Eight fp32 values as three planes of eight bf16, each rounded to nearest.
__device__ __forceinline__ void split8(const float (&x)[8], u32x4& hi, u32x4& mid, u32x4& lo) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float x0 = x[2 * q], x1 = x[2 * q + 1];
    hi[q] = pack_bf16x2(x0, x1);
    const float r0 = x0 - __uint_as_float(hi[q] << 16), r1 = x1 - __uint_as_float(hi[q] & 0xffff0000u);
    mid[q] = pack_bf16x2(r0, r1);
    lo[q] = pack_bf16x2(r0 - __uint_as_float(mid[q] << 16), r1 - __uint_as_float(mid[q] & 0xffff0000u));
  }
}

constexpr float kSplitMin = 0x1p-110f;  // smallest magnitude that three planes hold exactly

// One operand's path to LDS: U units of 64 outer indices, an item = 8 reduction elements of one of them,
// U items per thread and stage.  KC: the reduction index is the contiguous one.
template <bool KC, int U>
struct Loader {
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t voff[U];
  uint32_t lds[U];
  uint32_t k_bytes;  // bytes between consecutive reduction elements
  int oct[U];
  float x[U][8];

  // src: outer index 0, reduction element 0 of the tile; bytes: what may be read from there; outers: indices
  // that exist (k contiguous: the last one is read for those that do not, which are never stored: zeros would
  // take every stage through holds_small)
  __device__ __forceinline__ void init(const unsigned char* src, int64_t ld, int64_t bytes, int64_t outers, int tid) {
    rsrc = make_rsrc(src, bytes);
    k_bytes = (uint32_t)(KC ? 4 : ld * 4);
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int id = tid + i * kGemmThreads;
      // k contiguous: 4 lanes read the 128 bytes of a row; otherwise a wavefront reads 64 columns
      const int outer = KC ? id >> 2 : id & (U * kUnit - 1);
      oct[i] = KC ? id & 3 : id / (U * kUnit);
      const int64_t from = outer < outers ? outer : outers - 1;
      voff[i] = KC ? (uint32_t)(from * ld * 4 + oct[i] * 32) : (uint32_t)(oct[i] * 8 * ld * 4 + outer * 4);
      lds[i] = (uint32_t)(oct[i] * OCTET + outer * 16);
    }
  }
  __device__ __forceinline__ void load(int64_t k0, int64_t K) {
    const uint32_t soff = (uint32_t)k0 * k_bytes;
#pragma unroll
    for (int i = 0; i < U; ++i) {
      if constexpr (KC) {
        const uint32_t vo = k0 + oct[i] * 8 < K ? voff[i] : kOob;
        const u32x4 v0 = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)vo, (int)soff, 0);
        const u32x4 v1 = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)vo, (int)soff + 16, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          x[i][q] = __uint_as_float(v0[q]);
          x[i][4 + q] = __uint_as_float(v1[q]);
        }
      } else {
#pragma unroll
        for (int q = 0; q < 8; ++q)
          x[i][q] = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(
              rsrc, (int)voff[i], (int)(soff + q * k_bytes), 0));
      }
    }
  }
  __device__ __forceinline__ void store(unsigned char* stage) const {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      u32x4 hi, mid, lo;
      split8(x[i], hi, mid, lo);
      *reinterpret_cast<u32x4*>(stage + lds[i]) = hi;
      *reinterpret_cast<u32x4*>(stage + PLANE + lds[i]) = mid;
      *reinterpret_cast<u32x4*>(stage + 2 * PLANE + lds[i]) = lo;
    }
  }
  // Smallest magnitude of the stage and `m`, zeros included; a NaN may hide the others, or be the result.
  __device__ __forceinline__ float smallest(float m) const {
#pragma unroll
    for (int i = 0; i < U; ++i)  // in one piece: the compiler pads every asm statement with a no-op
      asm("v_min3_f32 %0, |%2|, |%3|, %1\n\tv_min3_f32 %0, |%4|, |%5|, %0\n\t"
          "v_min3_f32 %0, |%6|, |%7|, %0\n\tv_min3_f32 %0, |%8|, |%9|, %0"
          : "=&v"(m)
          : "v"(m), "v"(x[i][0]), "v"(x[i][1]), "v"(x[i][2]), "v"(x[i][3]), "v"(x[i][4]), "v"(x[i][5]), "v"(x[i][6]),
            "v"(x[i][7]));
    return m;
  }
  // Whether the stage holds a value below kSplitMin that is not zero.
  __device__ __forceinline__ bool holds_small() const {
    uint32_t least = 0xffffffffu;  // of twice the bits, less one: zero wraps to the top
#pragma unroll
    for (int i = 0; i < U; ++i)
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const uint32_t v = __float_as_uint(x[i][q]) * 2u - 1u;
        least = v < least ? v : least;
      }
    return least < __float_as_uint(kSplitMin) * 2u - 1u;
  }
  // element (outer, k) for the fp32 MFMA; past the end of either reads as zero
  __device__ __forceinline__ float one(int outer, int64_t k, int64_t K, int64_t ld) const {
    const uint32_t off = KC ? (uint32_t)((outer * ld + k) * 4) : (uint32_t)((k * ld + outer) * 4);
    return __uint_as_float(
        (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(k < K ? off : kOob), 0, 0));
  }
};

struct Item {
  int e, nt;
  long long row0;      // first row of the expert
  int64_t n;           // rows of the expert
  int64_t first, cnt;  // output rows of the tile: [first, first + cnt) of the expert's (TN: of K)
  int piece;           // of the reduction, of p.pieces
};

template <int MODE, int EPI, int RF>
__device__ __forceinline__ void run_tile(const GmmParams& p, const Item& it, unsigned char* lds, int wave, int lane,
                                         int tid) {
  constexpr bool GLU_BWD = EPI == EPI_GLU_BWD_SILU || EPI == EPI_GLU_BWD_GELU;
  const int64_t M = p.M, red = MODE == MODE_TN ? it.n : p.K;
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t col0 = (int64_t)it.nt * BN;

  Loader<MODE != MODE_TN, RF> la;
  Loader<MODE == MODE_NT, 2> lb;
  const int64_t ld_a = p.K, ld_b = MODE == MODE_NT ? p.K : M;
  if constexpr (MODE == MODE_TN) {
    la.init(p.a + (it.row0 * p.K + it.first) * 4, ld_a, (it.n * p.K - it.first) * 4, it.cnt, tid);
    lb.init(p.b + (it.row0 * M + col0) * 4, ld_b, (it.n * M - col0) * 4, M - col0, tid);
  } else {
    la.init(p.a + (it.row0 + it.first) * p.K * 4, ld_a, it.cnt * p.K * 4, it.cnt, tid);
    if constexpr (MODE == MODE_NT)
      lb.init(p.b + ((int64_t)it.e * M + col0) * p.K * 4, ld_b, (M - col0) * p.K * 4, M - col0, tid);
    else
      lb.init(p.b + ((int64_t)it.e * p.K * M + col0) * 4, ld_b, (p.K * M - col0) * 4, M - col0, tid);
  }

  f32x16 sum[RF][2];
#pragma unroll
  for (int i = 0; i < RF; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) sum[i][j][v] = 0.f;

  const uint32_t frag = (uint32_t)((lane >> 5) * OCTET + (lane & 31) * 16);
  const unsigned char* fa = lds + frag + wm * RF * 32 * 16;
  const unsigned char* fb = lds + OPERAND + frag + wn * 64 * 16;
  // the stages of this tile's piece of the reduction
  constexpr bool CAN_SPLIT = MODE != MODE_TN && EPI == EPI_NONE;
  const int all_stages = (int)((red + BKT - 1) / BKT);
  int from = 0, stages = all_stages;
  if constexpr (CAN_SPLIT) {
    if (p.pieces > 1) {
      from = all_stages * it.piece / p.pieces;
      stages = all_stages * (it.piece + 1) / p.pieces;
    }
  }
  if (stages > from) {
    la.load((int64_t)from * BKT, red);
    lb.load((int64_t)from * BKT, red);
  }
  uint64_t small = 0;  // lanes
  for (int s = from; s < stages; ++s) {
    la.store(lds);
    lb.store(lds + OPERAND);
    if (__ballot(!(la.smallest(lb.smallest(kSplitMin)) >= kSplitMin)) != 0)
      small |= __ballot(la.holds_small() || lb.holds_small());
    __syncthreads();
    if (s + 1 < stages) {
      la.load((int64_t)(s + 1) * BKT, red);
      lb.load((int64_t)(s + 1) * BKT, red);
    }
    f32x16 blk[RF][2];
    u32x4 a1[2][RF], b1[2][2];
    static_for<0, 2>([&](auto ks_c) {
      constexpr int ks = decltype(ks_c)::value;
      u32x4 a2[RF], a3[RF], b2[2], b3[2];
#pragma unroll
      for (int i = 0; i < RF; ++i) {
        const unsigned char* f = fa + ks * 2 * OCTET + i * 32 * 16;
        a1[ks][i] = *reinterpret_cast<const u32x4*>(f);
        a2[i] = *reinterpret_cast<const u32x4*>(f + PLANE);
        a3[i] = *reinterpret_cast<const u32x4*>(f + 2 * PLANE);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const unsigned char* f = fb + ks * 2 * OCTET + j * 32 * 16;
        b1[ks][j] = *reinterpret_cast<const u32x4*>(f);
        b2[j] = *reinterpret_cast<const u32x4*>(f + PLANE);
        b3[j] = *reinterpret_cast<const u32x4*>(f + 2 * PLANE);
      }
      auto all = [&](const u32x4 (&a)[RF], const u32x4 (&b)[2], bool first) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RF; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            if (first) blk[i][j] = f32x16{};
            Mma<GMOE_BF16>::run(a[i], b[j], blk[i][j]);
          }
      };
      all(a3, b1[ks], ks == 0);
      all(a1[ks], b3, false);
      all(a2, b2, false);
      all(a2, b1[ks], false);
      all(a1[ks], b2, false);
    });
    static_for<0, 2>([&](auto ks_c) {
      constexpr int ks = decltype(ks_c)::value;
#pragma unroll
      for (int i = 0; i < RF; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) Mma<GMOE_BF16>::run(a1[ks][i], b1[ks][j], blk[i][j]);
    });
#pragma unroll
    for (int i = 0; i < RF; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) sum[i][j] += blk[i][j];
    __syncthreads();
  }

  // a small operand, an infinity or a NaN: the tile again on the fp32 MFMA
  int redo = small != 0;
#pragma unroll
  for (int i = 0; i < RF; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) redo |= sum[i][j][v] != sum[i][j][v];
  if (__builtin_expect(__syncthreads_or(redo), 0)) {
#pragma unroll
    for (int i = 0; i < RF; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) sum[i][j] = f32x16{};
    constexpr int kAhead = 2;  // pairs of reduction elements requested together
    const int64_t end = (int64_t)stages * BKT < red ? (int64_t)stages * BKT : red;
#pragma unroll 1
    for (int64_t k0 = (int64_t)from * BKT; k0 < end; k0 += 2 * kAhead) {
      float av[kAhead][RF], bv[kAhead][2];
#pragma unroll
      for (int q = 0; q < kAhead; ++q) {
        const int64_t k = k0 + 2 * q + (lane >> 5);
#pragma unroll
        for (int i = 0; i < RF; ++i) av[q][i] = la.one(wm * RF * 32 + i * 32 + (lane & 31), k, end, ld_a);
#pragma unroll
        for (int j = 0; j < 2; ++j) bv[q][j] = lb.one(wn * 64 + j * 32 + (lane & 31), k, end, ld_b);
      }
#pragma unroll
      for (int q = 0; q < kAhead; ++q)
#pragma unroll
        for (int i = 0; i < RF; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(bv[q][j], av[q][i], sum[i][j], 0, 0, 0);
    }
  }

  // a lane holds 4 consecutive columns of one row per accumulator quarter
#pragma unroll
  for (int i = 0; i < RF; ++i) {
    const int64_t m = wm * RF * 32 + i * 32 + (lane & 31);
    if (m >= it.cnt) continue;
    const int64_t n0 = col0 + wn * 64 + 4 * (lane >> 5);
    if constexpr (GLU_BWD) {
      // all loads of the row before its first store: they may alias as far as the compiler knows, and each
      // would wait for the stores before it
      constexpr bool gelu = EPI == EPI_GLU_BWD_GELU;
      const int64_t at = ((it.row0 + it.first + m) * 2 * M + n0) * 4;
      f32x4 g[8], u[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (n0 + q * 8 >= M) continue;
        g[q] = *reinterpret_cast<const f32x4*>(p.aux + at + q * 32);
        u[q] = *reinterpret_cast<const f32x4*>(p.aux + at + q * 32 + M * 4);
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (n0 + q * 8 >= M) continue;
        f32x4 dg, du;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float d = sum[i][q / 4][q % 4 * 4 + t];
          dg[t] = d * glu_act_grad(g[q][t], gelu) * u[q][t];
          du[t] = d * glu_act(g[q][t], gelu);
        }
        *reinterpret_cast<f32x4*>(p.c + at + q * 32) = dg;
        *reinterpret_cast<f32x4*>(p.c + at + q * 32 + M * 4) = du;
      }
    } else {
      const int64_t row = MODE == MODE_TN ? (int64_t)it.e * p.K + it.first + m : it.row0 + it.first + m;
      unsigned char* out = p.c;
      if constexpr (CAN_SPLIT) {
        if (p.pieces > 1) out = reinterpret_cast<unsigned char*>(p.ws + it.piece * p.N * M);
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (n0 + q * 8 >= M) continue;
        const f32x16& v = sum[i][q / 4];
        *reinterpret_cast<f32x4*>(out + (row * M + n0 + q * 8) * 4) =
            f32x4{v[q % 4 * 4], v[q % 4 * 4 + 1], v[q % 4 * 4 + 2], v[q % 4 * 4 + 3]};
      }
    }
  }
}

template <int MODE, int EPI>
__global__ __launch_bounds__(kGemmThreads, 2) void gmm_f32_kernel(GmmParams p) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  __shared__ int tile_cum[kMaxGroupsLds + 1];
  __shared__ int wave_tot[kGemmThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int E = p.E, nt_cnt = (int)((p.M + BN - 1) / BN);
  // output rows of an expert, in units; units are dealt as evenly as possible to the fewest tiles
  auto rows_of = [&](int e) -> int64_t {
    return MODE == MODE_TN ? p.K : (int64_t)(group_begin(p, e + 1) - group_begin(p, e));
  };
  auto units_of = [](int64_t n) { return (int)((n + kUnit - 1) / kUnit); };

  // tiles per expert -> exclusive prefix (a thread owns kPer consecutive experts)
  auto count_tiles = [&](int max_units) {
    constexpr int kPer = kMaxGroupsLds / kGemmThreads;
    int cnt[kPer], local = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int e = tid * kPer + j;
      cnt[j] = e >= E ? 0 : nt_cnt * ((units_of(rows_of(e)) + max_units - 1) / max_units);
      local += cnt[j];
    }
    int incl = local;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(incl, d);
      if (lane >= d) incl += o;
    }
    __syncthreads();
    if (lane == 63) wave_tot[wave] = incl;
    __syncthreads();
    int run = incl - local;
    for (int w = 0; w < wave; ++w) run += wave_tot[w];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int e = tid * kPer + j;
      if (e <= E) tile_cum[e] = run;
      run += cnt[j];
    }
    if (tid == kGemmThreads - 1) tile_cum[E] = run;
    __syncthreads();
  };
  int max_units = kMaxUnits;
  count_tiles(max_units);
  if ((int64_t)tile_cum[E] * p.pieces <= (int)gridDim.x / 2) {
    max_units = 1;
    count_tiles(max_units);
  }
  const int tiles_all = tile_cum[E], total = tiles_all * p.pieces;  // a piece's tiles are neighbours

  // XCD x takes the positions [x*G/8, (x+1)*G/8) of every whole round of G tiles; the last, partial
  // round is dealt to the XCDs in equal consecutive shares
  const int G = gridDim.x, per_xcd = G / 8;
  const int xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
  int e = 0;
  for (int base = 0; base < total; base += G) {
    int v = base + xcd * per_xcd + slot;
    if (total - base < G) {
      const int share = (total - base + 7) / 8;
      v = base + xcd * share + slot;
      if (slot >= share || v >= total) break;
    }
    Item it;
    it.piece = 0;
    if (p.pieces > 1) {
      it.piece = __builtin_amdgcn_readfirstlane(v / tiles_all);
      v -= it.piece * tiles_all;
      if (v < tile_cum[e]) e = 0;
    }
    while (tile_cum[e + 1] <= v) ++e;
    it.e = __builtin_amdgcn_readfirstlane(e);
    it.row0 = group_begin(p, it.e);
    it.n = group_begin(p, it.e + 1) - it.row0;
    const int64_t n_out = rows_of(it.e);
    const int all = units_of(n_out), tiles = (all + max_units - 1) / max_units;
    int c;
    strip_order(v - tile_cum[it.e], tiles, nt_cnt, c, it.nt);
    const int each = all / tiles, extra = all - each * tiles;
    const int units = each + (c < extra ? 1 : 0);
    it.first = (int64_t)(c * each + (c < extra ? c : extra)) * kUnit;
    it.cnt = n_out - it.first < units * kUnit ? n_out - it.first : units * kUnit;
    if (__builtin_amdgcn_readfirstlane(units) == 1) run_tile<MODE, EPI, 1>(p, it, lds, wave, lane, tid);
    else run_tile<MODE, EPI, 2>(p, it, lds, wave, lane, tid);
  }
}

// c = the sum of the pieces' results, which lie behind one another in the workspace, in ascending order.  Rows
// outside the groups have no pieces, and c keeps them.
__global__ __launch_bounds__(256) void f32_pieces_sum_kernel(GmmParams p) {
  const int64_t first = group_begin(p, 0) * p.M / 4, quads = group_begin(p, p.E) * p.M / 4, step = p.N * p.M / 4;
  const f32x4* ws = reinterpret_cast<const f32x4*>(p.ws);
  f32x4* out = reinterpret_cast<f32x4*>(p.c);
  for (int64_t i = first + (int64_t)blockIdx.x * 256 + threadIdx.x; i < quads; i += (int64_t)gridDim.x * 256) {
    f32x4 sum = ws[i];
#pragma unroll 4
    for (int s = 1; s < p.pieces; ++s) sum += ws[s * step + i];
    out[i] = sum;
  }
}

template <int MODE, int EPI>
static int launch_cfg(const GmmParams& p, hipStream_t st) {
  auto kern = gmm_f32_kernel<MODE, EPI>;
  static std::atomic<uint64_t> done_mask{0};
  if (!gmoe_once_per_device(done_mask, [&] {
        return hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES) == hipSuccess;
      }))
    return GMOE_ERR_LAUNCH;
  int grid = (gmoe_cu_count() / 8) * 8 * 2;
  if (grid < 8) grid = 8;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(kGemmThreads), LDS_BYTES, st, p);
  if (p.pieces > 1) {
    const int64_t blocks = (p.N * p.M / 4 + 255) / 256;
    hipLaunchKernelGGL(f32_pieces_sum_kernel, dim3((unsigned)(blocks < 4 * grid ? blocks : 4 * grid)), dim3(256), 0, st,
                       p);
  }
  return gmoe_launch_status();
}

}  // namespace f32s

int launch_gmm_f32(const GmmParams& p, int mode, int epi, hipStream_t st) {
  using namespace f32s;
  if (epi == EPI_GLU_BWD_SILU) return launch_cfg<MODE_NT, EPI_GLU_BWD_SILU>(p, st);
  if (epi == EPI_GLU_BWD_GELU) return launch_cfg<MODE_NT, EPI_GLU_BWD_GELU>(p, st);
  if (mode == MODE_NN) return launch_cfg<MODE_NN, EPI_NONE>(p, st);
  if (mode == MODE_NT) return launch_cfg<MODE_NT, EPI_NONE>(p, st);
  return launch_cfg<MODE_TN, EPI_NONE>(p, st);
}

}  // namespace gmoe
