// Grouped GEMM with row-adaptive tiles for 16-bit operands (bf16 / fp16) on gfx950: NN and NT of
// gmm.hip's contract, with the fused gated-activation epilogues, for a few dozen to a few hundred rows
// per expert (the rule with both sides' times is rows_rule.h).
//
//   * A tile is RF*64 rows (RF = 1..4, chosen per tile) x 256 columns of C.  An expert's rows are cut
//     into chunks of up to 256 (192, 128 where those fill the rounds better: best_max_units) that are as
//     equal as 64-row steps allow, so at most 63 rows per expert are padding: a fixed 128- or 256-row tile
//     multiplies a third of its rows for nothing at 380 rows per expert, and its operand stream is the larger the
//     smaller the tile.
//   * 2x2 wavefronts of (RF*32) x 128, one workgroup per CU.
//   * Operands go global -> LDS without staging registers (buffer_load ... lds) in stages of 32
//     reduction elements, 4 stages for 256 rows up to 7 for 64 rows; one barrier per stage.
//   * What bounds it: the operand stream.  Without the MFMAs the Mixtral-shape fc1 launch still takes
//     5.5 of 6.5 ms (42 GB/s per CU, whatever the number of stages; 72 GB/s when every stage hits L2),
//     without the copies 4.3 ms.  Hence the large tile, and the copies spread one by one between the
//     MFMAs of both K steps (a tile's copies in one burst: 4-9 % slower at full tiles).  Measured
//     without gain: 64-deep stages (128-byte pieces of the rows), a staggered start of the
//     workgroups' K walks, 128x256 tiles with two workgroups per CU (their operand stream is half
//     again as large: 700 instead of 860 TFLOP/s at 383 rows per expert).
#include "gmm_common.h"

namespace gmoe {

namespace rows {

constexpr int BN = 256;
constexpr int BKT = 32;  // reduction elements per stage
constexpr int B_BYTES = BN * BKT * 2;
constexpr int kUnit = 64;     // rows per unit: 32 for each of the two wavefront rows
constexpr int kMaxUnits = kRowsMaxUnits;  // units per tile

// LDS stages of a tile of RF units: as many as fit 144 KiB
template <int RF>
struct Stages {
  static constexpr int a_bytes = RF * kUnit * BKT * 2;
  static constexpr int bytes = a_bytes + B_BYTES;
  static constexpr int count = RF == 4 ? 4 : (RF == 3 ? 5 : (RF == 2 ? 6 : 7));
  static_assert(count * bytes <= 144 * 1024, "LDS");
};

typedef short s16x4 __attribute__((ext_vector_type(4)));

// Row chunks of an expert with n rows: units of kUnit rows dealt as evenly as possible to
// ceil(units / max_units) chunks.
__device__ __forceinline__ int unit_count(long long n) { return (int)((n + kUnit - 1) / kUnit); }
__device__ __forceinline__ int chunk_count(long long n, int max_units) {
  return (unit_count(n) + max_units - 1) / max_units;
}
// rows_chunk_units for the launch; units, chunks: of this thread's experts, summed over the workgroup here.
__device__ __forceinline__ int best_max_units(int units, const int (&chunks)[kMaxUnits + 1], int nt_cnt, int grid,
                                              int64_t K, int (*sums)[kMaxUnits + 1], int lane, int wave) {
  int v[kMaxUnits + 1] = {units, 0, chunks[2], chunks[3], chunks[4]};
#pragma unroll
  for (int i = 0; i <= kMaxUnits; ++i) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) v[i] += __shfl_xor(v[i], d);
    if (lane == 0) sums[wave][i] = v[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i <= kMaxUnits; ++i) {
    v[i] = 0;
#pragma unroll
    for (int w = 0; w < kGemmThreads / 64; ++w) v[i] += sums[w][i];
  }
  return rows_chunk_units(v, nt_cnt, grid, K);
}
// first unit and unit count of chunk c of cnt
__device__ __forceinline__ void chunk_units(long long n, int cnt, int c, int& first, int& units) {
  const int all = (int)((n + kUnit - 1) / kUnit);
  const int base = all / cnt, extra = all - base * cnt;
  first = c * base + (c < extra ? c : extra);
  units = base + (c < extra ? 1 : 0);
}

// Operand with the reduction index contiguous: LDS tile [rows][32 k], 64 bytes per row; the 16-byte
// piece c of row r sits in slot c ^ ((r >> 2) & 3), so 16 consecutive rows of a fragment read cover
// all 64 banks.  One copy instruction moves 16 rows.
template <int INSTR>  // copy instructions per wavefront and stage
struct KContig {
  u32x4 rsrc;
  uint32_t voff[INSTR];
  uint32_t lds_off;
  int kchunk;
  int64_t k_lim;
  uint32_t frag[2];  // byte offset of the lane's piece at K step 0 / 1, fragment 0

  // row0: first row of the tile; rows past o_lim read as zero
  __device__ __forceinline__ void init(const unsigned char* src, int64_t ld, int64_t o0, int64_t o_lim,
                                       int rows_max, int64_t k_limit, int wave, int lane,
                                       int frag_row0) {
    int64_t rows = o_lim - o0;
    rows = rows < 0 ? 0 : (rows > rows_max ? rows_max : rows);
    rsrc = make_raw_rsrc(src + o0 * ld * 2, rows * ld * 2);
    k_lim = k_limit;
    const int chunk = (lane & 3) ^ ((lane >> 4) & 3);
    kchunk = chunk * 8;
#pragma unroll
    for (int q = 0; q < INSTR; ++q) {
      const int blk = wave * INSTR + q;
      voff[q] = (uint32_t)(((int64_t)(blk * 16 + (lane >> 2)) * ld + chunk * 8) * 2);
    }
    lds_off = (uint32_t)(wave * INSTR * 1024);
    const int r = lane & 31, g = lane >> 5;
    frag[0] = (uint32_t)((frag_row0 + r) * 64 + ((g ^ ((r >> 2) & 3)) * 16));
    frag[1] = frag[0] ^ 32u;
  }
  __device__ __forceinline__ uint32_t offset(int kt) const { return stage_offset(rsrc[2], (uint32_t)kt, BKT * 2); }
  template <int q>
  __device__ __forceinline__ void issue(int kt, uint32_t off, uint32_t lds_tile, int) const {
    const bool kok = (int64_t)kt * BKT + kchunk < k_lim;
    dma16(lds_tile + lds_off + q * 1024, kok ? voff[q] : kOob, rsrc, off);
  }
  static constexpr int READS = 1;
  template <int j, int ks, int h>
  __device__ __forceinline__ void read(const unsigned char* tile, u32x4& f) const {
    f = *reinterpret_cast<const u32x4*>(tile + frag[ks] + j * 32 * 64);
  }
};

// Operand with the outer index contiguous: LDS tile [32 k][256 outer], 512 bytes per k row, segment
// swizzle and transposing reads as in gmm_dtl.hip.
struct OuterContig {
  u32x4 rsrc;
  uint32_t voff[4];
  uint32_t stage_bytes;  // global bytes between consecutive K tiles
  uint32_t frag_k;
  uint32_t frag_seg[4];

  // seg(j): 32-column segment of the lane's fragment j; gap > 0: tile columns 128..255 are outer
  // indices o0 + gap ..
  template <typename SegOf>
  __device__ __forceinline__ void init(const unsigned char* src, int64_t ld, int64_t o0, int64_t k_limit,
                                       int wave, int lane, SegOf&& seg, int64_t gap) {
    rsrc = make_raw_rsrc(src + o0 * 2, k_limit * ld * 2 - o0 * 2);
    stage_bytes = (uint32_t)(ld * 2 * BKT);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int krow = (wave * 4 + q) * 2 + (lane >> 5);
      const int f = (krow & 3) | ((krow >> 1) & 4);
      const int P = lane & 31;
      int64_t ct = ((((P >> 2) ^ f) << 2) + (P & 3)) * 8;
      if (gap > 0 && ct >= 128) ct += gap - 128;
      voff[q] = (uint32_t)(((int64_t)krow * ld + ct) * 2);
    }
    const int s = lane & 15, g = lane >> 5, half = (lane >> 4) & 1;
    frag_k = (uint32_t)((8 * g + (s >> 2)) * 512);
    const int f = (s >> 2) | (g << 2);
#pragma unroll
    for (int j = 0; j < 4; ++j) frag_seg[j] = (uint32_t)(((seg(j) ^ f) * 64) + half * 32 + (s & 3) * 8);
  }
  __device__ __forceinline__ uint32_t offset(int kt) const { return stage_offset(rsrc[2], (uint32_t)kt, stage_bytes); }
  template <int q>
  __device__ __forceinline__ void issue(int, uint32_t off, uint32_t lds_tile, int wave) const {
    dma16(lds_tile + (uint32_t)((wave * 4 + q) * 1024), voff[q], rsrc, off);
  }
  static constexpr int READS = 2;
  template <int j, int ks, int h>
  __device__ __forceinline__ void read(const unsigned char* tile, u32x4& f) const {
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4*)(lds_byte*)(tile + frag_k + frag_seg[j] +
                                                               (ks * 16 + h * 4) * 512));
    const u32x2 w = __builtin_bit_cast(u32x2, v);
    f[2 * h] = w[0];
    f[2 * h + 1] = w[1];
  }
};

// Row passes of the fused activation backward: the staged tile of d(act) with fc1 = [gate | up] gives
// d(fc1).  Out of line, as in gmm.hip: its registers are allocated apart from the main loop's, the
// pointers are cast to the global address space, and the loads carry no conditions (rows past the
// tile's last one repeat it), so each wait counts exactly the loads it needs.
template <int DT, bool GELU, int NP>
__attribute__((noinline)) __device__ void glu_bwd_rows(const unsigned char* lds, const unsigned char* fc1,
                                                       unsigned char* dfc1, int64_t F, int64_t n, int cc, int r0,
                                                       int64_t rows) {
  using CT = CTile<BN>;
  typedef __attribute__((address_space(1))) u32x4 global_u32x4;
  constexpr int PB = 2, NB = NP / PB;
  u32x4 gq[2][PB], uq[2][PB];
  auto request = [&](auto buf_c, int b) __attribute__((always_inline)) {
    constexpr int BUF = decltype(buf_c)::value;
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      int64_t row = (b * PB + j) * 8 + r0;
      row = row < rows ? row : rows - 1;
      const unsigned char* s = fc1 + (row * 2 * F + n) * 2;
      gq[BUF][j] = __builtin_nontemporal_load((const global_u32x4*)s);
      uq[BUF][j] = __builtin_nontemporal_load((const global_u32x4*)(s + F * 2));
    }
  };
  auto finish = [&](auto buf_c, int b) __attribute__((always_inline)) {
    constexpr int BUF = decltype(buf_c)::value;
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      const int row = (b * PB + j) * 8 + r0;
      float d[8], g[8], u[8], dg[8], du[8];
      Vec16<DT>::unpack(ctile_read16(lds + row * CT::pitch + cc * 16), d);
      Vec16<DT>::unpack(gq[BUF][j], g);
      Vec16<DT>::unpack(uq[BUF][j], u);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        dg[q] = d[q] * glu_act_grad(g[q], GELU) * u[q];
        du[q] = d[q] * glu_act(g[q], GELU);
      }
      if (row < rows) {
        unsigned char* o = dfc1 + ((int64_t)row * 2 * F + n) * 2;
        *(global_u32x4*)o = Vec16<DT>::pack(dg);
        *(global_u32x4*)(o + F * 2) = Vec16<DT>::pack(du);
      }
    }
  };
  request(std::integral_constant<int, 0>{}, 0);
  GMOE_SCHED_FENCE();
  static_for<0, NB>([&](auto b_c) __attribute__((always_inline)) {
    constexpr int b = decltype(b_c)::value;
    if constexpr (b + 1 < NB) request(std::integral_constant<int, (b + 1) & 1>{}, b + 1);
    GMOE_SCHED_FENCE();
    finish(std::integral_constant<int, b & 1>{}, b);
    GMOE_SCHED_FENCE();
  });
}

struct Item {
  int e, nt;
  long long row0;   // first row of the chunk, in the whole operand
  int64_t n;        // rows of the chunk that exist
};

// One tile: RF*64 rows x 256 columns, whole reduction, epilogue included.
template <int DT, int ODT, int MODE, int EPI, int RF>
__device__ __forceinline__ void run_tile(const GmmParams& p, const Item& it, unsigned char* lds, uint32_t lds0,
                                         int wave, int lane, int tid) {
  constexpr bool GLU = EPI == EPI_GLU_FWD_SILU || EPI == EPI_GLU_FWD_GELU;
  constexpr bool GLU_BWD = EPI == EPI_GLU_BWD_SILU || EPI == EPI_GLU_BWD_GELU;
  constexpr int A_BYTES = Stages<RF>::a_bytes, STAGE_BYTES = Stages<RF>::bytes, NST = Stages<RF>::count;
  constexpr int NLOAD = RF + 4;  // copy instructions per wavefront and stage
  typedef KContig<RF> OpA;
  typedef std::conditional_t<MODE == MODE_NT, KContig<4>, OuterContig> OpB;
  constexpr int RB = OpB::READS;
  constexpr int NREAD = RF + 4 * RB;
  constexpr int NM = RF * 4;
  const int64_t K = p.K, M = p.M;
  const int wm = wave >> 1, wn = wave & 1;

  f32x16 acc[RF][4];
#pragma unroll
  for (int i = 0; i < RF; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  OpA oa;
  OpB ob;
  oa.init(p.a + it.row0 * K * 2, K, 0, it.n, RF * kUnit, K, wave, lane, wm * RF * 32);
  if constexpr (MODE == MODE_NT)
    ob.init(p.b + (int64_t)it.e * M * K * 2, K, (int64_t)it.nt * BN, M, BN, K, wave, lane, wn * 128);
  else if constexpr (GLU)
    // fragments 0, 1: the wavefront's 64 gate columns, 2, 3: the up columns under them
    ob.init(p.b + (int64_t)it.e * K * M * 2, M, (int64_t)it.nt * 128, K, wave, lane,
            [&](int j) { return j < 2 ? 2 * wn + j : 4 + 2 * wn + (j - 2); }, p.F);
  else
    ob.init(p.b + (int64_t)it.e * K * M * 2, M, (int64_t)it.nt * BN, K, wave, lane,
            [&](int j) { return 4 * wn + j; }, 0);

  const int kt_cnt = (int)((K + BKT - 1) / BKT);
  u32x4 fa[2][RF], fb[2][4];

  auto issue = [&](auto op_c, int kt, uint32_t offa, uint32_t offb, uint32_t st) {
    constexpr int op = decltype(op_c)::value;
    if constexpr (op < RF) oa.template issue<op>(kt, offa, st, wave);
    else ob.template issue<op - RF>(kt, offb, st + A_BYTES, wave);
  };
  auto frag_read = [&](auto r_c, auto ks_c, auto buf_c, const unsigned char* stage) {
    constexpr int r = decltype(r_c)::value, ks = decltype(ks_c)::value, buf = decltype(buf_c)::value;
    if constexpr (r < RF) oa.template read<r, ks, 0>(stage, fa[buf][r]);
    else ob.template read<(r - RF) / RB, ks, (r - RF) % RB>(stage + A_BYTES, fb[buf][(r - RF) / RB]);
  };

  // One K step: the MFMAs with NREAD fragment reads and N copy requests spread evenly between them.
  // Requests issued in a burst (all of a tile's at the end of one step) cost 5-9 % of a large launch.
  auto k_step = [&](auto ks_c, auto n_c, auto&& read, auto&& request) {
    constexpr int ks = decltype(ks_c)::value, N = decltype(n_c)::value;
    static_for<0, NM>([&](auto m_c) {
      constexpr int m = decltype(m_c)::value;
      constexpr int mi = m / 4, mj = (mi & 1) ? 3 - m % 4 : m % 4;
      Mma<DT>::run(fa[ks][mi], fb[ks][mj], acc[mi][mj]);
      GMOE_SCHED_FENCE();
      static_for<(m * NREAD + NM - 1) / NM, ((m + 1) * NREAD + NM - 1) / NM>(read);
      static_for<(m * N + NM / 2) / NM, ((m + 1) * N + NM / 2) / NM>(request);
      GMOE_SCHED_FENCE();
    });
  };
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};

  static_for<0, NST - 1>([&](auto t_c) {
    constexpr int t = decltype(t_c)::value;
    const uint32_t offa = oa.offset(t), offb = ob.offset(t);
    static_for<0, NLOAD>([&](auto q) { issue(q, t, offa, offb, lds0 + t * STAGE_BYTES); });
  });
  wait_dma_outstanding<(NST - 2) * NLOAD>();
  __syncthreads();
  static_for<0, NREAD>([&](auto r) {
    frag_read(r, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, lds);
  });
  int s0 = 0;        // stage of tile kt
  int sl = NST - 1;  // stage of tile kt + NST - 1
  for (int kt = 0; kt < kt_cnt; ++kt) {
    const int s1 = s0 == NST - 1 ? 0 : s0 + 1;
    const unsigned char* cur = lds + s0 * STAGE_BYTES;
    const unsigned char* nxt = lds + s1 * STAGE_BYTES;
    const uint32_t stl = lds0 + (uint32_t)(sl * STAGE_BYTES);
    const int ktl = kt + NST - 1;
    const uint32_t offa = oa.offset(ktl), offb = ob.offset(ktl);
    // step 0: read step 1's fragments; request half of the tile kt+NST-1 into the stage tile kt-1 left
    k_step(c0, std::integral_constant<int, NLOAD / 2>{}, [&](auto r_c) { frag_read(r_c, c1, c1, cur); },
           [&](auto q_c) { issue(q_c, ktl, offa, offb, stl); });
    // tile kt+1 has landed (the later ones may be in flight); every wavefront has read this stage
    wait_dma_outstanding<(NST - 3) * NLOAD + NLOAD / 2>();
    __syncthreads();
    GMOE_SCHED_FENCE();
    // step 1: read step 0's fragments of tile kt+1; request the other half
    k_step(c1, std::integral_constant<int, NLOAD - NLOAD / 2>{}, [&](auto r_c) { frag_read(r_c, c0, c0, nxt); },
           [&](auto q_c) {
             issue(std::integral_constant<int, NLOAD / 2 + decltype(q_c)::value>{}, ktl, offa, offb, stl);
           });
    sl = s0;
    s0 = s1;
  }
  wait_dma_outstanding<0>();
  __syncthreads();

  // ---- epilogue ------------------------------------------------------------------------------
  constexpr int OES = Elem<ODT>::bytes;
  using CT = CTile<BN>;
  if constexpr (ODT == GMOE_F32) {
    unsigned char* c_base = p.c + it.row0 * M * OES;
#pragma unroll
    for (int i = 0; i < RF; ++i) {
      const int64_t m = wm * RF * 32 + i * 32 + (lane & 31);
      if (m >= it.n) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int vq = 0; vq < 4; ++vq) {
          const int64_t n = (int64_t)it.nt * BN + wn * 128 + j * 32 + 8 * vq + 4 * (lane >> 5);
          if (n < M)
            *reinterpret_cast<f32x4*>(c_base + (m * M + n) * OES) =
                f32x4{acc[i][j][4 * vq], acc[i][j][4 * vq + 1], acc[i][j][4 * vq + 2], acc[i][j][4 * vq + 3]};
        }
    }
    return;
  } else {
    stage_acc_lds<ODT, RF, 4, BN>(lds, acc, wm * RF * 32, wn * 128, lane);
    __syncthreads();
    if constexpr (GLU) {
      constexpr bool gelu = EPI == EPI_GLU_FWD_GELU;
      const int64_t F = p.F;
      unsigned char* fc1 = p.c + it.row0 * M * 2;
      unsigned char* act = p.c2 + it.row0 * F * 2;
      const int cc = tid & 15, r0 = tid >> 4;
      const int64_t n = (int64_t)it.nt * 128 + cc * 8;
      const int lcol = (cc >> 3) * 128 + (cc & 7) * 8;
#pragma unroll 4
      for (int q = 0; q < RF * 4; ++q) {
        const int row = q * 16 + r0;
        if (row >= it.n || n >= F) continue;
        const u32x4 gw = ctile_read16(lds + row * CT::pitch + lcol * 2);
        const u32x4 uw = ctile_read16(lds + row * CT::pitch + (lcol + 64) * 2);
        float g[8], u[8], o[8];
        Vec16<DT>::unpack(gw, g);
        Vec16<DT>::unpack(uw, u);
#pragma unroll
        for (int t = 0; t < 8; ++t) o[t] = glu_act(g[t], gelu) * u[t];
        st16(fc1 + (row * M + n) * 2, gw);
        st16(fc1 + (row * M + F + n) * 2, uw);
        st16(act + (row * F + n) * 2, Vec16<DT>::pack(o));
      }
    } else if constexpr (GLU_BWD) {
      const int cc = tid & 31, r0 = tid >> 5;
      const int64_t n = (int64_t)it.nt * BN + cc * 8;
      constexpr bool gelu = EPI == EPI_GLU_BWD_GELU;
      const int64_t F = M;
      const unsigned char* fc1 = p.aux + it.row0 * 2 * F * OES;
      unsigned char* dfc1 = p.c + it.row0 * 2 * F * OES;
      if (n < F) glu_bwd_rows<DT, gelu, RF * 8>(lds, fc1, dfc1, F, n, cc, r0, it.n);
    } else {
      const int cc = tid & 31, r0 = tid >> 5;
      const int64_t n = (int64_t)it.nt * BN + cc * 8;
      unsigned char* c_base = p.c + it.row0 * M * OES;
#pragma unroll 8
      for (int q = 0; q < RF * 8; ++q) {
        const int row = q * 8 + r0;
        if (row < it.n && n < M)
          st16(c_base + ((int64_t)row * M + n) * OES, ctile_read16(lds + row * CT::pitch + cc * 16));
      }
    }
    __syncthreads();
  }
}

template <int DT, int ODT, int MODE, int EPI>
__global__ __launch_bounds__(kGemmThreads, 1) void gmm_rows_kernel(GmmParams p) {
  constexpr bool GLU = EPI == EPI_GLU_FWD_SILU || EPI == EPI_GLU_FWD_GELU;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  __shared__ int tile_cum[kMaxGroupsLds + 1];
  __shared__ int wave_tot[kGemmThreads / 64];
  __shared__ int sums[kGemmThreads / 64][kMaxUnits + 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lds0 = lds_offset_of(lds);
  const int E = p.E;
  const int nt_cnt = GLU ? (int)((p.F + 127) / 128) : (int)((p.M + BN - 1) / BN);

  int max_units = kMaxUnits;
  {
    // tiles per expert -> exclusive prefix (a thread owns kPer consecutive experts)
    constexpr int kPer = kMaxGroupsLds / kGemmThreads;
    long long rows_of[kPer];
    int units = 0, chunks[kMaxUnits + 1] = {};
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int e = tid * kPer + j;
      rows_of[j] = e >= E ? 0 : group_begin(p, e + 1) - group_begin(p, e);
      units += unit_count(rows_of[j]);
#pragma unroll
      for (int u = 2; u <= kMaxUnits; ++u) chunks[u] += chunk_count(rows_of[j], u);
    }
    max_units = best_max_units(units, chunks, nt_cnt, (int)gridDim.x, p.K, sums, lane, wave);
    int cnt[kPer], local = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      cnt[j] = nt_cnt * chunk_count(rows_of[j], max_units);
      local += cnt[j];
    }
    int incl = local;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(incl, d);
      if (lane >= d) incl += o;
    }
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
  }
  __syncthreads();
  const int total = tile_cum[E];

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
    while (tile_cum[e + 1] <= v) ++e;
    Item it;
    it.e = __builtin_amdgcn_readfirstlane(e);
    const long long row0 = group_begin(p, e), n_e = group_begin(p, e + 1) - row0;
    const int chunks = chunk_count(n_e, max_units);
    int c, first, units;
    strip_order(v - tile_cum[e], chunks, nt_cnt, c, it.nt);
    chunk_units(n_e, chunks, c, first, units);
    it.row0 = row0 + (long long)first * kUnit;
    it.n = n_e - (long long)first * kUnit;
    if (it.n > units * kUnit) it.n = units * kUnit;
    switch (__builtin_amdgcn_readfirstlane(units)) {
      case 1: run_tile<DT, ODT, MODE, EPI, 1>(p, it, lds, lds0, wave, lane, tid); break;
      case 2: run_tile<DT, ODT, MODE, EPI, 2>(p, it, lds, lds0, wave, lane, tid); break;
      case 3: run_tile<DT, ODT, MODE, EPI, 3>(p, it, lds, lds0, wave, lane, tid); break;
      default: run_tile<DT, ODT, MODE, EPI, 4>(p, it, lds, lds0, wave, lane, tid); break;
    }
  }
}

template <int DT, int ODT, int MODE, int EPI>
static int launch_cfg(const GmmParams& p, hipStream_t st) {
  constexpr size_t stages = 144 * 1024, ctile = (size_t)256 * CTile<BN>::pitch;
  constexpr size_t smem = stages > ctile ? stages : ctile;
  auto kern = gmm_rows_kernel<DT, ODT, MODE, EPI>;
  static std::atomic<uint64_t> done_mask{0};
  if (!gmoe_once_per_device(done_mask, [&] {
        return hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) == hipSuccess;
      }))
    return GMOE_ERR_LAUNCH;
  int grid = (gmoe_cu_count() / 8) * 8;
  if (grid < 8) grid = 8;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(kGemmThreads), smem, st, p);
  return gmoe_launch_status();
}

template <int DT>
static int launch_dt(const GmmParams& p, int mode, int out_dtype, int epi, hipStream_t st) {
  if (mode == MODE_NN) {
    if (epi == EPI_GLU_FWD_SILU) return launch_cfg<DT, DT, MODE_NN, EPI_GLU_FWD_SILU>(p, st);
    if (epi == EPI_GLU_FWD_GELU) return launch_cfg<DT, DT, MODE_NN, EPI_GLU_FWD_GELU>(p, st);
    if (out_dtype == GMOE_F32) return launch_cfg<DT, GMOE_F32, MODE_NN, EPI_NONE>(p, st);
    return launch_cfg<DT, DT, MODE_NN, EPI_NONE>(p, st);
  }
  if (epi == EPI_GLU_BWD_SILU) return launch_cfg<DT, DT, MODE_NT, EPI_GLU_BWD_SILU>(p, st);
  if (epi == EPI_GLU_BWD_GELU) return launch_cfg<DT, DT, MODE_NT, EPI_GLU_BWD_GELU>(p, st);
  if (out_dtype == GMOE_F32) return launch_cfg<DT, GMOE_F32, MODE_NT, EPI_NONE>(p, st);
  return launch_cfg<DT, DT, MODE_NT, EPI_NONE>(p, st);
}

}  // namespace rows

int launch_gmm_rows(const GmmParams& p, int mode, int dtype, int out_dtype, int epi, hipStream_t st) {
  if (dtype == GMOE_BF16) return rows::launch_dt<GMOE_BF16>(p, mode, out_dtype, epi, st);
  if (dtype == GMOE_F16) return rows::launch_dt<GMOE_F16>(p, mode, out_dtype, epi, st);
  return GMOE_ERR_UNSUPPORTED;
}

}  // namespace gmoe
