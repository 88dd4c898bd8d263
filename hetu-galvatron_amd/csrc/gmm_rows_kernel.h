// Grouped GEMM with row-adaptive tiles for 16-bit operands (bf16 / fp16) on gfx950: NN and NT of
// gmm.hip's contract, with the fused gated-activation epilogues: from 96 rows per expert on what rows_rule.h prices cheaper
// here, with the activation from 4 rows on where the tiles fill their rounds, and its short launches from one row on.
//
//   * A tile is RF*64 rows (RF = 1..6, chosen per tile) x 256 columns of C.  An expert's rows are cut
//     into chunks of up to 384 (320 .. 128 where those fill the rounds better: best_max_units) that are as
//     equal as 64-row steps allow, so at most 63 rows per expert are padding.
//   * 2x2 wavefronts of (RF*32) x 128, one workgroup per CU.  Up to 24 accumulators of 32x32: 16 in the
//     256 accumulation registers, the other 8 in architectural ones (mma_vgpr), which leaves 128 of those for
//     two sets of fragments and the addresses.
//   * What bounds it: power, and the operand stream where an expert has a few hundred rows (fc1 of the
//     Mixtral shape at 383 rows per expert: matrix cores 60 % busy at 1.85 GHz; without three fifths of the
//     MFMAs 575 instead of 663 us at 2.4 GHz).  Both ask for fewer operand bytes per operation.  A 384-row tile
//     takes 17 % fewer than a 256-row one through L2 and LDS: 4096 rows per expert, 8 experts, us in chunks of up
//     to 256 / 384 rows, with activation 4096 x 28672 6255 / 5836, NN 14336 x 4096 2953 / 2790, NT 28672 x 4096
//     5978 / 5727.
//   * Operands go global -> LDS without staging registers (buffer_load ... lds).  Rows that are contiguous in
//     the reduction index are copied 64 elements at a time, whole cache lines: copies of 32, half lines, ask L2
//     one and a half times as often (NT 1024 rows per expert, 2816 x 2048, 64 experts 660 -> 637 us, 28672 x 4096, 8
//     experts of 383 753 -> 691).  Each operand has a ring of its own as deep as LDS allows; weights whose
//     reduction index is the slow dimension (NN) move 32 rows of 512 bytes at a time, which lets four to eight of
//     them be in flight beside two or three tiles of A (one ring of 64-deep tiles for both: with activation 383 rows,
//     4096 x 28672 734 instead of 686 us).  The copies are spread one by one between the MFMAs.
//   * Measured without gain: a staggered start of the workgroups' K walks, 128x256 tiles with two workgroups per
//     CU (their operand stream is half again as large: 700 instead of 860 TFLOP/s at 383 rows per expert).
#pragma once
#include "gmm_common.h"

namespace gmoe {

namespace rows {

constexpr int BN = 256;
constexpr int BKT = 64;    // reduction elements per round
constexpr int kUnit = 64;  // rows per unit: 32 for each of the two wavefront rows
constexpr int kLdsBytes = 160 * 1024;
constexpr int kMaxUnits = kTallMaxUnits;  // units per tile

// LDS: a ring of 64-deep tiles of A and one of B.  B's are 64 deep where its rows are contiguous in the reduction
// index (NT), as A's, and 32 deep where they are not (NN).
template <int MODE, int RF>
struct Rings {
  static constexpr bool nt = MODE == MODE_NT;
  static constexpr int a_bytes = RF * kUnit * BKT * 2, b_bytes = nt ? BN * BKT * 2 : BN * BKT;
  static constexpr int na = nt ? (RF >= 3 ? 2 : (RF == 2 ? 3 : 4)) : (RF >= 5 ? 2 : 3);
  static constexpr int nb = nt ? (RF >= 5 ? 2 : (RF >= 2 ? 3 : 4))
                               : (RF == 6 || RF == 4 ? 4 : (RF == 5 || RF == 3 ? 5 : (RF == 2 ? 7 : 8)));
  static_assert(na * a_bytes + nb * b_bytes <= kLdsBytes, "LDS");
};

typedef short s16x4 __attribute__((ext_vector_type(4)));

// Row chunks of an expert with n rows: units of kUnit rows dealt as evenly as possible to
// ceil(units / max_units) chunks.
__device__ __forceinline__ int unit_count(long long n) { return (int)((n + kUnit - 1) / kUnit); }
__device__ __forceinline__ int chunk_count(long long n, int max_units) {
  return (unit_count(n) + max_units - 1) / max_units;
}
// rows_chunk_units for the launch; v: units and chunks of this thread's experts, summed over the workgroup here.
template <int EPI>
__device__ __forceinline__ int best_max_units(int (&v)[kMaxUnits + 1], int nt_cnt, int grid, int E, int64_t K, int* sums,
                                              int lane, int wave) {
#pragma unroll
  for (int i = 0; i <= kMaxUnits; ++i) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) v[i] += __shfl_xor(v[i], d);
    if (lane == 0) sums[wave * (kMaxUnits + 1) + i] = v[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i <= kMaxUnits; ++i) {
    v[i] = 0;
#pragma unroll
    for (int w = 0; w < kGemmThreads / 64; ++w) v[i] += sums[w * (kMaxUnits + 1) + i];
  }
  constexpr bool bwd = EPI == EPI_GLU_BWD_SILU || EPI == EPI_GLU_BWD_GELU;
  return rows_chunk_units(v, nt_cnt, grid, K, chunk_costs(bwd, v[0], E));
}
// first unit and unit count of chunk c of cnt
__device__ __forceinline__ void chunk_units(long long n, int cnt, int c, int& first, int& units) {
  const int all = (int)((n + kUnit - 1) / kUnit);
  const int base = all / cnt, extra = all - base * cnt;
  first = c * base + (c < extra ? c : extra);
  units = base + (c < extra ? 1 : 0);
}

// Operand with the reduction index contiguous: LDS tile [rows][64 k], 128 bytes per row; the 16-byte
// piece c of row r sits in slot c ^ ((r >> 1) & 7), so 16 consecutive rows of a fragment read cover
// all 64 banks.  One copy instruction moves 8 rows, whole cache lines of them.
template <int INSTR>  // copy instructions per wavefront and stage
struct KContig {
  u32x4 rsrc;
  uint32_t voff[2];      // even and odd copy instructions, without their rows
  uint32_t row16_bytes;  // 16 rows of the operand
  uint32_t lds_off;
  int kchunk[2];
  int64_t k_lim;
  uint32_t frag;  // byte offset of the lane's piece at K step 0, fragment 0

  // o0: first row of the tile; rows past o_lim read as zero
  __device__ __forceinline__ void init(const unsigned char* src, int64_t ld, int64_t o0, int64_t o_lim,
                                       int rows_max, int64_t k_limit, int wave, int lane,
                                       int frag_row0) {
    int64_t rows = o_lim - o0;
    rows = rows < 0 ? 0 : (rows > rows_max ? rows_max : rows);
    rsrc = make_raw_rsrc(src + o0 * ld * 2, rows * ld * 2);
    k_lim = k_limit;
    row16_bytes = (uint32_t)(16 * ld * 2);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int row = (wave * INSTR + q) * 8 + (lane >> 3);
      const int chunk = (lane & 7) ^ ((row >> 1) & 7);
      kchunk[q] = chunk * 8;
      voff[q] = (uint32_t)((int64_t)row * ld * 2 + chunk * 16);
    }
    lds_off = (uint32_t)(wave * INSTR * 1024);
    const int r = lane & 31, g = lane >> 5;
    frag = (uint32_t)((frag_row0 + r) * 128 + ((g ^ ((r >> 1) & 7)) * 16));
  }
  __device__ __forceinline__ uint32_t offset(int kt) const { return (uint32_t)kt * (BKT * 2); }
  template <int q>
  __device__ __forceinline__ void issue(int kt, uint32_t off, uint32_t lds_tile, int) const {
    const bool kok = (int64_t)kt * BKT + kchunk[q & 1] < k_lim;
    const uint32_t o = off + (q >> 1) * row16_bytes;
    dma16(lds_tile + lds_off + q * 1024, kok ? voff[q & 1] : kOob, rsrc, o < rsrc[2] ? o : rsrc[2]);
  }
  static constexpr int READS = 1;
  template <int j, int ks, int h>
  __device__ __forceinline__ void read(const unsigned char* tile, u32x4& f) const {
    f = *reinterpret_cast<const u32x4*>(tile + (frag ^ (ks * 32u)) + j * 32 * 128);
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
    stage_bytes = (uint32_t)(ld * 2 * 32);
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

// acc += b a with the accumulators in architectural registers: the compiler puts those of the builtin into the
// accumulation registers, which hold 16 fragments.  It inserts no wait states around assembly: mma_ready and mma_settle bring
// those before the first and after the last, and in between no vector instruction may write an operand in the two wait
// states before, or touch the result in the 18 after, which the built kernels are tested for.  (The two wait states in
// front of each one: 1 % slower, NN and NT of 4096 rows, 14336 x 4096 and 28672 x 4096, 8 experts.)
template <int DT>
__device__ __forceinline__ void mma_vgpr(const u32x4& a, const u32x4& b, f32x16& acc) {
  if constexpr (DT == GMOE_BF16)
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(b), "v"(a));
  else
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(acc) : "v"(b), "v"(a));
}

// Between vector instructions that wrote operands of mma_vgpr and the first of them.
__device__ __forceinline__ void mma_ready() {
  GMOE_SCHED_FENCE();
  asm volatile("s_nop 1");
  GMOE_SCHED_FENCE();
}

// Before vector instructions read what mma_vgpr wrote: the compiler does not know how long that takes (up to 16 passes
// and 18 wait states; these are 24).
__device__ __forceinline__ void mma_settle(f32x16& acc) { asm volatile("s_nop 15\n\ts_nop 7" : "+v"(acc)); }

// Fragments I0 .. I0+IN-1 of both wavefront rows as a tile of 2 * IN * 32 rows.
template <int ODT, int RF, int I0, int IN>
__device__ __forceinline__ void stage_acc_part(unsigned char* lds, const f32x16 (&acc)[RF][4], int wm, int wn, int lane) {
#pragma unroll
  for (int i = 0; i < IN; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        const int row = wm * IN * 32 + i * 32 + (lane & 31), col = wn * 128 + j * 32 + 8 * vq + 4 * (lane >> 5);
        const f32x16& v = acc[I0 + i][j];
        *reinterpret_cast<u32x2*>(lds + row * CTile<BN>::pitch + col * 2) =
            pack4<ODT>(v[4 * vq], v[4 * vq + 1], v[4 * vq + 2], v[4 * vq + 3]);
      }
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
  // what depends on the lane is worked out by each tile size for itself: shared between them it would be spilled
  asm volatile("" : "+v"(lane), "+v"(tid));
  asm volatile("" : "+s"(wave), "+s"(lds0));
  constexpr bool GLU = EPI == EPI_GLU_FWD_SILU || EPI == EPI_GLU_FWD_GELU;
  constexpr bool GLU_BWD = EPI == EPI_GLU_BWD_SILU || EPI == EPI_GLU_BWD_GELU;
  typedef Rings<MODE, RF> R;
  constexpr int NA = R::na, NB = R::nb;
  constexpr int LA = 2 * RF, LB = R::nt ? 8 : 4;  // copy instructions per wavefront and tile of A / B
  typedef KContig<2 * RF> OpA;
  typedef std::conditional_t<MODE == MODE_NT, KContig<8>, OuterContig> OpB;
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
  unsigned char* const ring_b = lds + NA * R::a_bytes;
  const uint32_t lds_b = lds0 + NA * R::a_bytes;

  auto k_step = [&](auto ks_c, auto n_c, auto&& read, auto&& request) __attribute__((always_inline)) {
    constexpr int ks = decltype(ks_c)::value, N = decltype(n_c)::value;
    static_for<0, NM>([&](auto m_c) __attribute__((always_inline)) {
      constexpr int m = decltype(m_c)::value;
      constexpr int mi = m / 4, mj = (mi & 1) ? 3 - m % 4 : m % 4;
      if constexpr (mi < RF - 4) mma_vgpr<DT>(fa[ks & 1][mi], fb[ks & 1][mj], acc[mi][mj]);
      else Mma<DT>::run(fa[ks & 1][mi], fb[ks & 1][mj], acc[mi][mj]);
      GMOE_SCHED_FENCE();
      static_for<(m * NREAD + NM - 1) / NM, ((m + 1) * NREAD + NM - 1) / NM>(read);
      static_for<(m * N + NM / 2) / NM, ((m + 1) * N + NM / 2) / NM>(request);
      GMOE_SCHED_FENCE();
    });
  };
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  constexpr std::integral_constant<int, 2> c2{};
  constexpr std::integral_constant<int, 3> c3{};
  auto read_frags = [&](auto ks_c, const unsigned char* ta, const unsigned char* tb) {
    // reader of the fragments of K step ks, from A's tile ta and B's tile tb
    return [&, ta, tb](auto r_c) __attribute__((always_inline)) {
      constexpr int r = decltype(r_c)::value, ks = decltype(ks_c)::value, buf = ks & 1;
      if constexpr (r < RF) oa.template read<r, ks, 0>(ta, fa[buf][r]);
      else ob.template read<(r - RF) / RB, R::nt ? ks : (ks & 1), (r - RF) % RB>(tb, fb[buf][(r - RF) / RB]);
    };
  };
  auto next = [](int i, int n) { return i == n - 1 ? 0 : i + 1; };
  constexpr std::integral_constant<int, 0> none{};

  if constexpr (R::nt) {
    // Order of the copies of round p (64 reduction elements): tile p - 1 + NA of A, then tile p - 1 + NB of B, from
    // K step 3 of round p - 1 on; where B's ring has two tiles, early enough to land within the round.  Copies land
    // in order, so what may be in flight when a tile is needed is what was issued after it.
    constexpr int L = LA + LB;
    constexpr int N3 = NB == 2 ? L * 3 / 10 : L / 4, N0 = NB == 2 ? L * 4 / 10 : L / 4,
                  N1 = NB == 2 ? L - N3 - N0 : L / 4, N2 = L - N3 - N0 - N1;
    constexpr int a_end = (2 - NA) * L + LA, b_end = (3 - NB) * L;
    constexpr int wait_y = L - (a_end > b_end ? a_end : b_end);
    // copy op of round p: la, lb the slots of the two tiles
    auto issue = [&](auto op_c, int p, uint32_t offa, uint32_t offb, int la, int lb) __attribute__((always_inline)) {
      constexpr int op = decltype(op_c)::value;
      if constexpr (op < LA) oa.template issue<op>(p - 1 + NA, offa, lds0 + (uint32_t)la * R::a_bytes, wave);
      else ob.template issue<op - LA>(p - 1 + NB, offb, lds_b + (uint32_t)lb * R::b_bytes, wave);
    };
    static_for<0, NB>([&](auto i_c) {
      constexpr int r = decltype(i_c)::value + 1 - NB;  // rounds 1 - NB .. 0
      static_for<0, (r == 0 ? N3 : L)>([&](auto q) {
        if constexpr (decltype(q)::value >= LA || r - 1 + NA >= 0)
          issue(q, r, oa.offset(r - 1 + NA), ob.offset(r - 1 + NB), r - 1 + NA, r - 1 + NB);
      });
    });
    wait_dma_outstanding<wait_y + N3>();
    __syncthreads();
    static_for<0, NREAD>(read_frags(c0, lds, ring_b));
    if constexpr (RF > 4) mma_ready();
    int sa = 0, sb = 0;            // slots of tile kt
    int la = NA - 1, lb = NB - 1;  // slots of tiles kt - 1 + NA of A and kt - 1 + NB of B
    for (int kt = 0; kt < kt_cnt; ++kt) {
      const int sa1 = next(sa, NA), sb1 = next(sb, NB);
      const unsigned char *ca = lds + sa * R::a_bytes, *cb = ring_b + sb * R::b_bytes;
      const unsigned char *xa = lds + sa1 * R::a_bytes, *xb = ring_b + sb1 * R::b_bytes;
      {
        const uint32_t offa = oa.offset(kt - 1 + NA), offb = ob.offset(kt - 1 + NB);
        auto request = [&](auto first_c) {
          return [&](auto q_c) __attribute__((always_inline)) {
            issue(std::integral_constant<int, decltype(first_c)::value + decltype(q_c)::value>{}, kt, offa, offb, la, lb);
          };
        };
        k_step(c0, std::integral_constant<int, N0>{}, read_frags(c1, ca, cb), request(std::integral_constant<int, N3>{}));
        k_step(c1, std::integral_constant<int, N1>{}, read_frags(c2, ca, cb), request(std::integral_constant<int, N3 + N0>{}));
        k_step(c2, std::integral_constant<int, N2>{}, read_frags(c3, ca, cb), request(std::integral_constant<int, N3 + N0 + N1>{}));
      }
      // tiles kt + 1 have landed; every wavefront has read tiles kt
      wait_dma_outstanding<wait_y>();
      __syncthreads();
      GMOE_SCHED_FENCE();
      {
        const uint32_t offa = oa.offset(kt + NA), offb = ob.offset(kt + NB);
        k_step(c3, std::integral_constant<int, N3>{}, read_frags(c0, xa, xb),
               [&](auto q_c) { issue(q_c, kt + 1, offa, offb, sa, sb); });
      }
      la = sa;
      sa = sa1;
      lb = sb;
      sb = sb1;
    }
  } else {
    // Order of the copies of round p (64 reduction elements): tile p - 1 + NA of A in K steps 3 of round p - 1
    // and 0, tiles 2 p - 1 + NB and 2 p + NB of B in K steps 1 and 2.  Copies land in order, so what may be in
    // flight when a tile is needed is what was issued after it (positions in the order, relative to round 0).
    constexpr int L = LA + 2 * LB;
    constexpr auto half = [](int v) { return v < 0 ? -((1 - v) / 2) : v / 2; };
    constexpr int a_end = (2 - NA) * L + LA;  // tile 1 of A
    constexpr int b2_end = NB % 2 == 0 ? ((2 - NB) / 2 + 1) * L : half(3 - NB) * L + LA + LB;  // tile 2 of B
    constexpr int b1_end = NB % 2 == 0 ? half(2 - NB) * L + LA + LB : (half(1 - NB) + 1) * L;  // tile 1 of B
    constexpr int wait_y = L - (a_end > b2_end ? a_end : b2_end), wait_x = LA - b1_end;
    constexpr int A3 = LA / 2;
    auto issue_a = [&](auto q_c, int t, uint32_t off, int slot) __attribute__((always_inline)) {
      oa.template issue<decltype(q_c)::value>(t, off, lds0 + (uint32_t)slot * R::a_bytes, wave);
    };
    auto issue_b = [&](auto q_c, uint32_t off, int slot) __attribute__((always_inline)) {
      ob.template issue<decltype(q_c)::value>(0, off, lds_b + (uint32_t)slot * R::b_bytes, wave);
    };
    static_for<0, NB>([&](auto i_c) {
      constexpr int r = decltype(i_c)::value - NB;  // rounds -NB .. -1
      if constexpr (r - 1 + NA >= 0)
        static_for<0, LA>([&](auto q) { issue_a(q, r - 1 + NA, oa.offset(r - 1 + NA), r - 1 + NA); });
      if constexpr (2 * r - 1 + NB >= 0)
        static_for<0, LB>([&](auto q) { issue_b(q, ob.offset(2 * r - 1 + NB), 2 * r - 1 + NB); });
      if constexpr (2 * r + NB >= 0)
        static_for<0, LB>([&](auto q) { issue_b(q, ob.offset(2 * r + NB), 2 * r + NB); });
    });
    wait_dma_outstanding<wait_y>();
    __syncthreads();
    static_for<0, NREAD>(read_frags(c0, lds, ring_b));
    static_for<0, A3>([&](auto q) { issue_a(q, NA - 1, oa.offset(NA - 1), NA - 1); });
    if constexpr (RF > 4) mma_ready();
    int sa = 0, sb = 0;    // slots of tiles p of A and 2 p of B
    int la = NA - 1, lb = NB - 1;  // slots of tiles p - 1 + NA of A and 2 p - 1 + NB of B
    for (int p2 = 0; p2 < kt_cnt; ++p2) {
      const int sb1 = next(sb, NB), sb2 = next(sb1, NB), sa1 = next(sa, NA);
      const unsigned char *ca = lds + sa * R::a_bytes, *xa = lds + sa1 * R::a_bytes;
      const unsigned char *b0 = ring_b + sb * R::b_bytes, *b1 = ring_b + sb1 * R::b_bytes, *b2 = ring_b + sb2 * R::b_bytes;
      {
        const uint32_t off = oa.offset(p2 - 1 + NA);
        k_step(c0, std::integral_constant<int, LA - A3>{}, read_frags(c1, ca, b0), [&](auto q_c) {
          issue_a(std::integral_constant<int, A3 + decltype(q_c)::value>{}, p2 - 1 + NA, off, la);
        });
      }
      // tile 2 p + 1 of B has landed; every wavefront has read tile 2 p
      wait_dma_outstanding<wait_x>();
      __syncthreads();
      GMOE_SCHED_FENCE();
      {
        const uint32_t off = ob.offset(2 * p2 - 1 + NB);
        k_step(c1, std::integral_constant<int, LB>{}, read_frags(c2, ca, b1), [&](auto q_c) { issue_b(q_c, off, lb); });
      }
      {
        const uint32_t off = ob.offset(2 * p2 + NB);
        k_step(c2, std::integral_constant<int, LB>{}, read_frags(c3, ca, b1), [&](auto q_c) { issue_b(q_c, off, sb); });
      }
      // tiles p + 1 of A and 2 p + 2 of B have landed; every wavefront has read A's tile p and B's tile 2 p + 1
      wait_dma_outstanding<wait_y>();
      __syncthreads();
      GMOE_SCHED_FENCE();
      {
        const uint32_t off = oa.offset(p2 + NA);
        k_step(c3, std::integral_constant<int, A3>{}, read_frags(c0, xa, b2),
               [&](auto q_c) { issue_a(q_c, p2 + NA, off, sa); });
      }
      la = sa;
      sa = sa1;
      lb = sb1;
      sb = sb2;
    }
  }
  wait_dma_outstanding<0>();
  static_for<0, (RF > 4 ? RF - 4 : 0)>([&](auto i_c) {
    static_for<0, 4>([&](auto j_c) { mma_settle(acc[decltype(i_c)::value][decltype(j_c)::value]); });
  });
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
    // a tile of more than 256 rows is staged in two parts, each of some fragments of both wavefront rows
    constexpr int PARTS = RF > 4 ? 2 : 1;
    static_for<0, PARTS>([&](auto part_c) __attribute__((always_inline)) {
      constexpr int part = decltype(part_c)::value;
      constexpr int I0 = part * (RF + 1) / 2 * (PARTS - 1), IN = PARTS == 1 ? RF : (part == 0 ? (RF + 1) / 2 : RF / 2);
      stage_acc_part<ODT, RF, I0, IN>(lds, acc, wm, wn, lane);
      __syncthreads();
      constexpr int BLOCKS = PARTS == 1 ? 1 : 2, BROWS = PARTS == 1 ? RF * 64 : IN * 32;
#pragma unroll
      for (int w = 0; w < BLOCKS; ++w) {
        const int first = w * RF * 32 + I0 * 32;
        const int64_t rows = it.n - first;
        if (rows <= 0) continue;
        const int64_t row0 = it.row0 + first;
        const unsigned char* tile = lds + w * BROWS * CT::pitch;
        if constexpr (GLU) {
          constexpr bool gelu = EPI == EPI_GLU_FWD_GELU;
          const int64_t F = p.F;
          unsigned char* fc1 = p.c + row0 * M * 2;
          unsigned char* act = p.c2 + row0 * F * 2;
          const int cc = tid & 15, r0 = tid >> 4;
          const int64_t n = (int64_t)it.nt * 128 + cc * 8;
          const int lcol = (cc >> 3) * 128 + (cc & 7) * 8;
#pragma unroll 4
          for (int q = 0; q < BROWS / 16; ++q) {
            const int row = q * 16 + r0;
            if (row >= rows || n >= F) continue;
            const u32x4 gw = ctile_read16(tile + row * CT::pitch + lcol * 2);
            const u32x4 uw = ctile_read16(tile + row * CT::pitch + (lcol + 64) * 2);
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
          const unsigned char* fc1 = p.aux + row0 * 2 * F * OES;
          unsigned char* dfc1 = p.c + row0 * 2 * F * OES;
          if (n < F) glu_bwd_rows<DT, gelu, BROWS / 8>(tile, fc1, dfc1, F, n, cc, r0, rows);
        } else {
          const int cc = tid & 31, r0 = tid >> 5;
          const int64_t n = (int64_t)it.nt * BN + cc * 8;
          unsigned char* c_base = p.c + row0 * M * OES;
#pragma unroll 8
          for (int q = 0; q < BROWS / 8; ++q) {
            const int row = q * 8 + r0;
            if (row < rows && n < M)
              st16(c_base + ((int64_t)row * M + n) * OES, ctile_read16(tile + row * CT::pitch + cc * 16));
          }
        }
      }
      __syncthreads();
    });
  }
}

template <int DT, int ODT, int MODE, int EPI>
__global__ __launch_bounds__(kGemmThreads, 1) void gmm_rows_kernel(GmmParams p) {
  constexpr bool GLU = EPI == EPI_GLU_FWD_SILU || EPI == EPI_GLU_FWD_GELU;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lds0 = lds_offset_of(lds);
  const int E = p.E;
  const int nt_cnt = GLU ? (int)((p.F + 127) / 128) : (int)((p.M + BN - 1) / BN);

  // Tiles before and after each of this thread's kPer consecutive experts; the rings and the staged result take all
  // of the LDS, so the table stays in registers and LDS serves as scratch between tiles.
  constexpr int kPer = kMaxGroupsLds / kGemmThreads, kWaves = kGemmThreads / 64;
  int* const scratch = reinterpret_cast<int*>(lds);
  int tiles_before[kPer + 1], total, max_units;
  {
    long long rows_of[kPer];
    int v[kMaxUnits + 1] = {};
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int e = tid * kPer + j;
      rows_of[j] = e >= E ? 0 : group_begin(p, e + 1) - group_begin(p, e);
      v[0] += unit_count(rows_of[j]);
#pragma unroll
      for (int u = 2; u <= kMaxUnits; ++u) v[u] += chunk_count(rows_of[j], u);
    }
    max_units = best_max_units<EPI>(v, nt_cnt, (int)gridDim.x, E, p.K, scratch + kWaves, lane, wave);
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
    if (lane == 63) scratch[wave] = incl;
    __syncthreads();
    int run = incl - local;
    total = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      if (w < wave) run += scratch[w];
      total += scratch[w];
    }
    total = __builtin_amdgcn_readfirstlane(total);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      tiles_before[j] = run;
      run += cnt[j];
    }
    tiles_before[kPer] = run;
    __syncthreads();
  }

  // XCD x takes the positions [x*G/8, (x+1)*G/8) of every whole round of G tiles; the last, partial
  // round is dealt to the XCDs in equal consecutive shares
  const int G = gridDim.x, per_xcd = G / 8;
  const int xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
  for (int base = 0; base < total; base += G) {
    int v = base + xcd * per_xcd + slot;
    if (total - base < G) {
      const int share = (total - base + 7) / 8;
      v = base + xcd * share + slot;
      if (slot >= share || v >= total) break;
    }
    // the thread whose expert tile v belongs to says so
#pragma unroll
    for (int j = 0; j < kPer; ++j)
      if (v >= tiles_before[j] && v < tiles_before[j + 1]) {
        scratch[0] = tid * kPer + j;
        scratch[1] = v - tiles_before[j];
      }
    __syncthreads();
    Item it;
    it.e = __builtin_amdgcn_readfirstlane(scratch[0]);
    const int place = __builtin_amdgcn_readfirstlane(scratch[1]);
    __syncthreads();
    const long long row0 = group_begin(p, it.e), n_e = group_begin(p, it.e + 1) - row0;
    const int chunks = chunk_count(n_e, max_units);
    int c, first, units;
    strip_order(place, chunks, nt_cnt, c, it.nt);
    chunk_units(n_e, chunks, c, first, units);
    it.row0 = row0 + (long long)first * kUnit;
    it.n = n_e - (long long)first * kUnit;
    if (it.n > units * kUnit) it.n = units * kUnit;
    switch (__builtin_amdgcn_readfirstlane(units)) {
      case 1: run_tile<DT, ODT, MODE, EPI, 1>(p, it, lds, lds0, wave, lane, tid); break;
      case 2: run_tile<DT, ODT, MODE, EPI, 2>(p, it, lds, lds0, wave, lane, tid); break;
      case 3: run_tile<DT, ODT, MODE, EPI, 3>(p, it, lds, lds0, wave, lane, tid); break;
      case 4: run_tile<DT, ODT, MODE, EPI, 4>(p, it, lds, lds0, wave, lane, tid); break;
      case 5: run_tile<DT, ODT, MODE, EPI, 5>(p, it, lds, lds0, wave, lane, tid); break;
      default: run_tile<DT, ODT, MODE, EPI, 6>(p, it, lds, lds0, wave, lane, tid); break;
    }
  }
}

template <int DT, int ODT, int MODE, int EPI>
static int launch_cfg(const GmmParams& p, hipStream_t st) {
  constexpr size_t smem = kLdsBytes;
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
}  // namespace gmoe
