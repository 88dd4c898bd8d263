// Grouped GEMM, LDS-DMA variant for the dW product (TN) of 16-bit operands (bf16 / fp16) on gfx950:
//   c[e] = a[rows_e]^T @ b[rows_e],  a [N,K], b [N,M], c [E,K,M].
//
// Same contract, tile order and MFMA arrangement as gmm.hip (256x256 block tile, 2x2 wavefronts,
// 32x32x16 MFMAs, operands swapped so a lane owns 4 consecutive columns of C).  What differs is how
// operand tiles reach LDS and how deep the prefetch is:
//
//   * Global memory is copied straight into LDS by `buffer_load_dwordx4 ... lds` (no staging
//     registers, no ds_write).  A wavefront instruction deposits 64 x 16 bytes contiguously, so
//     there is no room for row padding; bank conflicts are avoided by permuting WHICH 16-byte
//     chunk a lane fetches (an XOR swizzle applied on the global side) and undoing it in the
//     fragment addresses.
//   * A K tile is 32 elements deep and LDS holds 4 stages (4 x 32 KiB): the copy of tile t+3 is
//     issued while tile t is multiplied, i.e. a request has about three tiles of MFMAs to land.
//     One barrier per K tile; the copies are tracked by hand (vmcnt), the compiler tracks the
//     LDS reads.
//   * The K tiles of all of a workgroup's output tiles form one sequence: the last three of a tile
//     request the first three of the next, and the stores of a tile are left in flight under the next
//     tile's MFMAs.
//   * Long reductions (STORE_SPREAD): a 16-bit result is rounded into half the registers while the next tile's
//     first MFMAs overwrite the accumulators, and stored piece by piece under the MFMAs after those, so that
//     the matrix cores see no epilogue (2-4 % at 1024 rows per expert, nothing at 4096, where the chip's power is
//     the bound; figures at launch_cfg).
//   * Large results are stored past the L2s' reusable lines (nontemporal), and few rows per expert read both
//     operands once beforehand (warm_operands): the launch is then bound by its writes.  4096 x 28672 over 8
//     experts, operands from HBM: 192 rows each 663 -> 483 us (3.9 TB/s of results), 384 rows 882 -> 740.
//   * Both operands have the reduction index (the token) as the slow dimension in memory; they are
//     stored in LDS as they are in memory, [k][outer], and the MFMA fragments are read with the
//     transposing LDS load ds_read_b64_tr_b16: a group of 16 lanes reads a 4(k) x 16(outer) block
//     and every lane receives the 4 k-values of its own column.
//
// NN and NT have a kernel of their own (gmm_rows_kernel.h): 32-deep copies of an operand whose reduction
// index is contiguous would be 64-byte row pieces, which the address path handles at half the rate of whole lines.
// What did not help: stores issued by two wavefronts and copies by the other two, so that no copy waits behind a
// store (5 to 7 % slower at 383 to 4096 rows per expert: 16 copies per K tile from one wavefront).
#include "gmm_common.h"

namespace gmoe {

namespace dtl {

constexpr int BM = 256, BN = 256;
constexpr int BKT = 32;                 // reduction elements per stage
constexpr int NST = 4;                  // LDS stages
constexpr int OPER_BYTES = 256 * BKT * 2;  // one operand tile: 16 KiB
constexpr int STAGE_BYTES = 2 * OPER_BYTES;
constexpr int LOADS_PER_TILE = 8;       // LDS-DMA instructions per wavefront per K tile (4 per operand)

constexpr int kNontemporal = 2;         // cache policy operand of a buffer store

typedef short s16x4 __attribute__((ext_vector_type(4)));
// ---- operand stored outer-contiguous: LDS tile [32 k][256 outer], 512 bytes per k row ----------
// The 64-byte segment sg of row k sits at segment position sg ^ f(k), f(k) = (k & 3) | ((k >> 1) & 4):
// the 8 rows one transposing read touches (k0..k0+3 and k0+8..k0+11) land in 8 different segments.
// What a lane needs of an operand whatever the output tile; the tile itself is a buffer resource.
struct TransOperand {
  uint32_t voff[4];
  uint32_t stage_bytes;  // global bytes between consecutive K tiles
  uint32_t frag_k;       // byte offset of the lane's first k row
  uint32_t frag_seg[4];  // byte offset of the lane's 8 bytes inside a k row, per fragment

  __device__ __forceinline__ void init(int64_t ld, int wave, int lane, int sub_col0) {
    stage_bytes = (uint32_t)(ld * 2 * BKT);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int krow = (wave * 4 + q) * 2 + (lane >> 5);
      const int f = (krow & 3) | ((krow >> 1) & 4);
      const int P = lane & 31;                      // 16-byte slot inside the k row
      const int ct = ((((P >> 2) ^ f) << 2) + (P & 3)) * 8;  // tile column this slot holds
      voff[q] = (uint32_t)(((int64_t)krow * ld + ct) * 2);
    }
    const int s = lane & 15, g = lane >> 5, half = (lane >> 4) & 1;
    frag_k = (uint32_t)((8 * g + (s >> 2)) * 512);
    const int f = (s >> 2) | (g << 2);
    const int seg0 = sub_col0 / 32;  // 128-column sub-tile: 0 or 4
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      frag_seg[j] = (uint32_t)((((seg0 + j) ^ f) * 64) + half * 32 + (s & 3) * 8);
    }
  }
  // Offset of K tile kt inside the resource, clamped to its end: whole K tiles past the last row read as zero.
  __device__ __forceinline__ uint32_t offset(const u32x4& rsrc, int kt) const {
    return stage_offset(rsrc[2], (uint32_t)kt, stage_bytes);
  }
  template <int q>
  __device__ __forceinline__ void issue(const u32x4& rsrc, uint32_t off, uint32_t lds_tile, int wave) const {
    dma16(lds_tile + (uint32_t)((wave * 4 + q) * 1024), voff[q], rsrc, off);
  }
  static constexpr int READS_PER_FRAG = 2;
  // half h (4 of the 8 k values) of fragment j of K step ks
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

// An accumulator element, read where it is used: left to the compiler, all 256 are copied to the vector
// registers at the head of the epilogue, which do not hold them beside the next tile's fragments.
__device__ __forceinline__ float acc_read(float a) {
  float v;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
  return v;
}

// One stretch of a workgroup's work: the reduction rows of one output tile, or of one segment of them (a
// buffer resource spans at most 2 GiB; an expert with more rows is walked in segments, the accumulators
// carried across).
struct Work {
  u32x4 ra, rb;  // the operands' rows, from the tile's first column on
  int kt_cnt;    // K tiles, at least MIN_KT (whole ones past the last row read as zero)
  int e, mt, nt; // e < 0: none left
  bool last;     // the tile's last stretch
};

// How a tile's result is stored (the rule is in launch_cfg): after its last K tile, with ordinary or with
// nontemporal stores, or nontemporally in four K tiles spread over the next tile.  A next tile of fewer than nine
// K tiles (an empty expert, or one of 256 rows and less) has no room for that: then at once.
enum { STORE_NOW, STORE_NOW_STREAM, STORE_SPREAD };
template <int DT, int ODT, int STORE>
__global__ __launch_bounds__(kGemmThreads) void gmm_dtl_kernel(GmmParams p) {
  typedef TransOperand OpA;
  typedef TransOperand OpB;
  typedef __attribute__((address_space(4))) const long long const_i64;
  constexpr int WT = 4;   // 32x32 accumulators per wavefront in each direction
  constexpr int NM = 16;  // MFMAs per K step
  constexpr int RA = OpA::READS_PER_FRAG, RB = OpB::READS_PER_FRAG;
  constexpr int NREAD = WT * RA + WT * RB;  // LDS reads per K step
  static_assert(ODT != GMOE_F32 || STORE == STORE_NOW, "32-bit results are stored from the accumulators");
  constexpr bool SPREAD = STORE == STORE_SPREAD;
  constexpr int STORES = 8;  // stores per wavefront and fragment row of a 16-bit result
  constexpr int MIN_KT = NST - 1;  // the copies reach one stretch ahead, never two
  constexpr int SPREAD_KT = 1 + 2 * WT;  // K tiles that the result of the tile before takes
  static_assert(NREAD == NM && LOADS_PER_TILE == NM / 2, "one read per MFMA, a copy after every fourth");

  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const uint32_t lds0 = lds_offset_of(lds);

  const int E = p.E;
  const int64_t K = p.K, M = p.M;
  const int nt_cnt = (int)((M + BN - 1) / BN);
  const int mt_cnt = (int)((K + BM - 1) / BM);

  // every expert has the same mt_cnt x nt_cnt grid of output tiles (32-bit: the output they tile is memory)
  const int per_expert = mt_cnt * nt_cnt;
  const int total_tiles = per_expert * E;
  // workgroup w runs on XCD w % 8: XCD x takes the positions [x*G/8, (x+1)*G/8) of every whole round
  // of G = gridDim.x tiles; the last, partial round is dealt to the XCDs in equal consecutive shares
  const int G = gridDim.x;
  const int xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
  const int whole = total_tiles / G * G;  // tiles in whole rounds
  auto tail_tile = [&]() -> int {
    const int share = (total_tiles - whole + 7) / 8;
    const int t = whole + xcd * share + slot;
    return (slot < share && t < total_tiles) ? t : -1;
  };
  const int first = xcd * (G / 8) + slot;
  const int64_t seg_rows = tn_segment_rows(K, M, 2);

  OpA oa;
  OpB ob;
  oa.init(K, wave, lane, wm * 128);
  ob.init(M, wave, lane, wn * 128);

  int s = first < whole ? first : tail_tile();  // the tile and segment `fetch` takes next
  int64_t seg0 = 0;
  auto fetch = [&](Work& w) {
    if (s < 0) {
      w.ra = w.rb = make_raw_rsrc(p.a, 0);
      w.e = -1;
      w.kt_cnt = 0;
      return;
    }
    const int e = s / per_expert;
    // scalar loads: a vector load's wait would drain the copies in flight
    const_i64* off = (const_i64*)(p.offsets);
    const long long row0 = off ? off[e] : 0, n_e = (off ? off[e + 1] : (long long)p.N) - row0;
    const int q = s - e * per_expert, strip = q / (mt_cnt * kStripTiles), rem = q - strip * mt_cnt * kStripTiles;
    const int n0 = strip * kStripTiles, width = nt_cnt - n0 < kStripTiles ? nt_cnt - n0 : kStripTiles;
    w.e = e;
    w.mt = rem / width;
    w.nt = n0 + rem % width;
    const int64_t left = n_e - seg0, k_lim = left < seg_rows ? left : seg_rows;
    w.ra = make_raw_rsrc(p.a + ((row0 + seg0) * K + (int64_t)w.mt * BM) * 2, (k_lim * K - (int64_t)w.mt * BM) * 2);
    w.rb = make_raw_rsrc(p.b + ((row0 + seg0) * M + (int64_t)w.nt * BN) * 2, (k_lim * M - (int64_t)w.nt * BN) * 2);
    const int kt = (int)((k_lim + BKT - 1) / BKT);
    w.kt_cnt = kt < MIN_KT ? MIN_KT : kt;
    w.last = left <= seg_rows;
    if (w.last) {
      s = s >= whole ? -1 : (s + G < whole ? s + G : tail_tile());
      seg0 = 0;
    } else {
      seg0 += seg_rows;
    }
  };

  f32x16 acc[WT][WT];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
      for (int j = 0; j < WT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  };
  u32x4 fa[2][WT], fb[2][WT];
  // read operation r of K step ks of the tile at `stage` into fragment buffer `buf`
  auto frag_read = [&](auto r_c, auto ks_c, auto buf_c, const unsigned char* stage) {
    constexpr int r = decltype(r_c)::value, ks = decltype(ks_c)::value, buf = decltype(buf_c)::value;
    if constexpr (r < WT * RA) {
      oa.template read<r / RA, ks, r % RA>(stage, fa[buf][r / RA]);
    } else {
      constexpr int rb = r - WT * RA;
      ob.template read<rb / RB, ks, rb % RB>(stage + OPER_BYTES, fb[buf][rb / RB]);
    }
  };

  if (p.warm) warm_operands(p);
  Work cur;
  fetch(cur);
  if (cur.e < 0) return;
  // ---- prologue, once per workgroup: K tiles 0..2 in flight, wait for tile 0, fragments of its step 0
  static_for<0, NST - 1>([&](auto t_c) {
    constexpr int t = decltype(t_c)::value;
    const uint32_t st = lds0 + t * STAGE_BYTES, offa = oa.offset(cur.ra, t), offb = ob.offset(cur.rb, t);
    static_for<0, 4>([&](auto q) { oa.template issue<decltype(q)::value>(cur.ra, offa, st, wave); });
    static_for<0, 4>([&](auto q) { ob.template issue<decltype(q)::value>(cur.rb, offb, st + OPER_BYTES, wave); });
  });
  wait_dma_outstanding<2 * LOADS_PER_TILE>();
  __syncthreads();
  static_for<0, NREAD>([&](auto r) {
    frag_read(r, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, lds);
  });

  // ---- the result of a tile: lane holds row (lane%32), columns 8*(v/4) + 4*(lane/32) + v%4 of each 32x32 ----
  // 16-bit results are rounded into `pk` (half the registers) and go to memory 32 rows x 128 columns at a time,
  // through 8 KiB of LDS of the wavefront's own: the 16-byte piece c of row r sits in slot c ^ (r & 15).  The
  // buffer stores carry no condition (rows and columns that do not exist are out of the resource), so each
  // fragment row leaves STORES of them in flight.
  constexpr int OES = Elem<ODT>::bytes;
  u32x2 pk[WT][WT][4];
  u32x4 sv[4];  // pieces on their way from LDS to memory
  const uint32_t mine = lds0 + NST * STAGE_BYTES + wave * 8192;
  // a lane's 8 bytes of slot 0 of its fragment row; its 16 bytes of rows 0..3
  uint32_t put = mine + (lane & 31) * 256 + (lane & 15) * 16 + 8 * (lane >> 5);
  uint32_t get = mine + (lane >> 4) * 256 + ((lane & 15) ^ (lane >> 4)) * 16;
  __amdgpu_buffer_rsrc_t rc;
  uint32_t vo = 0;
  const uint32_t four_rows = (uint32_t)(4 * M * OES);
  auto take = [&](auto i_c, auto j_c) {  // accumulator (i, j) -> pk
    constexpr int i = decltype(i_c)::value, j = decltype(j_c)::value;
#pragma unroll
    for (int vq = 0; vq < 4; ++vq) {
      pk[i][j][vq] = pack4<ODT>(acc_read(acc[i][j][4 * vq]), acc_read(acc[i][j][4 * vq + 1]),
                                acc_read(acc[i][j][4 * vq + 2]), acc_read(acc[i][j][4 * vq + 3]));
      asm volatile("" : "+v"(pk[i][j][vq]));  // rounded here: sunk to its use, the fp32 values spill
    }
  };
  auto stage_put = [&](auto i_c, auto m_c) {  // 4 columns of every row of fragment row i
    constexpr int i = decltype(i_c)::value, m = decltype(m_c)::value;
    *lds_at<u32x2>(put ^ (m * 16)) = pk[i][m / 4][m % 4];
  };
  auto stage_get = [&](auto t_c) {  // rows 4t .. 4t+3, 256 bytes each
    constexpr int t = decltype(t_c)::value;
    sv[t % 4] = *lds_at<const u32x4>((get ^ (t % 4 * 64)) + t * 1024);
  };
  auto stage_store = [&](auto t_c) {
    __builtin_amdgcn_raw_buffer_store_b128(sv[decltype(t_c)::value % 4], rc, (int)vo, 0,
                                           STORE == STORE_NOW ? 0 : kNontemporal);
    vo += four_rows;
  };
  auto locate = [&](const Work& w) {  // where the tile's result goes
    const int64_t c_rows = K - (int64_t)w.mt * BM, n = (int64_t)w.nt * BN + wn * 128 + (lane & 15) * 8;
    rc = __builtin_amdgcn_make_buffer_rsrc(p.c + ((int64_t)w.e * K + (int64_t)w.mt * BM) * M * OES, 0,
                                           (int)((c_rows < BM ? c_rows : BM) * M * OES), 0x00020000);
    vo = n < M ? (uint32_t)(((wm * 128 + (lane >> 4)) * M + n) * OES) : kOob;
  };

  // The K tiles of all stretches form one sequence through the NST stages: the last three of a stretch
  // request the first three of the next, so that neither the first copies of a tile nor the stores of the
  // tile before are waited for with idle matrix cores.
  int g = 0;  // K tiles done, all stretches
  Work nx;
  // One K tile.  kind PLAIN: MFMAs, fragment reads, copies; TAKE: also the result of the tile before out of
  // the accumulators; 0..3: also fragment row `kind` of it to memory.  `stores`: how many may be in flight
  // behind the copies of tile kt+1.
  constexpr int PLAIN = -1, TAKE = -2;
  auto k_tile = [&](auto kind_c, auto stores_c, int kt) __attribute__((always_inline)) {
    constexpr int kind = decltype(kind_c)::value;
    const unsigned char* here = lds + (g & (NST - 1)) * STAGE_BYTES;
    const unsigned char* nxt = lds + ((g + 1) & (NST - 1)) * STAGE_BYTES;
    const uint32_t st3 = lds0 + (uint32_t)(((g + 3) & (NST - 1)) * STAGE_BYTES);
    const bool own = kt + 3 < cur.kt_cnt;
    const int kt3 = own ? kt + 3 : kt + 3 - cur.kt_cnt;
    const u32x4 ra = own ? cur.ra : nx.ra, rb = own ? cur.rb : nx.rb;
    const uint32_t offa = oa.offset(ra, kt3), offb = ob.offset(rb, kt3);
    if constexpr (kind >= 0) asm volatile("" : "+v"(put), "+v"(get));  // the addresses made of them are not kept
    // ---- K step 0: MFMAs on buffer 0; read step 1 into buffer 1; request a of tile kt+3 ---
    // One fragment read per MFMA and a copy after every fourth: the stage of tile kt-1 is free for
    // both steps, and copies spread over both are 1-2 % faster than all eight at the end of this
    // one (dW of fc1 on the Mixtral shape 6.20 -> 6.14 ms, 1.09 -> 1.06 ms for 8192 x 2048 x 11264).
    static_for<0, NM>([&](auto m_c) {
      constexpr int m = decltype(m_c)::value;
      // boustrophedon order over the fragments: one operand changes per MFMA
      constexpr int mi = m / WT, mj = (mi & 1) ? WT - 1 - m % WT : m % WT;
      if constexpr (kind == TAKE) {
        // written 16 MFMAs ago, so complete
        take(std::integral_constant<int, mi>{}, std::integral_constant<int, mj>{});
        GMOE_SCHED_FENCE();
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[mi][mj][v] = 0.f;
      }
      Mma<DT>::run(fa[0][mi], fb[0][mj], acc[mi][mj]);
      GMOE_SCHED_FENCE();
      frag_read(m_c, std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{}, here);
      if constexpr (kind >= 0) stage_put(kind_c, m_c);
      if constexpr (m % 4 == 2) oa.template issue<m / 4>(ra, offa, st3, wave);
      GMOE_SCHED_FENCE();
    });
    // tile kt+1 must have landed (kt+2, the half of kt+3 and stores issued since may still be in flight);
    // the barrier also tells everyone that this tile's stage has been read for the last time
    wait_dma_outstanding<LOADS_PER_TILE + 4 + decltype(stores_c)::value>();
    __syncthreads();
    GMOE_SCHED_FENCE();
    // ---- K step 1: MFMAs on buffer 1; read step 0 of tile kt+1 into buffer 0; request b of kt+3
    static_for<0, NM>([&](auto m_c) {
      constexpr int m = decltype(m_c)::value;
      constexpr int mi = m / WT, mj = (mi & 1) ? WT - 1 - m % WT : m % WT;
      Mma<DT>::run(fa[1][mi], fb[1][mj], acc[mi][mj]);
      GMOE_SCHED_FENCE();
      if constexpr (kind >= 0) {
        if constexpr (m >= 4 && m < 12) stage_store(std::integral_constant<int, m - 4>{});
        if constexpr (m < 8) stage_get(m_c);
      }
      frag_read(m_c, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, nxt);
      if constexpr (m % 4 == 2) ob.template issue<m / 4>(rb, offb, st3 + OPER_BYTES, wave);
      GMOE_SCHED_FENCE();
    });
    ++g;
  };
  constexpr std::integral_constant<int, PLAIN> plain{};
  constexpr std::integral_constant<int, 0> none{};
  constexpr std::integral_constant<int, STORES> some{};
  constexpr std::integral_constant<int, WT * STORES> all{};
  // fragment row i at once, with no MFMAs beside it
  auto store_row = [&](auto i_c) {
    GMOE_SCHED_FENCE();
    static_for<0, WT>([&](auto j_c) { take(i_c, j_c); });
    static_for<0, 16>([&](auto m_c) { stage_put(i_c, m_c); });
    static_for<0, 2>([&](auto h_c) {
      constexpr int h = decltype(h_c)::value;
      static_for<4 * h, 4 * h + 4>(stage_get);
      static_for<4 * h, 4 * h + 4>(stage_store);
    });
    GMOE_SCHED_FENCE();
  };

  // The K tiles of `cur` from kt on, its further stretches included.
  auto finish = [&](int kt) __attribute__((always_inline)) {
    for (;;) {
      for (; kt < cur.kt_cnt; ++kt) k_tile(plain, none, kt);
      if (cur.last) break;
      cur = nx;
      fetch(nx);
      kt = 0;
    }
  };

  bool stored = false;  // the stores of a tile before are in flight
  for (;;) {
    fetch(nx);
    int kt = 0;
    clear();
    // the copies of the first two tiles were requested before the stores
    if (ODT != GMOE_F32 && stored)
      for (; kt < 2; ++kt) k_tile(plain, all, kt);
    finish(kt);
    // a loop of its own: the accumulators must not meet those of another path, of which there is no copy
    while (SPREAD && nx.kt_cnt >= SPREAD_KT) {
      locate(cur);
      cur = nx;
      fetch(nx);
      kt = 0;
      const int stride = (cur.kt_cnt - 1) / WT;
      k_tile(std::integral_constant<int, TAKE>{}, none, kt++);
      static_for<0, WT>([&](auto i_c) __attribute__((always_inline)) {
        k_tile(i_c, none, kt++);
        k_tile(plain, some, kt++);
        if constexpr (decltype(i_c)::value + 1 < WT)
          for (int r = 2; r < stride; ++r) k_tile(plain, none, kt++);
      });
      finish(kt);
    }
    if constexpr (ODT != GMOE_F32) {
      locate(cur);
      asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last MFMA's result, read by acc_read
      asm volatile("" : "+v"(put), "+v"(get));
      static_for<0, WT>(store_row);
      stored = true;
    } else {
      unsigned char* c_tile = p.c + ((int64_t)cur.e * K + (int64_t)cur.mt * BM) * M * OES;
      const int64_t c_rows = K - (int64_t)cur.mt * BM;
#pragma unroll
      for (int i = 0; i < WT; ++i) {
        const int64_t m = wm * 128 + i * 32 + (lane & 31);
        if (m >= c_rows) continue;
#pragma unroll
        for (int j = 0; j < WT; ++j)
#pragma unroll
          for (int vq = 0; vq < 4; ++vq) {
            const int64_t n = (int64_t)cur.nt * BN + wn * 128 + j * 32 + 8 * vq + 4 * (lane >> 5);
            if (n < M)
              *reinterpret_cast<f32x4*>(c_tile + (m * M + n) * OES) =
                  f32x4{acc[i][j][4 * vq], acc[i][j][4 * vq + 1], acc[i][j][4 * vq + 2], acc[i][j][4 * vq + 3]};
          }
      }
      wait_dma_outstanding<0>();  // an unknown number of stores: the counted waits start anew
    }
    if (nx.e < 0) break;
    cur = nx;
  }
  wait_dma_outstanding<0>();  // nothing may land in LDS after the workgroup has ended
}

template <int DT, int ODT, int STORE>
static int launch_kernel(const GmmParams& p, hipStream_t st) {
  constexpr size_t smem = (size_t)NST * STAGE_BYTES + (ODT == GMOE_F32 ? 0 : 4 * 8192)  /* a wavefront's staging */;
  auto kern = gmm_dtl_kernel<DT, ODT, STORE>;
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

// n = rows per expert, us, operands from HBM and a result buffer of its own for every launch (into one buffer, the
// part of it that the memory-side cache still holds favours ordinary stores):
//   * stores after the tile / spread over the next one: n 1024 811 / 789 (14336 x 4096, 8 experts), 1621 / 1581
//     (7168 x 4096, 32), 662 / 653 (2048 x 2816, 64), 185 / 175 (1024 x 5632, 16); n 900 326 / 308 (1408 x 2048,
//     64).  At n 640 as often behind as ahead (457 / 465, 252 / 245, 124 / 126).  A store covers four rows, and
//     where those lie 14 KB and more apart, the copies wait behind the spread ones until a tile is long: n 1024
//     1596 / 1656, n 1408 2100 / 2112, n 1600 2352 / 2339 (4096 x 28672, 8); n 1024 1347 / 1380, n 1408 1773 / 1770
//     (6144 x 16384, 8); n 1024 820 / 827, n 1408 1072 / 1067 (2048 x 7168, 32).
//     In whole steps with fc1's result stored after the tile / spread, fc2's spread: 8 experts of 8192, hidden
//     4096, n 1100 5184 / 5274; of 14336, n 1024 8264 / 8295, n 1300 9843 / 9841.
//   * ordinary / nontemporal stores after the tile: n 256 742 / 634, n 448 897 / 851 (4096 x 28672, 8), n 256 264 /
//     246, n 512 387 / 394 (2048 x 2816, 64), n 256 99 / 84 (4096 x 4096, 8, 256 MB); smaller results either way: n
//     256 74 / 71 (1024 x 5632, 16), 53 / 57 (1024 x 1024, 64), n 1152 100 / 112 (2816 x 1024, 16).
constexpr int64_t kSpreadRows = 900, kSpreadRowsWide = 1408, kSpreadWide = 7168;

template <int DT, int ODT>
static int launch_cfg(const GmmParams& p, hipStream_t st) {
  if constexpr (ODT == GMOE_F32) {
    return launch_kernel<DT, ODT, STORE_NOW>(p, st);
  } else {
    if (p.N / (p.E > 0 ? p.E : 1) >= (p.M >= kSpreadWide ? kSpreadRowsWide : kSpreadRows))
      return launch_kernel<DT, ODT, STORE_SPREAD>(p, st);
    if (gmm_tn_streams(p)) return launch_kernel<DT, ODT, STORE_NOW_STREAM>(p, st);
    return launch_kernel<DT, ODT, STORE_NOW>(p, st);
  }
}

}  // namespace dtl

int launch_gmm_dtl_tn(const GmmParams& p, int dtype, int out_dtype, hipStream_t st) {
  if (dtype == GMOE_BF16 && out_dtype == GMOE_BF16) return dtl::launch_cfg<GMOE_BF16, GMOE_BF16>(p, st);
  if (dtype == GMOE_BF16 && out_dtype == GMOE_F32) return dtl::launch_cfg<GMOE_BF16, GMOE_F32>(p, st);
  if (dtype == GMOE_F16 && out_dtype == GMOE_F16) return dtl::launch_cfg<GMOE_F16, GMOE_F16>(p, st);
  if (dtype == GMOE_F16 && out_dtype == GMOE_F32) return dtl::launch_cfg<GMOE_F16, GMOE_F32>(p, st);
  return GMOE_ERR_UNSUPPORTED;
}

}  // namespace gmoe
