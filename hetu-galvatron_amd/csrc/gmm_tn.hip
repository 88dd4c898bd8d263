// Grouped weight-gradient product (TN) of 16-bit operands for short reductions on gfx950:
//   c[e] = a[rows_e]^T @ b[rows_e],  a [N,K], b [N,M], c [E,K,M]: the contract of gmm_dtl.hip.
//
// For outputs of less than a round of 256x256 tiles, whose CUs then have nothing to hide a tile's prologue
// and epilogue under, and for a few dozen rows per expert, where a launch is all prologue and epilogue.  Here a tile
// is 128x256 and two workgroups share a CU (72 KiB of LDS, at most 256 registers each): one multiplies while the
// other copies its first stages or writes its result.
// Results are stored nontemporally, whatever their size (us with ordinary stores / so: 7 MB of them 9.5 / 8.7, 31 MB
// 15.4 / 13.7, 64 MB 22.4 / 22.0, 192 MB 73 / 71, 350 MB 117 / 99).  A launch that reads a result of 30 to 250 MB
// next loses as much as is gained here (with a pass over it: 51 MB 36 / 38, 128 MB 82 / 85), beyond that it gains
// too (552 MB 375 / 330); weight gradients are not read before the backward has ended. The price is half again as
// much operand traffic per product, so long reductions and large outputs stay with gmm_dtl.hip (the rule with both
// sides' times is gmm_tn_short_pays in gmm.hip).
#include "gmm_common.h"

namespace gmoe {

namespace tn {

constexpr int BM = 128, BN = 256;
constexpr int BKT = 32;  // reduction elements per stage
constexpr int NST = 3;   // LDS stages
constexpr int A_BYTES = BM * BKT * 2;
constexpr int B_BYTES = BN * BKT * 2;
constexpr int STAGE_BYTES = A_BYTES + B_BYTES;

typedef short s16x4 __attribute__((ext_vector_type(4)));

// Operand with the outer index contiguous, 128 wide: LDS tile [32 k][128 outer], 256 bytes per k row,
// the 64-byte segment sg of row k in place sg ^ (k & 3); fragments by transposing reads.
struct Outer128 {
  u32x4 rsrc;
  uint32_t voff[2];
  uint32_t stage_bytes;  // global bytes between consecutive K tiles
  uint32_t frag[4];
  __device__ __forceinline__ void init(const unsigned char* src, int64_t ld, int64_t o0, int64_t k_limit,
                                       int wave, int lane) {
    rsrc = make_raw_rsrc(src + o0 * 2, k_limit * ld * 2 - o0 * 2);
    stage_bytes = (uint32_t)(ld * 2 * BKT);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int krow = (wave * 2 + q) * 4 + (lane >> 4);
      const int P = lane & 15;
      const int ct = ((((P >> 2) ^ (krow & 3)) << 2) + (P & 3)) * 8;
      voff[q] = (uint32_t)(((int64_t)krow * ld + ct) * 2);
    }
    const int s = lane & 15, g = lane >> 5, half = (lane >> 4) & 1;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      frag[j] = (uint32_t)((8 * g + (s >> 2)) * 256 + ((j ^ (s >> 2)) * 64) + half * 32 + (s & 3) * 8);
  }
  __device__ __forceinline__ uint32_t offset(int kt) const { return stage_offset(rsrc[2], (uint32_t)kt, stage_bytes); }
  template <int q>
  __device__ __forceinline__ void issue(uint32_t off, uint32_t lds_tile, int wave) const {
    dma16(lds_tile + (uint32_t)((wave * 2 + q) * 1024), voff[q], rsrc, off);
  }
  static constexpr int READS = 2;
  template <int j, int ks, int h>
  __device__ __forceinline__ void read(const unsigned char* tile, u32x4& f) const {
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4*)(lds_byte*)(tile + frag[j] + (ks * 16 + h * 4) * 256));
    const u32x2 w = __builtin_bit_cast(u32x2, v);
    f[2 * h] = w[0];
    f[2 * h + 1] = w[1];
  }
};

// Operand with the outer index contiguous: LDS tile [32 k][256 outer], 512 bytes per k row, segment
// swizzle as in gmm_dtl.hip; a wavefront owns the 64 columns from 64 * wave.
struct Outer256 {
  u32x4 rsrc;
  uint32_t voff[4];
  uint32_t stage_bytes;  // global bytes between consecutive K tiles
  uint32_t frag_k;
  uint32_t frag_seg[2];

  __device__ __forceinline__ void init(const unsigned char* src, int64_t ld, int64_t o0, int64_t k_limit,
                                       int wave, int lane) {
    rsrc = make_raw_rsrc(src + o0 * 2, k_limit * ld * 2 - o0 * 2);
    stage_bytes = (uint32_t)(ld * 2 * BKT);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int krow = (wave * 4 + q) * 2 + (lane >> 5);
      const int f = (krow & 3) | ((krow >> 1) & 4);
      const int P = lane & 31;
      const int ct = ((((P >> 2) ^ f) << 2) + (P & 3)) * 8;
      voff[q] = (uint32_t)(((int64_t)krow * ld + ct) * 2);
    }
    const int s = lane & 15, g = lane >> 5, half = (lane >> 4) & 1;
    frag_k = (uint32_t)((8 * g + (s >> 2)) * 512);
    const int f = (s >> 2) | (g << 2);
    frag_seg[0] = (uint32_t)((((2 * wave) ^ f) * 64) + half * 32 + (s & 3) * 8);
    frag_seg[1] = (uint32_t)((((2 * wave + 1) ^ f) * 64) + half * 32 + (s & 3) * 8);
  }
  __device__ __forceinline__ uint32_t offset(int kt) const { return stage_offset(rsrc[2], (uint32_t)kt, stage_bytes); }
  template <int q>
  __device__ __forceinline__ void issue(uint32_t off, uint32_t lds_tile, int wave) const {
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

template <int DT, int ODT>
__global__ __launch_bounds__(kGemmThreads, 2) void gmm_tn_kernel(GmmParams p) {
  constexpr int WM = 4, WN = 2, NM = WM * WN;
  constexpr int NLOAD = 6;             // copy instructions per wavefront and stage: 2 for a, 4 for b
  constexpr int NREAD = 2 * WM + 2 * WN;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lds0 = lds_offset_of(lds);
  const int64_t K = p.K, M = p.M;
  const int nt_cnt = (int)((M + BN - 1) / BN), mt_cnt = (int)((K + BM - 1) / BM);
  const long long per_expert = (long long)mt_cnt * nt_cnt, total = per_expert * p.E;
  // XCD x takes the positions [x*G/8, (x+1)*G/8) of every whole round of G tiles; the last, partial
  // round is dealt to the XCDs in equal consecutive shares
  const int G = gridDim.x, per_xcd = G / 8;
  const int xcd = blockIdx.x % 8, slot = blockIdx.x / 8;

  if (p.warm) warm_operands(p);
  for (long long base = 0; base < total; base += G) {
    long long v = base + (long long)xcd * per_xcd + slot;
    if (total - base < G) {
      const long long share = (total - base + 7) / 8;
      v = base + xcd * share + slot;
      if (slot >= share || v >= total) break;
    }
    const int e = (int)(v / per_expert);
    const long long row0 = group_begin(p, e), n_e = group_begin(p, e + 1) - row0;
    int mt, nt;
    strip_order(v - e * per_expert, mt_cnt, nt_cnt, mt, nt);

    f32x16 acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.f;

    // a buffer resource spans at most 2 GiB: an expert with more rows is walked in segments
    const int64_t seg_rows = tn_segment_rows(K, M, 2);
    for (int64_t seg0 = 0; seg0 < n_e; seg0 += seg_rows) {
      const int64_t k_lim = n_e - seg0 < seg_rows ? n_e - seg0 : seg_rows;
      Outer128 oa;
      Outer256 ob;
      oa.init(p.a + (row0 + seg0) * K * 2, K, (int64_t)mt * BM, k_lim, wave, lane);
      ob.init(p.b + (row0 + seg0) * M * 2, M, (int64_t)nt * BN, k_lim, wave, lane);
      const int kt_cnt = (int)((k_lim + BKT - 1) / BKT);
      u32x4 fa[2][WM], fb[2][WN];
      auto issue = [&](auto op_c, uint32_t offa, uint32_t offb, uint32_t st) {
        constexpr int op = decltype(op_c)::value;
        if constexpr (op < 2) oa.template issue<op>(offa, st, wave);
        else ob.template issue<op - 2>(offb, st + A_BYTES, wave);
      };
      auto frag_read = [&](auto r_c, auto ks_c, auto buf_c, const unsigned char* stage) {
        constexpr int r = decltype(r_c)::value, ks = decltype(ks_c)::value, buf = decltype(buf_c)::value;
        if constexpr (r < 2 * WN) ob.template read<r / 2, ks, r % 2>(stage + A_BYTES, fb[buf][r / 2]);
        else oa.template read<(r - 2 * WN) / 2, ks, (r - 2 * WN) % 2>(stage, fa[buf][(r - 2 * WN) / 2]);
      };
      auto k_step = [&](auto ks_c, auto&& op_of, auto n_ops_c) {
        constexpr int ks = decltype(ks_c)::value, n_ops = decltype(n_ops_c)::value;
        static_for<0, NM>([&](auto m_c) {
          constexpr int m = decltype(m_c)::value;
          constexpr int mi = m / WN, mj = (mi & 1) ? 1 - m % WN : m % WN;
          Mma<DT>::run(fa[ks][mi], fb[ks][mj], acc[mi][mj]);
          GMOE_SCHED_FENCE();
          constexpr int op_begin = (m * n_ops + NM - 1) / NM, op_end = ((m + 1) * n_ops + NM - 1) / NM;
          static_for<op_begin, op_end>(op_of);
          GMOE_SCHED_FENCE();
        });
      };
      constexpr std::integral_constant<int, 0> c0{};
      constexpr std::integral_constant<int, 1> c1{};

      static_for<0, NLOAD>([&](auto q) { issue(q, 0u, 0u, lds0); });
      static_for<0, NLOAD>([&](auto q) { issue(q, oa.offset(1), ob.offset(1), lds0 + STAGE_BYTES); });
      wait_dma_outstanding<NLOAD>();
      __syncthreads();
      static_for<0, NREAD>([&](auto r) { frag_read(r, c0, c0, lds); });
      int s0 = 0;  // stage of tile kt
      for (int kt = 0; kt < kt_cnt; ++kt) {
        const int s1 = s0 == NST - 1 ? 0 : s0 + 1, s2 = s1 == NST - 1 ? 0 : s1 + 1;
        const unsigned char* cur = lds + s0 * STAGE_BYTES;
        const unsigned char* nxt = lds + s1 * STAGE_BYTES;
        const uint32_t st2 = lds0 + (uint32_t)(s2 * STAGE_BYTES);
        const uint32_t offa = oa.offset(kt + 2), offb = ob.offset(kt + 2);
        // step 0: read step 1's fragments, request tile kt+2 into the stage tile kt-1 has left
        k_step(c0, [&](auto op_c) {
          constexpr int op = decltype(op_c)::value;
          if constexpr (op < NREAD) frag_read(op_c, c1, c1, cur);
          else issue(std::integral_constant<int, op - NREAD>{}, offa, offb, st2);
        }, std::integral_constant<int, NREAD + NLOAD>{});
        // tile kt+1 has landed (kt+2 may be in flight) and every wavefront has read this stage
        wait_dma_outstanding<NLOAD>();
        __syncthreads();
        GMOE_SCHED_FENCE();
        k_step(c1, [&](auto op_c) { frag_read(op_c, c0, c0, nxt); }, std::integral_constant<int, NREAD>{});
        s0 = s1;
      }
      // every copy has landed and every wavefront is done with LDS before it is reused
      wait_dma_outstanding<0>();
      __syncthreads();
    }

    constexpr int OES = Elem<ODT>::bytes;
    unsigned char* c_base = p.c + ((int64_t)e * K + (int64_t)mt * BM) * M * OES;
    const int64_t c_rows = K - (int64_t)mt * BM;
    if constexpr (ODT != GMOE_F32) {
      using CT = CTile<BN>;
      stage_acc_lds<ODT, WM, WN, BN>(lds, acc, 0, wave * 64, lane);
      __syncthreads();
      const int cc = tid % CT::chunks, r0 = tid / CT::chunks;
      const int64_t n = (int64_t)nt * BN + cc * 8;
#pragma unroll 4
      for (int it = 0; it < BM / CT::rows_per_pass; ++it) {
        const int row = it * CT::rows_per_pass + r0;
        if (row < c_rows && n < M)
          st16_nt(c_base + ((int64_t)row * M + n) * OES, ctile_read16(lds + row * CT::pitch + cc * 16));
      }
      __syncthreads();  // the next tile's copies overwrite the staged values
    } else {
#pragma unroll
      for (int i = 0; i < WM; ++i) {
        const int64_t m = i * 32 + (lane & 31);
        if (m >= c_rows) continue;
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
          for (int vq = 0; vq < 4; ++vq) {
            const int64_t n = (int64_t)nt * BN + wave * 64 + j * 32 + 8 * vq + 4 * (lane >> 5);
            if (n < M)
              *reinterpret_cast<f32x4*>(c_base + (m * M + n) * OES) =
                  f32x4{acc[i][j][4 * vq], acc[i][j][4 * vq + 1], acc[i][j][4 * vq + 2], acc[i][j][4 * vq + 3]};
          }
      }
    }
  }
}

template <int DT, int ODT>
static int launch_cfg(const GmmParams& p, hipStream_t st) {
  constexpr size_t stages = (size_t)NST * STAGE_BYTES, ctile = (size_t)BM * CTile<BN>::pitch;
  constexpr size_t smem = stages > ctile ? stages : ctile;
  auto kern = gmm_tn_kernel<DT, ODT>;
  static std::atomic<uint64_t> done_mask{0};
  if (!gmoe_once_per_device(done_mask, [&] {
        return hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) == hipSuccess;
      }))
    return GMOE_ERR_LAUNCH;
  int grid = (gmoe_cu_count() / 8) * 8 * 2;
  if (grid < 8) grid = 8;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(kGemmThreads), smem, st, p);
  return gmoe_launch_status();
}

}  // namespace tn

int launch_gmm_tn_short(const GmmParams& p, int dtype, int out_dtype, hipStream_t st) {
  if (dtype == GMOE_BF16 && out_dtype == GMOE_BF16) return tn::launch_cfg<GMOE_BF16, GMOE_BF16>(p, st);
  if (dtype == GMOE_BF16 && out_dtype == GMOE_F32) return tn::launch_cfg<GMOE_BF16, GMOE_F32>(p, st);
  if (dtype == GMOE_F16 && out_dtype == GMOE_F16) return tn::launch_cfg<GMOE_F16, GMOE_F16>(p, st);
  if (dtype == GMOE_F16 && out_dtype == GMOE_F32) return tn::launch_cfg<GMOE_F16, GMOE_F32>(p, st);
  return GMOE_ERR_UNSUPPORTED;
}

}  // namespace gmoe
