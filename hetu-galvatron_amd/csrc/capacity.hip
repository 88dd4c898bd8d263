// Expert-capacity selection for gfx950: keep at most `capacity` tokens per expert
// (topk_softmax_with_capacity, moe/moe_utils.py:519-544).  The reference takes a top-`capacity`
// along the token axis of the dense gate matrix ("probs" policy) or of the 0/1 routing map
// ("position" policy) with torch.topk, whose order among equal values is unspecified; here the
// rule is fixed: among equal keys the lowest token index wins.
//
// One workgroup per expert column.  The capacity-th largest key is found by a radix selection, 8 bits a
// pass, with an LDS histogram: 4 passes for fp32, 2 for 16-bit gates (ordered by their own bits), 1 for
// the map.  Then every key above the threshold is kept and, in token order, the first `need` keys equal
// to it.
//
// Latency-bound: E workgroups, and the steps of a selection follow each other.  So every step is short:
//   * the keys of up to 16384 tokens stay in LDS (more are read again in every pass; in registers, with
//     every loop unrolled for it, they spilled and the code outgrew the instruction cache: 47 us where
//     this form takes 9.7);
//   * the bin that holds the threshold is found by one wavefront, four bins per lane and a scan;
//   * most gates are zero, and LDS atomics of one address take turns: a wavefront adds its first two
//     distinct digits as counts (two ballots), only the rest one by one;
//   * the ranks of equal keys come from one scan of all (block of tokens, wavefront) counts.
// 2048 tokens x 16 experts fp16 56 -> 9.7 us, fp32 56 -> 12.3, by the map 63 -> 8.1; 8192 x 64 bf16 90 -> 32;
// 16384 x 8 fp32 111 -> 48; 40000 x 8 bf16 187 -> 84.  Before, one thread walked the 256 bins and the keys
// were read in every pass.
#include "gmoe_common.h"

namespace gmoe {

constexpr int kCapThreads = 1024;
constexpr int kCapWaves = kCapThreads / 64;
constexpr int kCapKeys = 16;  // tokens per thread whose keys fit the LDS array
constexpr int kCapGroup = 4;  // tokens per thread loaded together
static_assert(kCapKeys * kCapWaves == 256, "the scans take 4 entries per lane of one wavefront");

// Order-preserving image of a value in unsigned integers: 32 bits of fp32, 16 of the 16-bit types.
template <int DT>
__device__ __forceinline__ uint32_t sort_key(const unsigned char* p, int64_t i) {
  if constexpr (DT == GMOE_F32) {
    const uint32_t b = reinterpret_cast<const uint32_t*>(p)[i];
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  } else {
    const uint32_t b = reinterpret_cast<const uint16_t*>(p)[i];
    return (b & 0x8000u) ? (~b & 0xffffu) : (b | 0x8000u);
  }
}

// Sum over the lanes below this one.
__device__ __forceinline__ unsigned int wave_exclusive_sum(unsigned int v, int lane) {
  unsigned int x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned int y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  return x - v;
}

template <int PDT>
__global__ __launch_bounds__(kCapThreads) void capacity_select_kernel(
    const unsigned char* probs, const uint8_t* routing_map, int64_t T, int E, int64_t capacity,
    int by_position, int pad, unsigned char* out_probs, uint8_t* out_map) {
  __shared__ unsigned int hist[256];  // the histogram, then the counts of equal keys [block][wavefront]
  __shared__ unsigned int sel[2];     // chosen byte, remaining count; then the number of equal keys
  const int e = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int64_t kSpan = (int64_t)kCapKeys * kCapThreads;
  const bool one_span = T <= kSpan;

  __shared__ uint32_t keys[kCapKeys * kCapThreads];  // read by the thread that wrote them
  auto blocks_at = [&](int64_t base) {  // blocks of kCapThreads tokens of the span at base
    const int64_t n = (T - base + kCapThreads - 1) / kCapThreads;
    return (int)(n < kCapKeys ? n : kCapKeys);
  };
  auto load_keys = [&](int64_t base) {
    const int n = blocks_at(base);
    for (int i = 0; i < n; i += kCapGroup) {
      uint32_t k[kCapGroup];
#pragma unroll
      for (int q = 0; q < kCapGroup; ++q) {
        const int64_t t = base + (i + q) * kCapThreads + tid;
        k[q] = 0u;
        if (t < T) k[q] = by_position ? (routing_map[t * E + e] ? 1u : 0u) : sort_key<PDT>(probs, t * E + e);
      }
#pragma unroll
      for (int q = 0; q < kCapGroup; ++q) keys[(i + q) * kCapThreads + tid] = k[q];
    }
  };
  if (one_span) load_keys(0);

  // ---- threshold: the capacity-th largest key -------------------------------------------------
  uint32_t prefix = 0, known = 0;
  unsigned int need = (unsigned int)capacity;  // 1 <= capacity <= T (checked by the host)
  for (int pass = by_position ? 0 : (PDT == GMOE_F32 ? 3 : 1); pass >= 0; --pass) {
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
    for (int64_t base = 0; base < T; base += kSpan) {
      if (!one_span) load_keys(base);
      const int n = blocks_at(base);
#pragma unroll 1
      for (int i = 0; i < n; ++i) {
        const uint32_t key = keys[i * kCapThreads + tid], digit = (key >> (8 * pass)) & 255u;
        bool open = base + i * kCapThreads + tid < T && (key & known) == prefix;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const uint64_t left = __ballot(open);
          if (left == 0) break;
          const int first = __builtin_ctzll(left);
          const uint32_t d = (uint32_t)__builtin_amdgcn_readlane((int)digit, first);
          const uint64_t same = __ballot(open && digit == d);
          if (lane == first) atomicAdd(&hist[d], (unsigned int)__popcll(same));
          open = open && digit != d;
        }
        if (open) atomicAdd(&hist[digit], 1u);
      }
    }
    __syncthreads();
    if (wave == 0) {
      // lane l: bins 255 - 4l down to 252 - 4l
      unsigned int h[4], sum = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) sum += h[q] = hist[255 - 4 * lane - q];
      unsigned int cum = wave_exclusive_sum(sum, lane);
      if (cum < need && cum + sum >= need) {  // one lane: the passes before left `need` keys or more
        int q = 0;
        while (q < 3 && cum + h[q] < need) cum += h[q++];
        sel[0] = (unsigned int)(255 - 4 * lane - q);
        sel[1] = need - cum;
      }
    }
    __syncthreads();
    prefix |= sel[0] << (8 * pass);
    known |= 0xffu << (8 * pass);
    need = sel[1];
  }
  const uint32_t thr = prefix;  // `need` keys equal to thr are kept, in token order

  // ---- selection in token order -----------------------------------------------------------------
  unsigned int eq_before = 0;
  for (int64_t base = 0; base < T; base += kSpan) {
    if (!one_span) load_keys(base);
    const int n = blocks_at(base);
#pragma unroll 1
    for (int i = 0; i < kCapKeys; ++i) {
      const uint64_t eq =
          __ballot(i < n && base + i * kCapThreads + tid < T && keys[i * kCapThreads + tid] == thr);
      if (lane == 0) hist[i * kCapWaves + wave] = (unsigned int)__popcll(eq);
    }
    __syncthreads();
    if (wave == 0) {
      unsigned int h[4], sum = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) sum += h[q] = hist[4 * lane + q];
      unsigned int cum = wave_exclusive_sum(sum, lane);
      if (lane == 63) sel[0] = cum + sum;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        hist[4 * lane + q] = cum;
        cum += h[q];
      }
    }
    __syncthreads();
#pragma unroll 1
    for (int i = 0; i < n; i += kCapGroup) {
      float p[kCapGroup];
      bool mapped[kCapGroup];
#pragma unroll
      for (int q = 0; q < kCapGroup; ++q) {
        const int64_t t = base + (i + q) * kCapThreads + tid;
        p[q] = t < T ? Elem<PDT>::load(probs, t * E + e) : 0.f;
        mapped[q] = pad || (t < T && routing_map[t * E + e] != 0);
      }
#pragma unroll
      for (int q = 0; q < kCapGroup; ++q) {
        const int64_t t = base + (i + q) * kCapThreads + tid;
        const uint32_t key = keys[(i + q) * kCapThreads + tid];
        const bool eq = t < T && key == thr;
        const uint64_t bal = __ballot(eq);
        const unsigned int rank = eq_before + hist[(i + q) * kCapWaves + wave] +
                                  (unsigned int)__popcll(bal & ((1ull << lane) - 1ull));
        const bool keep = (key > thr || (eq && rank < need)) && mapped[q];
        if (t < T) {
          out_map[t * E + e] = keep ? 1 : 0;
          Elem<PDT>::store(out_probs, t * E + e, keep ? p[q] : 0.f);
        }
      }
    }
    eq_before += sel[0];
    __syncthreads();  // before the next span writes hist and sel
  }
}

}  // namespace gmoe

extern "C" int gmoe_capacity_select(const void* probs, int probs_dtype, const uint8_t* routing_map,
                                    int64_t T, int E, int64_t capacity, int by_position, int pad,
                                    void* out_probs, uint8_t* out_map, void* stream) {
  using namespace gmoe;
  GMOE_CHECK_ARG(T >= 0 && E >= 1 && capacity >= 1);
  if (T == 0) return GMOE_OK;
  GMOE_CHECK_ARG(probs && routing_map && out_probs && out_map);
  if (capacity > T) capacity = T;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)E), block(kCapThreads);
  const unsigned char* pp = static_cast<const unsigned char*>(probs);
  unsigned char* op = static_cast<unsigned char*>(out_probs);
  switch (probs_dtype) {
    case GMOE_F32:
      hipLaunchKernelGGL((capacity_select_kernel<GMOE_F32>), grid, block, 0, st, pp, routing_map, T, E,
                         capacity, by_position, pad, op, out_map);
      break;
    case GMOE_BF16:
      hipLaunchKernelGGL((capacity_select_kernel<GMOE_BF16>), grid, block, 0, st, pp, routing_map, T, E,
                         capacity, by_position, pad, op, out_map);
      break;
    case GMOE_F16:
      hipLaunchKernelGGL((capacity_select_kernel<GMOE_F16>), grid, block, 0, st, pp, routing_map, T, E,
                         capacity, by_position, pad, op, out_map);
      break;
    default:
      return GMOE_ERR_UNSUPPORTED;
  }
  return gmoe_launch_status();
}
