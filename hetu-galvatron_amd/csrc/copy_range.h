// Where the LDS-DMA copies of a K tile begin inside their buffer resource.  The copies run a few tiles ahead, so
// past an operand's last row too.  The bounds check compares a lane's offset with what num_records leaves after
// the scalar offset; that this difference may be negative is nowhere promised.  At num_records itself, every lane
// is out of range, reads zero and touches no memory.
#pragma once
#include <cstdint>

namespace gmoe {

// kt: K tile, stage_bytes: global bytes between consecutive ones, bytes: of the resource.  A K tile is at most
// 256 MiB (256 rows of an operand stay below 2 GiB), a resource at most 2 GiB, and the copies run up to seven tiles
// past it, so the product fits 32 bits.
__host__ __device__ constexpr uint32_t stage_offset(uint32_t bytes, uint32_t kt, uint32_t stage_bytes) {
  const uint32_t o = kt * stage_bytes;
  return o < bytes ? o : bytes;
}

}  // namespace gmoe
