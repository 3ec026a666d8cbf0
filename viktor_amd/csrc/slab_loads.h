// Offsets of the large products' direct loads (gemm_big.hip): instruction i of wavefront wid brings rows
// 8 (wid + nwaves i) .. + 7 of an operand's row block, 16 bytes a lane, of the 64-wide K slab kt into LDS. Plain integer
// code, so that a host program can check every offset against a descriptor's range.
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define VK_SLAB_FN __host__ __device__ __forceinline__
#else
#define VK_SLAB_FN inline
#endif

namespace vk {

constexpr int SLAB_ROWS = 8;          // rows per instruction
constexpr uint32_t SLAB_BYTES = 128;  // bytes of a row per slab

// Bytes of a descriptor over `rows` whole rows of K bf16.
VK_SLAB_FN uint32_t slab_bytes(uint32_t rows, uint32_t K) { return rows * K * 2; }

// The vector offset: the lane's row and its chunk of the slab (the one that belongs into its LDS slot, lane % 8). The row
// stands here and only the slab in the scalar offset: whether the range check counts the scalar offset or not, a
// row inside the descriptor is then read, at every slab, and a row past its end reads as zero (its offset alone is past
// the end, and the scalar offset is below one row's bytes, so end minus scalar does not wrap). With the row block in the
// scalar offset a check that leaves it out would let whole blocks past the end through.
VK_SLAB_FN uint32_t slab_vector_offset(int wid, int nwaves, int i, int lane, uint32_t K) {
  const uint32_t r = SLAB_ROWS * static_cast<uint32_t>(wid + nwaves * i) + (static_cast<uint32_t>(lane) >> 3);
  return r * K * 2 + 16 * ((static_cast<uint32_t>(lane) & 7) ^ ((r >> 1) & 7));
}
VK_SLAB_FN uint32_t slab_scalar_offset(int kt) { return static_cast<uint32_t>(kt) * SLAB_BYTES; }

}  // namespace vk
