// Where the batched Q8_0 GEMM's kernels (fkv_gemm.hip) read: byte offsets of their buffer
// loads from the resource's base. Plain integer functions, for the host too.
//
// Both kernels load a few steps ahead of the sums, so past the end of a row. Every step is
// bounded here by the last pair of blocks (the last block pair of the activation), which is
// then read once more and never used: each load stays inside its matrix or workspace by
// itself, and nothing is left to the buffer's range check, which counts the lane offset but
// is not documented alike for the scalar offset that these loads grow by.
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define FKV_AT __host__ __device__ __forceinline__ constexpr
#else
#define FKV_AT constexpr
#endif

namespace fkv {
namespace gemm_at {

constexpr uint32_t kPairBytes = 68;  // two Q8_0 blocks of 34 bytes

FKV_AT uint32_t lower(uint32_t a, uint32_t b) { return a < b ? a : b; }

// Weights: a pair of blocks of a row is 17 dwords; units of 16 bytes from dwords 0, 4, 9
// and 13, and dword 8 by itself.
FKV_AT uint32_t weight_unit(uint32_t unit) { return unit * 16u + (unit >= 2u ? 4u : 0u); }
constexpr uint32_t kWeightDword8 = 32;
FKV_AT uint32_t last_pair(uint32_t np) { return (np - 1u) * kPairBytes; }
// pair p of a row of np, bounded; as a scalar, and for a lane's own pair
FKV_AT uint32_t pair(uint32_t p, uint32_t np) { return lower(p * kPairBytes, last_pair(np)); }
// row r of a tile whose last row that the matrix has is last_row
FKV_AT uint32_t row(uint32_t r, uint32_t last_row, uint32_t row_bytes) {
  return lower(r, last_row) * row_bytes;
}

// gemm_q8_tile_kernel: chunks of 4 blocks. Lanes:
FKV_AT uint32_t tile_weights(uint32_t wave, uint32_t lane, uint32_t last_row, uint32_t row_bytes) {
  return row(16u * wave + lane / 4u, last_row, row_bytes) + weight_unit((lane & 3u) ^ (lane >> 4));
}
FKV_AT uint32_t tile_dwords8(uint32_t lane, uint32_t last_row, uint32_t row_bytes) {
  return row(lane, last_row, row_bytes) + kWeightDword8;
}
// the 16-token tile of a lane's token, of those from the workgroup's first on (at most 4)
FKV_AT uint32_t tile_of(uint32_t wave, uint32_t lane, uint32_t last_tile) {
  return lower(2u * (wave & 1u) + (lane & 31u) / 16u, last_tile);
}
FKV_AT uint32_t tile_quants(uint32_t wave, uint32_t lane, uint32_t last_tile, uint32_t nb) {
  return tile_of(wave, lane, last_tile) * nb * 512u + (lane >> 5) * 256u + (lane & 15u) * 16u;
}
FKV_AT uint32_t tile_scales(uint32_t wave, uint32_t lane, uint32_t last_tile, uint32_t nb) {
  return tile_of(wave, lane, last_tile) * nb * 64u + (lane >> 5) * 64u + (lane & 15u) * 4u;
}
// Scalars of chunk k: its first block of the wave's two (even), bounded; quants of block
// b + i at (b + i) * 512, the scales of both at b * 64.
FKV_AT uint32_t tile_block(uint32_t k, uint32_t wave, uint32_t nb) {
  return lower(4u * k + 2u * (wave >> 1), nb - 2u);
}

// gemm_q8_rows_kernel, the wave that stages weights: chunks of 4 pairs, 16 rows.
FKV_AT uint32_t rows_weights(uint32_t lane, uint32_t last_row, uint32_t row_bytes) {
  return row(lane / 4u, last_row, row_bytes) + weight_unit((lane & 3u) ^ (lane >> 4));
}
FKV_AT uint32_t rows_dwords8(uint32_t lane, uint32_t last_row, uint32_t row_bytes) {
  return row(lane & 15u, last_row, row_bytes) + kWeightDword8;
}
// and the computing waves: group g of 4 blocks of one 16-token tile. Pair p's quants:
FKV_AT uint32_t rows_quants(uint32_t p, uint32_t np) { return lower(p, np - 1u) * 1024u; }
// The scales of 4 blocks, a lane's block 4g + lane / 16: whole groups by a scalar, or, where
// the last group is not whole, each lane by itself.
FKV_AT uint32_t rows_scales(uint32_t g, uint32_t nb) { return lower(g, nb / 4u - 1u) * 256u; }
FKV_AT uint32_t rows_scales_lane(uint32_t g, uint32_t lane, uint32_t nb) {
  return lower(g * 256u + lane * 4u, (nb - 1u) * 64u + (lane & 15u) * 4u);
}

}  // namespace gemm_at
}  // namespace fkv
