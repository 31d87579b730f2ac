// Which kernel a batched Q8_0 GEMM (fkv_gemm.hip) runs, and its grids. Plain integer
// functions of the sizes, for the host.
#pragma once
#include <cstdint>

namespace fkv {

// HIP refuses a launch of more threads than this along a grid's x.
constexpr uint64_t kMaxGridThreads = 0xffffffffull;

// The activation quantizer: 8 values a thread, of whole 16-token tiles.
constexpr uint32_t kGemmActThreads = 64;
constexpr uint64_t gemm_act_threads(uint32_t cols, uint32_t n_tokens) {
  const uint64_t items = ((uint64_t)n_tokens + 15u) / 16u * 16u * (cols / 8u);
  return (items + kGemmActThreads - 1u) / kGemmActThreads * kGemmActThreads;
}

// The 64 x 64 kernel: row tiles are dealt to the 8 XCDs in turn, so whole eights of them.
constexpr uint32_t kGemmTileRows = 64;
constexpr uint32_t kGemmTileThreads = 256;
constexpr uint64_t gemm_tile_wgs(uint64_t row_tiles, uint32_t n_tokens) {
  return (row_tiles + 7u) / 8u * 8u * (((uint64_t)n_tokens + 63u) / 64u);
}

// A workgroup of the 64 x 64 kernel takes about as long alone on its CU as with two others
// (4,096 columns: 25 us at one a CU, 34 us at three), so it wins once every CU has one:
// at 256 workgroups and 4,096 x 4,096 weights 28.1 us against 30.5 for 16 x 16 tiles (256
// tokens), at 192 27.0 against 24.3 (192 tokens); 2,048 and 14,336 columns turn at the same
// count (17.4 / 19.4 and 77.5 / 85.7 us at 256). And the tokens have to use more than half
// of its 64: 28,672 rows, 32 tokens 48.5 us against 47.2, 64 tokens 50 against 69. Launches
// past one grid's threads (134 million tokens of a few rows) run the other kernel, whose
// token tiles are the grid's y.
constexpr uint64_t kTileMinWgs = 256;
constexpr uint32_t kTileMinTokens = 33;
constexpr bool gemm_tile_fills(uint64_t row_tiles, uint32_t n_tokens) {
  return n_tokens >= kTileMinTokens &&
         row_tiles * (((uint64_t)n_tokens + 63u) / 64u) >= kTileMinWgs &&
         gemm_tile_wgs(row_tiles, n_tokens) * kGemmTileThreads <= kMaxGridThreads;
}

}  // namespace fkv
