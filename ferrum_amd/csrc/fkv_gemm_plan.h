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

// The 16 x 16 kernel: 16 rows a workgroup, up to 4 tiles of 16 tokens, one a wave, and one
// more wave that streams the weights.
constexpr uint32_t kGemmRowTile = 16;
// Token tiles a workgroup: as few workgroups as four allow, and no wave that has no tile but
// the last one's.
constexpr uint32_t gemm_row_wg_tiles(uint32_t n_tiles) {
  const uint32_t groups = (n_tiles + 3u) / 4u;
  return (n_tiles + groups - 1u) / groups;
}

// Which of the two. Chains: the ordered sums that the 16 x 16 kernel runs, 16 rows x 16
// tokens each, idle waves and blocks past the row's end with them; its time grows with them.
// A workgroup of the 64 x 64 kernel takes nearly as long alone on its CU as with another, so
// it wins where the launch fills the CUs. us with weights from HBM, 64 x 64 / 16 x 16:
// - up to 256 workgroups and over 64 tokens, past 3,072 chains, three a SIMD: 4,096 x 4,096
//   26.6 / 23.4 (192 tokens, 3,072), 26.9 / 28.6 (200, 4,096), 5,120 x 5,120 32.4 / 34.7 (160
//   tokens, 3,840), 14,336 columns 78.8 / 65.5 (192) and 78.4 / 83.6 (200);
// - up to 64 tokens, where the weights' stream bounds both, past 192 workgroups too: 12,288 x
//   4,096 28.7 / 25.8 (192, 33 tokens), 14,336 x 4,096 29.1 / 33.0 (224);
// - 257 to 512 workgroups, two a CU here and there, past 5,120 chains: 8,192 x 8,192 74.1 /
//   66.8 (129 tokens, 4,608), 75.2 / 74.9 (160, 6,144), 10,240 x 4,096 46.3 / 38.8 (128,
//   5,120), 41.6 / 45.6 (129, 5,760), 4,096 x 14,336 123.4 / 100.7 (320, 5,120), 124.5 /
//   128.1 (384, 6,144), 20,480 x 4,096 48.8 / 41 (33, 3,840), 50.0 / 44.3 (64, 5,120),
//   22,528 x 4,096 50.0 / 50.4 (64, 5,632);
// - 513 to 640, the third a CU, past 6,912: 17,408 x 4,096 57.5 / 48.5 (65 tokens, 6,528),
//   12,288 x 4,096 54.7 / 53.8 (129, 6,912), q/k/v 47.9 / 57.0 (384, 9,216); 64 x 64 beyond.
// And the tokens have to use more than half of its 64: 28,672 rows, 32 tokens 48.5 us
// against 47.2. Launches past one grid's threads (134 million tokens of a few rows) run the
// 16 x 16 kernel, whose token tiles are the grid's y.
constexpr uint64_t gemm_row_chains(uint64_t row_tiles, uint32_t cols, uint32_t n_tokens) {
  const uint32_t n_tiles = (uint32_t)(((uint64_t)n_tokens + 15u) / 16u);
  const uint32_t w = gemm_row_wg_tiles(n_tiles), nb = cols / 32u;
  const uint64_t chains = row_tiles * ((n_tiles + w - 1u) / w * w);
  return chains * ((nb + 15u) / 16u * 16u) / nb;
}
// tile_rows and row_tiles: the launch's row tiles of 64 and of 16.
constexpr uint32_t kTileMinTokens = 33;
constexpr bool gemm_tile_wins(uint64_t tile_rows, uint64_t row_tiles, uint32_t cols,
                              uint32_t n_tokens) {
  if (n_tokens < kTileMinTokens ||
      gemm_tile_wgs(tile_rows, n_tokens) * kGemmTileThreads > kMaxGridThreads)
    return false;
  const uint64_t wgs = tile_rows * (((uint64_t)n_tokens + 63u) / 64u);
  const uint64_t chains = gemm_row_chains(row_tiles, cols, n_tokens);
  if (wgs > 256u) return wgs > 640u || chains > (wgs > 512u ? 6912u : 5120u);
  return n_tokens <= 64u ? wgs > 192u || chains >= 3072u : chains > 3072u;
}

// How the 16 x 16 kernel of `tiles` token tiles a workgroup runs; us with weights from HBM.
// wide: a ring of 2 chunks of 16 blocks, for 3 of 8. Three and four tiles' waves hide more of
// a chunk's wait and share its barrier (3 of 8 / 2 of 16: 16.2 / 15.9 q/k/v for 64 tokens,
// 23.9 / 22.8 for 128, down 50.3 / 43.6 for 128, 11,264 rows of 2,048 columns 16.4 / 15.6 for
// 64); one tile's fill the first chunk sooner (q/k/v 12.3 / 12.9 for 16 tokens), and two's,
// but for eight groups ahead (8,192 x 8,192 28.5 / 26.8 for 32 tokens).
// ahead: the groups of 4 blocks whose activation a wave loads ahead. Its loads queue behind
// the weights' in the CU's memory path, so in long rows from HBM four groups wait on it: down
// took 30.7 us for 16 tokens, with eight 26.4; 8,192 x 8,192 23.5, 21.4; down for 32 tokens
// 33.6, 28.3, for 64 35.8, 30.5; 5,120 columns gain nothing. Eight are 35 registers more. Up to
// two workgroups a CU the CU holds the waves all the same, and one of three tiles or four,
// which gain by it only where each streams its own rows (1,024 x 8,192 for 192 tokens 20.5
// against 20.3). Past that four are the quicker: 11,264 rows of 2,048 columns (704) 11.9
// against 12.6 for 32 tokens, q/k/v (384) 15.8 against 20.1 for 64.
// spare_lds: LDS that a launch asks for and leaves alone, so that a CU holds three
// workgroups. Launches that CUs work through in turn read from HBM the slower, the more rows
// are read at once: one tile, 8 workgroups a CU or 3: 22,528 x 4,096 35.5 / 30.6 (16 tokens),
// 40,960 x 4,096 61.4 / 53.0; three tiles, 4 or 3: 17,408 x 4,096 38.3 / 35.9 (33 tokens);
// two, 5 or 3, with eight groups ahead: 128,256 x 4,096 190.1 / 175.3 (32 tokens), 28,672 x
// 8,192 86.0 / 82.2. Launches that the CUs hold at once are slower for it (14,336 x 4,096,
// 3.5 a CU: 23.0 / 27.5 for 16 tokens).
struct GemmRowsCut {
  bool wide;
  uint32_t ahead, spare_lds;
};
constexpr GemmRowsCut gemm_rows_cut(uint32_t tiles, uint32_t cols, uint64_t row_tiles, uint64_t wgs) {
  const bool long_rows = cols >= 8192u;
  if (tiles == 1u) {
    if (wgs > 4u * 256u) return GemmRowsCut{false, 4u, 35840u};
    return GemmRowsCut{false, long_rows && wgs <= 512u ? 8u : 4u, 0u};
  }
  if (tiles == 2u) {
    if (wgs > 5u * 256u) return GemmRowsCut{true, 8u, 35840u};
    return long_rows && wgs <= 512u ? GemmRowsCut{true, 8u, 0u} : GemmRowsCut{false, 4u, 0u};
  }
  if (tiles == 3u && wgs > 4u * 256u) return GemmRowsCut{true, 4u, 35840u};
  return GemmRowsCut{true, long_rows && wgs <= 256u && row_tiles > 192u ? 8u : 4u, 0u};
}

}  // namespace fkv
