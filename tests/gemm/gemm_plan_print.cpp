// "rows cols tokens" lines in; whether the batched GEMM runs in 64 x 64 tiles, their grid's
// threads and the quantizer's, and the 16 x 16 kernel's token tiles a workgroup, wide chunks,
// groups loaded ahead and spare LDS out.
#include "../../ferrum_amd/csrc/fkv_gemm_plan.h"

#include <cstdio>

int main() {
  unsigned rows, cols, tokens;
  while (std::scanf("%u %u %u", &rows, &cols, &tokens) == 3) {
    const unsigned tile_rows = (rows + 63) / 64, row_tiles = (rows + 15) / 16, n_tiles = (tokens + 15) / 16;
    const unsigned w = fkv::gemm_row_wg_tiles(n_tiles);
    const fkv::GemmRowsCut cut = fkv::gemm_rows_cut(w, cols, row_tiles, (unsigned long long)row_tiles * ((n_tiles + w - 1) / w));
    std::printf("%d %llu %llu %u %d %u %u\n", fkv::gemm_tile_wins(tile_rows, row_tiles, cols, tokens),
                (unsigned long long)fkv::gemm_tile_wgs(tile_rows, tokens) * fkv::kGemmTileThreads,
                (unsigned long long)fkv::gemm_act_threads(cols, tokens), w, cut.wide, cut.ahead, cut.spare_lds);
  }
  return 0;
}
