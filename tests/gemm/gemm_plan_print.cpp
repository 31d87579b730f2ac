// "row_tiles cols tokens" lines in; whether the batched GEMM runs in 64 x 64 tiles, their
// grid's threads and the quantizer's out.
#include "../../ferrum_amd/csrc/fkv_gemm_plan.h"

#include <cstdio>

int main() {
  unsigned row_tiles, cols, tokens;
  while (std::scanf("%u %u %u", &row_tiles, &cols, &tokens) == 3)
    std::printf("%d %llu %llu\n", fkv::gemm_tile_fills(row_tiles, tokens),
                (unsigned long long)fkv::gemm_tile_wgs(row_tiles, tokens) * fkv::kGemmTileThreads,
                (unsigned long long)fkv::gemm_act_threads(cols, tokens));
  return 0;
}
