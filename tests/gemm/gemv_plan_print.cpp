// "rows cols tokens" lines in; the GEMV's tokens a workgroup and row split of each out.
#include "../../ferrum_amd/csrc/fkv_gemv_plan.h"

#include <cstdio>

int main() {
  unsigned rows, cols, tokens;
  while (std::scanf("%u %u %u", &rows, &cols, &tokens) == 3) {
    const fkv::GemvCut c = fkv::gemv_cut(tokens, cols, (rows + fkv::kGemvRowsPerWg - 1) / fkv::kGemvRowsPerWg);
    std::printf("%u %u\n", c.tokens, c.split);
  }
  return 0;
}
