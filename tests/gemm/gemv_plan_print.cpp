// "rows cols tokens" lines in; the GEMV's tokens a workgroup and row split of each out, and
// whether all its workgroups run at once.
#include "../../ferrum_amd/csrc/fkv_gemv_plan.h"

#include <cstdio>

int main() {
  unsigned rows, cols, tokens;
  while (std::scanf("%u %u %u", &rows, &cols, &tokens) == 3) {
    const unsigned n_wg = (rows + fkv::kGemvRowsPerWg - 1) / fkv::kGemvRowsPerWg;
    const fkv::GemvCut c = fkv::gemv_cut(tokens, cols, n_wg);
    std::printf("%u %u %d\n", c.tokens, c.split, fkv::gemv_runs_at_once(tokens, cols, n_wg));
  }
  return 0;
}
