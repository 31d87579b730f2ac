// How one Q8_0 GEMV launch (fkv_gemv.hip) is cut up: LDS, tokens a workgroup, lanes a row.
// Plain integer functions of the sizes, for the host and the kernels.
#pragma once
#include <cstddef>
#include <cstdint>

#ifdef __HIPCC__
#define FKV_PLAN __host__ __device__ constexpr
#else
#define FKV_PLAN constexpr
#endif

namespace fkv {

// LDS one workgroup may hold on gfx950.
constexpr size_t kGemvMaxLds = 163840;
constexpr uint32_t kGemvRowsPerWg = 16;  // of a workgroup of 4 waves, 16 lanes a row
constexpr int kGemvPipe = 4;             // 16-block steps in flight
// LDS dwords per (token, block): aligned q[0..8) | shifted q[0..8) | two tail pairs,
// aligned (q[8] = 0, xs) and shifted (q[8], xs).
constexpr uint32_t kGemvXDw = 20;

// LDS blocks a token: the step count rounded up to whole groups of kGemvPipe iterations
// (an iteration is S steps of 16 blocks), so every step a group runs reads inside the
// array.
FKV_PLAN uint32_t gemv_padded_blocks(uint32_t nb, uint32_t S = 1) {
  return (nb + 16u * S * kGemvPipe - 1u) / (16u * S * kGemvPipe) * (16u * S * kGemvPipe);
}
FKV_PLAN size_t gemv_lds_bytes(uint32_t tokens, uint32_t cols, uint32_t S = 1) {
  return (size_t)tokens * gemv_padded_blocks(cols / 32u, S) * kGemvXDw * 4u;
}

// tokens: those a workgroup takes with each weight it reads; split: 2 where the 16-lane
// rows of a wave take every other step of half the rows, twice the workgroups.
struct GemvCut {
  uint32_t tokens, split;
};

// Launches of one token whose S = 1 grid would leave SIMDs with fewer than two waves
// (under 512 workgroups of 4 waves on 256 CUs) take S = 2, when its LDS fits as well.
constexpr uint32_t kGemvSplitBelowWgs = 512;
FKV_PLAN uint32_t gemv_split(uint32_t cols, uint32_t n_wg) {
  return n_wg < kGemvSplitBelowWgs && gemv_lds_bytes(1, cols, 2) <= 65536u ? 2u : 1u;
}

// Tokens a workgroup takes with each weight it reads, for a launch of n_wg workgroups of 16
// rows. Four read the weights least often, but their ordered sums are four times the VALU
// work of a wave, so they win only where the launch has workgroups enough at four tokens
// each; smaller ones run two, twice the workgroups. us at 2 / 4 tokens a workgroup (w:
// workgroups of four):
// - up to 4 tokens, 4,096 columns: 6,144 rows 10.7 / 12.9 (384), 8,192 13.4 / 13.2 (512),
//   11,264 19.3 / 17.4 (704), 28,672 45.1 / 36.1;
// - over 4,096 columns a CU holds two workgroups of four, and two tokens win up to about
//   1,500 of them: 5,632 columns, 8,192 rows 31.2 / 32.3 for 8 tokens (w 1,024), 44.1 /
//   45.7 (11,264 rows, 1,408), 64.2 / 60.9 (16,384 rows, 2,048);
// - narrower ones turn from about 700 workgroups of four, and there by whole rounds of the
//   256 CUs, a round of four costing 1.8 of two: 2,048 columns 9.3 / 9.0 (4,096 rows, 12
//   tokens, w 768), 12.9 / 11.8 (20 tokens, 1,280), but 9.5 / 10.2 (8,192 rows, 5 tokens: 4
//   rounds against 6); 4,096 columns 20.1 / 18.1 (8,192 rows, 7 tokens, 1,024), 20.8 / 21.8
//   (6,144 rows, 12 tokens: 5 against 9), 30.4 / 25.5 (11,264 rows, 7 tokens: 6 against 11).
// Four tokens' activation has to fit 64 KiB of LDS, two tokens' half a CU's 160.
constexpr uint64_t kGemvFourMinWgs = 1500;
constexpr uint64_t kGemvFourMinWgsNarrow = 700;
constexpr uint32_t kGemvFourMinRowWgs = 512;  // launches of one slice of tokens
FKV_PLAN bool gemv_four_wins(uint32_t n_tokens, uint32_t cols, uint32_t n_wg) {
  if (n_tokens <= 4u) return n_tokens >= 3u && n_wg >= kGemvFourMinRowWgs;
  const uint64_t four = (uint64_t)n_wg * ((n_tokens + 3u) / 4u),
                 two = (uint64_t)n_wg * ((n_tokens + 1u) / 2u);
  if (four >= kGemvFourMinWgs) return true;
  const bool narrow = 3u * gemv_lds_bytes(4, cols) <= kGemvMaxLds;
  return narrow && four >= kGemvFourMinWgsNarrow &&
         9u * ((four + 255u) / 256u) < 5u * ((two + 255u) / 256u);
}
// Where two tokens' activation takes more than 64 KiB (12,320 to 16,384 columns) a CU holds
// two workgroups of two tokens, and a launch that leaves most of them out is bound by the
// chain of a row's ordered sum: one token with split rows has half of it. 14,336 columns, us
// at one / two tokens: 16 workgroups of rows and 8 tokens 9.5 / 13.9, 32 and 8 (256) 12.0 /
// 14.2, 64 and 6 (384) 14.6 / 14.4, 64 and 8 (512) 17.0 / 14.4, 256 and 4 (1,024) 40.7 / 25.9.
constexpr uint64_t kGemvOneMaxWgs = 384;
FKV_PLAN uint32_t gemv_tokens(uint32_t n_tokens, uint32_t cols, uint32_t n_wg) {
  if (n_tokens == 1u) return 1u;
  if (gemv_lds_bytes(4, cols) <= 65536u && gemv_four_wins(n_tokens, cols, n_wg)) return 4u;
  if (gemv_lds_bytes(2, cols) <= 65536u) return 2u;
  return gemv_lds_bytes(2, cols) <= kGemvMaxLds / 2u && (uint64_t)n_wg * n_tokens > kGemvOneMaxWgs
             ? 2u
             : 1u;
}

FKV_PLAN GemvCut gemv_cut(uint32_t n_tokens, uint32_t cols, uint32_t n_wg) {
  const uint32_t t = gemv_tokens(n_tokens, cols, n_wg);
  return GemvCut{t, t == 1u ? gemv_split(cols, n_wg) : 1u};
}

// Batches (8 tokens or more) that the matrix cores could take as well (fkv_gemm.hip): a GEMV
// all of whose workgroups run at once, up to three a CU, is the quicker one. It is one
// launch where those are two, and its chain of ordered sums is half as long a block. us as
// a GEMV / on the matrix cores, w its workgroups: 256 rows of 576 columns 3.7 / 5.8 (8
// tokens, w 64), 6.2 / 6.6 (128, 1,024), 10.4 / 6.8 (256, 2,048); 1,024 of 4,096 9.3 / 10.7
// (24, 768), 11.2 / 10.4 (32, 1,024); 2,048 of 2,752 8.6 / 8.7 (12, 768), 10.3 / 8.6 (16,
// 1,024); 256 of 14,336 8.9 / 22.4 (8, 128).
constexpr uint64_t kGemvAtOnceWgsPerCu = 3;
FKV_PLAN bool gemv_runs_at_once(uint32_t n_tokens, uint32_t cols, uint32_t n_wg) {
  const GemvCut c = gemv_cut(n_tokens, cols, n_wg);
  if (c.tokens == 4u) return false;  // over 1,300 workgroups of two
  const uint64_t wgs = (uint64_t)n_wg * c.split * ((n_tokens + c.tokens - 1u) / c.tokens);
  const uint64_t held = kGemvMaxLds / gemv_lds_bytes(c.tokens, cols, c.split);
  return wgs <= 256u * (held < kGemvAtOnceWgsPerCu ? held : kGemvAtOnceWgsPerCu);
}

}  // namespace fkv
