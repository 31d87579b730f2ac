// Every byte that the batched GEMM's buffer loads read, from its kernels' own offset
// functions (fkv_gemm_at.h), against the matrix or workspace part it belongs to: for each
// width, rows left in the tile and tokens left, all chunks the kernels stage (their
// read-ahead past the row's end with them), all lanes. Lane and scalar offset together have
// to end inside, and a load that is used has to name its own row, pair and block.
#include "../../ferrum_amd/csrc/fkv_gemm_at.h"

#include <cstdio>
#include <cstdlib>
#include <initializer_list>

using namespace fkv::gemm_at;

static unsigned long checks = 0;
static const char* where = "";
static void inside(uint64_t at, uint32_t size, uint64_t bytes, const char* what) {
  ++checks;
  if (at + size <= bytes) return;
  std::printf("%s: %s reads %llu..%llu of %llu\n", where, what, (unsigned long long)at,
              (unsigned long long)(at + size), (unsigned long long)bytes);
  std::exit(1);
}
static void same(uint64_t got, uint64_t want, const char* what) {
  ++checks;
  if (got == want) return;
  std::printf("%s: %s at %llu, expected %llu\n", where, what, (unsigned long long)got,
              (unsigned long long)want);
  std::exit(1);
}

// Dword of a pair that its unit starts at, and dword 8 apart.
static const uint32_t kUnitDword[4] = {0, 4, 9, 13};

static void tile_kernel(uint32_t nb, uint32_t rows_left, uint32_t tiles_left) {
  const uint32_t np = nb / 2, nc = (np + 1) / 2, row_bytes = nb * 34;
  const uint64_t w_bytes = (uint64_t)rows_left * row_bytes, q_bytes = (uint64_t)tiles_left * nb * 512,
                 s_bytes = (uint64_t)tiles_left * nb * 64;
  const uint32_t last_row = rows_left - 1, last_tile = tiles_left - 1;
  for (uint32_t k = 0; k < nc + 3; ++k)
    for (uint32_t wave = 0; wave < 4; ++wave) {
      const uint32_t b = tile_block(k, wave, nb);
      for (uint32_t lane = 0; lane < 64; ++lane) {
        const uint32_t w = tile_weights(wave, lane, last_row, row_bytes);
        for (uint32_t i = 0; i < 2; ++i) {
          const uint64_t at = (uint64_t)w + pair(2 * k + i, np);
          inside(at, 16, w_bytes, "weights");
          const uint32_t r = 16 * wave + lane / 4, unit = (lane % 4) ^ (r / 4) % 4;
          if (2 * k + i < np && r < rows_left)
            same(at, (uint64_t)r * row_bytes + (2 * k + i) * 68 + kUnitDword[unit] * 4, "weights");
          const uint64_t xq = (uint64_t)tile_quants(wave, lane, last_tile, nb) + (b + i) * 512;
          inside(xq, 16, q_bytes, "quants");
          const uint32_t blk = 4 * k + 2 * (wave / 2) + i, t = 2 * (wave % 2) + lane % 32 / 16;
          if (blk < nb && t < tiles_left)
            same(xq, ((uint64_t)t * nb + blk) * 512 + lane / 32 * 256 + lane % 16 * 16, "quants");
        }
        const uint64_t e = (uint64_t)tile_dwords8(lane, last_row, row_bytes) + pair(2 * k + wave % 2, np);
        inside(e, 4, w_bytes, "dwords 8");
        if (2 * k + wave % 2 < np && lane < rows_left)
          same(e, (uint64_t)lane * row_bytes + (2 * k + wave % 2) * 68 + 32, "dwords 8");
        const uint64_t xs = (uint64_t)tile_scales(wave, lane, last_tile, nb) + b * 64;
        inside(xs, 4, s_bytes, "scales");
        const uint32_t blk = 4 * k + 2 * (wave / 2) + lane / 32, t = 2 * (wave % 2) + lane % 32 / 16;
        if (blk < nb && t < tiles_left)
          same(xs, ((uint64_t)t * nb + blk) * 64 + lane % 16 * 4, "scales");
      }
    }
}

static void rows_kernel(uint32_t nb, uint32_t rows_left, uint32_t pairs, uint32_t ring, uint32_t ahead) {
  const uint32_t np = nb / 2, ng = (nb + 3) / 4, n4 = (ng + 3) / 4, row_bytes = nb * 34;
  const uint64_t w_bytes = (uint64_t)rows_left * row_bytes;
  const uint32_t last_row = rows_left - 1;
  // barriers, and the chunks staged before the first
  const uint32_t chunks = (pairs == 4 ? 2 : 1) + 4 * n4 * 2 / pairs + ring - 1;
  for (uint32_t lane = 0; lane < 64; ++lane) {
    for (uint32_t k = 0; k < chunks; ++k) {
      for (uint32_t i = 0; i < pairs; ++i) {
        const uint64_t at = (uint64_t)rows_weights(lane, last_row, row_bytes) + pair(pairs * k + i, np);
        inside(at, 16, w_bytes, "weights");
        const uint32_t r = lane / 4, unit = (lane % 4) ^ (r / 4) % 4;
        if (pairs * k + i < np && r < rows_left)
          same(at, (uint64_t)r * row_bytes + (pairs * k + i) * 68 + kUnitDword[unit] * 4, "weights");
      }
      for (uint32_t i = 0; i < pairs; i += 4) {
        const uint32_t p = pairs * k + i + lane / 16;
        const uint64_t e = (uint64_t)rows_dwords8(lane, last_row, row_bytes) + pair(p, np);
        inside(e, 4, w_bytes, "dwords 8");
        if (p < np && lane % 16 < rows_left)
          same(e, (uint64_t)(lane % 16) * row_bytes + p * 68 + 32, "dwords 8");
      }
    }
    for (uint32_t g = 0; g < 4 * n4 + 1 + ahead; ++g) {
      for (uint32_t i = 0; i < 2; ++i) {
        const uint64_t at = (uint64_t)lane * 16 + rows_quants(2 * g + i, np);
        inside(at, 16, (uint64_t)np * 1024, "quants");
        if (2 * g + i < np) same(at, (uint64_t)(2 * g + i) * 1024 + lane * 16, "quants");
      }
      const uint32_t blk = 4 * g + lane / 16;
      const uint64_t whole = (uint64_t)lane * 4 + (nb % 16 ? 0 : rows_scales(g, nb)),
                     own = rows_scales_lane(g, lane, nb);
      if (nb % 16 == 0) inside(whole, 4, (uint64_t)nb * 64, "scales of whole groups");
      inside(own, 4, (uint64_t)nb * 64, "scales");
      if (blk < nb) {
        if (nb % 16 == 0) same(whole, (uint64_t)blk * 64 + lane % 16 * 4, "scales of whole groups");
        same(own, (uint64_t)blk * 64 + lane % 16 * 4, "scales");
      }
    }
  }
}

int main() {
  static char text[96];
  where = text;
  const uint32_t wide[] = {128, 176, 318, 448, 1022, 4608};  // blocks of wider rows
  for (uint32_t i = 0; i < 40 + sizeof(wide) / sizeof(*wide); ++i) {
    const uint32_t nb = i < 40 ? 2 * (i + 1) : wide[i - 40];
    for (uint32_t rows : {1u, 2u, 15u, 16u, 17u, 33u, 63u, 64u, 200u}) {
      for (uint32_t tiles = 1; tiles <= 5; ++tiles) {
        std::snprintf(text, sizeof text, "32 x 32 tiles, %u blocks, %u rows, %u tiles", nb, rows, tiles);
        tile_kernel(nb, rows, tiles);
      }
      std::snprintf(text, sizeof text, "16 x 16 tiles, %u blocks, %u rows", nb, rows);
      for (uint32_t ahead : {4u, 8u}) {
        rows_kernel(nb, rows, 4, 3, ahead);
        rows_kernel(nb, rows, 8, 2, ahead);
      }
    }
  }
  std::printf("ok\n");
  return checks > 1000000 ? 0 : 1;
}
