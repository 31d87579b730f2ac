// Batched Q8_0 GEMM on the matrix cores of gfx950, for batches of activation rows (a
// decode step's sequences, a prefill chunk): the GEMV reads every weight once per 1
// to 4 tokens. The activation is quantized once, into a workspace; then one of two kernels,
// 32 x 32 tiles first.
//
// The result is the GEMV's (fkv_gemv.hip) bit for bit: per output, starting from +0 and
// for each 32-value block in order, acc += f32(sumi) * (w_scale * x_scale)
// (crates/kernels/src/q8_dot.rs:72-109), the product and the sum each rounded once.
//
// What bounds it: one v_mfma_i32_32x32x32_i8 (32 cycles) gives a block's integer dots of
// 1,024 outputs, and then the VALU has to round and add each output by itself, 16 a lane.
// So every instruction per output counts. Written as in the reference there are four
// (convert, the product of the scales, the product, the sum); here three:
// - the accumulator input of the integer MFMA is the bit pattern of M = 1.5 * 2^23, so
//   its result, read as an f32, is M + sumi exactly (|sumi| <= 32 * 128 * 128 < 2^22),
//   and one subtraction (exact; 2 a 4-cycle slot from two waves, a v_cvt_f32_i32 only
//   one) gives f32(sumi);
// - w_scale * x_scale of 1,024 outputs and two blocks is one v_mfma_f32_32x32x4_2b_f16
//   whose second to fourth terms are zero: the product of two binary16 values is exact in
//   f32, Inf and NaN included. (The f32 form of the same outer product held up the VALU:
//   780 against 953 TFLOP/s in a register-only loop of these instructions.)
// Measured at 512 tokens on Llama-3-8B's projections (the 32 x 32 kernel alone, from a kernel
// trace; distinct weights each call): q/k/v 54.8 us, attn_output 39.5, gate/up 218 (551
// TFLOP/s), down 130; the four calls with their quantizers 443 us, where 16 x 16 tiles, one a
// wave, on the four-instruction epilogue took 642. Three waves a SIMD take 223 cycles a block
// together, 94% of them issue VALU instructions, and the clock is about 1.9 GHz under that
// load.
#include "fkv_device.h"
#include "fkv_gemm_at.h"
#include "fkv_gemm_plan.h"
#include "fkv_gemv_plan.h"
#include "fkv_q8_act.h"

namespace fkv {
namespace {

typedef float f32x4a __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4a __attribute__((ext_vector_type(4), aligned(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x32 __attribute__((ext_vector_type(32)));

constexpr uint32_t kQ8Bytes = 34;
static_assert(gemm_at::kPairBytes == 2 * kQ8Bytes, "a pair of blocks");
constexpr uint32_t kTileRows = kGemmTileRows;
[[maybe_unused]] constexpr uint32_t kMagicBits = 0x4b400000u;
[[maybe_unused]] constexpr float kMagic = 12582912.0f;    // 1.5 * 2^23

// The activation in the workspace, per 16-token tile (tokens past n_tokens quantize to
// zeros): 512 bytes a block of quants in 16-byte units, then, after every tile's quants,
// the scales, binary16 bits in 32, [tile][block][token]. An even block's quants are in the
// order its weights are read in (Chunk): 0, 1, 30, 31, then 2 .. 29. A unit, for the
// 32 x 32 kernel, is (block, half of the block, token); for the 16 x 16 kernel (kPairs)
// (pair of blocks, quarter, token): that quarter's 8 quants of both blocks.
__host__ __device__ constexpr uint64_t act_quant_bytes(uint32_t n_tiles, uint32_t nb) {
  return (uint64_t)n_tiles * nb * 512u;
}

constexpr uint32_t kActThreads = kGemmActThreads;

template <bool kPairs>
__global__ __launch_bounds__(kActThreads) void q8_act_tile_kernel(const float* __restrict__ x,
                                                                  uint32_t cols, uint32_t n_tokens,
                                                                  uint32_t n_tiles,
                                                                  uint8_t* __restrict__ ws) {
  // Item i: token t = i / (cols/8), values 8j .. 8j + 7 with j = i % (cols/8): quarter
  // j % 4 of block j / 4, so a quad of lanes holds a block.
  const uint32_t per = cols / 8u, nb = cols / 32u;
  const uint64_t i = (uint64_t)blockIdx.x * kActThreads + threadIdx.x;
  if (i >= (uint64_t)n_tiles * 16u * per) return;
  const uint32_t t = (uint32_t)(i / per), j = (uint32_t)(i % per);
  f32x4a a = {0.0f, 0.0f, 0.0f, 0.0f}, b = {0.0f, 0.0f, 0.0f, 0.0f};
  if (t < n_tokens) {
    const float* src = x + (uint64_t)t * cols + 8u * j;
    a = *(const f32x4a*)src;
    b = *(const f32x4a*)(src + 4);
  }
  float m = __builtin_fmaxf(__builtin_fabsf(a.x), __builtin_fabsf(a.y));
  m = __builtin_fmaxf(m, __builtin_fabsf(a.z));
  m = __builtin_fmaxf(m, __builtin_fabsf(a.w));
  m = __builtin_fmaxf(m, __builtin_fabsf(b.x));
  m = __builtin_fmaxf(m, __builtin_fabsf(b.y));
  m = __builtin_fmaxf(m, __builtin_fabsf(b.z));
  m = __builtin_fmaxf(m, __builtin_fabsf(b.w));
  m = __builtin_fmaxf(m, 0.0f);  // all NaN: 0, as the reference's amax = 0 start
  m = __builtin_fmaxf(m, dev::dpp<0xB1>(m));
  m = __builtin_fmaxf(m, dev::dpp<0x4E>(m));
  const float d = dev::div127(m);
  const float id = (d != 0.0f) ? 1.0f / d : 0.0f;
  const uint32_t qa = dev::q8_byte(a.x * id) | (dev::q8_byte(a.y * id) << 8) |
                      (dev::q8_byte(a.z * id) << 16) | (dev::q8_byte(a.w * id) << 24);
  const uint32_t qb = dev::q8_byte(b.x * id) | (dev::q8_byte(b.y * id) << 8) |
                      (dev::q8_byte(b.z * id) << 16) | (dev::q8_byte(b.w * id) << 24);
  const uint32_t tt = t / 16u, c = t % 16u, blk = j / 4u, quarter = j % 4u;
  const uint64_t at = (uint64_t)tt * nb + blk;
  uint32_t lo = qa, hi = qb;
  if (blk % 2u == 0u) {
    // quads rotate: the lane before (the last one's for the first) holds 2 of these bytes
    const uint32_t prev = (uint32_t)__builtin_amdgcn_mov_dpp((int)qb, 0x93, 0xf, 0xf, true);
    lo = quarter == 0u ? (qa & 0xffffu) | (prev & 0xffff0000u) : __builtin_amdgcn_alignbit(qa, prev, 16);
    hi = __builtin_amdgcn_alignbit(qb, qa, 16);
  }
  const uint64_t to = kPairs ? (at - blk % 2u) * 512u + (quarter * 16u + c) * 16u + (blk % 2u) * 8u
                             : at * 512u + (quarter / 2u) * 256u + c * 16u + (quarter % 2u) * 8u;
  *(uint2*)(ws + to) = make_uint2(lo, hi);
  if (quarter == 0u)
    ((uint32_t*)(ws + act_quant_bytes(n_tiles, nb)))[at * 16u + c] = dev::f16_bits_away(d);
}

// A buffer of `bytes` at p. Every load stays inside it by its own offsets (gemm_at).
[[maybe_unused]] __device__ __forceinline__ __amdgpu_buffer_rsrc_t lds_source(const void* p,
                                                                             uint64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(
      (void*)p, (short)0, (int)(bytes < 0x7fffffffu ? bytes : 0x7fffffffu), 0x00020000);
}

// A chunk of 4 blocks (2 pairs) in LDS. A pair of a weight row is 17 dwords, [scale 0 |
// quants 0, 1] [2 .. 5] ... [26 .. 29] [30, 31 | scale 1] and 8 of the odd block's quants:
// as 16-byte units, dwords 0-3, 4-7, 9-12 and 13-16, and dword 8 by itself. The units of
// the odd block are its quants; the even block's are too, but for dword 0, which with
// dword 8 gives quants 0, 1, 30, 31 (one v_perm, a second one the scales): a dot does not
// depend on the order of its terms, so nothing is realigned.
// A row's units lie at unit ^ (row / 4) % 4: a wave stages 16 rows' with one load (4 lanes
// a row, 64 consecutive bytes) and reads one unit of 32 rows, both over all banks.
struct Chunk {
  uint4 wq[2][kTileRows][4];   // [pair][row][unit, at unit ^ (row / 4) % 4]
  uint4 xq[2][4][2][32];       // [token half][block][half of the block][token]
  uint32_t we[2][kTileRows];   // [pair][row]
  uint32_t xs[2][2][2][32];    // [pair][token half][block][token]
};

// A workgroup: 64 weight rows x 64 tokens, a wave 32 x 32; 3 workgroups a CU (154 VGPRs,
// 52.5 KiB of LDS). Everything is staged by loads straight into LDS, two to three chunks
// ahead (three buffers), so that no wave spends registers or instructions on it. (Weights
// through registers with the repacking done by the computing waves: gate/up 285 us; by two
// or four further waves: 264-300.)
// Tokens are the MFMA rows and weight rows its columns, so a lane's results are one
// column of y and 32 consecutive lanes store 128 consecutive bytes.
__global__ __launch_bounds__(256, 2) void gemm_q8_tile_kernel(const GemvBatch bat, uint32_t cols,
                                                              uint32_t n_tokens, uint32_t n_tiles,
                                                              uint32_t row_tiles,
                                                              uint32_t token_tiles,
                                                              const uint8_t* __restrict__ ws) {
#ifdef __HIP_DEVICE_COMPILE__  // the host pass needs the kernel's stub only
  // Workgroups are dealt to the 8 XCDs in turn; the token tiles of one row tile follow
  // each other on one XCD, whose L2 then reads the weights once.
  const uint32_t xcd = blockIdx.x % 8u, j8 = blockIdx.x / 8u;
  const uint32_t rt = (j8 / token_tiles) * 8u + xcd, ty = j8 % token_tiles;
  if (rt >= row_tiles) return;
  uint32_t mi = 0;
#pragma unroll
  for (int j = 1; j < kGemvMaxMats; ++j)
    if ((uint32_t)j < bat.n && rt >= bat.m[j].wg0) mi = (uint32_t)j;
  const GemvMat M = mi == 0u ? bat.m[0] : mi == 1u ? bat.m[1] : mi == 2u ? bat.m[2] : bat.m[3];
  const uint32_t rows = M.rows, row0 = (rt - M.wg0) * kTileRows;
  const uint32_t nb = cols / 32u, np = nb / 2u, nc = (np + 1u) / 2u;
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t c32 = lane & 31u, half = lane >> 5;
  const uint32_t wr = wave & 1u, wt = wave >> 1;

  __shared__ Chunk s0, s1, s2;

  // Staging: loads straight into LDS, 6 a wave and chunk. Rows past the matrix, tokens past
  // the batch and blocks past the row's end read the last one (never used; gemm_at). An
  // address is a lane's register and a scalar, bounded by one scalar minimum for each of a
  // chunk's two pairs and one for its activation.
  const uint64_t row_bytes = (uint64_t)nb * kQ8Bytes;
  const uint32_t last_row = rows - 1u - row0;
  const uint32_t t16 = ty * 4u;
  const uint64_t left = (uint64_t)(n_tiles - t16) * nb;  // blocks of this and the later tiles
  const __amdgpu_buffer_rsrc_t rw = lds_source(M.w + row0 * row_bytes, (rows - row0) * row_bytes);
  const __amdgpu_buffer_rsrc_t rq = lds_source(ws + (uint64_t)t16 * nb * 512u, left * 512u);
  const __amdgpu_buffer_rsrc_t rs =
      lds_source(ws + act_quant_bytes(n_tiles, nb) + (uint64_t)t16 * nb * 64u, left * 64u);
  const uint32_t last_tile = n_tiles - 1u - t16;
  // weights: wave w stages rows 16w .. 16w + 15, 4 lanes a row
  const uint32_t w_off = gemm_at::tile_weights(wave, lane, last_row, (uint32_t)row_bytes);
  // their dwords 8: waves w and w + 2 pair w (the same ones), a lane a row
  const uint32_t e_off = gemm_at::tile_dwords8(lane, last_row, (uint32_t)row_bytes);
  // activation: wave w blocks 2 * (w / 2), + 1 of token half w % 2, and their scales
  const uint32_t xq_off = gemm_at::tile_quants(wave, lane, last_tile, nb);
  const uint32_t xs_off = gemm_at::tile_scales(wave, lane, last_tile, nb);
#define FKV_LDS(p) (__attribute__((address_space(3))) void*)(p)
  const uint32_t xb0 = 2u * (wave >> 1);
  auto stage = [&](uint32_t k, Chunk& L) __attribute__((always_inline)) {
    const uint32_t wo[2] = {gemm_at::pair(2u * k, np), gemm_at::pair(2u * k + 1u, np)};
    const uint32_t b = gemm_at::tile_block(k, wave, nb);
#pragma unroll
    for (uint32_t i = 0; i < 2u; ++i) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, FKV_LDS(&L.wq[i][16u * wave][0]), 16, w_off,
                                               (int)wo[i], 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rq, FKV_LDS(&L.xq[wave & 1u][xb0 + i][0][0]), 16,
                                               xq_off, (int)((b + i) * 512u), 0, 0);
    }
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, FKV_LDS(&L.we[wave & 1u][0]), 4, e_off,
                                             (int)(wave & 1u ? wo[1] : wo[0]), 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, FKV_LDS(&L.xs[wave >> 1][wave & 1u][0][0]), 4,
                                             xs_off, (int)(b * 64u), 0, 0);
  };
#undef FKV_LDS
  // This wave's reads of the chunk to be overwritten are done, and its loads of the next
  // chunk have landed (those of the chunk after it, the last 6, may still be in flight);
  // then every wave's.
  auto sync = [&]() __attribute__((always_inline)) {
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0076);  // vmcnt(6) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
  };

  float acc[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  i32x16 magic;
#pragma unroll
  for (int r = 0; r < 16; ++r) magic[r] = (int)kMagicBits;
  __asm__("" : "+v"(magic));  // kept in registers: not written anew for every product

  // A pair's operands, and its products: the integer dots of its blocks and both blocks'
  // products of scales.
  i32x2 w1 = {0, 0}, x1 = {0, 0};
  i32x4 wq0, wq1, xq0, xq1;
  uint32_t we;
  f32x32 P;
  i32x16 D0, D1;
  const f32x32 zero = {};
  const uint32_t row_l = wr * 32u + c32, u0 = half ^ (c32 / 4u) % 4u;
  // v_perm selectors of the even block's first dword (lanes 0-31: quants 0, 1, 30, 31;
  // the others' is as stored) and of the scale (lanes 0-31 the even block's)
  const uint32_t sel_q = half ? 0x03020100u : 0x05040302u, sel_s = half ? 0x0c0c0706u : 0x0c0c0100u;
  auto read_0 = [&](const Chunk& L, int s) __attribute__((always_inline)) {
    wq0 = __builtin_bit_cast(i32x4, L.wq[s][row_l][u0]);
    we = L.we[s][row_l];
    xq0 = __builtin_bit_cast(i32x4, L.xq[wt][2 * s][half][c32]);
    x1[0] = (int)L.xs[s][wt][half][c32];
  };
  auto read_1 = [&](const Chunk& L, int s) __attribute__((always_inline)) {
    wq1 = __builtin_bit_cast(i32x4, L.wq[s][row_l][u0 ^ 2u]);
    xq1 = __builtin_bit_cast(i32x4, L.xq[wt][2 * s + 1][half][c32]);
  };
  auto dots_0 = [&]() __attribute__((always_inline)) {
    w1[0] = (int)__builtin_amdgcn_perm(we, (uint32_t)wq0[0], sel_s);
    wq0[0] = (int)__builtin_amdgcn_perm(we, (uint32_t)wq0[0], sel_q);
    D0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(xq0, wq0, magic, 0, 0, 0);
  };
  auto scales = [&]() __attribute__((always_inline)) {
    P = __builtin_amdgcn_mfma_f32_32x32x4f16(__builtin_bit_cast(f16x4, x1),
                                             __builtin_bit_cast(f16x4, w1), zero, 0, 0, 0);
  };
  auto sub16 = [&](f32x16& f) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) f[r] = f[r] - kMagic;
    __builtin_amdgcn_sched_barrier(0);
  };
  auto mul16 = [&](f32x16& f, int o) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) f[r] = f[r] * P[o + r];
    __builtin_amdgcn_sched_barrier(0);
  };
  auto add16 = [&](float (&a)[16], const f32x16& f) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) a[r] = a[r] + f[r];
    __builtin_amdgcn_sched_barrier(0);
  };
  // A pair from P, D0, D1; each is replaced by the next pair's as soon as it is used up,
  // from the operands in registers, which are then read anew for the pair after that
  // (pair s of L). What an MFMA writes is used 32 to 64 instructions later.
  auto pair = [&](const Chunk& L, int s, auto between) __attribute__((always_inline)) {
    f32x16 f = __builtin_bit_cast(f32x16, D0);
    sub16(f);
    mul16(f, 0);
    add16(acc, f);
    dots_0();
    __builtin_amdgcn_sched_barrier(0);
    f = __builtin_bit_cast(f32x16, D1);
    sub16(f);
    mul16(f, 16);
    scales();
    __builtin_amdgcn_sched_barrier(0);
    between();
    read_0(L, s);
    __builtin_amdgcn_sched_barrier(0);
    add16(acc, f);
    D1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(xq1, wq1, magic, 0, 0, 0);
    read_1(L, s);
    __builtin_amdgcn_sched_barrier(0);
  };
  // Chunk k while chunk k + 1 (N) is read and chunk k + 3 staged into L, whose reads all
  // waves have finished.
  auto chunk = [&](Chunk& L, Chunk& N, uint32_t k) __attribute__((always_inline)) {
    pair(N, 0, [&]() __attribute__((always_inline)) {
      sync();
      stage(k + 3u, L);
    });
    if (2u * k + 1u < np) pair(N, 1, [] {});
  };

  stage(0, s0);
  stage(1, s1);
  sync();
  stage(2, s2);
  read_0(s0, 0);
  read_1(s0, 0);
  dots_0();
  scales();
  D1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(xq1, wq1, magic, 0, 0, 0);
  read_0(s0, 1);
  read_1(s0, 1);
  for (uint32_t k = 0;; k += 3u) {
    chunk(s0, s1, k);
    if (k + 1u >= nc) break;
    chunk(s1, s2, k + 1u);
    if (k + 2u >= nc) break;
    chunk(s2, s0, k + 2u);
    if (k + 3u >= nc) break;
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // no load into LDS outlives the workgroup

  const uint32_t row = row0 + wr * 32u + c32;
  if (row >= rows) return;
  const uint32_t tok0 = (ty * 2u + wt) * 32u + 4u * half;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const uint32_t tok = tok0 + 8u * (uint32_t)(r / 4) + (uint32_t)(r % 4);
    if (tok < n_tokens) M.y[(uint64_t)tok * rows + row] = acc[r];
  }
#endif
}

// ---------------------------------------------------------------------------
// Few workgroups of 64 x 64: 16 weight rows x 64 tokens a workgroup, 16 x 16 a wave.
// ---------------------------------------------------------------------------
//
// The same sums (integer dots from v_mfma_i32_16x16x32_i8, four blocks' products of scales
// from one v_mfma_f32_16x16x4_4b_f16, three VALU instructions per output and block), for
// launches that would leave CUs without work in 64 x 64 tiles, or most of their tokens
// unused. The ordered sum makes a row tile one chain, a wave takes 95 cycles a block at best
// (one row tile, weights from cache) and about 120 with a CU's weights from HBM, and a CU has
// few waves: the chain bounds launches of few rows (down of Llama-3-8B, 448 blocks: 23 us at
// 16 tokens where the weights alone stream in 10), and what matters is that nothing else is
// waited for. A further wave streams the weights through a ring of chunks in LDS by direct
// loads; the computing waves load the activation, which the L2 holds, four or eight groups of
// blocks ahead into registers. Loads retire in order, so with the weight loads in the
// computing waves each activation load would wait for HBM. Against the kernel before (one variant with and one without such a wave,
// weights through registers, four VALU instructions), us with weights from HBM, 16 tokens:
// q/k/v 14.3 -> 12.1, attn_output 12.9 -> 11.4, gate/up 40.8 -> 40.0, down 29.3 -> 26.4; 64
// tokens: 19.0 -> 15.9, 14.5 -> 13.3, gate/up in 64 x 64 tiles, 35.0 -> 30.1.
// Chunk, ring and the groups loaded ahead are the launch's (gemm_rows_cut).
[[maybe_unused]] constexpr uint32_t kGroup = 4;    // blocks of a step
constexpr uint32_t kRowTile = kGemmRowTile;

template <uint32_t kPairs>
struct RowChunk {
  uint4 wq[kPairs][kRowTile][4];   // as Chunk's
  uint32_t we[kPairs][kRowTile];
};

// kTail: columns not a multiple of 512. The blocks that fill the row's last 16 up get
// scales of zero (the row's last pair is read for them), so they add +0.
// W computing waves, a 16-token tile each. Chunks of kPairs pairs, a ring of kRing; kAhead
// groups of activation in registers.
template <int W, bool kTail, uint32_t kPairs, uint32_t kRing, int kAhead>
__global__ __launch_bounds__((W + 1) * 64, kAhead == 4 ? 4 : 2) void gemm_q8_rows_kernel(
    const GemvBatch bat, uint32_t cols, uint32_t n_tokens, uint32_t n_tiles,
    const uint8_t* __restrict__ ws) {
#ifdef __HIP_DEVICE_COMPILE__  // the host pass needs the kernel's stub only
  uint32_t mi = 0;
#pragma unroll
  for (int j = 1; j < kGemvMaxMats; ++j)
    if ((uint32_t)j < bat.n && blockIdx.x >= bat.m[j].wg0) mi = (uint32_t)j;
  const GemvMat M = mi == 0u ? bat.m[0] : mi == 1u ? bat.m[1] : mi == 2u ? bat.m[2] : bat.m[3];
  const uint32_t rows = M.rows, row0 = (blockIdx.x - M.wg0) * kRowTile;
  const uint32_t nb = cols / 32u, np = nb / 2u;
  // groups, runs of 4 groups
  const uint32_t ng = (nb + kGroup - 1u) / kGroup, n4 = (ng + 3u) / 4u;
  constexpr int kGroups = (int)kPairs / 2;  // of a chunk
  static_assert(kGroups == 2 || kGroups == 4, "whole chunks a run of 4 groups");
  static_assert(kAhead == 4 || kAhead == 8, "whole runs a turn of the registers");
  // barriers: one a chunk, and the chunks read past the row's end (up to 3 groups ahead)
  const uint32_t n_bar = (kGroups == 2 ? 2u : 1u) + n4 * (4u / (uint32_t)kGroups);
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t c = lane & 15u, grp = lane >> 4;

  using Rows = RowChunk<kPairs>;
  __shared__ Rows ring[kRing];
  auto barrier = [] {
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
  };

  if (wave == (uint32_t)W) {
    // Rows past the matrix and pairs past the row's end load the last one (never used, or
    // met by zero scales; gemm_at).
    const uint64_t row_bytes = (uint64_t)nb * kQ8Bytes;
    const uint32_t last_row = rows - 1u - row0;
    const __amdgpu_buffer_rsrc_t rw = lds_source(M.w + row0 * row_bytes, (rows - row0) * row_bytes);
    const uint32_t w_off = gemm_at::rows_weights(lane, last_row, (uint32_t)row_bytes);
    const uint32_t e_off = gemm_at::rows_dwords8(lane, last_row, (uint32_t)row_bytes);
    auto stage = [&](uint32_t k) __attribute__((always_inline)) {
      Rows& L = ring[k % kRing];
#pragma unroll
      for (uint32_t i = 0; i < kPairs; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rw, (__attribute__((address_space(3))) void*)&L.wq[i][0][0], 16, w_off,
            (int)gemm_at::pair(k * kPairs + i, np), 0, 0);
#pragma unroll
      for (uint32_t i = 0; i < kPairs; i += 4u)  // 4 pairs' dwords 8
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rw, (__attribute__((address_space(3))) void*)&L.we[i][0], 4,
            e_off + gemm_at::pair(k * kPairs + i + grp, np), 0, 0, 0);
    };
    for (uint32_t k = 0; k + 1u < kRing; ++k) stage(k);
    // Before barrier k: chunk k has landed (kRing - 2 later ones may be in flight). After
    // it every wave is done with chunk k - 1, whose buffer takes chunk k - 1 + kRing.
    constexpr uint32_t kInFlight = (kPairs + kPairs / 4u) * (kRing - 2u);
    static_assert(kInFlight < 16u, "the wait's field");
    for (uint32_t k = 0; k < n_bar; ++k) {
      __builtin_amdgcn_s_waitcnt(0x0f70 | kInFlight);  // vmcnt
      barrier();
      stage(k + kRing - 1u);
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);  // no load into LDS outlives the workgroup
    return;
  }

  const uint32_t tt = blockIdx.y * (uint32_t)W + wave;
  if (tt >= n_tiles) {  // wave-uniform
    for (uint32_t k = 0; k < n_bar; ++k) barrier();
    return;
  }

  // Activation of group g: a unit of each of its two pairs, and the scale of block
  // 4g + grp; past the row's end the last one's (never used, or met by zero scales).
  const __amdgpu_buffer_rsrc_t rq = lds_source(ws + (uint64_t)tt * np * 1024u, np * 1024u);
  const __amdgpu_buffer_rsrc_t rs =
      lds_source(ws + act_quant_bytes(n_tiles, nb) + (uint64_t)tt * nb * 64u, nb * 64u);
  const int32_t blocks_left = (int32_t)nb - (int32_t)grp;
  const uint32_t xq_off = lane * 16u;
  uint4 xq[kAhead][2];
  uint32_t xs[kAhead];
  auto load_x = [&](uint32_t g, int slot) __attribute__((always_inline)) {
    xq[slot][0] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rq, xq_off, gemm_at::rows_quants(2u * g, np), 0));
    xq[slot][1] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rq, xq_off, gemm_at::rows_quants(2u * g + 1u, np), 0));
    xs[slot] = kTail ? __builtin_amdgcn_raw_buffer_load_b32(rs, gemm_at::rows_scales_lane(g, lane, nb), 0, 0)
                     : __builtin_amdgcn_raw_buffer_load_b32(rs, lane * 4u, gemm_at::rows_scales(g, nb), 0);
  };

  // Weights of a group: 8 quants of row c of each block (unit grp / 2 of the block), the
  // pairs' dwords 8 and the scale of block grp.
  const uint32_t f = c / 4u;
  const uint32_t o_even = c * 64u + ((grp / 2u) ^ f) * 16u + (grp % 2u) * 8u, o_odd = o_even ^ 32u;
  const uint32_t o_we = (uint32_t)offsetof(Rows, we) + c * 4u;
  const bool s_odd = grp % 2u != 0u;
  const uint32_t o_s = s_odd ? o_we + (grp / 2u) * 64u + 2u : (grp / 2u) * 1024u + c * 64u + f * 16u;
  const uint32_t s_step = s_odd ? 128u : 2048u;  // a group on
  uint2 wb[2][4];
  uint32_t we[2][2], sw[2];
  uint32_t a_even = o_even, a_odd = o_odd, a_we = o_we, a_s = o_s;  // in the chunk being read
  auto at_chunk = [&](uint32_t base) __attribute__((always_inline)) {
    a_even = base + o_even;
    a_odd = base + o_odd;
    a_we = base + o_we;
    a_s = base + o_s;
  };
  auto read_w = [&](int g) __attribute__((always_inline)) {  // group g % kGroups of the chunk
    const uint8_t* L = (const uint8_t*)ring;
    const int j = g % kGroups, t = g % 2;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      wb[t][2 * i] = *(const uint2*)(L + a_even + (2 * j + i) * 1024);
      wb[t][2 * i + 1] = *(const uint2*)(L + a_odd + (2 * j + i) * 1024);
      we[t][i] = *(const uint32_t*)(L + a_we + (2 * j + i) * 64);
    }
    sw[t] = *(const uint16_t*)(L + a_s);
    a_s += s_step;
  };

  float acc[4] = {};
  i32x4 magic = {(int)kMagicBits, (int)kMagicBits, (int)kMagicBits, (int)kMagicBits};
  __asm__("" : "+v"(magic));
  const f32x16 zero = {};
  const uint32_t sel_q = grp == 0u ? 0x05040302u : 0x03020100u;
  f32x16 P;
  i32x4 D[4];
  // Blocks 2h and 2h + 1 of the group in slot: tokens are the MFMA rows.
  auto dots = [&](int h, int slot) __attribute__((always_inline)) {
    const uint4 x = xq[slot][h];
    const uint2* w = wb[slot % 2];
    const uint32_t w0 = __builtin_amdgcn_perm(we[slot % 2][h], w[2 * h].x, sel_q);
    auto l64 = [](uint32_t lo, uint32_t hi) { return (long)(((uint64_t)hi << 32) | lo); };
    D[2 * h] = __builtin_amdgcn_mfma_i32_16x16x32_i8(l64(x.x, x.y), l64(w0, w[2 * h].y), magic, 0, 0, 0);
    D[2 * h + 1] = __builtin_amdgcn_mfma_i32_16x16x32_i8(
        l64(x.z, x.w), l64(w[2 * h + 1].x, w[2 * h + 1].y), magic, 0, 0, 0);
  };
  auto scales = [&](uint32_t g, int slot) __attribute__((always_inline)) {
    i32x2 x1 = {(int)xs[slot], 0}, w1 = {(int)sw[slot % 2], 0};
    if (kTail && (int32_t)(kGroup * g) >= blocks_left) x1[0] = w1[0] = 0;
    P = __builtin_amdgcn_mfma_f32_16x16x4f16(__builtin_bit_cast(f16x4, x1),
                                             __builtin_bit_cast(f16x4, w1), zero, 0, 0, 0);
  };
  float v[8];
  auto products = [&](int h) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r] = __int_as_float(D[2 * h + r / 4][r % 4]) - kMagic;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r] = v[r] * P[8 * h + r];
    __builtin_amdgcn_sched_barrier(0);
  };
  auto add = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 8; ++r) acc[r % 4] = acc[r % 4] + v[r];
  };

#pragma unroll
  for (int j = 0; j < kAhead; ++j) load_x((uint32_t)j, j);
  barrier();  // chunk 0
  read_w(0);
  dots(0, 0);
  dots(1, 0);
  scales(0, 0);
  load_x((uint32_t)kAhead, 0);
  read_w(1);
  uint32_t base = 0;
  auto next_chunk = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave has read the last one
    barrier();
    base = base + sizeof(Rows) < sizeof(ring) ? base + (uint32_t)sizeof(Rows) : 0u;
    at_chunk(base);
  };
  if (kGroups == 2) next_chunk();
  read_w(2);
  for (uint32_t k = 0; k < n4; k += (uint32_t)kAhead / 4u) {
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      if (j == 4 && k + 1u >= n4) break;
      // Group g, while group g + 1's products go through the matrix cores from the operands
      // in registers, which then take group g + 3's weights and g + 1 + kAhead's activation.
      const uint32_t g = 4u * k + (uint32_t)j;
      const int n = (j + 1) % kAhead;
      __builtin_amdgcn_sched_barrier(0);
      products(0);
      add();
      __builtin_amdgcn_sched_barrier(0);
      dots(0, n);
      __builtin_amdgcn_sched_barrier(0);
      products(1);
      scales(g + 1u, n);
      __builtin_amdgcn_sched_barrier(0);
      add();
      __builtin_amdgcn_sched_barrier(0);
      dots(1, n);
      load_x(g + 1u + (uint32_t)kAhead, n);
      if ((j + 3) % kGroups == 0) next_chunk();
      read_w((j + 3) % 4);
    }
  }

  const uint32_t row = row0 + c;
  if (row >= rows) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const uint32_t tok = tt * 16u + 4u * grp + (uint32_t)r;
    if (tok < n_tokens) M.y[(uint64_t)tok * rows + row] = acc[r];
  }
#endif
}

}  // namespace

bool gemm_mfma_eligible(const GemvBatch& b, uint32_t cols, uint32_t n_tokens) {
  if (n_tokens < kGemmMfmaMinTokens || cols % 64u != 0u) return false;
  for (uint32_t m = 0; m < b.n; ++m)
    if ((uintptr_t)b.m[m].w % 4u != 0u) return false;
  return true;
}

bool gemm_mfma_needs_workspace(const GemvBatch& b, uint32_t cols) {
  if (cols % 1024u != 0u) return false;
  for (uint32_t m = 0; m < b.n; ++m)
    if ((uintptr_t)b.m[m].w % 16u != 0u) return false;
  return true;
}

bool gemm_mfma_pays(const GemvBatch& b, uint32_t cols, uint32_t n_tokens) {
  uint32_t n_wg = 0;
  for (uint32_t m = 0; m < b.n; ++m) n_wg += (b.m[m].rows + kGemvRowsPerWg - 1u) / kGemvRowsPerWg;
  return !gemv_runs_at_once(n_tokens, cols, n_wg) &&
         gemm_act_threads(cols, n_tokens) <= kMaxGridThreads;
}

uint64_t gemm_mfma_workspace_bytes(uint32_t cols, uint32_t n_tokens) {
  const uint32_t n_tiles = (n_tokens + 15u) / 16u, nb = cols / 32u;
  return act_quant_bytes(n_tiles, nb) + (uint64_t)n_tiles * nb * 16u * 4u;
}

template <int W, uint32_t kPairs, uint32_t kRing, int kAhead>
static void launch_rows_as(const GemvBatch& b, dim3 grid, uint32_t spare_lds, uint32_t cols,
                           uint32_t n_tokens, uint32_t n_tiles, const uint8_t* ws, hipStream_t s) {
  const auto kernel = cols % 512u != 0u ? gemm_q8_rows_kernel<W, true, kPairs, kRing, kAhead>
                                        : gemm_q8_rows_kernel<W, false, kPairs, kRing, kAhead>;
  kernel<<<grid, (W + 1) * 64, spare_lds, s>>>(b, cols, n_tokens, n_tiles, ws);
}
template <int W>
static void launch_rows(const GemvBatch& b, uint32_t row_tiles, uint32_t cols, uint32_t n_tokens,
                        uint32_t n_tiles, const uint8_t* ws, hipStream_t s) {
  const dim3 grid(row_tiles, (n_tiles + W - 1u) / W);
  const GemmRowsCut cut = gemm_rows_cut(W, cols, row_tiles, (uint64_t)grid.x * grid.y);
  if constexpr (W <= 2) {
    if (!cut.wide && cut.ahead == 4u)
      return launch_rows_as<W, 4, 3, 4>(b, grid, cut.spare_lds, cols, n_tokens, n_tiles, ws, s);
  }
  if constexpr (W == 1) {
    launch_rows_as<W, 4, 3, 8>(b, grid, cut.spare_lds, cols, n_tokens, n_tiles, ws, s);
  } else {
    if constexpr (W >= 3) {
      if (cut.ahead == 4u)
        return launch_rows_as<W, 8, 2, 4>(b, grid, cut.spare_lds, cols, n_tokens, n_tiles, ws, s);
    }
    launch_rows_as<W, 8, 2, 8>(b, grid, cut.spare_lds, cols, n_tokens, n_tiles, ws, s);
  }
}

hipError_t launch_gemm_q8_mfma(GemvBatch b, uint32_t cols, const float* x, uint32_t n_tokens,
                               void* workspace, hipStream_t s) {
  uint64_t tile_rows = 0, row_tiles_16 = 0;
  for (uint32_t m = 0; m < b.n; ++m) {
    tile_rows += (b.m[m].rows + kTileRows - 1u) / kTileRows;
    row_tiles_16 += (b.m[m].rows + kRowTile - 1u) / kRowTile;
  }
  const bool tiles = gemm_tile_wins(tile_rows, row_tiles_16, cols, n_tokens);
  const uint32_t row_tile = tiles ? kTileRows : kRowTile;
  uint32_t row_tiles = 0;
  for (uint32_t m = 0; m < b.n; ++m) {
    b.m[m].wg0 = row_tiles;
    row_tiles += (b.m[m].rows + row_tile - 1u) / row_tile;
  }
  for (uint32_t m = b.n; m < (uint32_t)kGemvMaxMats; ++m) b.m[m] = b.m[0];
  const uint32_t n_tiles = (n_tokens + 15u) / 16u, token_tiles = (n_tiles + 3u) / 4u;
  const uint32_t act_grid = (uint32_t)(gemm_act_threads(cols, n_tokens) / kActThreads);
  uint8_t* wsp = (uint8_t*)workspace;
  if (tiles)
    q8_act_tile_kernel<false><<<act_grid, kActThreads, 0, s>>>(x, cols, n_tokens, n_tiles, wsp);
  else
    q8_act_tile_kernel<true><<<act_grid, kActThreads, 0, s>>>(x, cols, n_tokens, n_tiles, wsp);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (tiles)
    gemm_q8_tile_kernel<<<(uint32_t)gemm_tile_wgs(row_tiles, n_tokens), kGemmTileThreads, 0, s>>>(
        b, cols, n_tokens, n_tiles, row_tiles, token_tiles, wsp);
  else
    switch (gemm_row_wg_tiles(n_tiles)) {
      case 1: launch_rows<1>(b, row_tiles, cols, n_tokens, n_tiles, wsp, s); break;
      case 2: launch_rows<2>(b, row_tiles, cols, n_tokens, n_tiles, wsp, s); break;
      case 3: launch_rows<3>(b, row_tiles, cols, n_tokens, n_tiles, wsp, s); break;
      default: launch_rows<4>(b, row_tiles, cols, n_tokens, n_tiles, wsp, s);
    }
  return hipGetLastError();
}

}  // namespace fkv
