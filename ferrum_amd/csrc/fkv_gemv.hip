// Q8_0 weight GEMV/GEMM on gfx950: Ferrum's ggml q8_0 x q8_0 product
// (crates/kernels/src/q8_dot.rs:35-109; scalar.rs:84-116,191-204), bit for bit.
//
// Per token the f32 activation row is quantized as Q8Activation::quantize_into
// (q8_dot.rs:35-61): per 32 values amax = max|v| (NaN ignored), d = amax/127,
// id = d != 0 ? 1/d : 0, q = clamp(round_half_away(v * id)), and the scale kept is
// f16(d) through the reference's own ties-away encoder (q8_dot.rs:111-139). Every
// output is then dot_q8_row_q8_act (q8_dot.rs:72-109):
//   acc = 0; for b = 0, 1, ...: acc += f32(sumi_b) * (w_scale_b * x_scale_b)
// where sumi_b is the int32 dot of the two 32-byte runs. The integer dots have no
// rounding, so any order gives the same sumi_b; w_scale * x_scale is exact (two
// binary16 significands fit in 22 bits); f32(sumi_b) * that rounds once, as in the
// reference (no FMA anywhere: -ffp-contract=off); and the f32 sum keeps the
// reference's left-to-right block order through a DPP broadcast chain.
//
// Layout: weights row-major, row r = cols/32 blocks of 34 bytes ([f16 scale LE]
// [32 x i8]) at w + r * (cols/32) * 34 (Ferrum's tensor bytes, dtype.rs:19-21); x is
// [n_tokens][cols] f32, y is [n_tokens][rows] f32 (GemmArgs, par.rs:9-26).
//
// Work split: a workgroup of 4 waves owns 16 consecutive rows of one of the launch's
// matrices (up to four that share the activation), a wave 4 rows, one per 16-lane DPP
// row. Lane l of a row group takes blocks l, l+16, l+32, ... of its
// row, so a 16-block step of the wave reads four runs of 544 contiguous bytes.
// Up to kPipe steps of loads are in flight per wave.
//
// Alignment without realignment: a block is only 2-byte aligned (34 = 2 mod 4), and
// the parity of its address is the same for every step of a lane (16 * 34 = 0 mod
// 4). A lane reads the 8 dwords that start at the first dword boundary of its block
// and the 16-bit word they leave out, and dots those 9 dwords as they are against
// one of two copies of the quantized activation block kept in LDS:
//   block at 2 mod 4: dwords = q0..q31, word = scale -> aligned copy (x0..x31, 0)
//   block at 0 mod 4: dwords = (scale, q0 q1), (q2..q5) ... (q26..q29), word = (q30,
//                     q31) -> copy shifted by two bytes ((0, 0, x0, x1), ..., (x30,
//                     x31, 0, 0)); the scale bytes meet zeros.
// The activation is quantized into LDS by each workgroup; its loads are issued
// before any weight load (loads retire in issue order, so activation loads behind
// a wave's weight prefetch would wait for all of it).
#include <utility>

#include "fkv_device.h"
#include "fkv_gemv_plan.h"
#include "fkv_q8_act.h"

namespace fkv {
namespace {

using dev::div127;
using dev::f16_bits_away;
using dev::q8_byte;

typedef float f32x4a __attribute__((ext_vector_type(4), aligned(4)));

constexpr uint32_t kQ8Bytes = 34;
constexpr int kGemvWaves = 4;
constexpr int kGemvThreads = 64 * kGemvWaves;
constexpr int kRowsPerWave = 4;                             // 16 lanes per row
constexpr uint32_t kRowsPerWg = kGemvRowsPerWg;
static_assert(kRowsPerWg == kGemvWaves * kRowsPerWave, "rows of a workgroup");
constexpr int kPipe = kGemvPipe;
// A (token, block) record in LDS is kGemvXDw dwords: each copy's first 8 dwords are
// 16-byte aligned. The tail pairs trade places in blocks with bit 3 set
// (tail_dw): lanes l and l + 8 read blocks 8 records = 160 dwords apart, a multiple
// of 32 banks, and would otherwise hit the same banks with their 8-byte tail reads.
constexpr uint32_t kXDw = kGemvXDw;
__device__ __forceinline__ uint32_t tail_dw(bool aligned, uint32_t block) {
  const uint32_t swap = (block >> 3) & 1u;
  return aligned ? 16u + 2u * swap : 18u - 2u * swap;
}
// Activation passes (8 values a lane) loaded up front: 2 by default, 4 for two-token
// launches and 8 for one-token launches of more than 4096 columns (measured: more
// passes up front slowed the 3- and 4-token launches).
constexpr int kXRegs = 2;
constexpr int kXRegsWide = 8;

struct RawBlock {
  uint32_t d[8];
  uint32_t tail;
};

typedef unsigned int v4u __attribute__((ext_vector_type(4)));
// Buffer descriptor word 3 for raw 32-bit access on gfx9 (the data format that
// makes out-of-range reads return zero); offsets at or past kOobOffset are out of
// range (the resource never spans more than kOobOffset - 1 bytes).
constexpr int kBufferWord3 = 0x00020000;
constexpr uint32_t kOobOffset = 0x80000000u;

template <int L>
__device__ __forceinline__ float row_bcast(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + L, 0xf, 0xf, true));
}

// acc + p(lane 0) + p(lane 1) + ... + p(lane 15) of this lane's 16-lane row, in that
// order, one rounding per add (one v_add_f32_dpp row_newbcast each).
template <int... L>
__device__ __forceinline__ float chain16(float acc, float p, std::integer_sequence<int, L...>) {
  ((acc = acc + row_bcast<L>(p)), ...);
  return acc;
}

// Activation quantization into LDS. Pass q covers token t = q / C of the launch
// (C = ceil((cols/8) / 256) passes a token), items j = (q % C) * 256 + thread:
// values 8j .. 8j+8 of the token; four consecutive lanes (a quad) own one 32-value
// block. Token and chunk are uniform, so no lane divides.
template <int XR>
struct XRegs {
  f32x4a v[2 * XR];
};

struct XPlan {
  uint32_t per_tok;  // cols / 8 items a token
  uint32_t chunks;   // passes a token
  uint32_t passes;   // nt * chunks
};

// Issues the loads of passes [q0, q0 + XR) (none past the last pass: a uniform
// test). Items past a token's end read its last item (in bounds; never stored).
template <int XR>
__device__ __forceinline__ void load_x(const float* x, uint32_t cols, uint32_t t0,
                                       const XPlan& pl, uint32_t q0, XRegs<XR>& r) {
#pragma unroll
  for (int k = 0; k < XR; ++k) {
    const uint32_t q = q0 + (uint32_t)k;
    if (q >= pl.passes) break;  // uniform
    const uint32_t t = q / pl.chunks, c = q - t * pl.chunks;
    uint32_t j = c * kGemvThreads + threadIdx.x;
    j = j < pl.per_tok ? j : pl.per_tok - 1u;
    const float* src = x + (uint64_t)(t0 + t) * cols + 8u * j;
    r.v[2 * k] = *(const f32x4a*)src;
    r.v[2 * k + 1] = *(const f32x4a*)(src + 4);
  }
}

template <int XR>
__device__ __forceinline__ void quantize_x(const XRegs<XR>& r, uint32_t nb, const XPlan& pl,
                                           uint32_t q0, uint32_t* lds) {
#pragma unroll
  for (int k = 0; k < XR; ++k) {
    const uint32_t q = q0 + (uint32_t)k;
    if (q >= pl.passes) break;  // uniform
    const uint32_t t = q / pl.chunks, c = q - t * pl.chunks;
    const uint32_t j = c * kGemvThreads + threadIdx.x;
    const f32x4a a = r.v[2 * k], b = r.v[2 * k + 1];
    // Rust's max ignores NaN; so does fmaxf (maxnum: a NaN operand, quiet or
    // signaling, yields the other one).
    float m = __builtin_fmaxf(__builtin_fabsf(a.x), __builtin_fabsf(a.y));
    m = __builtin_fmaxf(m, __builtin_fabsf(a.z));
    m = __builtin_fmaxf(m, __builtin_fabsf(a.w));
    m = __builtin_fmaxf(m, __builtin_fabsf(b.x));
    m = __builtin_fmaxf(m, __builtin_fabsf(b.y));
    m = __builtin_fmaxf(m, __builtin_fabsf(b.z));
    m = __builtin_fmaxf(m, __builtin_fabsf(b.w));
    m = __builtin_fmaxf(m, 0.0f);  // all NaN: 0, as the reference's amax = 0 start
    // max over the quad; a quad is entirely below or past per_tok (a multiple of 4)
    m = __builtin_fmaxf(m, dev::dpp<0xB1>(m));
    m = __builtin_fmaxf(m, dev::dpp<0x4E>(m));
    const float d = div127(m);
    const float id = (d != 0.0f) ? 1.0f / d : 0.0f;
    const uint32_t qa = q8_byte(a.x * id) | (q8_byte(a.y * id) << 8) |
                        (q8_byte(a.z * id) << 16) | (q8_byte(a.w * id) << 24);
    const uint32_t qb = q8_byte(b.x * id) | (q8_byte(b.y * id) << 8) |
                        (q8_byte(b.z * id) << 16) | (q8_byte(b.w * id) << 24);
    // the previous lane's qb (quad_perm [0,0,1,2]); nothing before the first lane
    const uint32_t sub = threadIdx.x & 3u;
    uint32_t prev = (uint32_t)__builtin_amdgcn_mov_dpp((int)qb, 0x90, 0xf, 0xf, true);
    prev = sub == 0u ? 0u : prev;
    if (j < pl.per_tok) {
      uint32_t* blk = lds + ((uint64_t)t * nb + j / 4u) * kXDw;
      *(uint2*)(blk + 2u * sub) = make_uint2(qa, qb);
      *(uint2*)(blk + 8u + 2u * sub) = make_uint2(__builtin_amdgcn_alignbit(qa, prev, 16),
                                                  __builtin_amdgcn_alignbit(qb, qa, 16));
      const uint32_t ta = tail_dw(true, j / 4u), ts = tail_dw(false, j / 4u);
      if (sub == 0u) {
        const float xs = dev::f16_bits_to_f32(f16_bits_away(d));
        *(uint2*)(blk + ta) = make_uint2(0u, __float_as_uint(xs));
        blk[ts + 1u] = __float_as_uint(xs);
      }
      if (sub == 3u) blk[ts] = qb >> 16;
    }
  }
}

// Four waves a SIMD (at most 128 VGPRs) keep every wave of a 14336-row matrix
// resident at once, so its weight stream never pauses between rounds of waves.
// S = 2 (launches with few rows): a weight row takes two 16-lane DPP rows, h = 0 the
// even 16-block steps and h = 1 the odd ones, so a wave holds 2 weight rows and the
// launch twice the waves. Each iteration's two steps are added in order by both DPP
// rows (the products of the other one brought over by a lane swap), so the sum is
// the same as S = 1's, bit for bit.
template <int T, int S, int XR>
__global__ __launch_bounds__(kGemvThreads) void gemv_q8_kernel(const GemvBatch bat, uint32_t cols,
                                                               const float* x, uint32_t n_tokens) {
  // This workgroup's matrix (uniform: scalar selects over the launch's few matrices).
  uint32_t mi = 0;
#pragma unroll
  for (int j = 1; j < kGemvMaxMats; ++j)
    if ((uint32_t)j < bat.n && blockIdx.x >= bat.m[j].wg0) mi = (uint32_t)j;
  const GemvMat M = mi == 0u ? bat.m[0] : mi == 1u ? bat.m[1] : mi == 2u ? bat.m[2] : bat.m[3];
  const uint8_t* __restrict__ w = M.w;
  float* __restrict__ y = M.y;
  const uint32_t rows = M.rows;
  const uint32_t wg = blockIdx.x - M.wg0;
  extern __shared__ uint32_t lds[];  // [T][nb][kXDw]
  const uint32_t nb = cols / 32u;
  const uint32_t t0 = blockIdx.y * T;
  const uint32_t nt = n_tokens - t0 < (uint32_t)T ? n_tokens - t0 : (uint32_t)T;

  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t l = lane & 15u;
  const uint32_t h = (lane >> 4) % (uint32_t)S;  // which steps of its row this DPP row takes
  constexpr uint32_t kRowsWg = kRowsPerWg / S;
  const uint32_t row = wg * kRowsWg + wave * (kRowsPerWave / S) + (lane >> 4) / S;
  const bool row_ok = row < rows;
  const uint32_t n_it = (nb + 16u * S - 1u) / (16u * S);  // iterations (S steps) a row
  const uint32_t nbp = gemv_padded_blocks(nb, S);         // LDS blocks a token (whole groups)

  // Weights through a buffer resource based at this workgroup's first row: a lane
  // whose block lies past its row's end asks for an offset beyond the resource, which
  // reads zeros without touching memory. So no load is clamped or branched around,
  // and every step's loads are a lane offset plus an immediate.
  const uint64_t row_bytes = (uint64_t)nb * kQ8Bytes;
  const uint32_t row0 = wg * kRowsWg;
  const uint64_t base = (uint64_t)(uintptr_t)w + row0 * row_bytes;
  const uint64_t left = (uint64_t)rows * row_bytes - row0 * row_bytes;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(uintptr_t)base, (short)0, (int)(left < kOobOffset ? left : kOobOffset - 1u),
      kBufferWord3);
  // A row past the end reads the last row (its results are not stored).
  const uint32_t lane_off = (uint32_t)((uint64_t)((row_ok ? row : rows - 1u) - row0) * row_bytes) +
                            (h * 16u + l) * kQ8Bytes;
  // Which activation copy this lane's blocks pair with (the parity of a lane's block
  // addresses is the same at every step), as LDS dword offsets of its 8 quant dwords
  // and of its (9th dword, scale) pair; and its byte offsets of the 8 dwords and of
  // the 16-bit word.
  const bool aligned = ((base + lane_off) & 2u) != 0u;
  // a step's blocks start at a multiple of 16, so bit 3 of lane l's block is bit 3 of l
  const uint32_t q_dw = aligned ? 0u : 8u, t_dw = tail_dw(aligned, l);
  const uint32_t dw_off = lane_off + (aligned ? 2u : 0u);
  const uint32_t tail_off = lane_off + (aligned ? 0u : 32u);

  XPlan pl;
  pl.per_tok = cols / 8u;
  pl.chunks = (pl.per_tok + kGemvThreads - 1u) / kGemvThreads;
  pl.passes = nt * pl.chunks;
  XRegs<XR> xr;
  load_x<XR>(x, cols, t0, pl, 0, xr);
  // Keep these loads ahead of the weight prefetch: no load moves across an asm
  // statement that may touch memory (x is not __restrict__, so that covers it).
  __asm__ volatile("" ::: "memory");

  // Iteration it's loads: blocks (it*S + h)*16 + l; beyond the row (or the step count)
  // none.
  auto load_step = [&](uint32_t it, RawBlock& rb) {
    const bool in = (it * S + h) * 16u + l < nb;
    const uint32_t o = it * (16u * S * kQ8Bytes);
    const uint32_t od = in ? dw_off + o : kOobOffset;
    const uint32_t ot = in ? tail_off + o : kOobOffset;
    const v4u a = __builtin_amdgcn_raw_buffer_load_b128(rsrc, od, 0, 0);
    const v4u b = __builtin_amdgcn_raw_buffer_load_b128(rsrc, od + 16u, 0, 0);
    rb.d[0] = a[0]; rb.d[1] = a[1]; rb.d[2] = a[2]; rb.d[3] = a[3];
    rb.d[4] = b[0]; rb.d[5] = b[1]; rb.d[6] = b[2]; rb.d[7] = b[3];
    rb.tail = __builtin_amdgcn_raw_buffer_load_b16(rsrc, ot, 0, 0);
  };

  RawBlock buf[kPipe];
#pragma unroll
  for (int k = 0; k < kPipe; ++k) load_step((uint32_t)k, buf[k]);

  quantize_x<XR>(xr, nbp, pl, 0, lds);
  for (uint32_t q0 = XR; q0 < pl.passes; q0 += XR) {
    load_x<XR>(x, cols, t0, pl, q0, xr);
    quantize_x<XR>(xr, nbp, pl, q0, lds);
  }
  __syncthreads();

  float acc[T];
#pragma unroll
  for (int t = 0; t < T; ++t) acc[t] = 0.0f;

  // Step it into acc: lane L's block is the L-th added. Blocks past the row's end
  // (loaded as zeros, paired with LDS padding) add +0: acc starts at +0 and a zero
  // sum is +0 under round-to-nearest, so acc is never -0 and acc + 0 == acc.
  const uint32_t* lane_x = lds + (uint64_t)(h * 16u + l) * kXDw;
  auto consume = [&](uint32_t it, const RawBlock& rb) {
    const bool ok = (it * S + h) * 16u + l < nb;
    const float ws = dev::f16_bits_to_f32(aligned ? rb.tail : rb.d[0]);
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const uint32_t* xb = lane_x + ((uint64_t)t * nbp + it * 16u * S) * kXDw;
      const uint4 x0 = *(const uint4*)(xb + q_dw);
      const uint4 x1 = *(const uint4*)(xb + q_dw + 4u);
      const uint2 xt = *(const uint2*)(xb + t_dw);
      int s = 0;
      s = __builtin_amdgcn_sdot4((int)rb.d[0], (int)x0.x, s, false);
      s = __builtin_amdgcn_sdot4((int)rb.d[1], (int)x0.y, s, false);
      s = __builtin_amdgcn_sdot4((int)rb.d[2], (int)x0.z, s, false);
      s = __builtin_amdgcn_sdot4((int)rb.d[3], (int)x0.w, s, false);
      s = __builtin_amdgcn_sdot4((int)rb.d[4], (int)x1.x, s, false);
      s = __builtin_amdgcn_sdot4((int)rb.d[5], (int)x1.y, s, false);
      s = __builtin_amdgcn_sdot4((int)rb.d[6], (int)x1.z, s, false);
      s = __builtin_amdgcn_sdot4((int)rb.d[7], (int)x1.w, s, false);
      s = __builtin_amdgcn_sdot4((int)rb.tail, (int)xt.x, s, false);
      float p = (float)s * (ws * __uint_as_float(xt.y));
      p = ok ? p : 0.0f;
      if constexpr (S == 1) {
        acc[t] = chain16(acc[t], p, std::make_integer_sequence<int, 16>{});
      } else {
        // this lane's product and the other DPP row's for the same lane index: step
        // it*2 (h = 0's) first, then step it*2 + 1 (h = 1's)
        const float o = __shfl_xor(p, 16);
        const float first = h == 0u ? p : o, second = h == 0u ? o : p;
        acc[t] = chain16(acc[t], first, std::make_integer_sequence<int, 16>{});
        acc[t] = chain16(acc[t], second, std::make_integer_sequence<int, 16>{});
      }
    }
  };

  // Groups of kPipe steps: consume each step, then load the step kPipe ahead into
  // its buffer (loads past the last step read nothing).
  for (uint32_t g = 0; g < n_it; g += kPipe) {
#pragma unroll
    for (int k = 0; k < kPipe; ++k) {
      consume(g + (uint32_t)k, buf[k]);
      load_step(g + (uint32_t)k + kPipe, buf[k]);
    }
  }

  if (row_ok && l == 0u && h == 0u) {
#pragma unroll
    for (int t = 0; t < T; ++t)
      if ((uint32_t)t < nt) y[(uint64_t)(t0 + t) * rows + row] = acc[t];
  }
}

template <int T, int S, int XR = kXRegs>
hipError_t launch_t(const GemvBatch& b, uint32_t n_wg, uint32_t cols, const float* x,
                    uint32_t n_tokens, hipStream_t s) {
  const dim3 grid(n_wg, (n_tokens + T - 1u) / T);
  const size_t lds = gemv_lds_bytes(T, cols, S);
  if (lds > 65536u) {
    const hipError_t e = hipFuncSetAttribute((const void*)gemv_q8_kernel<T, S, XR>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((gemv_q8_kernel<T, S, XR>), grid, dim3(kGemvThreads), lds, s, b, cols, x,
                     n_tokens);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_gemv_q8(GemvBatch b, uint32_t cols, const float* x, uint32_t n_tokens,
                          hipStream_t s) {
  uint32_t n_wg = 0;
  for (uint32_t m = 0; m < b.n; ++m) n_wg += (b.m[m].rows + kRowsPerWg - 1u) / kRowsPerWg;
  const GemvCut cut = gemv_cut(n_tokens, cols, n_wg);
  const uint32_t S = cut.split;
  n_wg = 0;
  for (uint32_t m = 0; m < b.n; ++m) {
    b.m[m].wg0 = n_wg;
    n_wg += (b.m[m].rows + kRowsPerWg / S - 1u) / (kRowsPerWg / S);
  }
  for (uint32_t m = b.n; m < (uint32_t)kGemvMaxMats; ++m) b.m[m] = b.m[0];
  switch (cut.tokens) {
    case 4: return launch_t<4, 1>(b, n_wg, cols, x, n_tokens, s);
    case 2: return launch_t<2, 1, 4>(b, n_wg, cols, x, n_tokens, s);
    default:
      if (cols > 4096u)
        return S == 2u ? launch_t<1, 2, kXRegsWide>(b, n_wg, cols, x, n_tokens, s)
                       : launch_t<1, 1, kXRegsWide>(b, n_wg, cols, x, n_tokens, s);
      return S == 2u ? launch_t<1, 2>(b, n_wg, cols, x, n_tokens, s)
                     : launch_t<1, 1>(b, n_wg, cols, x, n_tokens, s);
  }
}

}  // namespace fkv
