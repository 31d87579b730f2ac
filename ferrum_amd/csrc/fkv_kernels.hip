// HIP kernels of the paged KV-cache hot path, written for gfx950 (CDNA4,
// wave64). Host-side validation lives in fkv_api.cpp; every launcher here
// assumes the shapes it is given were checked there.
//
// Reference semantics these kernels implement on the GPU:
//   append        KvPool::append_layer      crates/kvcache/src/pool.rs:122-153
//   gather        KvPool::k / KvPool::v     crates/kvcache/src/pool.rs:174-204
//   f16 decode    f16_to_f32                crates/core-types/src/dtype.rs:135-154
//   Q8_0 encode   Q8Activation::quantize_into crates/kernels/src/q8_dot.rs:46-59
//   attention     forward_one_token loop    crates/model/src/llama.rs:220-247
//   softmax       scalar softmax            crates/kernels/src/scalar.rs:125-141
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fkv_device.h"
#include "fkv_internal.h"

namespace fkv {
namespace {

using namespace dev;

// ---------------------------------------------------------------------------
// Q8_0 block quantiser (q8_dot.rs:46-59)
// ---------------------------------------------------------------------------

// x[32] -> 32 int8 packed in q[8] (little-endian bytes) and the f16 scale bits.
__device__ __forceinline__ uint32_t q8_quantize(const float (&x)[32], int rounding,
                                                uint32_t (&q)[8]) {
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < 32; j++) amax = __builtin_fmaxf(amax, __builtin_fabsf(x[j]));
  float id;
  const float d = q8_scale(amax, id);
#pragma unroll
  for (int w = 0; w < 8; w++) {
    uint32_t packed = 0;
#pragma unroll
    for (int b = 0; b < 4; b++) packed |= ((uint32_t)q8_quant(x[w * 4 + b], id) & 0xffu) << (8 * b);
    q[w] = packed;
  }
  return encode_f16(d, rounding);
}

// ---------------------------------------------------------------------------
// Append (paged KvPool::append_layer)
// ---------------------------------------------------------------------------

// F32 storage, head_dim % 8 == 0, 16-byte aligned k/v: one thread moves 8
// values of one (token, kv, head) row (32 B in, 32 B out).
__global__ void __launch_bounds__(256) append_f32_kernel(Geom g, uint32_t layer,
                                                         const float* __restrict__ k,
                                                         const float* __restrict__ v,
                                                         const int64_t* __restrict__ slots,
                                                         uint32_t n_tokens) {
  const uint32_t cpr = g.head_dim / 8;
  const uint32_t cph = g.n_kv_heads * cpr;
  const uint64_t total = (uint64_t)n_tokens * 2u * cph;
  const uint64_t cap = g.num_blocks * g.block_size;
  for (uint64_t u = (uint64_t)blockIdx.x * 256u + threadIdx.x; u < total;
       u += (uint64_t)gridDim.x * 256u) {
    uint32_t token = (uint32_t)(u / (2u * cph));
    uint32_t rem = (uint32_t)(u % (2u * cph));
    uint32_t kv = rem / cph, r2 = rem % cph, h = r2 / cpr, c = r2 % cpr;
    int64_t slot = slots[token];
    if (slot < 0) continue;
    if ((uint64_t)slot >= cap) {
      if (rem == 0) raise_fault(g.fault, kFaultSlot);
      continue;
    }
    const float* src = (kv ? v : k) + ((uint64_t)token * g.n_kv_heads + h) * g.head_dim + c * 8u;
    uint8_t* tile = tile_ptr(g, (uint64_t)slot / g.block_size, layer, kv, h);
    float4* dst = (float4*)(tile + (((uint64_t)slot % g.block_size) * g.head_dim + c * 8u) * 4u);
    dst[0] = *(const float4*)src;
    dst[1] = *(const float4*)(src + 4);
  }
}

// F16 storage, head_dim % 16 == 0, 16-byte aligned k/v. Workgroups [0, k_groups)
// write K: one thread per 8 dims of a (token, head) row, one 16-byte store into
// run c of the [D/8][B][8] tile. The rest write V into the [D][B] tile: one wave
// per (16 input tokens, head, 16 dims), lane (t, g) holding dims 4g..4g+3 of
// token t, so each 2-byte store instruction fills whole 32-byte dim rows when
// the 16 tokens sit at consecutive offsets of one block (prefill), and is still
// exact for any other slot mapping.
__global__ void __launch_bounds__(256) append_f16_kernel(Geom g, uint32_t layer,
                                                         const float* __restrict__ k,
                                                         const float* __restrict__ v,
                                                         const int64_t* __restrict__ slots,
                                                         uint32_t n_tokens, uint32_t k_groups) {
  const uint32_t D = g.head_dim, Bs = g.block_size;
  const uint64_t cap = g.num_blocks * Bs;
  if (blockIdx.x < k_groups) {
    const uint32_t cpr = D / 8, cph = g.n_kv_heads * cpr;
    const uint64_t u = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (u >= (uint64_t)n_tokens * cph) return;
    const uint32_t token = (uint32_t)(u / cph), r2 = (uint32_t)(u % cph);
    const uint32_t h = r2 / cpr, c = r2 % cpr;
    const int64_t slot = slots[token];
    if (slot < 0) return;
    if ((uint64_t)slot >= cap) {
      if (r2 == 0) raise_fault(g.fault, kFaultSlot);
      return;
    }
    const float* src = k + ((uint64_t)token * g.n_kv_heads + h) * D + c * 8u;
    const float4 a = *(const float4*)src, b = *(const float4*)(src + 4);
    uint8_t* tile = tile_ptr(g, (uint64_t)slot / Bs, layer, 0, h);
    const uint4 w = make_uint4(encode_f16(a.x, g.rounding) | (encode_f16(a.y, g.rounding) << 16),
                               encode_f16(a.z, g.rounding) | (encode_f16(a.w, g.rounding) << 16),
                               encode_f16(b.x, g.rounding) | (encode_f16(b.y, g.rounding) << 16),
                               encode_f16(b.z, g.rounding) | (encode_f16(b.w, g.rounding) << 16));
    *(uint4*)(tile + ((uint64_t)c * Bs + (uint64_t)slot % Bs) * 16u) = w;
    if (f16x2_nonfinite(w.x) || f16x2_nonfinite(w.y) || f16x2_nonfinite(w.z) ||
        f16x2_nonfinite(w.w))
      mark_block(g, (uint64_t)slot / Bs);  // chunked prefill's leak-safe instance reads it
    return;
  }
  const uint32_t dgs = D / 16;  // 16-dim groups per head
  const uint64_t wv = ((uint64_t)(blockIdx.x - k_groups) * 256u + threadIdx.x) / 64u;
  const uint32_t lane = threadIdx.x % 64u, t = lane % 16u, grp = lane / 16u;
  const uint64_t tb = wv / ((uint64_t)g.n_kv_heads * dgs);
  const uint32_t rem = (uint32_t)(wv % ((uint64_t)g.n_kv_heads * dgs));
  const uint32_t h = rem / dgs, dg = rem % dgs;
  const uint64_t token = tb * 16u + t;
  if (token >= n_tokens) return;
  const int64_t slot = slots[token];
  if (slot < 0) return;
  if ((uint64_t)slot >= cap) {
    if (rem == 0 && grp == 0) raise_fault(g.fault, kFaultSlot);
    return;
  }
  const uint32_t d0 = dg * 16u + grp * 4u;
  const float4 x = *(const float4*)(v + (token * g.n_kv_heads + h) * D + d0);
  uint16_t* vt = (uint16_t*)tile_ptr(g, (uint64_t)slot / Bs, layer, 1, h) + (uint64_t)d0 * Bs +
                 (uint64_t)slot % Bs;
  const uint32_t e0 = encode_f16(x.x, g.rounding), e1 = encode_f16(x.y, g.rounding);
  const uint32_t e2 = encode_f16(x.z, g.rounding), e3 = encode_f16(x.w, g.rounding);
  vt[0] = (uint16_t)e0;
  vt[Bs] = (uint16_t)e1;
  vt[2 * Bs] = (uint16_t)e2;
  vt[3 * Bs] = (uint16_t)e3;
  if (f16_nonfinite(e0) || f16_nonfinite(e1) || f16_nonfinite(e2) || f16_nonfinite(e3))
    mark_block(g, (uint64_t)slot / Bs);  // chunked prefill's leak-safe instance reads it
}

// F16 storage, block_size 16, head_dim 64 or 128, 16-byte aligned k/v: one workgroup
// per 16 consecutive input tokens (a window) x 256 / (2 D) KV heads; thread (c, o)
// of a head holds dims 8c .. 8c+7 of window token o, tokens fastest, so a wave's
// loads cover whole 128-byte lines of four token rows.
// - K: the thread's 16-byte run goes to run c of its token's [D/8][16][8] tile;
//   tokens at consecutive slots of one block make a wave's stores contiguous.
// - V: the window's rows are transposed through LDS ([dim][token]); thread (d, hh)
//   then stores tokens 8hh .. 8hh+7 of dim d: one 16-byte store when they sit at
//   offsets 0..7 or 8..15 of one block (the whole half of the tile's row d), else one
//   2-byte store per token (any slot mapping, slots < 0 skipped).
// Encoding and fault rules are append_f16_kernel's, bit for bit.
template <int D>
__global__ void __launch_bounds__(256) append_f16_tile_kernel(Geom g, uint32_t layer,
                                                              const float* __restrict__ k,
                                                              const float* __restrict__ v,
                                                              const int64_t* __restrict__ slots,
                                                              uint32_t n_tokens) {
  constexpr int kRuns = D / 8;           // 8-dim runs of a row
  constexpr int kTph = 16 * kRuns;       // threads per (window, head)
  constexpr int kHpw = 256 / kTph;       // heads per workgroup
  static_assert(kHpw * kTph == 256, "head_dim 64 or 128");
  __shared__ int64_t s_slot[16];
  __shared__ __align__(16) uint16_t s_v[kHpw][D][16];

  const uint32_t hgroups = (g.n_kv_heads + kHpw - 1) / kHpw;
  const uint32_t win = blockIdx.x / hgroups, hg = blockIdx.x % hgroups;
  const uint32_t hl = threadIdx.x / kTph, u = threadIdx.x % kTph;
  const uint32_t h = hg * kHpw + hl;
  const bool head_ok = h < g.n_kv_heads;
  const uint64_t cap = g.num_blocks * 16u;
  if (threadIdx.x < 16) {
    const uint64_t t = (uint64_t)win * 16u + threadIdx.x;
    int64_t sl = t < n_tokens ? slots[t] : -1;
    if (sl >= 0 && (uint64_t)sl >= cap) {
      raise_fault(g.fault, kFaultSlot);
      sl = -1;
    }
    s_slot[threadIdx.x] = sl;
  }
  __syncthreads();

  const uint32_t c = u / 16u, o = u % 16u;
  const int64_t slot = s_slot[o];
  uint32_t ve[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (slot >= 0 && head_ok) {
    const uint64_t row = ((uint64_t)win * 16u + o) * g.n_kv_heads + h;
    const float* ks = k + row * D + c * 8u;
    const float* vs = v + row * D + c * 8u;
    const float4 a = *(const float4*)ks, b = *(const float4*)(ks + 4);
    const float4 x = *(const float4*)vs, y = *(const float4*)(vs + 4);
    uint8_t* kt = tile_ptr(g, (uint64_t)slot / 16u, layer, 0, h);
    const uint4 kw = make_uint4(encode_f16(a.x, g.rounding) | (encode_f16(a.y, g.rounding) << 16),
                                encode_f16(a.z, g.rounding) | (encode_f16(a.w, g.rounding) << 16),
                                encode_f16(b.x, g.rounding) | (encode_f16(b.y, g.rounding) << 16),
                                encode_f16(b.z, g.rounding) | (encode_f16(b.w, g.rounding) << 16));
    *(uint4*)(kt + ((uint64_t)c * 16u + (uint64_t)slot % 16u) * 16u) = kw;
    ve[0] = encode_f16(x.x, g.rounding); ve[1] = encode_f16(x.y, g.rounding);
    ve[2] = encode_f16(x.z, g.rounding); ve[3] = encode_f16(x.w, g.rounding);
    ve[4] = encode_f16(y.x, g.rounding); ve[5] = encode_f16(y.y, g.rounding);
    ve[6] = encode_f16(y.z, g.rounding); ve[7] = encode_f16(y.w, g.rounding);
    bool nf = f16x2_nonfinite(kw.x) || f16x2_nonfinite(kw.y) || f16x2_nonfinite(kw.z) ||
              f16x2_nonfinite(kw.w);
#pragma unroll
    for (int e = 0; e < 8; e++) nf = nf || f16_nonfinite(ve[e]);
    if (nf) mark_block(g, (uint64_t)slot / 16u);  // chunked prefill's leak-safe instance reads it
  }
#pragma unroll
  for (int e = 0; e < 8; e++) s_v[hl][c * 8u + e][o] = (uint16_t)ve[e];
  __syncthreads();

  if (!head_ok) return;
  // V row d of each destination tile. The window's tokens split into segments: maximal
  // runs of consecutive slots inside one 8-aligned group of a block (a whole group when
  // the window is aligned with the blocks, else two or three per group where a sequence
  // begins mid-window). Thread (d, hh) stores the segments that start at its tokens
  // hh*8 .. hh*8+7 with the widest aligned stores the run allows.
  const uint32_t d = u / 2u, hh = u % 2u;
  const uint16_t* vrow = s_v[hl][d];
  for (uint32_t i = hh * 8u; i < hh * 8u + 8u; i++) {
    const int64_t s0 = s_slot[i];
    if (s0 < 0 || (i > 0 && s0 % 8 != 0 && s_slot[i - 1] == s0 - 1)) continue;
    uint32_t len = 1;
    while (i + len < 16u && (s0 + len) % 8 != 0 && s_slot[i + len] == s0 + (int64_t)len) len++;
    uint8_t* row = tile_ptr(g, (uint64_t)s0 / 16u, layer, 1, h) + (uint64_t)d * 32u;
    uint32_t p = (uint32_t)(s0 % 16), j = i;
    const uint32_t end = p + len;
    while (p < end) {
      const uint32_t n = end - p;
      if (p % 8 == 0 && n >= 8) {
        *(uint4*)(row + p * 2u) =
            make_uint4(vrow[j] | ((uint32_t)vrow[j + 1] << 16), vrow[j + 2] | ((uint32_t)vrow[j + 3] << 16),
                       vrow[j + 4] | ((uint32_t)vrow[j + 5] << 16), vrow[j + 6] | ((uint32_t)vrow[j + 7] << 16));
        p += 8; j += 8;
      } else if (p % 4 == 0 && n >= 4) {
        *(uint2*)(row + p * 2u) =
            make_uint2(vrow[j] | ((uint32_t)vrow[j + 1] << 16), vrow[j + 2] | ((uint32_t)vrow[j + 3] << 16));
        p += 4; j += 4;
      } else if (p % 2 == 0 && n >= 2) {
        *(uint32_t*)(row + p * 2u) = vrow[j] | ((uint32_t)vrow[j + 1] << 16);
        p += 2; j += 2;
      } else {
        *(uint16_t*)(row + p * 2u) = vrow[j];
        p += 1; j += 1;
      }
    }
  }
}

// Any head_dim, F32/F16 storage: one element per thread.
__global__ void __launch_bounds__(256) append_scalar_kernel(Geom g, uint32_t layer,
                                                            const float* __restrict__ k,
                                                            const float* __restrict__ v,
                                                            const int64_t* __restrict__ slots,
                                                            uint32_t n_tokens) {
  const uint32_t D = g.head_dim;
  const uint32_t per_kv = g.n_kv_heads * D;
  const uint64_t total = (uint64_t)n_tokens * 2u * per_kv;
  const uint64_t cap = g.num_blocks * g.block_size;
  for (uint64_t u = (uint64_t)blockIdx.x * 256u + threadIdx.x; u < total;
       u += (uint64_t)gridDim.x * 256u) {
    uint32_t token = (uint32_t)(u / (2u * per_kv));
    uint32_t rem = (uint32_t)(u % (2u * per_kv));
    uint32_t kv = rem / per_kv, e = rem % per_kv, h = e / D, d = e % D;
    int64_t slot = slots[token];
    if (slot < 0) continue;
    if ((uint64_t)slot >= cap) {
      if (rem == 0) raise_fault(g.fault, kFaultSlot);
      continue;
    }
    float x = (kv ? v : k)[(uint64_t)token * per_kv + e];
    uint8_t* tile = tile_ptr(g, (uint64_t)slot / g.block_size, layer, kv, h);
    const uint64_t off = (uint64_t)slot % g.block_size;
    if (g.dtype == kDtypeF16) {
      const uint32_t e = encode_f16(x, g.rounding);
      ((uint16_t*)tile)[kv ? (uint64_t)d * g.block_size + off
                           : ((uint64_t)(d / 8) * g.block_size + off) * 8 + d % 8] = (uint16_t)e;
      if (f16_nonfinite(e)) mark_block(g, (uint64_t)slot / g.block_size);
    } else
      ((float*)tile)[off * D + d] = x;
  }
}

// Q8_0 storage: one thread quantises one 32-value run of a (token, kv, head) row.
template <bool kAligned>
__global__ void __launch_bounds__(256) append_q8_kernel(Geom g, uint32_t layer,
                                                        const float* __restrict__ k,
                                                        const float* __restrict__ v,
                                                        const int64_t* __restrict__ slots,
                                                        uint32_t n_tokens) {
  const uint32_t D = g.head_dim, B = g.block_size;
  const uint32_t cpr = D / 32;
  const uint32_t cph = g.n_kv_heads * cpr;
  const uint64_t total = (uint64_t)n_tokens * 2u * cph;
  const uint64_t cap = g.num_blocks * B;
  for (uint64_t u = (uint64_t)blockIdx.x * 256u + threadIdx.x; u < total;
       u += (uint64_t)gridDim.x * 256u) {
    uint32_t token = (uint32_t)(u / (2u * cph));
    uint32_t rem = (uint32_t)(u % (2u * cph));
    uint32_t kv = rem / cph, r2 = rem % cph, h = r2 / cpr, c = r2 % cpr;
    int64_t slot = slots[token];
    if (slot < 0) continue;
    if ((uint64_t)slot >= cap) {
      if (rem == 0) raise_fault(g.fault, kFaultSlot);
      continue;
    }
    const float* src = (kv ? v : k) + ((uint64_t)token * g.n_kv_heads + h) * D + c * 32u;
    float x[32];
    if constexpr (kAligned) {
#pragma unroll
      for (int j = 0; j < 8; j++) {
        float4 t = ((const float4*)src)[j];
        x[4 * j] = t.x; x[4 * j + 1] = t.y; x[4 * j + 2] = t.z; x[4 * j + 3] = t.w;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 32; j++) x[j] = src[j];
    }
    uint32_t q[8];
    uint32_t sc = q8_quantize(x, g.rounding, q);
    uint32_t off = (uint32_t)((uint64_t)slot % B);
    uint8_t* tile = tile_ptr(g, (uint64_t)slot / B, layer, kv, h);
    if (kv == 0) {  // K: dims c*32 + g*8 .. +7 are one 8-byte run per g
#pragma unroll
      for (uint32_t gg = 0; gg < 4; gg++)
        *(uint2*)(tile + q8_quant_offset(0, off, c * 32u + gg * 8u, D)) =
            make_uint2(q[2 * gg], q[2 * gg + 1]);
    } else {  // V: one byte per dim
#pragma unroll
      for (uint32_t j = 0; j < 32; j++)
        tile[q8_quant_offset(1, off, c * 32u + j, D)] = (uint8_t)(q[j / 4] >> (8 * (j % 4)));
    }
    ((uint16_t*)(tile + (uint64_t)B * D))[off * cpr + c] = (uint16_t)sc;
    // A scale of 512 or more marks the block (attention over it takes the exact
    // instance); one past the binary16 range (|x| >= 65520 * 127) is stored as +-inf,
    // as the reference's encoder stores it, and flagged.
    if (q8_wide_scale(sc)) {
      mark_block(g, (uint64_t)slot / B);
      if ((sc & 0x7c00u) == 0x7c00u) raise_fault(g.fault, kFaultRange);
    }
  }
}

// Lanes 0 .. 15 hold the slots of a window's tokens: -1 where a later lane names the same
// slot. Slots that rise from lane to lane hold none, so most windows take one comparison.
template <int N>
__device__ __forceinline__ bool slot_repeats(int64_t sl) {
  if constexpr (N == 16) {
    return false;
  } else {
    const int lo = __builtin_amdgcn_update_dpp(-1, (int)(uint32_t)sl, 0x100 + N, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(-1, (int)(sl >> 32), 0x100 + N, 0xf, 0xf, false);
    const bool same = lo == (int)(uint32_t)sl && hi == (int)(sl >> 32);  // row_shl:N
    return same | slot_repeats<N + 1>(sl);
  }
}
__device__ __forceinline__ int64_t drop_repeated_slot(int64_t sl) {
  const int lo = __builtin_amdgcn_update_dpp(-1, (int)(uint32_t)sl, 0x101, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(-1, (int)(sl >> 32), 0x101, 0xf, 0xf, false);
  const int64_t next = ((int64_t)hi << 32) | (uint32_t)lo;
  if (__ballot(threadIdx.x % 16u != 15u && sl >= next) == 0) return sl;
  return sl >= 0 && slot_repeats<1>(sl) ? -1 : sl;
}

// Q8_0 storage, head_dim 64 or 128, 16-byte aligned k/v: one workgroup per 16
// consecutive tokens x 128 / D KV heads. Bound by HBM: it reads 8 bytes a K/V element
// pair and writes 2 and a scale's share. So loads are coalesced and many: thread
// (token o, run r) takes dims 8r .. 8r + 7 of K and of V, a quad of lanes a Q8_0 block
// (its amax by two DPP steps; the encoding is append_q8_kernel's), and D / 8 lanes a
// whole row. (A thread that quantised 64 dims by itself read 256-byte strips, 64 lines
// an instruction, from 1/4 of the waves.)
// Quants go out through LDS in the tile's operand order. K: a 16-byte unit holds an
// 8-dim run of both blocks of a 64-dim pair for one token. V: one holds dims j, j + 16,
// j + 32, j + 48 of 4 consecutive tokens; for each segment of the window (a maximal run
// of consecutive slots inside one 4-aligned token group) it is stored whole when the
// segment is the whole group and by single bytes otherwise.
// Measured with 8 KV heads of 128 dims, 8,192 tokens (84 MB): 30.6 -> 24.9 us, 3.4 TB/s;
// 24,000 tokens 54.2 -> 49.4 (5.0 TB/s). (Scales stored before the barrier, and repeated
// slots looked for before the rows are asked for: 27.1 and 52.2.)
// A slot named twice in a window goes to the last of its tokens (drop_repeated_slot): its
// scales and quants are stored by different waves.
template <int D>
__global__ void __launch_bounds__(256) append_q8_tile_kernel(Geom g, uint32_t layer,
                                                             const float* __restrict__ k,
                                                             const float* __restrict__ v,
                                                             const int64_t* __restrict__ slots,
                                                             uint32_t n_tokens) {
  constexpr uint32_t kRuns = D / 8;          // threads of a row
  constexpr uint32_t kHpw = 16 / kRuns;      // heads per workgroup
  constexpr uint32_t kPairs = D / 64;        // 64-dim pairs of Q8_0 blocks per row
  constexpr uint32_t kUnits = D / 16;        // K units of a token
  static_assert(kHpw * kRuns == 16, "head_dim 64 or 128");
  constexpr uint32_t cpr = D / 32;
  __shared__ int64_t s_slot[16], s_keep[16];  // and without the repeated ones
  // rows of 16 tokens' K units and of a token's V quants, padded so that the strided
  // side of each transpose meets distinct banks
  __shared__ __align__(16) uint8_t s_k[kHpw][kUnits][16 * 16 + 16];
  __shared__ __align__(16) uint8_t s_v[kHpw][16][D + 4];

  const uint32_t hgroups = (g.n_kv_heads + kHpw - 1) / kHpw;
  const uint32_t win = blockIdx.x / hgroups, hg = blockIdx.x % hgroups;
  const uint32_t r = threadIdx.x % kRuns, o = (threadIdx.x / kRuns) % 16u,
                 hl = threadIdx.x / (16u * kRuns);
  const uint32_t h = hg * kHpw + hl;
  const uint32_t B = g.block_size;
  const uint64_t cap = g.num_blocks * B;
  if (threadIdx.x < 16) {
    const uint64_t t = (uint64_t)win * 16u + threadIdx.x;
    int64_t sl = t < n_tokens ? slots[t] : -1;
    if (sl >= 0 && (uint64_t)sl >= cap) {
      raise_fault(g.fault, kFaultSlot);
      sl = -1;
    }
    s_slot[threadIdx.x] = sl;
  }
  __syncthreads();

  const bool live = s_slot[o] >= 0 && h < g.n_kv_heads;
  float x[2][8] = {};
  if (live) {
    const uint64_t at = (((uint64_t)win * 16u + o) * g.n_kv_heads + h) * D + r * 8u;
#pragma unroll
    for (int kv = 0; kv < 2; kv++) {
      const float4* src = (const float4*)((kv ? v : k) + at);
      const float4 a = src[0], b = src[1];
      x[kv][0] = a.x; x[kv][1] = a.y; x[kv][2] = a.z; x[kv][3] = a.w;
      x[kv][4] = b.x; x[kv][5] = b.y; x[kv][6] = b.z; x[kv][7] = b.w;
    }
  }
  // (while the rows are on their way)
  if (threadIdx.x < 16) s_keep[threadIdx.x] = drop_repeated_slot(s_slot[threadIdx.x]);
  uint32_t sc[2];
#pragma unroll
  for (int kv = 0; kv < 2; kv++) {
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++) amax = __builtin_fmaxf(amax, __builtin_fabsf(x[kv][j]));
    amax = __builtin_fmaxf(amax, dpp<0xB1>(amax));
    amax = __builtin_fmaxf(amax, dpp<0x4E>(amax));
    float id;
    const float d = q8_scale(amax, id);
    uint32_t q[2] = {0, 0};
#pragma unroll
    for (int j = 0; j < 8; j++)
      q[j / 4] |= ((uint32_t)q8_quant(x[kv][j], id) & 0xffu) << (8 * (j % 4));
    sc[kv] = encode_f16(d, g.rounding);
    if (kv == 0) {  // unit (pair r / 8, run r % 4), half of the block
      *(uint2*)&s_k[hl][r / 8u * 4u + r % 4u][o * 16u + (r / 4u) % 2u * 8u] = make_uint2(q[0], q[1]);
    } else {
      uint32_t* dst = (uint32_t*)&s_v[hl][o][r * 8u];
      dst[0] = q[0];
      dst[1] = q[1];
    }
  }
  __syncthreads();

  const int64_t slot = s_keep[o];
  if (slot >= 0 && h < g.n_kv_heads && r % 4u == 0u) {
    const uint64_t blk = (uint64_t)slot / B;
    const uint32_t off = (uint32_t)((uint64_t)slot % B);
#pragma unroll
    for (int kv = 0; kv < 2; kv++) {
      ((uint16_t*)(tile_ptr(g, blk, layer, kv, h) + (uint64_t)B * D))[off * cpr + r / 4u] = (uint16_t)sc[kv];
      // A scale of 512 or more marks the block (attention over it takes the exact
      // instance); one past the binary16 range is stored as +-inf, as the reference's
      // encoder stores it, and flagged.
      if (q8_wide_scale(sc[kv])) {
        mark_block(g, blk);
        if ((sc[kv] & 0x7c00u) == 0x7c00u) raise_fault(g.fault, kFaultRange);
      }
    }
  }

  const uint32_t t = threadIdx.x % 128u;  // 128 units of K (waves 0, 1) and of V (2, 3)
  if (threadIdx.x < 128u) {
    const uint32_t e = t % 16u, un = (t / 16u) % kUnits, uh = t / (16u * kUnits);
    const int64_t sl = s_keep[e];
    if (sl < 0 || hg * kHpw + uh >= g.n_kv_heads) return;
    uint8_t* tile = tile_ptr(g, (uint64_t)sl / B, layer, 0, hg * kHpw + uh);
    *(uint4*)(tile + q8_quant_offset(0, (uint32_t)((uint64_t)sl % B), un / 4u * 64u + un % 4u * 8u, D)) =
        *(const uint4*)&s_k[uh][un][e * 16u];
    return;
  }
  // Segments that start at tokens 4 * part .. + 3 of the window (one of them where the
  // window is a block's slots in order).
  const uint32_t j = t % 16u, part = (t / 16u) % 4u, vi = (t / 64u) % kPairs,
                 vh = t / (64u * kPairs);
  const uint32_t hv = hg * kHpw + vh;
  if (hv >= g.n_kv_heads) return;
  for (uint32_t e0 = 4u * part; e0 < 4u * part + 4u; e0++) {
    const int64_t s0 = s_keep[e0];
    if (s0 < 0 || (e0 > 0 && s0 % 4 != 0 && s_keep[e0 - 1] == s0 - 1)) continue;
    uint32_t len = 1;
    while (e0 + len < 16u && (s0 + len) % 4 != 0 && s_keep[e0 + len] == s0 + (int64_t)len) len++;
    const uint32_t off = (uint32_t)((uint64_t)s0 % B);
    uint8_t* unit = tile_ptr(g, (uint64_t)s0 / B, layer, 1, hv) +
                    (q8_quant_offset(1, off, vi * 64u + j, D) & ~(uint64_t)15);
    const uint8_t* src = &s_v[vh][e0][vi * 64u + j];
    constexpr uint32_t kRow = D + 4;
    if (len == 4) {  // the whole 4-token group: bytes mm*4 + e = token e0+e, dim j + 16mm
      uint32_t w[4];
#pragma unroll
      for (uint32_t mm = 0; mm < 4; mm++)
        w[mm] = (uint32_t)src[16 * mm] | ((uint32_t)src[kRow + 16 * mm] << 8) |
                ((uint32_t)src[2 * kRow + 16 * mm] << 16) | ((uint32_t)src[3 * kRow + 16 * mm] << 24);
      *(uint4*)unit = make_uint4(w[0], w[1], w[2], w[3]);
    } else {
      for (uint32_t e = 0; e < len; e++)
#pragma unroll
        for (uint32_t mm = 0; mm < 4; mm++)
          unit[mm * 4u + (off + e) % 4u] = src[e * kRow + 16 * mm];
    }
  }
}

// ---------------------------------------------------------------------------
// Gather (paged KvPool::k / v): one unit = one (row, kv, head, chunk)
// ---------------------------------------------------------------------------

// Copies/decodes chunk c of the (blk, off, kv, h) row into `dst_row` (the
// output row of head h). Chunk = 8 values (F32/F16) or 32 values (Q8_0).
__device__ __forceinline__ void gather_chunk(const Geom& g, uint32_t layer, uint64_t blk,
                                             uint32_t off, uint32_t kv, uint32_t h,
                                             uint32_t c, int format, uint8_t* dst_row,
                                             bool aligned) {
  const uint32_t D = g.head_dim;
  const uint8_t* tile = tile_ptr(g, blk, layer, kv, h);
  if (g.dtype == kDtypeQ8) {
    uint32_t sc = ((const uint16_t*)(tile + (uint64_t)g.block_size * D))[off * (D / 32u) + c];
    auto qv = [&](uint32_t j) { return tile[q8_quant_offset(kv, off, c * 32u + j, D)]; };
    if (format == 0) {
      float s = f16_bits_to_f32(sc);
      float* o = (float*)dst_row + c * 32u;
      for (uint32_t j = 0; j < 32; j++) o[j] = s * (float)(int8_t)qv(j);
    } else {
      // Ferrum's 34-byte Q8_0 block: f16 scale (LE) then 32 x i8 (dtype.rs:19-21).
      uint16_t* o = (uint16_t*)(dst_row + (uint64_t)c * 34u);
      o[0] = (uint16_t)sc;
      for (uint32_t j = 0; j < 16; j++) o[1 + j] = (uint16_t)(qv(2 * j) | (qv(2 * j + 1) << 8));
    }
    return;
  }
  if (g.dtype == kDtypeF16 && kv == 1) {  // V tile [D][B]: dims are rows
    const uint16_t* src = (const uint16_t*)tile + (uint64_t)c * 8u * g.block_size + off;
    const uint32_t B = g.block_size;
    if (format == 0) {
      float* o = (float*)dst_row + c * 8u;
      for (int j = 0; j < 8; j++) o[j] = f16_bits_to_f32(src[j * B]);
    } else {
      uint16_t* o = (uint16_t*)dst_row + c * 8u;
      for (int j = 0; j < 8; j++) o[j] = src[j * B];
    }
    return;
  }
  if (g.dtype == kDtypeF16) {  // K tile [D/8][B][8]: run c of token off
    const uint16_t* src = (const uint16_t*)tile + ((uint64_t)c * g.block_size + off) * 8u;
    if (format == 0) {
      float* o = (float*)dst_row + c * 8u;
      if (aligned) {
        uint4 w = *(const uint4*)src;
        ((float4*)o)[0] = make_float4(f16_bits_to_f32(w.x & 0xffffu), f16_bits_to_f32(w.x >> 16),
                                      f16_bits_to_f32(w.y & 0xffffu), f16_bits_to_f32(w.y >> 16));
        ((float4*)o)[1] = make_float4(f16_bits_to_f32(w.z & 0xffffu), f16_bits_to_f32(w.z >> 16),
                                      f16_bits_to_f32(w.w & 0xffffu), f16_bits_to_f32(w.w >> 16));
      } else {
        for (int j = 0; j < 8; j++) o[j] = f16_bits_to_f32(src[j]);
      }
    } else {
      uint16_t* o = (uint16_t*)dst_row + c * 8u;
      if (aligned) *(uint4*)o = *(const uint4*)src;
      else for (int j = 0; j < 8; j++) o[j] = src[j];
    }
    return;
  }
  const float* src = (const float*)tile + (uint64_t)off * D + c * 8u;
  float* o = (float*)dst_row + c * 8u;
  if (aligned) {
    ((float4*)o)[0] = ((const float4*)src)[0];
    ((float4*)o)[1] = ((const float4*)src)[1];
  } else {
    for (int j = 0; j < 8; j++) o[j] = src[j];
  }
}

// Output bytes per head row in `format`.
__device__ __forceinline__ uint64_t out_head_bytes(const Geom& g, int format) {
  if (format == 0) return (uint64_t)g.head_dim * 4u;
  if (g.dtype == kDtypeF32) return (uint64_t)g.head_dim * 4u;
  if (g.dtype == kDtypeF16) return (uint64_t)g.head_dim * 2u;
  return (uint64_t)g.head_dim / 32u * 34u;
}

__device__ __forceinline__ uint32_t chunk_values(const Geom& g) {
  return g.dtype == kDtypeQ8 ? 32u : 8u;
}

__global__ void __launch_bounds__(256) gather_slots_kernel(Geom g, uint32_t layer,
                                                           const int64_t* __restrict__ slots,
                                                           uint32_t n_tokens, int format,
                                                           uint8_t* out_k, uint8_t* out_v,
                                                           bool aligned) {
  const uint32_t cpr = g.head_dim / chunk_values(g);
  const uint32_t cph = g.n_kv_heads * cpr;
  const uint64_t total = (uint64_t)n_tokens * 2u * cph;
  const uint64_t cap = g.num_blocks * g.block_size;
  const uint64_t hb = out_head_bytes(g, format);
  for (uint64_t u = (uint64_t)blockIdx.x * 256u + threadIdx.x; u < total;
       u += (uint64_t)gridDim.x * 256u) {
    uint32_t token = (uint32_t)(u / (2u * cph));
    uint32_t rem = (uint32_t)(u % (2u * cph));
    uint32_t kv = rem / cph, r2 = rem % cph, h = r2 / cpr, c = r2 % cpr;
    int64_t slot = slots[token];
    if (slot < 0) continue;
    if ((uint64_t)slot >= cap) {
      if (rem == 0) raise_fault(g.fault, kFaultSlot);
      continue;
    }
    uint8_t* row = (kv ? out_v : out_k) + ((uint64_t)token * g.n_kv_heads + h) * hb;
    gather_chunk(g, layer, (uint64_t)slot / g.block_size,
                 (uint32_t)((uint64_t)slot % g.block_size), kv, h, c, format, row, aligned);
  }
}

// Gather whole sequences through their block tables; blockIdx.y = sequence.
__global__ void __launch_bounds__(256) gather_tables_kernel(
    Geom g, uint32_t layer, const int32_t* __restrict__ tables, uint32_t max_blocks,
    const int32_t* __restrict__ ctx_lens, const int64_t* __restrict__ out_offsets, int format,
    uint8_t* out_k, uint8_t* out_v, bool aligned) {
  const uint32_t seq = blockIdx.y;
  const uint32_t cpr = g.head_dim / chunk_values(g);
  const uint32_t cph = g.n_kv_heads * cpr;
  int32_t ctx = ctx_lens[seq];
  const int32_t cap = (int32_t)(max_blocks * g.block_size);
  if (ctx < 0 || ctx > cap) {
    if (blockIdx.x == 0 && threadIdx.x == 0) raise_fault(g.fault, kFaultCtx);
    ctx = ctx < 0 ? 0 : cap;
  }
  const uint64_t total = (uint64_t)ctx * 2u * cph;
  const uint64_t hb = out_head_bytes(g, format);
  const int64_t base_row = out_offsets[seq];
  for (uint64_t u = (uint64_t)blockIdx.x * 256u + threadIdx.x; u < total;
       u += (uint64_t)gridDim.x * 256u) {
    uint32_t pos = (uint32_t)(u / (2u * cph));
    uint32_t rem = (uint32_t)(u % (2u * cph));
    uint32_t kv = rem / cph, r2 = rem % cph, h = r2 / cpr, c = r2 % cpr;
    int32_t blk = tables[(uint64_t)seq * max_blocks + pos / g.block_size];
    if (blk < 0 || (uint64_t)blk >= g.num_blocks) {
      if (rem == 0) raise_fault(g.fault, kFaultBlock);
      continue;
    }
    uint8_t* row = (kv ? out_v : out_k) + ((uint64_t)(base_row + pos) * g.n_kv_heads + h) * hb;
    gather_chunk(g, layer, (uint64_t)blk, pos % g.block_size, kv, h, c, format, row, aligned);
  }
}

// ---------------------------------------------------------------------------
// Gather, tile path: one workgroup per 16 tokens of one 16-token block x kHpw KV heads
// (block size 16, head_dim 64 or 128, F16 or Q8_0 storage, 16-byte aligned outputs).
// The output rows of the 16 tokens are consecutive (row0 + o for token o), as both
// entry points lay them out: a sequence's positions (by block table) or a window of 16
// slots that are one whole block (by slot).
// ---------------------------------------------------------------------------

// Heads per workgroup: F16 one 16-byte unit of each tile a thread (1 at D = 128, 2 at
// 64); Q8_0 tiles are half the bytes and taken whole, so 4 (8) heads keep as many bytes
// in flight per workgroup (one head a workgroup ran at 43% of a device copy).
constexpr uint32_t gather_heads_per_wg(int dtype, uint32_t d) {
  return dtype == kDtypeF16 ? 256u / (2u * d) : 512u / d;
}

template <int DT, int D>
struct GatherShape {
  static constexpr int kTph = 2 * D;            // F16 threads per (block, head) tile
  static constexpr int kHpw = (int)gather_heads_per_wg(DT, D);
  static constexpr int kTile = DT == kDtypeF16 ? 16 * D * 2 : 16 * D + 16 * (D / 32) * 2;
  static constexpr int kUnits = kTile / 16;     // 16-byte units of a tile
  static constexpr int kVRow = D + 4;           // F16 V transpose row (halves): rows 8 apart
                                                // fall 16 banks apart
};

// Bytes of a Q8_0 workgroup's heads in one output row: kHpw heads of D / 32 34-byte
// blocks, 16 x 34 at head_dim 64 and 128 alike.
constexpr uint32_t kGatherQ8Span = 16u * 34u;

constexpr int kFmtF32 = 0;  // FKV_GATHER_F32
constexpr int kFmtRaw = 1;  // FKV_GATHER_RAW

// LDS of the tile path: F16 the V tiles transposed to [token][dim]; Q8_0 to f32 the K and
// V tile of each head as stored; Q8_0 raw the workgroup's output records
// [kv][token][span], token rows 560 bytes apart and V's 16 bytes past a whole number of
// K's (the stores of one instruction then meet few banks twice).
template <int DT, int D, int FMT>
struct __align__(16) GatherLds {  // 16-byte unit stores into q
  using S = GatherShape<DT, D>;
  static constexpr bool kF16 = DT == kDtypeF16;
  static constexpr bool kRec = DT == kDtypeQ8 && FMT == kFmtRaw;
  static constexpr uint32_t kRecRow = kGatherQ8Span + 16u;
  static constexpr uint32_t kRecKv = 16u * kRecRow + 16u;
  union {
    uint16_t v[kF16 ? S::kHpw : 1][kF16 ? 16 : 1][S::kVRow];
    uint8_t q[DT == kDtypeQ8 && !kRec ? S::kHpw * 2 * S::kTile : 16];
    uint8_t rec[kRec ? 2u * kRecKv : 16u];
  };
  __device__ uint8_t* rec_at(uint32_t kv, uint32_t o, uint32_t b) {
    return rec + kv * kRecKv + o * kRecRow + b;
  }
};

// Stores 8 binary16 values (one 16-byte unit) as FMT requires: RAW the 16 bytes, F32
// the 8 decoded floats (32 bytes).
template <int FMT>
__device__ __forceinline__ void store_f16_unit(uint8_t* dst, uint4 w) {
  if constexpr (FMT == kFmtRaw) {
    *(uint4*)dst = w;
  } else {
    ((float4*)dst)[0] = make_float4(f16_bits_to_f32(w.x & 0xffffu), f16_bits_to_f32(w.x >> 16),
                                    f16_bits_to_f32(w.y & 0xffffu), f16_bits_to_f32(w.y >> 16));
    ((float4*)dst)[1] = make_float4(f16_bits_to_f32(w.z & 0xffffu), f16_bits_to_f32(w.z >> 16),
                                    f16_bits_to_f32(w.w & 0xffffu), f16_bits_to_f32(w.w >> 16));
  }
}

// The value of the quad's lane that kCtrl (a quad_perm) names.
template <int kCtrl>
__device__ __forceinline__ uint32_t quad_lane(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, kCtrl, 0xf, 0xf, true);
}

// One tile group: head hl of the workgroup is KV head h (h_ok false past the last head);
// kt / vt the head's K and V tiles (null when the block's table entry is outside the
// pool: nothing is written); tokens o < n are written to rows row0 + o of out_k / out_v
// (row_bytes apart; head h at h * head_bytes within a row). All 256 threads call this.
template <int DT, int D, int FMT>
__device__ __forceinline__ void gather_tile(GatherLds<DT, D, FMT>& lds, const Geom& g, uint32_t layer,
                                            int64_t blk, uint32_t h0, int32_t n,
                                            uint8_t* out_k, uint8_t* out_v, uint64_t row0) {
  using S = GatherShape<DT, D>;
  constexpr uint64_t kHeadBytes = FMT == kFmtF32 ? (uint64_t)D * 4u
                                  : DT == kDtypeF16      ? (uint64_t)D * 2u
                                                         : (uint64_t)D / 32u * 34u;
  const uint64_t row_bytes = (uint64_t)g.n_kv_heads * kHeadBytes;
  const bool blk_ok = blk >= 0 && (uint64_t)blk < g.num_blocks;
  if constexpr (DT == kDtypeF16) {
    const uint32_t hl = threadIdx.x / S::kTph, u = threadIdx.x % S::kTph;
    const uint32_t h = h0 + hl;
    const bool live = blk_ok && h < g.n_kv_heads;
    uint4 kw = make_uint4(0, 0, 0, 0), vw = make_uint4(0, 0, 0, 0);
    if (live) {
      // unit u of each tile: K run c = u / 16 of token u % 16; V dim u / 2, tokens 8(u % 2) ..
      kw = *(const uint4*)(tile_ptr(g, (uint64_t)blk, layer, 0, h) + (uint64_t)u * 16u);
      vw = *(const uint4*)(tile_ptr(g, (uint64_t)blk, layer, 1, h) + (uint64_t)u * 16u);
    }
    const uint32_t d = u / 2u, t8 = (u % 2u) * 8u;
    const uint32_t vh[8] = {vw.x & 0xffffu, vw.x >> 16, vw.y & 0xffffu, vw.y >> 16,
                            vw.z & 0xffffu, vw.z >> 16, vw.w & 0xffffu, vw.w >> 16};
#pragma unroll
    for (int j = 0; j < 8; j++) lds.v[hl][t8 + j][d] = (uint16_t)vh[j];
    const uint32_t o = u % 16u, c = u / 16u;
    if (live && (int32_t)o < n) {
      const uint64_t off = (row0 + o) * row_bytes + (uint64_t)h * kHeadBytes;
      constexpr uint32_t kUnitOut = FMT == kFmtF32 ? 32u : 16u;
      store_f16_unit<FMT>(out_k + off + (uint64_t)c * kUnitOut, kw);
    }
    __syncthreads();
    if (live && (int32_t)o < n) {
      const uint16_t* r = &lds.v[hl][o][c * 8u];
      const uint4 w = make_uint4(r[0] | ((uint32_t)r[1] << 16), r[2] | ((uint32_t)r[3] << 16),
                                 r[4] | ((uint32_t)r[5] << 16), r[6] | ((uint32_t)r[7] << 16));
      const uint64_t off = (row0 + o) * row_bytes + (uint64_t)h * kHeadBytes;
      constexpr uint32_t kUnitOut = FMT == kFmtF32 ? 32u : 16u;
      store_f16_unit<FMT>(out_v + off + (uint64_t)c * kUnitOut, w);
    }
    __syncthreads();  // the LDS is reused by the caller's next tile group
  } else if constexpr (FMT == kFmtRaw) {
    // Ferrum's 34-byte blocks (dtype.rs:19-21: f16 scale, then 32 x i8). Bound by HBM, so
    // what counts is bytes in flight: every thread loads 2 units of K and 2 of V straight
    // into registers, and LDS holds the output records alone (18 KiB, 8 workgroups a CU;
    // with the tiles staged too it was 37 KiB and 4). The records then go out as whole
    // 16-byte units: a token's heads of the workgroup are one contiguous span of its
    // output row. Blocks start 34 bytes apart, so an even one's quants lie 2 off a dword
    // bound and an odd one's on it.
    // Measured with 8 KV heads of 128 dims, 32,192 tokens of 16 sequences (140 MB): 38.8 ->
    // 30.1 us, 4.65 TB/s.
    constexpr uint32_t kNb = D / 32u;
    constexpr uint32_t kQUnits = S::kHpw * D;       // quant units of the heads' K (V) tiles
    constexpr uint32_t kSUnits = 2u * kNb;          // scale units of a tile
    static_assert(kQUnits == 512u && S::kHpw * 2u * kSUnits == 64u, "units a thread");
    uint4 kw[2] = {}, vw[2] = {}, sw = make_uint4(0, 0, 0, 0);
    const uint32_t s_hl = threadIdx.x / (2u * kSUnits), s_kv = threadIdx.x / kSUnits % 2u,
                   s_un = threadIdx.x % kSUnits;
    if (blk_ok) {
#pragma unroll
      for (uint32_t i = 0; i < 2; i++) {
        const uint32_t un = threadIdx.x + 256u * i, h = h0 + un / D, at = un % D * 16u;
        if (h < g.n_kv_heads) {
          kw[i] = *(const uint4*)(tile_ptr(g, (uint64_t)blk, layer, 0, h) + at);
          vw[i] = *(const uint4*)(tile_ptr(g, (uint64_t)blk, layer, 1, h) + at);
        }
      }
      if (threadIdx.x < 64u && h0 + s_hl < g.n_kv_heads)
        sw = *(const uint4*)(tile_ptr(g, (uint64_t)blk, layer, s_kv, h0 + s_hl) + 16u * D + s_un * 16u);
    }
    // 8 scales a unit, in (token, block) order
    if (threadIdx.x < 64u) {
      const uint32_t w[4] = {sw.x, sw.y, sw.z, sw.w};
#pragma unroll
      for (uint32_t e = 0; e < 8; e++) {
        const uint32_t at = s_un * 8u + e;
        *(uint16_t*)lds.rec_at(s_kv, at / kNb, s_hl * (uint32_t)kHeadBytes + at % kNb * 34u) =
            (uint16_t)(w[e / 2u] >> (16u * (e % 2u)));
      }
    }
#pragma unroll
    for (uint32_t i = 0; i < 2; i++) {
      const uint32_t un = threadIdx.x + 256u * i, p = un % D / 64u;
      const uint32_t head = un / D * (uint32_t)kHeadBytes + 68u * p;  // blocks 2p, 2p + 1
      {  // K unit (run, token): 8 quants of each block
        uint8_t* dst = lds.rec_at(0u, un % 16u, head + 2u + un / 16u % 4u * 8u);
        *(uint16_t*)dst = (uint16_t)kw[i].x;
        *(uint32_t*)(dst + 2) = (kw[i].x >> 16) | (kw[i].y << 16);
        *(uint16_t*)(dst + 6) = (uint16_t)(kw[i].y >> 16);
        ((uint32_t*)(dst + 34))[0] = kw[i].z;
        ((uint32_t*)(dst + 34))[1] = kw[i].w;
      }
      // V unit (token group, dim j): dword mm holds the 4 tokens of dim 16mm + j. A quad of
      // lanes has 4 dims; lane e takes token e's byte from each (4 x 4 byte transpose).
      const uint32_t e = threadIdx.x % 4u;
      uint8_t* dst = lds.rec_at(1u, un / 16u % 4u * 4u + e, head + 2u + un % 16u / 4u * 4u);
      const uint32_t w[4] = {vw[i].x, vw[i].y, vw[i].z, vw[i].w};
      const uint32_t sel = 0x0c0c0400u + e * 0x0101u;  // byte e of both operands
#pragma unroll
      for (uint32_t mm = 0; mm < 4; mm++) {
        const uint32_t l0 = quad_lane<0x00>(w[mm]), l1 = quad_lane<0x55>(w[mm]),
                       l2 = quad_lane<0xAA>(w[mm]), l3 = quad_lane<0xFF>(w[mm]);
        const uint32_t t = __builtin_amdgcn_perm(l1, l0, sel) |
                           (__builtin_amdgcn_perm(l3, l2, sel) << 16);
        uint8_t* to = dst + mm / 2u * 34u + mm % 2u * 16u;
        if (mm < 2u) {
          ((uint16_t*)to)[0] = (uint16_t)t;
          ((uint16_t*)to)[1] = (uint16_t)(t >> 16);
        } else {
          *(uint32_t*)to = t;
        }
      }
    }
    __syncthreads();
    if (blk_ok) {
      // The span of the group's heads that exist, at h0 * kHeadBytes = a multiple of 544
      // bytes into the row: whole 16-byte units where the rows keep that alignment,
      // dwords otherwise (records are dword multiples).
      const uint32_t nh = g.n_kv_heads - h0 < (uint32_t)S::kHpw ? g.n_kv_heads - h0 : (uint32_t)S::kHpw;
      const uint32_t span = nh * (uint32_t)kHeadBytes;
      const uint64_t col0 = (uint64_t)h0 * kHeadBytes;
      auto put = [&](auto unit, uint32_t per) {
        using U = decltype(unit);
        const uint32_t half = (uint32_t)n * per;
        for (uint32_t i = threadIdx.x; i < 2u * half; i += 256u) {
          const uint32_t kv = i >= half ? 1u : 0u, r = i - (kv ? half : 0u);
          const uint32_t o = r / per, u = r % per;
          *(U*)((kv ? out_v : out_k) + (row0 + o) * row_bytes + col0 + u * (uint32_t)sizeof(U)) =
              *(const U*)lds.rec_at(kv, o, u * (uint32_t)sizeof(U));
        }
      };
      if (span == kGatherQ8Span && row_bytes % 16u == 0) put(uint4{}, kGatherQ8Span / 16u);
      else if (span % 16u == 0 && row_bytes % 16u == 0) put(uint4{}, span / 16u);
      else put(uint32_t{}, span / 4u);
    }
    __syncthreads();
  } else {
    // Q8_0 to f32: both tiles of every head to LDS as stored, then each output unit from
    // there.
    for (uint32_t i = threadIdx.x; i < (uint32_t)(S::kHpw * 2 * S::kUnits); i += 256u) {
      const uint32_t hl = i / (2u * S::kUnits), r = i % (2u * S::kUnits);
      const uint32_t kv = r / S::kUnits, un = r % S::kUnits;
      const uint32_t h = h0 + hl;
      if (blk_ok && h < g.n_kv_heads)
        *(uint4*)&lds.q[(hl * 2u + kv) * S::kTile + un * 16u] =
            *(const uint4*)(tile_ptr(g, (uint64_t)blk, layer, kv, h) + (uint64_t)un * 16u);
    }
    __syncthreads();
    if (blk_ok) {
      // f16_to_f32(scale) * (i8 as f32), scalar.rs:268-275: 8 dims a step
      constexpr uint32_t kPer = 2u * 16u * (D / 8u);
      for (uint32_t i = threadIdx.x; i < (uint32_t)S::kHpw * kPer; i += 256u) {
        const uint32_t hl = i / kPer, r = i % kPer;
        const uint32_t kv = r / (16u * (D / 8u)), o = (r / (D / 8u)) % 16u, c8 = r % (D / 8u);
        const uint32_t h = h0 + hl;
        if (h >= g.n_kv_heads || (int32_t)o >= n) continue;
        const uint8_t* t = lds.q + (hl * 2u + kv) * S::kTile;
        const float sc =
            f16_bits_to_f32(*(const uint16_t*)&t[16u * D + (o * (D / 32u) + c8 / 4u) * 2u]);
        float x[8];
#pragma unroll
        for (uint32_t e = 0; e < 8; e++)
          x[e] = sc * (float)(int8_t)t[q8_quant_offset(kv, o, c8 * 8u + e, D)];
        float4* dst = (float4*)((kv ? out_v : out_k) + (row0 + o) * row_bytes +
                                (uint64_t)h * kHeadBytes + c8 * 32u);
        dst[0] = make_float4(x[0], x[1], x[2], x[3]);
        dst[1] = make_float4(x[4], x[5], x[6], x[7]);
      }
    }
    __syncthreads();
  }
}

// By block table: workgroup (x, y) takes sequence y, block x / head_groups of its table
// (positions 16j .. 16j + 15, clamped to the context), head group x % head_groups.
template <int DT, int D, int FMT>
__global__ void __launch_bounds__(256) gather_tables_tile_kernel(
    Geom g, uint32_t layer, const int32_t* __restrict__ tables, uint32_t max_blocks,
    const int32_t* __restrict__ ctx_lens, const int64_t* __restrict__ out_offsets,
    uint8_t* out_k, uint8_t* out_v) {
  using S = GatherShape<DT, D>;
  __shared__ GatherLds<DT, D, FMT> lds;
  const uint32_t hgroups = (g.n_kv_heads + S::kHpw - 1) / S::kHpw;
  const uint32_t seq = blockIdx.y, j = blockIdx.x / hgroups, hg = blockIdx.x % hgroups;
  int32_t ctx = ctx_lens[seq];
  const int32_t cap = (int32_t)(max_blocks * 16u);
  if (ctx < 0 || ctx > cap) {
    if (blockIdx.x == 0 && threadIdx.x == 0) raise_fault(g.fault, kFaultCtx);
    ctx = ctx < 0 ? 0 : cap;
  }
  const int32_t n = ctx - (int32_t)j * 16 < 16 ? ctx - (int32_t)j * 16 : 16;
  if (n <= 0) return;  // uniform over the workgroup
  const int32_t blk = tables[(uint64_t)seq * max_blocks + j];
  if ((blk < 0 || (uint64_t)blk >= g.num_blocks) && hg == 0 && threadIdx.x == 0)
    raise_fault(g.fault, kFaultBlock);
  gather_tile<DT, D, FMT>(lds, g, layer, blk, hg * S::kHpw, n, out_k, out_v,
                          (uint64_t)(out_offsets[seq] + (int64_t)j * 16));
}

// By slot: workgroup x takes input tokens 16w .. 16w + 15 (w = x / head_groups). When
// they are the 16 slots of one block in order (a sequence read block by block) they go
// through the tile path; any other window (a partial or scattered one) takes the
// per-chunk path of gather_slots_kernel for its tokens.
template <int DT, int D, int FMT>
__global__ void __launch_bounds__(256) gather_slots_tile_kernel(
    Geom g, uint32_t layer, const int64_t* __restrict__ slots, uint32_t n_tokens,
    uint8_t* out_k, uint8_t* out_v) {
  using S = GatherShape<DT, D>;
  __shared__ GatherLds<DT, D, FMT> lds;
  __shared__ int32_t s_whole;
  const uint32_t hgroups = (g.n_kv_heads + S::kHpw - 1) / S::kHpw;
  const uint32_t win = blockIdx.x / hgroups, hg = blockIdx.x % hgroups;
  const uint64_t t0 = (uint64_t)win * 16u;
  const uint64_t cap = g.num_blocks * 16u;
  if (threadIdx.x == 0) s_whole = 1;
  __syncthreads();
  if (threadIdx.x < 16) {
    const uint64_t t = t0 + threadIdx.x;
    const int64_t sl = t < n_tokens ? slots[t] : -1;
    const int64_t s0 = t0 < n_tokens ? slots[t0] : -1;
    if (sl < 0 || (uint64_t)sl >= cap || s0 < 0 || s0 % 16 != 0 || sl != s0 + (int64_t)threadIdx.x)
      s_whole = 0;
  }
  __syncthreads();
  if (s_whole) {
    gather_tile<DT, D, FMT>(lds, g, layer, slots[t0] / 16, hg * S::kHpw, 16, out_k, out_v, t0);
    return;
  }
  constexpr uint32_t kCv = DT == kDtypeQ8 ? 32u : 8u;  // values per chunk
  constexpr uint32_t kCpr = D / kCv;
  constexpr uint64_t kHeadBytes = FMT == kFmtF32 ? (uint64_t)D * 4u
                                  : DT == kDtypeF16      ? (uint64_t)D * 2u
                                                         : (uint64_t)D / 32u * 34u;
  const uint32_t units = 16u * 2u * S::kHpw * kCpr;
  for (uint32_t i = threadIdx.x; i < units; i += 256u) {
    const uint32_t o = i / (2u * S::kHpw * kCpr), r = i % (2u * S::kHpw * kCpr);
    const uint32_t kv = r / (S::kHpw * kCpr), hl = (r / kCpr) % S::kHpw, c = r % kCpr;
    const uint32_t h = hg * S::kHpw + hl;
    const uint64_t t = t0 + o;
    if (t >= n_tokens || h >= g.n_kv_heads) continue;
    const int64_t slot = slots[t];
    if (slot < 0) continue;
    if ((uint64_t)slot >= cap) {
      if (hg == 0 && r == 0) raise_fault(g.fault, kFaultSlot);
      continue;
    }
    uint8_t* row = (kv ? out_v : out_k) + (t * g.n_kv_heads + h) * kHeadBytes;
    gather_chunk(g, layer, (uint64_t)slot / 16u, (uint32_t)((uint64_t)slot % 16u), kv, h, c, FMT,
                 row, true);
  }
}

// ---------------------------------------------------------------------------
// copy_blocks / fill / device copy
// ---------------------------------------------------------------------------

// Native clang vector (the nontemporal builtins do not take HIP's uint4 struct).
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kCopyUnroll = 4;
constexpr uint64_t kCopyChunkVecs = 256u * kCopyUnroll;  // 16 KiB per workgroup step

__global__ void __launch_bounds__(256) copy_blocks_kernel(Geom g, const int64_t* __restrict__ pairs,
                                                          uint32_t n_pairs) {
  const uint64_t vecs = g.block_bytes / 16u;
  const uint64_t cpb = (vecs + kCopyChunkVecs - 1) / kCopyChunkVecs;
  const uint64_t total = (uint64_t)n_pairs * cpb;
  for (uint64_t w = blockIdx.x; w < total; w += gridDim.x) {
    uint64_t pr = w / cpb, ch = w % cpb;
    int64_t src = pairs[2 * pr], dst = pairs[2 * pr + 1];
    if (src < 0 || dst < 0 || (uint64_t)src >= g.num_blocks || (uint64_t)dst >= g.num_blocks) {
      if (ch == 0 && threadIdx.x == 0) raise_fault(g.fault, kFaultBlock);
      continue;
    }
    if (ch == 0 && threadIdx.x == 0) {  // the block's mark goes with its bytes
      const uint32_t m = g.bmark[src] ? 1u : 0u;
      const uint32_t old = atomicExch(g.bmark + dst, m);
      if (m != (old ? 1u : 0u)) atomicAdd(g.fault + 1, m ? 1u : 0xffffffffu);
    }
    const u32x4* s = (const u32x4*)(g.base + (uint64_t)src * g.block_bytes);
    u32x4* d = (u32x4*)(g.base + (uint64_t)dst * g.block_bytes);
    uint64_t i0 = ch * kCopyChunkVecs + threadIdx.x;
    u32x4 r[kCopyUnroll];
#pragma unroll
    for (uint32_t j = 0; j < kCopyUnroll; j++) {
      uint64_t i = i0 + j * 256u;
      if (i < vecs) r[j] = __builtin_nontemporal_load(s + i);
    }
#pragma unroll
    for (uint32_t j = 0; j < kCopyUnroll; j++) {
      uint64_t i = i0 + j * 256u;
      if (i < vecs) __builtin_nontemporal_store(r[j], d + i);
    }
  }
}

// Every device block's mark = m, and the count of marked blocks with it.
__global__ void __launch_bounds__(256) marks_fill_kernel(Geom g, uint32_t m) {
  for (uint64_t b = (uint64_t)blockIdx.x * 256u + threadIdx.x; b < g.num_blocks;
       b += (uint64_t)gridDim.x * 256u)
    g.bmark[b] = m;
  if (blockIdx.x == 0 && threadIdx.x == 0) g.fault[1] = m ? (uint32_t)g.num_blocks : 0u;
}

// swap_out (out): host block p.host[i] takes device block p.dev[i]'s mark; swap_in: the
// reverse, keeping the count of marked device blocks.
__global__ void __launch_bounds__(256) marks_swap_kernel(Geom g, MarkPairs p, bool out) {
  const uint32_t i = threadIdx.x;
  if (i >= p.n) return;
  if (out) {
    g.hmark[p.host[i]] = g.bmark[p.dev[i]] ? 1u : 0u;
  } else {
    const uint32_t m = g.hmark[p.host[i]] ? 1u : 0u;
    const uint32_t old = atomicExch(g.bmark + p.dev[i], m);
    if (m != (old ? 1u : 0u)) atomicAdd(g.fault + 1, m ? 1u : 0xffffffffu);
  }
}

__global__ void __launch_bounds__(256) marks_apply_kernel(Geom g, uint64_t first, uint64_t n,
                                                          const uint8_t* __restrict__ ops) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * 256u) {
    if (ops[i] == 0) continue;
    const uint32_t m = ops[i] == 1 ? 1u : 0u;
    const uint32_t old = atomicExch(g.bmark + first + i, m);
    if (m != (old ? 1u : 0u)) atomicAdd(g.fault + 1, m ? 1u : 0xffffffffu);
  }
}

__global__ void __launch_bounds__(256) fill_kernel(uint8_t* dst, uint32_t word, uint64_t bytes) {
  const uint64_t vecs = bytes / 16u;
  uint4 w = make_uint4(word, word, word, word);
  for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < vecs;
       i += (uint64_t)gridDim.x * 256u)
    ((uint4*)dst)[i] = w;
  uint64_t tail = vecs * 16u + (uint64_t)blockIdx.x * 256u + threadIdx.x;
  if (tail < bytes && blockIdx.x == 0) dst[tail] = (uint8_t)word;
}

__global__ void __launch_bounds__(256) device_copy_kernel(u32x4* __restrict__ dst,
                                                          const u32x4* __restrict__ src,
                                                          uint64_t vecs) {
  for (uint64_t i0 = (uint64_t)blockIdx.x * kCopyChunkVecs + threadIdx.x; i0 < vecs;
       i0 += (uint64_t)gridDim.x * kCopyChunkVecs) {
    u32x4 r[kCopyUnroll];
#pragma unroll
    for (uint32_t j = 0; j < kCopyUnroll; j++) {
      uint64_t i = i0 + j * 256u;
      if (i < vecs) r[j] = __builtin_nontemporal_load(src + i);
    }
#pragma unroll
    for (uint32_t j = 0; j < kCopyUnroll; j++) {
      uint64_t i = i0 + j * 256u;
      if (i < vecs) __builtin_nontemporal_store(r[j], dst + i);
    }
  }
}

__global__ void copy_tail_kernel(uint8_t* dst, const uint8_t* src, uint64_t from, uint64_t bytes) {
  uint64_t i = from + threadIdx.x;
  if (i < bytes) dst[i] = src[i];
}

inline uint32_t grid_for(uint64_t units, uint32_t max_wg = 8192) {
  uint64_t wg = (units + 255) / 256;
  if (wg < 1) wg = 1;
  return (uint32_t)(wg < max_wg ? wg : max_wg);
}

}  // namespace

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------

hipError_t launch_append(const Geom& g, uint32_t layer, const float* k, const float* v,
                         const int64_t* slots, uint32_t n_tokens, hipStream_t s) {
  if (n_tokens == 0) return hipSuccess;
  const bool aligned = ((uintptr_t)k % 16 == 0) && ((uintptr_t)v % 16 == 0);
  if (g.dtype == kDtypeQ8 && (g.head_dim == 64 || g.head_dim == 128) && aligned) {
    const uint32_t hpw = 128u / g.head_dim;
    const uint64_t wgs = ((uint64_t)n_tokens + 15u) / 16u * ((g.n_kv_heads + hpw - 1) / hpw);
    if (wgs > 0x7fffffffull) return hipErrorInvalidValue;
    if (g.head_dim == 128)
      append_q8_tile_kernel<128><<<(uint32_t)wgs, 256, 0, s>>>(g, layer, k, v, slots, n_tokens);
    else
      append_q8_tile_kernel<64><<<(uint32_t)wgs, 256, 0, s>>>(g, layer, k, v, slots, n_tokens);
  } else if (g.dtype == kDtypeQ8) {
    uint64_t units = (uint64_t)n_tokens * 2u * g.n_kv_heads * (g.head_dim / 32u);
    if (aligned)
      append_q8_kernel<true><<<grid_for(units), 256, 0, s>>>(g, layer, k, v, slots, n_tokens);
    else
      append_q8_kernel<false><<<grid_for(units), 256, 0, s>>>(g, layer, k, v, slots, n_tokens);
  } else if (g.dtype == kDtypeF16 && g.block_size == 16 && (g.head_dim == 64 || g.head_dim == 128) &&
             aligned) {
    const uint32_t hpw = gather_heads_per_wg(g.dtype, g.head_dim);
    const uint64_t wgs = ((uint64_t)n_tokens + 15u) / 16u * ((g.n_kv_heads + hpw - 1) / hpw);
    if (wgs > 0x7fffffffull) return hipErrorInvalidValue;
    if (g.head_dim == 128)
      append_f16_tile_kernel<128><<<(uint32_t)wgs, 256, 0, s>>>(g, layer, k, v, slots, n_tokens);
    else
      append_f16_tile_kernel<64><<<(uint32_t)wgs, 256, 0, s>>>(g, layer, k, v, slots, n_tokens);
  } else if (g.dtype == kDtypeF16 && g.head_dim % 16 == 0 && aligned) {
    const uint64_t k_threads = (uint64_t)n_tokens * g.n_kv_heads * (g.head_dim / 8u);
    const uint64_t v_waves =
        ((uint64_t)n_tokens + 15u) / 16u * g.n_kv_heads * (g.head_dim / 16u);
    const uint64_t k_groups = (k_threads + 255u) / 256u, v_groups = (v_waves + 3u) / 4u;
    if (k_groups + v_groups > 0x7fffffffull) return hipErrorInvalidValue;
    append_f16_kernel<<<(uint32_t)(k_groups + v_groups), 256, 0, s>>>(g, layer, k, v, slots,
                                                                      n_tokens, (uint32_t)k_groups);
  } else if (g.dtype == kDtypeF32 && g.head_dim % 8 == 0 && aligned) {
    uint64_t units = (uint64_t)n_tokens * 2u * g.n_kv_heads * (g.head_dim / 8u);
    append_f32_kernel<<<grid_for(units), 256, 0, s>>>(g, layer, k, v, slots, n_tokens);
  } else {
    uint64_t units = (uint64_t)n_tokens * 2u * g.n_kv_heads * g.head_dim;
    append_scalar_kernel<<<grid_for(units), 256, 0, s>>>(g, layer, k, v, slots, n_tokens);
  }
  return hipGetLastError();
}

// The chunked gather path needs head_dim % 8 == 0 (F32/F16); callers with other
// head dims use it through the per-element fallback below.
__global__ void __launch_bounds__(256) gather_slots_scalar_kernel(Geom g, uint32_t layer,
                                                                  const int64_t* __restrict__ slots,
                                                                  uint32_t n_tokens, int format,
                                                                  uint8_t* out_k, uint8_t* out_v) {
  const uint32_t D = g.head_dim;
  const uint32_t per_kv = g.n_kv_heads * D;
  const uint64_t total = (uint64_t)n_tokens * 2u * per_kv;
  const uint64_t cap = g.num_blocks * g.block_size;
  for (uint64_t u = (uint64_t)blockIdx.x * 256u + threadIdx.x; u < total;
       u += (uint64_t)gridDim.x * 256u) {
    uint32_t token = (uint32_t)(u / (2u * per_kv));
    uint32_t rem = (uint32_t)(u % (2u * per_kv));
    uint32_t kv = rem / per_kv, e = rem % per_kv, h = e / D, d = e % D;
    int64_t slot = slots[token];
    if (slot < 0) continue;
    if ((uint64_t)slot >= cap) {
      if (rem == 0) raise_fault(g.fault, kFaultSlot);
      continue;
    }
    const uint8_t* tile = tile_ptr(g, (uint64_t)slot / g.block_size, layer, kv, h);
    const uint64_t off = (uint64_t)slot % g.block_size;
    uint64_t idx = off * D + d;
    uint8_t* o = kv ? out_v : out_k;
    uint64_t oi = (uint64_t)token * per_kv + e;
    if (g.dtype == kDtypeF16) {
      uint16_t bits = ((const uint16_t*)tile)[kv ? (uint64_t)d * g.block_size + off
                                                 : ((uint64_t)(d / 8) * g.block_size + off) * 8 + d % 8];
      if (format == 0) ((float*)o)[oi] = f16_bits_to_f32(bits);
      else ((uint16_t*)o)[oi] = bits;
    } else {
      ((float*)o)[oi] = ((const float*)tile)[idx];
    }
  }
}

// The tile path's shapes: F16 or Q8_0, block size 16, head_dim 64 or 128, 16-byte
// aligned outputs.
static bool gather_tile_ok(const Geom& g, const void* out_k, const void* out_v) {
  return (g.dtype == kDtypeF16 || g.dtype == kDtypeQ8) && g.block_size == 16 &&
         (g.head_dim == 64 || g.head_dim == 128) && (uintptr_t)out_k % 16 == 0 &&
         (uintptr_t)out_v % 16 == 0;
}

#define FKV_GATHER_TILE_DISPATCH(KERNEL, GRID, ...)                                    \
  do {                                                                                  \
    const bool raw = format == kFmtRaw;                                                 \
    if (g.dtype == kDtypeF16 && g.head_dim == 128) {                                    \
      if (raw) KERNEL<kDtypeF16, 128, kFmtRaw><<<GRID, 256, 0, s>>>(__VA_ARGS__);       \
      else KERNEL<kDtypeF16, 128, kFmtF32><<<GRID, 256, 0, s>>>(__VA_ARGS__);           \
    } else if (g.dtype == kDtypeF16) {                                                  \
      if (raw) KERNEL<kDtypeF16, 64, kFmtRaw><<<GRID, 256, 0, s>>>(__VA_ARGS__);        \
      else KERNEL<kDtypeF16, 64, kFmtF32><<<GRID, 256, 0, s>>>(__VA_ARGS__);            \
    } else if (g.head_dim == 128) {                                                     \
      if (raw) KERNEL<kDtypeQ8, 128, kFmtRaw><<<GRID, 256, 0, s>>>(__VA_ARGS__);        \
      else KERNEL<kDtypeQ8, 128, kFmtF32><<<GRID, 256, 0, s>>>(__VA_ARGS__);            \
    } else {                                                                            \
      if (raw) KERNEL<kDtypeQ8, 64, kFmtRaw><<<GRID, 256, 0, s>>>(__VA_ARGS__);         \
      else KERNEL<kDtypeQ8, 64, kFmtF32><<<GRID, 256, 0, s>>>(__VA_ARGS__);             \
    }                                                                                   \
  } while (0)

hipError_t launch_gather_slots(const Geom& g, uint32_t layer, const int64_t* slots,
                               uint32_t n_tokens, int format, void* out_k, void* out_v,
                               hipStream_t s) {
  if (n_tokens == 0) return hipSuccess;
  if (gather_tile_ok(g, out_k, out_v)) {
    const uint32_t hpw = gather_heads_per_wg(g.dtype, g.head_dim);
    const uint64_t wgs = ((uint64_t)n_tokens + 15u) / 16u * ((g.n_kv_heads + hpw - 1) / hpw);
    if (wgs > 0x7fffffffull) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)wgs);
    FKV_GATHER_TILE_DISPATCH(gather_slots_tile_kernel, grid, g, layer, slots, n_tokens,
                             (uint8_t*)out_k, (uint8_t*)out_v);
    return hipGetLastError();
  }
  if (g.dtype != kDtypeQ8 && g.head_dim % 8 != 0) {
    uint64_t units = (uint64_t)n_tokens * 2u * g.n_kv_heads * g.head_dim;
    gather_slots_scalar_kernel<<<grid_for(units), 256, 0, s>>>(
        g, layer, slots, n_tokens, format, (uint8_t*)out_k, (uint8_t*)out_v);
    return hipGetLastError();
  }
  const bool aligned = ((uintptr_t)out_k % 16 == 0) && ((uintptr_t)out_v % 16 == 0);
  uint32_t cv = g.dtype == kDtypeQ8 ? 32u : 8u;
  uint64_t units = (uint64_t)n_tokens * 2u * g.n_kv_heads * (g.head_dim / cv);
  gather_slots_kernel<<<grid_for(units), 256, 0, s>>>(g, layer, slots, n_tokens, format,
                                                      (uint8_t*)out_k, (uint8_t*)out_v, aligned);
  return hipGetLastError();
}

hipError_t launch_gather_tables(const Geom& g, uint32_t layer, const int32_t* tables,
                                uint32_t max_blocks, const int32_t* ctx_lens,
                                const int64_t* out_offsets, uint32_t n_seqs,
                                uint32_t max_ctx_len, int format, void* out_k, void* out_v,
                                hipStream_t s) {
  if (n_seqs == 0 || max_ctx_len == 0) return hipSuccess;
  if (gather_tile_ok(g, out_k, out_v)) {
    const uint32_t hpw = gather_heads_per_wg(g.dtype, g.head_dim);
    const uint64_t wgs = ((uint64_t)max_ctx_len + 15u) / 16u * ((g.n_kv_heads + hpw - 1) / hpw);
    if (wgs > 0x7fffffffull) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)wgs, n_seqs);
    FKV_GATHER_TILE_DISPATCH(gather_tables_tile_kernel, grid, g, layer, tables, max_blocks,
                             ctx_lens, out_offsets, (uint8_t*)out_k, (uint8_t*)out_v);
    return hipGetLastError();
  }
  const bool aligned = ((uintptr_t)out_k % 16 == 0) && ((uintptr_t)out_v % 16 == 0);
  uint32_t cv = g.dtype == kDtypeQ8 ? 32u : 8u;
  uint64_t units = (uint64_t)max_ctx_len * 2u * g.n_kv_heads * (g.head_dim / cv);
  dim3 grid(grid_for(units, 4096), n_seqs);
  gather_tables_kernel<<<grid, 256, 0, s>>>(g, layer, tables, max_blocks, ctx_lens, out_offsets,
                                            format, (uint8_t*)out_k, (uint8_t*)out_v, aligned);
  return hipGetLastError();
}

hipError_t launch_copy_blocks(const Geom& g, const int64_t* pairs, uint32_t n_pairs,
                              hipStream_t s) {
  if (n_pairs == 0) return hipSuccess;
  uint64_t vecs = g.block_bytes / 16u;
  uint64_t total = (uint64_t)n_pairs * ((vecs + kCopyChunkVecs - 1) / kCopyChunkVecs);
  uint32_t grid = (uint32_t)(total < 16384 ? total : 16384);
  copy_blocks_kernel<<<grid, 256, 0, s>>>(g, pairs, n_pairs);
  return hipGetLastError();
}

// Moves the FKV_FAULT_* word into the staging word fault[3] and clears it in one
// atomic exchange, so a bit that a kernel on another stream raises meanwhile is kept
// for the next read.
__global__ void take_fault_kernel(uint32_t* fault) {
  if (threadIdx.x == 0) fault[3] = atomicExch(fault, 0u);
}

hipError_t launch_take_fault(uint32_t* fault, hipStream_t s) {
  take_fault_kernel<<<1, 64, 0, s>>>(fault);
  return hipGetLastError();
}

hipError_t launch_fill(void* dst, uint8_t byte, uint64_t bytes, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  uint32_t word = 0x01010101u * byte;
  fill_kernel<<<grid_for(bytes / 16 + 1, 16384), 256, 0, s>>>((uint8_t*)dst, word, bytes);
  return hipGetLastError();
}

hipError_t launch_marks_fill(const Geom& g, uint32_t mark, hipStream_t s) {
  marks_fill_kernel<<<grid_for(g.num_blocks, 1024), 256, 0, s>>>(g, mark ? 1u : 0u);
  return hipGetLastError();
}

hipError_t launch_marks_swap(const Geom& g, const MarkPairs& p, bool out, hipStream_t s) {
  if (p.n == 0) return hipSuccess;
  if (p.n > kMarkPairs) return hipErrorInvalidValue;
  marks_swap_kernel<<<1, 256, 0, s>>>(g, p, out);
  return hipGetLastError();
}

hipError_t launch_marks_apply(const Geom& g, uint64_t first, uint64_t n, const uint8_t* ops,
                              hipStream_t s) {
  if (n == 0) return hipSuccess;
  marks_apply_kernel<<<grid_for(n, 1024), 256, 0, s>>>(g, first, n, ops);
  return hipGetLastError();
}

hipError_t launch_device_copy(void* dst, const void* src, uint64_t bytes, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  uint64_t vecs = bytes / 16u;
  if (vecs) {
    uint64_t wg = (vecs + kCopyChunkVecs - 1) / kCopyChunkVecs;
    device_copy_kernel<<<(uint32_t)(wg < 16384 ? wg : 16384), 256, 0, s>>>(
        (u32x4*)dst, (const u32x4*)src, vecs);
  }
  if (bytes % 16)
    copy_tail_kernel<<<1, 64, 0, s>>>((uint8_t*)dst, (const uint8_t*)src, vecs * 16u, bytes);
  return hipGetLastError();
}

}  // namespace fkv
