// Steps of the activation quantiser of the Q8_0 products (GEMV and batched GEMM), one
// Q8Activation::quantize_into value or scale each (crates/kernels/src/q8_dot.rs:35-61).
#pragma once

#include "fkv_device.h"

namespace fkv {
namespace dev {

// amax / 127 correctly rounded for every amax >= 0: q = amax * RN(1/127) corrected
// once by its FMA residual equals the IEEE quotient for all finite amax (checked
// exhaustively over all 2^31 of them); +Inf, where the residual is NaN, maps to +Inf.
__device__ __forceinline__ float div127(float a) {
  const float c = 1.0f / 127.0f;
  const float q = a * c;
  const float r = __builtin_fmaf(-q, 127.0f, a);
  const float q1 = __builtin_fmaf(r, c, q);
  return a == __builtin_inff() ? a : q1;
}

// Rust's round (half away from zero) as trunc(y + copysign(0.5 - 2^-25, y)): equal
// for every f32 y (checked exhaustively over all 2^32).
__device__ __forceinline__ float round_away(float y) {
  return __builtin_truncf(y + __builtin_copysignf(0.49999997f, y));
}

// clamp(round(y) as i32, -128, 127) as a byte. v_cvt_i32_f32 is Rust's `as i32`:
// it saturates and takes NaN to 0 (written as asm: the C++ cast of NaN is undefined).
__device__ __forceinline__ uint32_t q8_byte(float y) {
  int q;
  __asm__("v_cvt_i32_f32 %0, %1" : "=v"(q) : "v"(round_away(y)));
  q = q < -128 ? -128 : (q > 127 ? 127 : q);  // v_med3_i32
  return (uint32_t)q & 0xffu;
}

// binary16 bits of d >= 0 (never NaN), ties away from zero (q8_dot.rs:111-139): the
// round-toward-zero neighbour and the next binary16 up, compared by distance (both
// differences exact near a tie). 65504 < d < 65520 stays 65504; d >= 65520 -> Inf.
__device__ __forceinline__ uint32_t f16_bits_away(float d) {
  auto pk = __builtin_amdgcn_cvt_pkrtz(d, 0.0f);
  const uint32_t lo = __builtin_bit_cast(uint32_t, pk) & 0xffffu;
  const float lo_v = f16_bits_to_f32(lo);
  const float hi_v = (lo == 0x7bffu) ? 65536.0f : f16_bits_to_f32(lo + 1u);
  return (hi_v - d <= d - lo_v) ? lo + 1u : lo;
}

}  // namespace dev
}  // namespace fkv
