// Decode of the tiled weight's codes into MFMA B fragments, and the fp16
// forms of activations, shared by the kernels that run few activation rows.
#pragma once

#include "../mlq_layout.h"
#include "device_common.h"

namespace mlq {

// Exact fp16 decode of 8 codes of one quarter-block (MFMA B fragment).
template <int QT>
__device__ __forceinline__ h8_t decode8(uint32_t w0, uint32_t w1) {
  uint4 o;
  if (QT == MLQ_Q8_0) {
    const h2_t bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    uint32_t p0, p1, p2, p3;
    q8_pairs(w0, p0, p1);
    q8_pairs(w1, p2, p3);
    o.x = as_u32(as_h2(p0) - bias);
    o.y = as_u32(as_h2(p1) - bias);
    o.z = as_u32(as_h2(p2) - bias);
    o.w = as_u32(as_h2(p3) - bias);
  } else {
    const float lo = QT == MLQ_Q4_0 ? 1032.0f : 1024.0f;
    const float hi = QT == MLQ_Q4_0 ? 72.0f : 64.0f;
    const h2_t blo = {(_Float16)lo, (_Float16)lo};
    const h2_t bhi = {(_Float16)hi, (_Float16)hi};
    const Q4Pairs p = q4_pairs(w0);
    o.x = as_u32(as_h2(p.p0) - blo);
    o.y = as_u32(as_h2(p.p1) - bhi);
    o.z = as_u32(as_h2(p.p2) - blo);
    o.w = as_u32(as_h2(p.p3) - bhi);
  }
  return __builtin_bit_cast(h8_t, o);
}

__device__ __forceinline__ _Float16 half_at(uint2 s, int j) {
  const uint32_t w = (j & 2) ? s.y : s.x;
  return __builtin_bit_cast(_Float16,
                            (uint16_t)((j & 1) ? (w >> 16) : (w & 0xffffu)));
}

__device__ __forceinline__ h2_t splat(uint2 s, int b) {
  const _Float16 v = half_at(s, b);
  return (h2_t){v, v};
}

// The two words of block b's quarter in a unit's line(s): one word (q4) in
// q, two (q8) in q (blocks 0, 1) or q2 (blocks 2, 3).
__device__ __forceinline__ uint32_t q4_word(uint4 q, int b) {
  return b == 0 ? q.x : b == 1 ? q.y : b == 2 ? q.z : q.w;
}
template <int QT>
__device__ __forceinline__ h8_t decode_exact(uint4 q, uint4 q2, int b) {
  if constexpr (QT == MLQ_Q8_0) {
    const uint4 v = b < 2 ? q : q2;
    return decode8<QT>((b & 1) ? v.z : v.x, (b & 1) ? v.w : v.y);
  } else {
    return decode8<QT>(q4_word(q, b), 0u);
  }
}

// B fragment of block b: 8 codes of quarter lane/16 of row lane%16, decoded
// exactly, then scaled by d (q4_1: fused with + m) in fp16, one rounding.
template <int QT>
__device__ __forceinline__ h8_t decode_scaled(uint4 q, uint4 q2, uint2 d, uint2 m, int b) {
  const uint4 c = __builtin_bit_cast(uint4, decode_exact<QT>(q, q2, b));
  const h2_t d2 = splat(d, b);
  uint4 o;
  if constexpr (QT == MLQ_Q4_1) {
    const h2_t m2 = splat(m, b);
    o.x = as_u32(__builtin_elementwise_fma(as_h2(c.x), d2, m2));
    o.y = as_u32(__builtin_elementwise_fma(as_h2(c.y), d2, m2));
    o.z = as_u32(__builtin_elementwise_fma(as_h2(c.z), d2, m2));
    o.w = as_u32(__builtin_elementwise_fma(as_h2(c.w), d2, m2));
  } else {
    o.x = as_u32(as_h2(c.x) * d2);
    o.y = as_u32(as_h2(c.y) * d2);
    o.z = as_u32(as_h2(c.z) * d2);
    o.w = as_u32(as_h2(c.w) * d2);
  }
  return __builtin_bit_cast(h8_t, o);
}

// fp32 pair -> fp16 hi pair + fp16 lo pair with hi + lo = (a, b) to ~2^-22.
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi,
                                       uint32_t& lo) {
  const h2_t h = __builtin_convertvector((f2_t){a, b}, h2_t);
  const h2_t l = __builtin_convertvector(
      (f2_t){a - (float)h.x, b - (float)h.y}, h2_t);
  hi = as_u32(h);
  lo = as_u32(l);
}

// Largest |x| of four values joined to m; NaN propagates (a NaN row's
// output is NaN whatever its scale). Two v_maximum3_f32 with abs modifiers.
__device__ __forceinline__ float abs_maximum4(float m, float4 v) {
  m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, __builtin_fabsf(v.x)),
                                    __builtin_fabsf(v.y));
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, __builtin_fabsf(v.z)),
                                       __builtin_fabsf(v.w));
}

}  // namespace mlq
