// FP32 products on the bf16 matrix cores.
//
// A float is the exact sum of three bf16 values cut from its mantissa 8 bits
// at a time, x = h + m + l (h = x with its low 16 bits cleared, m the same of
// x - h, l the rest; both differences are exact).  A product keeps the six
// terms h h, h m, m h, m m, h l, l h; what is dropped, m l + l m + l l, is
// below 2^-23 of |x y| (2^-25 on average), the size of one f32 rounding.  Each
// term is an exact f32 product inside the MFMA.  On gfx950 a bf16 MFMA does 16
// times the work of the f32 one per cycle, so six of them cost 3/8 of the f32
// instructions they replace.  Infinite and NaN inputs give NaN.
#pragma once

#include "common.hpp"

namespace tpf {

struct Split8 {
  bf16x8 h, m, l;
};
struct Split4 {
  bf16x4 h, m, l;
};

// The upper halves of two floats as a bf16 pair (x0 in the low half).
__device__ __forceinline__ uint32_t hi_pair(float x0, float x1) {
  return __builtin_amdgcn_perm(__float_as_uint(x1), __float_as_uint(x0), 0x07060302u);
}
// (Forming x - h by a dot product with the packed pair, 7 instructions per
// pair instead of 11, measured slower: 208 against 195 us on the attention
// forward at N = 384.)
__device__ __forceinline__ float below_hi(float x) {
  return x - __uint_as_float(__float_as_uint(x) & 0xFFFF0000u);
}
__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t& h, uint32_t& m,
                                           uint32_t& l) {
  h = hi_pair(x0, x1);
  const float r0 = below_hi(x0), r1 = below_hi(x1);
  m = hi_pair(r0, r1);
  l = hi_pair(below_hi(r0), below_hi(r1));
}
__device__ __forceinline__ Split8 split8(const float (&x)[8]) {
  u32x4 h, m, l;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    uint32_t a, b, c;
    split_pair(x[2 * e], x[2 * e + 1], a, b, c);
    h[e] = a;
    m[e] = b;
    l[e] = c;
  }
  return Split8{__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m),
                __builtin_bit_cast(bf16x8, l)};
}
__device__ __forceinline__ Split4 split4(const f32x4& x) {
  u32x2 h, m, l;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    uint32_t a, b, c;
    split_pair(x[2 * e], x[2 * e + 1], a, b, c);
    h[e] = a;
    m[e] = b;
    l[e] = c;
  }
  return Split4{__builtin_bit_cast(bf16x4, h), __builtin_bit_cast(bf16x4, m),
                __builtin_bit_cast(bf16x4, l)};
}

// c + a b, the small terms first.
__device__ __forceinline__ f32x16 mfma32_split(const Split8& a, const Split8& b, f32x16 c) {
  c = mfma32(a.l, b.h, c);
  c = mfma32(a.h, b.l, c);
  c = mfma32(a.m, b.m, c);
  c = mfma32(a.m, b.h, c);
  c = mfma32(a.h, b.m, c);
  return mfma32(a.h, b.h, c);
}

}  // namespace tpf
