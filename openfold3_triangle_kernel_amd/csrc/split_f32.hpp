// FP32 products on the bf16 matrix cores, by the three-term bfloat16 splitting
// of Henry, Tang and Heinecke ("Leveraging the bfloat16 Artificial Intelligence
// Datatype For Higher-Precision Computations", ARITH 2019).
//
// A float is the exact sum of three bf16 values, x = h + m + l: h is x rounded
// to nearest, m the rounded x - h, l the rest (both differences are exact and
// l has at most 8 significant bits).  With x in [1, 2) 2^e, |m| <= 2^-8 2^e and
// |l| <= 2^-17 2^e, of either sign.  A product keeps the six terms h h, h m,
// m h, m m, h l, l h; what is dropped, m l + l m + l l, is below 2^-24 |x y|
// (1 + 2^-9), half a unit in the last place of an f32 product, and of either
// sign, so it averages out over a sum.  Each kept term is an exact f32 product
// inside the MFMA, whose sums round within one unit in the last place.
//
// Error against 64 bits in 2^-24 of sum |x y|, rms over 2^18 sums: K = 16
// operands of one sign 0.65 (f32 MFMA: 1.05), close to 1 + 2^-7 0.73 (1.03), of
// both signs 0.21 (0.46); K = 384: 3.3 (4.7), 3.6 (4.9), 0.40 (0.47).  A product
// alone is worse, 0.56 (0.42) and at most 2.4 (1.0).  Parts cut instead of
// rounded all have x's sign: the dropped terms reach 2^-21 of every product,
// one way (3.9 close to 1 + 2^-7 at K = 16), for 2 % less time (197 against
// 201 us for the attention forward at N = 384).  Operands below 2^-109 have
// parts that are subnormal in bf16, which the matrix cores read as zero: an
// error of up to 2^-126 times the other operand.
//
// On gfx950 a bf16 MFMA does 16 times the work of the f32 one per cycle, so
// six of them cost 3/8 of the f32 instructions they replace; the split takes
// 11 VALU instructions per pair of elements.
#pragma once

#include "common.hpp"

namespace tpf {

struct Split8 {
  bf16x8 h, m, l;
};
struct Split4 {
  bf16x4 h, m, l;
};

// Two floats rounded to a bf16 pair (x0 in the low half), and its halves as
// floats.  The pair passes through an asm: left alone, the compiler rounds x0
// a second time for its half (13 instructions per pair).
__device__ __forceinline__ uint32_t bf_pair(float x0, float x1) {
  uint32_t p = __builtin_bit_cast(uint32_t, bf16x2{f2bf(x0), f2bf(x1)});
  asm("" : "+v"(p));
  return p;
}
__device__ __forceinline__ float pair_lo(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float pair_hi(uint32_t p) { return __uint_as_float(p & 0xFFFF0000u); }
// Two floats split.  False where a part is NaN: for a NaN, an infinity, or a
// float above the largest bf16 (h rounds to infinity).
//
// ALL splits those too, so that products are those of f32 arithmetic: an
// infinity is (+-1, 0, +-inf), whose l meets only the other operand's h (of the
// same sign, 0 if the operand is 0: NaN as it should be) and whose h and m
// meet finite parts or the other infinity; a large float takes the largest
// bf16 as h.
template <bool ALL>
__device__ __forceinline__ bool split_pair(float x0, float x1, uint32_t& h, uint32_t& m,
                                           uint32_t& l) {
  if constexpr (ALL) {
    const float big = __uint_as_float(0x7F7F0000u);
    const bool i0 = __builtin_isinf(x0), i1 = __builtin_isinf(x1);
    auto head = [&](float x, bool inf) {
      return inf || fabsf(x) > big ? copysignf(inf ? 1.f : big, x) : x;
    };
    h = bf_pair(head(x0, i0), head(x1, i1));
    const float r0 = i0 ? 0.f : x0 - pair_lo(h), r1 = i1 ? 0.f : x1 - pair_hi(h);
    m = bf_pair(r0, r1);
    l = bf_pair(i0 ? x0 : r0 - pair_lo(m), i1 ? x1 : r1 - pair_hi(m));
    return true;
  } else {
    h = bf_pair(x0, x1);
    x0 -= pair_lo(h);
    x1 -= pair_hi(h);
    m = bf_pair(x0, x1);
    x0 -= pair_lo(m);
    x1 -= pair_hi(m);
    l = bf_pair(x0, x1);
    return !__builtin_isunordered(x0, x1);
  }
}
template <bool ALL = false>
__device__ __forceinline__ Split8 split8(const float (&x)[8], bool* ok = nullptr) {
  u32x4 h, m, l;
  bool good = true;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    uint32_t a, b, c;
    good &= split_pair<ALL>(x[2 * e], x[2 * e + 1], a, b, c);
    h[e] = a;
    m[e] = b;
    l[e] = c;
  }
  if (ok) *ok = good;
  return Split8{__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m),
                __builtin_bit_cast(bf16x8, l)};
}
template <bool ALL = false>
__device__ __forceinline__ Split4 split4(const f32x4& x, bool* ok = nullptr) {
  u32x2 h, m, l;
  bool good = true;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    uint32_t a, b, c;
    good &= split_pair<ALL>(x[2 * e], x[2 * e + 1], a, b, c);
    h[e] = a;
    m[e] = b;
    l[e] = c;
  }
  if (ok) *ok = good;
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
