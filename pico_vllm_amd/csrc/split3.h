// A float32 number as three bfloat16 ones, x = h + m + l exactly: h is x rounded to its upper 8 bits, m what is left of it rounded
// likewise, l what is left then (24 bits in three times 8).  Products of such pieces are exact in float32, so a float32 product
// runs on the bfloat16 matrix instruction, which does 16 times the float32 one's work:
//
//   a w = ah wh  +  (ah wm + am wh)  +  (am wm + ah wl + al wh)  +  (am wl + al wm + al wl)
//
// with the last three, 2^-26 of the product and less, left out: a float32 sum rounds by more at every addition.  The small terms
// are summed apart from ah wh, where their rounding is 2^-8 of its.
//
// bfloat16 has float32's exponents, so the lower pieces of numbers below 2^-110 would end at the smallest number that there is, and a number
// below 2^-134 would have none at all.  Both operands are therefore taken 2^48 times as large, where all of float32's numbers below 2^80 have their
// 24 bits in the pieces, and the sums are scaled back.  A larger number, a sum of 2^32 and more, infinities and NaN make the sum not
// finite.  Such sums are made again in float32 by who uses this (s3_redo).
#pragma once
#include "common.h"

typedef __bf16 s3_bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t s3_u32x4 __attribute__((ext_vector_type(4)));
typedef float s3_f32x16 __attribute__((ext_vector_type(16)));

struct Split8 {
  s3_u32x4 h, m, l;                    // eight numbers' pieces
};

constexpr float S3_SCALE = 0x1p48f, S3_BACK = 0x1p-96f;

// A sum (scaled back) that has to be made again in float32
__device__ __forceinline__ bool s3_redo(float sum) { return !(fabsf(sum) < INFINITY); }

__device__ __forceinline__ float s3_low(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float s3_high(uint32_t p) { return __uint_as_float(p & 0xffff0000u); }

__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  a *= S3_SCALE;
  b *= S3_SCALE;
  h = pack2_bf16(a, b);
  a -= s3_low(h);
  b -= s3_high(h);
  m = pack2_bf16(a, b);
  l = pack2_bf16(a - s3_low(m), b - s3_high(m));
}

template <typename V>                  // V: four floats
__device__ __forceinline__ Split8 split8(const V& a, const V& b) {
  Split8 s;
  uint32_t h, m, l;
  split2(a.x, a.y, h, m, l); s.h[0] = h; s.m[0] = m; s.l[0] = l;
  split2(a.z, a.w, h, m, l); s.h[1] = h; s.m[1] = m; s.l[1] = l;
  split2(b.x, b.y, h, m, l); s.h[2] = h; s.m[2] = m; s.l[2] = l;
  split2(b.z, b.w, h, m, l); s.h[3] = h; s.m[3] = m; s.l[3] = l;
  return s;
}

__device__ __forceinline__ s3_f32x16 mfma16(const s3_u32x4& a, const s3_u32x4& b, const s3_f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(s3_bf16x8, a), __builtin_bit_cast(s3_bf16x8, b), c, 0, 0, 0);
}

// 16 k of a 32 x 32 block: the large terms to `big`, the others to `small`.  EXACT: a's numbers are bfloat16 themselves (m = l = 0).
template <bool EXACT = false>
__device__ __forceinline__ void split_multiply(const Split8& a, const Split8& w, s3_f32x16& big, s3_f32x16& small) {
  if (!EXACT) small = mfma16(a.l, w.h, small);
  small = mfma16(a.h, w.l, small);
  if (!EXACT) small = mfma16(a.m, w.m, small);
  if (!EXACT) small = mfma16(a.m, w.h, small);
  small = mfma16(a.h, w.m, small);
  big = mfma16(a.h, w.h, big);
}
