// rqf_split.h -- fp32 products on the bf16 matrix cores.
//
// A float is exactly h + m + l with h, m, l bf16 values: h = bf16(x) to nearest,
// m = bf16(x - h), l = x - h - m, and both differences are exact (24 significant
// bits are three times 8).  With |m| <= 2^-8 |x| and |l| <= 2^-17 |x|, a product
// x y needs hh + hm + mh + mm + hl + lh; the three left out are below
// 2^-24 |x y| together, and of random sign.  bf16 has float's exponents, so the last
// part of a value below 2^-110 would fall under its smallest value: both operands
// are split scaled by 2^16, which covers every normal float, and the sums carry 2^32.
// What is left is a value past 2^111, a sum past 2^95, an infinity or a NaN: the scaled
// sum is infinite or NaN, and the caller then takes the fp32 instructions.
#pragma once

#include "rqf_device.h"

namespace rqf {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr float kFltMax = 3.402823466e38f;
constexpr float kSplitScale = 65536.0f;  // of each operand
constexpr float kSplitUnscale = 1.0f / kSplitScale / kSplitScale;  // of a sum of products

// Eight values as three bf16 operands of an MFMA with 8 k per lane.
struct Split8 {
  u32x4 h, m, l;
};

__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
  f32x2 v;
  v.x = a;
  v.y = b;
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float bf16_lo(uint32_t p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t p) {
  return __builtin_bit_cast(float, p & 0xffff0000u);
}

// Values 2p and 2p + 1.
__device__ __forceinline__ void split_pair(const float (&x)[8], int p, Split8& s) {
  const uint32_t h = pk_bf16(x[2 * p], x[2 * p + 1]);
  float a = x[2 * p] - bf16_lo(h), b = x[2 * p + 1] - bf16_hi(h);
  const uint32_t m = pk_bf16(a, b);
  a -= bf16_lo(m);
  b -= bf16_hi(m);
  s.h[p] = h;
  s.m[p] = m;
  s.l[p] = pk_bf16(a, b);
}
__device__ __forceinline__ void split8_scaled(const float (&x)[8], Split8& s) {
  float y[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) y[j] = kSplitScale * x[j];
#pragma unroll
  for (int p = 0; p < 4; ++p) split_pair(y, p, s);
}

__device__ __forceinline__ v4f mfma_bf16(u32x4 a, u32x4 b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// c + one of the six products of a and b; t = 0..5, the smallest first.
__device__ __forceinline__ v4f mfma_part(int t, const Split8& a, const Split8& b, v4f c) {
  switch (t) {
    case 0: return mfma_bf16(a.l, b.h, c);
    case 1: return mfma_bf16(a.m, b.m, c);
    case 2: return mfma_bf16(a.h, b.l, c);
    case 3: return mfma_bf16(a.m, b.h, c);
    case 4: return mfma_bf16(a.h, b.m, c);
    default: return mfma_bf16(a.h, b.h, c);
  }
}

}  // namespace rqf
