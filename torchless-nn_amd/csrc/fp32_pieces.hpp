// fp32 values as three bf16 pieces for the bf16 matrix cores: x = x1 + x2 + x3, each piece the
// rounding of what the pieces before it leave (8 + 8 + 8 significand bits and the signs cover
// fp32's 24, so the split is exact while x3 is representable, |x| >= 2^-110), and
//   a b = a1 b1 + (a1 b2 + a2 b1) + (a1 b3 + a2 b2 + a3 b1) + O(2^-24 a b):
// the three products left out are below half an fp32 ulp of a b. bf16 products are exact and
// accumulate in fp32. An infinity, a NaN or a value that rounds past bf16's largest makes NaN
// sums; pieces of tiny values underflow.
#pragma once

#include "tl_internal.hpp"

namespace tl {

// Two fp32 values -> their bf16 roundings, packed.
__device__ __forceinline__ uint32_t pack_bf2(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
}

// 8 fp32 values -> three 16-byte chunks of bf16 pieces.
__device__ __forceinline__ void split8(const float (&x)[8], uint4& p1, uint4& p2, uint4& p3) {
  uint32_t w1[4], w2[4], w3[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = x[2 * i], b = x[2 * i + 1];
    w1[i] = pack_bf2(a, b);
    const float ra = a - __uint_as_float(w1[i] << 16), rb = b - __uint_as_float(w1[i] & 0xffff0000u);
    w2[i] = pack_bf2(ra, rb);
    const float sa = ra - __uint_as_float(w2[i] << 16), sb = rb - __uint_as_float(w2[i] & 0xffff0000u);
    w3[i] = pack_bf2(sa, sb);
  }
  p1 = make_uint4(w1[0], w1[1], w1[2], w1[3]);
  p2 = make_uint4(w2[0], w2[1], w2[2], w2[3]);
  p3 = make_uint4(w3[0], w3[1], w3[2], w3[3]);
}

// The six products, smallest first: pieces kPieceA[t] of one operand, kPieceB[t] of the other.
constexpr int kPieceA[6] = {2, 1, 0, 1, 0, 0}, kPieceB[6] = {0, 1, 2, 0, 1, 0};

// Whether a sum of such products has to be taken again in fp32: not finite, or so small that
// underflowing pieces could show.
__device__ __forceinline__ bool pieces_doubtful(float v) {
  const float a = fabsf(v);
  return !(a < __builtin_inff()) || (a > 0.f && a < 0x1p-60f);
}

}  // namespace tl
