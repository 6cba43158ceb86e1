// fp32 values as three bf16 pieces for the bf16 matrix cores: x = x1 + x2 + x3, each piece the
// rounding of what the pieces before it leave (8 + 8 + 8 significand bits and the signs cover
// fp32's 24, so the split is exact while x3 is representable, |x| >= 2^-110), and
//   a b = a1 b1 + (a1 b2 + a2 b1) + (a1 b3 + a2 b2 + a3 b1) + O(2^-24 a b):
// the three products left out are below half an fp32 ulp of a b. bf16 products are exact and
// accumulate in fp32. An infinity, a NaN or a value that rounds past bf16's largest makes NaN
// sums.
//
// Pieces below 2^-126 may be lost: up to 2^-125.9 of an element, in absolute terms, which is
// nothing beside ordinary partners but all of a product such as 2^-124 x 2^124. A sum of n
// products whose operands are at most `most` in magnitude is therefore off by less than
// n 2^-125 most, which is below 2^-28 of every sum from n 2^-97 most on. Kernels keep the
// largest magnitude they split (half an instruction per element) and take smaller sums again in
// fp32 (pieces_least, pieces_doubtful). A sum that is exactly 0 (one in some ten million, by
// cancellation, or a row of zeros) has lost something only if one of its operands is tiny
// (pieces_tiny): a product of two others does not underflow.
#pragma once

#include "tl_internal.hpp"

namespace tl {

// Two fp32 values -> their bf16 roundings, packed.
__device__ __forceinline__ uint32_t pack_bf2(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
}

// max(m, |a|, |b|), a quiet NaN among them ignored. In assembly: fmaxf would first quiet each of
// the loaded values, at an instruction each.
__device__ __forceinline__ float max3_abs(float m, float a, float b) {
  float r;
  asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
  return r;
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

// The same, with `most` raised to the largest magnitude among them.
__device__ __forceinline__ void split8(const float (&x)[8], uint4& p1, uint4& p2, uint4& p3, float& most) {
  split8(x, p1, p2, p3);
#pragma unroll
  for (int i = 0; i < 4; ++i) most = max3_abs(most, x[2 * i], x[2 * i + 1]);
}

// The six products, smallest first: pieces kPieceA[t] of one operand, kPieceB[t] of the other.
constexpr int kPieceA[6] = {2, 1, 0, 1, 0, 0}, kPieceB[6] = {0, 1, 2, 0, 1, 0};

// The least magnitude at which a sum of n products is as good as an fp32 one, for operands of at
// most `most` (infinite: none is).
__device__ __forceinline__ float pieces_least(float most, int n) {
  return fmaxf(0x1p-60f, (float)n * (most * 0x1p-96f));
}

// Whether a sum has to be looked at: not finite, or below `least`; if it is not 0, it has to be
// taken again in fp32.
__device__ __forceinline__ bool pieces_doubtful(float v, float least) {
  const float a = fabsf(v);
  return !(a >= least && a < __builtin_inff());
}

// 0 < |x| < 2^-63
__device__ __forceinline__ bool pieces_tiny(float x) {
  return (__float_as_uint(x) << 1) - 1u < (64u << 24) - 1u;
}

}  // namespace tl
