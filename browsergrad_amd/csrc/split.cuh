// float32 products on the bf16 matrix core: every float32 value is the exact
// sum of three bf16 values, x = x1 + x2 + x3 (round to nearest at each step:
// 24 significand bits as 8 + 8 + 8 with signed remainders), and a product is
// taken as x1 y1 + x1 y2 + x2 y1 + x2 y2 + x1 y3 + x3 y1.  |x2| <= 2^-8 |x| and
// |x3| <= 2^-17 |x|, so what is dropped, x2 y3 + x3 y2 + x3 y3, is at most
// 2^-24 |x y| (a unit of float32 rounding, reached near x = y = 1 + 2^-8) and
// below 2^-26 |x y| for 97% of random pairs.  Sums stay in float32 accumulators
// and round once for 8 or 16 terms, which more than makes up for it from five
// terms on.
#pragma once

#include "common.cuh"

namespace bgk {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4s __attribute__((ext_vector_type(4)));

// Operands are split times kSplitScale: the third part of x reaches down to
// 2^-23 |x|, and the last place of any float32, 2^-149, becomes 2^-125, so that
// every part of every finite value is a normal bf16 number.  A sum of products
// comes out times kSplitScale^2.  (Unscaled, values below 2^-109, such as
// softmax tails, cannot be held: kernels that redid their tiles for them took
// 2 to 170 times as long with a single such value in an operand.)  Infinities,
// NaN, values of 2^104 and more and results of 2^80 and more leave sums that are
// not finite; such a tile is redone in float32.
constexpr float kSplitScale = 16777216.f;                // 2^24
constexpr float kSplitUnscale = 1.f / (16777216.f * 16777216.f);  // 2^-48

// Splits two values, already times kSplitScale, into the packed bf16 parts.
__device__ __forceinline__ void split2(float x0, float x1, uint32_t& p1, uint32_t& p2, uint32_t& p3) {
  const f32x2 v = {x0, x1};
  p1 = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  const f32x2 r = {x0 - __uint_as_float(p1 << 16), x1 - __uint_as_float(p1 & 0xffff0000u)};
  p2 = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
  const f32x2 q = {r[0] - __uint_as_float(p2 << 16), r[1] - __uint_as_float(p2 & 0xffff0000u)};
  p3 = __builtin_bit_cast(uint32_t, __builtin_convertvector(q, bf16x2));
}

// Splits eight consecutive values times `scale` (1 or kSplitScale).
__device__ __forceinline__ void split8(const float (&x)[8], float scale, u32x4s& p1, u32x4s& p2, u32x4s& p3) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t a, b, c;
    split2(x[2 * i] * scale, x[2 * i + 1] * scale, a, b, c);
    p1[i] = a;
    p2[i] = b;
    p3[i] = c;
  }
}

// The float32 redo: one 16-deep stage of float32 MFMAs from k-major LDS rows
// (LA and LB floats long; as and bs at the wavefront's first row and column).
template <int LA, int LB, int TM, int TN, typename Acc>
__device__ __forceinline__ void mul_stage_f32(const float* as, const float* bs, Acc (&acc)[TM][TN]) {
  const int l32 = threadIdx.x & 31, hi = (threadIdx.x >> 5) & 1;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    float a[TM], b[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) a[i] = as[(2 * q + hi) * LA + i * 32 + l32];
#pragma unroll
    for (int j = 0; j < TN; ++j) b[j] = bs[(2 * q + hi) * LB + j * 32 + l32];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
  }
}

}  // namespace bgk
