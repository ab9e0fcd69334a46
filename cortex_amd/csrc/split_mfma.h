// split_mfma.h -- float products on the bfloat16 matrix cores, of operands that are held to the last bit.
//
// v_mfma_f32_*_f32 multiplies 157 TFLOP/s, v_mfma_f32_*_bf16 2500.  A float has 24 significant bits, a bfloat16 eight and
// the same range of exponents: x = hi + mid + lo, each piece the rest of the one before it rounded to nearest, holds every
// float exactly, so that
//   a * b = hi hi + (hi mid + mid hi) + (hi lo + mid mid + lo hi) + (mid lo + lo mid + lo lo)
// (the decomposition of Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", 2019).  The last bracket is less than 2^-24 of the product (0.99 of that in the square of
// 1 + 2^-8 - 2^-17, a sixth on average) and is left out: six products in place of one, each exact in the matrix cores' float
// sums.  hi hi is summed apart from the rest, in two accumulators that are added at the end: the rounding errors of the five
// small ones are 2^-8 of the large one's.  A float sum rounds after every product, these once for eight: from two terms on
// that is more than what is left out, and a product by itself is formed from the floats.  Error against 64 bits, relative
// 2-norm over normal operands (k terms; the library's float product in brackets): k 784 1.6e-7 (2.6e-7), 1024 1.9e-7
// (5.7e-7), 4096 4.0e-7 (1.15e-6).
//
// Range.  The pieces of a small float would be denormal and those of the smallest would not be held at all, so operands
// are multiplied by 2^16 on the way in (any float, denormals included, is then a multiple of 2^-133, the least bfloat16)
// and sums by 2^-32 on the way out.  Pieces below 2^-126 remain, of floats below about 2^-118: neither the conversion nor
// v_dot2_f32_bf16 nor the matrix cores flush them.  A float of 2^112 or more, an infinity or a NaN becomes an infinity or a
// NaN in its row's or column's sums (an infinity's rest is NaN), and so does a result of 2^96 or more: a block that finds one
// in its sums forms them again from the floats themselves, on v_mfma_f32_32x32x2_f32, and stores that.
#pragma once

#include "common.h"

namespace cthip {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kSplitScale = 65536.f;
constexpr float kSplitUnscale = 1.f / (kSplitScale * kSplitScale);
constexpr int kSplitPieces = 3;
// The six products, smallest first: piece kSplitLeft[i] of the left operand by piece kSplitRight[i] of the right one.
constexpr int kSplitProducts = 6;
constexpr int kSplitLeft[kSplitProducts] = {0, 2, 1, 0, 1, 0};
constexpr int kSplitRight[kSplitProducts] = {2, 0, 1, 1, 0, 0};

// The weights {-1, 0} and {0, -1}, in registers: as an inline constant -1.0 stands for the upper half alone.
struct SplitWeights {
  bf16x2 low, high;
  __device__ __forceinline__ SplitWeights() {
    uint32_t l = 0x0000bf80u, h = 0xbf800000u;
    asm("" : "+s"(l));
    asm("" : "+s"(h));
    low = __builtin_bit_cast(bf16x2, l);
    high = __builtin_bit_cast(bf16x2, h);
  }
};

__device__ __forceinline__ uint32_t round_to_bf16(float a, float b) {
  bf16x2 v;
  v[0] = (__bf16)a;
  v[1] = (__bf16)b;
  return __builtin_bit_cast(uint32_t, v);
}

// Four floats as elements at .. at + 3 of eight of each piece.  v_dot2_f32_bf16 takes a rounded pair's half off the float it
// came from in one instruction (shift or mask, and subtract, are two: 6.5 in place of 4.5 vector instructions a float); the
// difference of a float and its rounding is exact.
__device__ __forceinline__ void split4(f32x4 x, u32x4 (&pieces)[kSplitPieces], int at, const SplitWeights& w) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    float a = x[2 * i] * kSplitScale, b = x[2 * i + 1] * kSplitScale;
#pragma unroll
    for (int p = 0; p < kSplitPieces; ++p) {
      const uint32_t pair = round_to_bf16(a, b);
      pieces[p][at / 2 + i] = pair;
      if (p + 1 < kSplitPieces) {
        a = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), w.low, a, false);
        b = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), w.high, b, false);
      }
    }
  }
}

__device__ __forceinline__ f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.f;
  return z;
}

__device__ __forceinline__ bool not_finite(float x) { return (__builtin_bit_cast(uint32_t, x) & 0x7f800000u) == 0x7f800000u; }

}  // namespace cthip
