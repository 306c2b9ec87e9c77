// Float32 products at the bfloat16 rate of the matrix cores, 16 times that of float32: operands split three ways,
// x = x1 + x2 + x3 with x1 the upper 8 mantissa bits, x2 the next 8 and x3 the last 8 (each a bfloat16, whose range is
// that of float32: the sum is exact from 2^-110 on, whatever the other terms of a sum are), and
// x y = x1 y1 + (x1 y2 + x2 y1) + (x1 y3 + x2 y2 + x3 y1) + O(2^-21 x y): six products, exact each, summed in
// float32, i.e. about the accuracy of a float32 product at 6/16 of its cost.
// (Two float16 parts with a scale for all terms of a sum take three products, but hold a term to 2^-37 of the largest
// operand of its row however large its partner is: opposed spreads of 2^20 left no digit.)
//
// The errors of these sums lie to one side, downwards whatever the sign of the sum (measured, sums of 250 007 terms in 128
// parts, normal values: mean -1.07e-6 of the sums' rms, also with all terms negated), and there are six additions a block
// of sixteen terms.  So a stretch of a sum is taken by itself where the registers allow it, the small products first and
// x1 y1 last, and added to the rest by a vector instruction, which rounds to nearest; or every other part is summed with
// its sign turned, so that the errors cancel.
#pragma once
#include "common.h"

namespace e3j_amd {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct Split3 {
    bf16x8 term[3];
};

// the upper halves of two floats side by side; what is left of them
__device__ __forceinline__ uint32_t take_upper(float &x, float &y) {
    const uint32_t a = __float_as_uint(x) & 0xffff0000u, b = __float_as_uint(y) & 0xffff0000u;
    x -= __uint_as_float(a);
    y -= __uint_as_float(b);
    return (a >> 16) | b;
}
// eight floats into their three bfloat16 parts (truncation keeps every part exact)
__device__ __forceinline__ Split3 split3(const float (&x)[8]) {
    Split3 out;
    float rest[8];
#pragma unroll
    for (int m = 0; m < 8; m++) rest[m] = x[m];
#pragma unroll
    for (int t = 0; t < 3; t++) {
        u32x4 packed;
#pragma unroll
        for (int m = 0; m < 8; m += 2) packed[m / 2] = take_upper(rest[m], rest[m + 1]);
        out.term[t] = __builtin_bit_cast(bf16x8, packed);
    }
    return out;
}
// The same with every part rounded to the nearest bfloat16: what is left out of a product is then 2^-26 of it and of
// either sign.  The last bits below the smallest bfloat16, infinities, NaN and what rounds to an infinity do not
// split: `lost` is then not zero.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t take_nearest(float &x, float &y) {
    const uint32_t both = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x, y}, bf16x2));
    x -= __uint_as_float(both << 16);
    y -= __uint_as_float(both & 0xffff0000u);
    return both;
}
__device__ __forceinline__ Split3 split3_nearest(const float (&x)[8], uint32_t &lost) {
    Split3 out;
    float rest[8];
#pragma unroll
    for (int m = 0; m < 8; m++) rest[m] = x[m];
#pragma unroll
    for (int t = 0; t < 3; t++) {
        u32x4 packed;
#pragma unroll
        for (int m = 0; m < 8; m += 2) packed[m / 2] = take_nearest(rest[m], rest[m + 1]);
        out.term[t] = __builtin_bit_cast(bf16x8, packed);
    }
#pragma unroll
    for (int m = 0; m < 8; m++) lost |= __float_as_uint(rest[m]);
    return out;
}
// the partial products, smallest first
constexpr int kPairs[6][2] = {{0, 2}, {1, 1}, {2, 0}, {0, 1}, {1, 0}, {0, 0}};

}  // namespace
}  // namespace e3j_amd
