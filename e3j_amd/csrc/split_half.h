// Float32 products at the half-precision rate of the matrix cores, 16 times that of float32: operands scaled by powers
// of two into the range of float16 and split two ways, x 2^k = hi + lo with 11 bits each and lo signed, so that the
// last bit of x is lost at most (2^-23 of x, for one value in four), and x y = hi hi + (hi lo + lo hi) + O(2^-22 x y):
// three products, exact each, summed in float32, at 3/16 of the cost of a float32 product.  With a scale for all terms
// of a sum the largest of them lies in [2^12, 2^15], and what another one loses at the lower end of the range is
// 2^-37 of the largest or less.
#pragma once
#include "common.h"

namespace e3j_amd {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
constexpr int kScaleTop = 125;         // the largest exponent of a scale; also that of a sum without terms
constexpr float kScaledMax = 32768.f;  // a scaled term above this asks for a smaller scale

struct Split2 {
    f16x8 term[2];
};
__device__ __forceinline__ float pow2(int k) { return __uint_as_float((uint32_t)(k + 127) << 23); }
// the exponent that takes a largest term of m to [2^12, 2^13)
__device__ __forceinline__ int scale_exponent(float m) {
    const int k = 139 - (int)((__float_as_uint(m) >> 23) & 255u);
    return k < kScaleTop ? k : kScaleTop;
}
__device__ __forceinline__ Split2 split2(const float (&x)[8], float scale) {
    Split2 out;
#pragma unroll
    for (int m = 0; m < 8; m++) {
        const _Float16 hi = (_Float16)(x[m] * scale);
        out.term[0][m] = hi;
        out.term[1][m] = (_Float16)__builtin_fmaf(x[m], scale, -(float)hi);
    }
    return out;
}
__device__ __forceinline__ float max_abs(const float (&x)[8]) {
    float m = fabsf(x[0]);
#pragma unroll
    for (int i = 1; i < 8; i++) m = fmaxf(m, fabsf(x[i]));
    return m;
}
// the partial products, smallest first
constexpr int kPairs[3][2] = {{0, 1}, {1, 0}, {0, 0}};

}  // namespace
}  // namespace e3j_amd
