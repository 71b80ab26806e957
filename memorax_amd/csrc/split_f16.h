// A float32 value as the sum of two float16 ones, for products on the float16 matrix units.
//
// The matrix units multiply float32 at a sixteenth of the float16 rate.  A value scaled by a power of two so that the largest of its row (or
// column) lies far up in float16's range is hi + lo with |x - hi - lo| <= 2^-23 |x|, and
//     x y = hi hi' + hi lo' + lo hi'   up to 2^-22 |x y|, zero on average,
// every product exact and every sum in float32: three products in the time of three sixteenths of a float32 one.  An inner product of n terms
// rounds its running sum n / 16 times instead of n / 4 times or more, which is what a float32 product's error is made of.  Error against float64 (2-norm,
// normal operands) here / the array library's float32 products, by terms: 64 0.77e-7 / 1.06e-7, 128 0.88e-7 / 1.51e-7, 256 1.03e-7 / 2.07e-7, 512
// 1.31e-7 / 2.9e-7, 2056 in four layers 3.3e-7 / 5.0e-7; sums over 32768 rows 2.6e-7 / 8.1e-7.  Values below 2^-16 of their row's (column's)
// largest keep an absolute error of 2^-39 of that.
#pragma once
#include "common.h"

namespace mrx {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float sf32x4 __attribute__((ext_vector_type(4)));

struct Split4 {
    f16x4 hi, lo;
};
__device__ __forceinline__ Split4 split4(sf32x4 v, float scale)
{
    const sf32x4 x = v * scale;
    Split4 r;
    r.hi = __builtin_convertvector(x, f16x4);
    r.lo = __builtin_convertvector(x - __builtin_convertvector(r.hi, sf32x4), f16x4);
    return r;
}
__device__ __forceinline__ f16x8 join(f16x4 a, f16x4 b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }

// floor(log2 |x|) of a normal float; -127 below, 128 for an infinity
__device__ __forceinline__ int exponent(float x) { return (int)(__float_as_uint(x) >> 23 & 0xff) - 127; }
__device__ __forceinline__ float power_of_two(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }   // -126 .. 127
__device__ __forceinline__ float max4(float m, sf32x4 v)
{
    return fmaxf(fmaxf(m, fmaxf(fabsf(v[0]), fabsf(v[1]))), fmaxf(fabsf(v[2]), fabsf(v[3])));
}
__device__ __forceinline__ sf32x4 mma_f16(f16x8 a, f16x8 b, sf32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

}  // namespace
}  // namespace mrx
