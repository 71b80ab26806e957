// A float32 value as the sum of three bfloat16 ones, for products on the bfloat16 matrix units.
//
// The matrix units multiply float32 at a sixteenth of the bfloat16 rate.  A value rounded to bfloat16, what that leaves rounded again, and what is left then
// are eight bits each: x = h + m + l, exactly, for |x| from 2^-110 to BF16_MOST (below, within 2^-134, where bfloat16 ends).  No scale is shared with
// other values, so that nothing is lost beside an outlier.  Of the nine products of two such sums,
//     x y = h h' + (h m' + m h') + (h l' + l h' + m m')
// leaves out m l' + l m' + l l', at most 2^-26 |x y| and zero on average: less than float32 rounds off one product.  Every product is exact and every sum in
// float32: six products in the time of six sixteenths of a float32 one.  The five small ones are added up by themselves first, so that the running sum is
// rounded twice in 32 terms, a float32 product's eight times or more.  Error against float64 (2-norm, normal operands), here / the array
// library's float32 products, by terms: 64 0.54e-7 / 1.43e-7, 256 0.78e-7 / 2.05e-7, 1024 1.5e-7 / 4.1e-7, 2056 in four layers 3.1e-7 / 5.0e-7; sums
// over 32768 rows 2.3e-7 / 8.1e-7.
// (Two float16 parts under a scale for each row and column are three products and took 142, 143 and 190 us where these take 184, 180 and 259, the cases below, but lose
// what lies 2^16 below the largest of its row, or 2^12 below the largest of its column: 1.3e-3 in a column of gradients beside one outlier of 1e8.)
#pragma once
#include "chunk_common.h"

namespace mrx {
namespace {

constexpr float BF16_MOST = 3.38953139e38f;   // the largest of bfloat16; what lies beyond, infinities among it, has no parts
constexpr int PARTS = 3;

// Two values in the parts of a word each: packed conversions, of whole words (element-wise access would undo them).
__device__ __forceinline__ void split2(float x, float y, uint32_t &h, uint32_t &m, uint32_t &l)
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    auto part = [&]() {
        const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x, y}, bf16x2));
        x -= __uint_as_float(w << 16), y -= __uint_as_float(w & 0xffff0000u);
        return w;
    };
    h = part(), m = part();
    l = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x, y}, bf16x2));
}
template <int W> struct Words {
    typedef uint32_t type __attribute__((ext_vector_type(W)));
};
// W pairs of values, W words a part
template <int W> __device__ __forceinline__ void split_parts(const f32x4 *v, typename Words<W>::type (&p)[PARTS])
{
#pragma unroll
    for (int i = 0; i < W; ++i) {
        uint32_t h, m, l;
        split2(v[i / 2][2 * (i % 2)], v[i / 2][2 * (i % 2) + 1], h, m, l);
        p[0][i] = h, p[1][i] = m, p[2][i] = l;
    }
}
__device__ __forceinline__ float max4(float m, f32x4 v)
{
    return fmaxf(fmaxf(m, fmaxf(fabsf(v[0]), fabsf(v[1]))), fmaxf(fabsf(v[2]), fabsf(v[3])));
}
__device__ __forceinline__ f32x4 mma_bf16(bf16x8 a, bf16x8 b, f32x4 c) { return TT<__bf16>::mma(a, b, c); }

// The products of two values' parts that are formed, the smallest first; the last one goes to the running sum.
constexpr int PRODUCTS = 6;
__device__ constexpr int PART_A[PRODUCTS] = {2, 0, 1, 1, 0, 0}, PART_B[PRODUCTS] = {0, 2, 1, 0, 1, 0};

}  // namespace
}  // namespace mrx
