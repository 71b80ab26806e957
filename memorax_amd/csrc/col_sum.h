// Sums over the rows of a (nparts, D) block of partial results, in a fixed order (run-to-run identical): what a kernel
// that keeps its parameters' gradients as per-workgroup partial sums needs afterwards.
#pragma once
#include "common.h"

namespace mrx {
namespace {

// out_y[col] = sum over the nparts rows of block y of parts (y = 0: out0, y = 1: out1): 64 columns per workgroup,
// sixteen threads per column that each add every sixteenth row, four independent sums in flight per thread.
constexpr int CS_GROUPS = 16;
__global__ void __launch_bounds__(64 * CS_GROUPS) column_sum_kernel(const float *__restrict__ parts, float *__restrict__ out0,
                                                                 float *__restrict__ out1, int nparts, int D)
{
    __shared__ float red[CS_GROUPS][64];
    const int c = threadIdx.x & 63, g = threadIdx.x >> 6, col = blockIdx.x * 64 + c;
    parts += (int64_t)blockIdx.y * nparts * D;
    float *out = blockIdx.y ? out1 : out0;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    if (col < D) {
        int p = g;
        for (; p + 3 * CS_GROUPS < nparts; p += 4 * CS_GROUPS)
#pragma unroll
            for (int u = 0; u < 4; ++u) s[u] += parts[(int64_t)(p + u * CS_GROUPS) * D + col];
        for (; p < nparts; p += CS_GROUPS) s[0] += parts[(int64_t)p * D + col];
    }
    red[g][c] = (s[0] + s[1]) + (s[2] + s[3]);
    __syncthreads();
    if (g == 0 && col < D) {
        float t[CS_GROUPS];   // in pairs: a running sum would round the whole total sixteen times
#pragma unroll
        for (int j = 0; j < CS_GROUPS; ++j) t[j] = red[j][c];
#pragma unroll
        for (int half = CS_GROUPS / 2; half > 0; half /= 2)
#pragma unroll
            for (int j = 0; j < half; ++j) t[j] += t[j + half];
        out[col] = t[0];
    }
}

inline int launch_column_sum(hipStream_t st, const float *parts, float *out0, float *out1, int nparts, int D)
{
    return launch_kernel(column_sum_kernel, dim3((unsigned)((D + 63) / 64), out1 ? 2u : 1u), dim3(64 * CS_GROUPS), 0, st, parts, out0, out1,
                         nparts, D);
}

}  // namespace
}  // namespace mrx
