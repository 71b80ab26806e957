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

// The same for many rows of few columns, where a workgroup's chain of loads is the time: 16 columns per workgroup, 64 threads
// per column, eight sums in flight per thread (the partial sums of a norm's gradients in an update, 1024 x 256: 7.4 -> 4.7 us).
__global__ void __launch_bounds__(1024) column_sum_tall_kernel(const float *__restrict__ parts, float *__restrict__ out0, float *__restrict__ out1,
                                                               int nparts, int D)
{
    __shared__ float red[16][16];
    const int c = threadIdx.x & 15, g = threadIdx.x >> 4, lane = threadIdx.x & 63, w = threadIdx.x >> 6, col = blockIdx.x * 16 + c;
    parts += (int64_t)blockIdx.y * nparts * D;
    float *out = blockIdx.y ? out1 : out0;
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (col < D)
        for (int p = g; p < nparts; p += 8 * 64)
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int r = p + u * 64;
                s[u] += r < nparts ? parts[(int64_t)r * D + col] : 0.f;
            }
    float x = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    x += __shfl_xor(x, 16);  // the wave's four threads of a column
    x += __shfl_xor(x, 32);
    if (lane < 16) red[w][c] = x;
    __syncthreads();
    if (w == 0) {
        const int j = lane >> 4;
        float t = (red[j][c] + red[j + 4][c]) + (red[j + 8][c] + red[j + 12][c]);
        t += __shfl_xor(t, 16);
        t += __shfl_xor(t, 32);
        if (j == 0 && col < D) out[col] = t;
    }
}

inline int launch_column_sum(hipStream_t st, const float *parts, float *out0, float *out1, int nparts, int D)
{
    // Where the rows are many and one workgroup per compute unit covers the columns (us, 64-wide / 16-wide: 512 x 256 2.79 / 2.53, 1024 x 256
    // 3.82 / 2.94, 4096 x 1024 10.1 / 6.3; not 256 x 256 2.25 / 2.44, nor 4096 x 16384 36.9 / 81.5, whose 64-byte rows of loads are read at half the rate)
    if (nparts >= 512 && D <= (out1 ? 2048 : 4096))
        return launch_kernel(column_sum_tall_kernel, dim3((unsigned)((D + 15) / 16), out1 ? 2u : 1u), dim3(1024), 0, st, parts, out0, out1, nparts, D);
    return launch_kernel(column_sum_kernel, dim3((unsigned)((D + 63) / 64), out1 ? 2u : 1u), dim3(64 * CS_GROUPS), 0, st, parts, out0, out1,
                         nparts, D);
}

}  // namespace
}  // namespace mrx
