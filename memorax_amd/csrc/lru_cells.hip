// What the LRU cell's layer (lru.py:32-108) has beside its recurrence (scan.hip) and its two products (dense_split.hip): the maps from its
// parameters to the decay and to the real matrices of interleaved components that the products read, their gradients, and the gradient of
// the skip vector.  As array operations the maps are some thirty launches forward and backward, each of a few thousand
// elements: an update of a small layer is bound by the host's calls, of which these were two thirds (64 x 64 rows of 128, a hidden width of
// 128: 560 -> 240 us an update).  Here they are one launch each way, and the skip's gradient one and a column sum.
#include "col_sum.h"

namespace mrx {
namespace {

constexpr int LC_THREADS = 256;

struct LruParams {
    const float *nu, *theta, *gamma, *b_re, *b_im, *c_re, *c_im;   // (N), (N), (N), (N,F), (N,F), (F,N), (F,N)
    int N, F;
};
struct LruMaps {
    float2 *decay;   // (N)
    float *wb;       // (2N,F): rows 2n, 2n + 1 = exp(gamma) (B_re, B_im)
    float2 *wc;      // (F,N): (C_re, -C_im)
};

__global__ void __launch_bounds__(LC_THREADS) lru_params_fwd_kernel(LruParams p, LruMaps m)
{
    const int64_t total = (int64_t)p.N * p.F, stride = (int64_t)gridDim.x * LC_THREADS;
    for (int64_t e = (int64_t)blockIdx.x * LC_THREADS + threadIdx.x; e < total; e += stride) {
        const int64_t n = e / p.F, f = e - n * p.F;
        const float s = expf(p.gamma[n]);
        m.wb[2 * n * p.F + f] = p.b_re[e] * s;
        m.wb[(2 * n + 1) * p.F + f] = p.b_im[e] * s;
        m.wc[e] = float2{p.c_re[e], -p.c_im[e]};
        if (e < p.N) {
            const float r = expf(-expf(p.nu[e]));
            float sin, cos;
            sincosf(expf(p.theta[e]), &sin, &cos);
            m.decay[e] = float2{r * cos, r * sin};
        }
    }
}

struct LruGrads {
    const float2 *decay;   // (N)
    const float *wb;       // (2N,F)
    const float2 *wc;      // (F,N)
    float *nu, *theta, *gamma, *b_re, *b_im, *c_re, *c_im;
};

// Workgroups 0 .. N - 1: a state's row of B and its scalars; the others: C.
__global__ void __launch_bounds__(LC_THREADS) lru_params_bwd_kernel(LruParams p, LruGrads g)
{
    const int tid = threadIdx.x;
    if ((int)blockIdx.x < p.N) {
        __shared__ float red[LC_THREADS / 64];
        const int n = blockIdx.x;
        const float s = expf(p.gamma[n]);
        float dot = 0.f;
        for (int f = tid; f < p.F; f += LC_THREADS) {
            const int64_t e = (int64_t)n * p.F + f;
            const float re = g.wb[(int64_t)2 * n * p.F + f] * s, im = g.wb[((int64_t)2 * n + 1) * p.F + f] * s;
            g.b_re[e] = re, g.b_im[e] = im;
            dot += re * p.b_re[e] + im * p.b_im[e];
        }
        for (int off = 32; off > 0; off >>= 1) dot += __shfl_xor(dot, off);
        if ((tid & 63) == 0) red[tid >> 6] = dot;
        __syncthreads();
        if (tid == 0) {
            float total = 0.f;
#pragma unroll
            for (int w = 0; w < LC_THREADS / 64; ++w) total += red[w];
            g.gamma[n] = total;
            const float en = expf(p.nu[n]), et = expf(p.theta[n]), r = expf(-en);
            float sin, cos;
            sincosf(et, &sin, &cos);
            const float2 d = g.decay[n];
            g.nu[n] = -(d.x * cos + d.y * sin) * r * en;
            g.theta[n] = (d.y * cos - d.x * sin) * r * et;
        }
        return;
    }
    const int64_t total = (int64_t)p.N * p.F, stride = (int64_t)(gridDim.x - p.N) * LC_THREADS;
    for (int64_t e = (int64_t)(blockIdx.x - p.N) * LC_THREADS + tid; e < total; e += stride) {
        const float2 d = g.wc[e];
        g.c_re[e] = d.x, g.c_im[e] = -d.y;
    }
}

// parts[slab][c] = sum over the slab's rows of a b: 64 columns and sixteen rows at a time a workgroup.
constexpr int CP_ROWS = 16, CP_PARTS = 128;
__global__ void __launch_bounds__(64 * CP_ROWS) column_product_kernel(const float *__restrict__ a, const float *__restrict__ b, float *__restrict__ parts,
                                                                      int64_t rows, int64_t slab, int D)
{
    __shared__ float red[CP_ROWS][64];
    const int c = threadIdx.x & 63, q = threadIdx.x >> 6, col = blockIdx.x * 64 + c;
    const int64_t r0 = blockIdx.y * slab, r1 = r0 + slab < rows ? r0 + slab : rows;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    if (col < D) {
        int64_t r = r0 + q;
        for (; r + 3 * CP_ROWS < r1; r += 4 * CP_ROWS)
#pragma unroll
            for (int u = 0; u < 4; ++u) s[u] += a[(r + u * CP_ROWS) * D + col] * b[(r + u * CP_ROWS) * D + col];
        for (; r < r1; r += CP_ROWS) s[0] += a[r * D + col] * b[r * D + col];
    }
    red[q][c] = (s[0] + s[1]) + (s[2] + s[3]);
    __syncthreads();
    if (q == 0 && col < D) {
        float t[CP_ROWS];
#pragma unroll
        for (int j = 0; j < CP_ROWS; ++j) t[j] = red[j][c];
#pragma unroll
        for (int half = CP_ROWS / 2; half > 0; half /= 2)
#pragma unroll
            for (int j = 0; j < half; ++j) t[j] += t[j + half];
        parts[(int64_t)blockIdx.y * D + col] = t[0];
    }
}
int slabs_of(int64_t rows) { return (int)(rows >= 64 * CP_PARTS ? CP_PARTS : (rows + 63) / 64); }

bool lru_sizes_ok(int64_t N, int64_t F) { return N > 0 && F > 0 && N <= (1 << 20) && F <= (1 << 20); }

}  // namespace
}  // namespace mrx

extern "C" int mrx_lru_params_fwd(void *stream, const float *const *params, void *decay, float *wb, float *wc, int64_t N, int64_t F)
{
    using namespace mrx;
    if (!params || !decay || !wb || !wc || !lru_sizes_ok(N, F) || !aligned(decay, 8) || !aligned(wc, 8)) return MRX_ERR_INVALID_ARG;
    for (int i = 0; i < 7; ++i)
        if (!params[i]) return MRX_ERR_INVALID_ARG;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    const LruParams p{params[0], params[1], params[2], params[3], params[4], params[5], params[6], (int)N, (int)F};
    const int64_t wgs = (N * F + LC_THREADS - 1) / LC_THREADS;
    return launch_kernel(lru_params_fwd_kernel, dim3((unsigned)(wgs < 1024 ? wgs : 1024)), dim3(LC_THREADS), 0, static_cast<hipStream_t>(stream), p,
                         LruMaps{static_cast<float2 *>(decay), wb, reinterpret_cast<float2 *>(wc)});
}

extern "C" int mrx_lru_params_bwd(void *stream, const float *const *params, const void *ddecay, const float *dwb, const float *dwc, float *const *grads,
                                  int64_t N, int64_t F)
{
    using namespace mrx;
    if (!params || !ddecay || !dwb || !dwc || !grads || !lru_sizes_ok(N, F) || !aligned(ddecay, 8) || !aligned(dwc, 8)) return MRX_ERR_INVALID_ARG;
    for (int i = 0; i < 7; ++i)
        if (!params[i] || !grads[i]) return MRX_ERR_INVALID_ARG;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    const LruParams p{params[0], params[1], params[2], params[3], params[4], params[5], params[6], (int)N, (int)F};
    const LruGrads g{static_cast<const float2 *>(ddecay), dwb, reinterpret_cast<const float2 *>(dwc), grads[0], grads[1], grads[2], grads[3], grads[4], grads[5], grads[6]};
    const int64_t wgs = (N * F + LC_THREADS - 1) / LC_THREADS;
    return launch_kernel(lru_params_bwd_kernel, dim3((unsigned)(N + (wgs < 1024 ? wgs : 1024))), dim3(LC_THREADS), 0, static_cast<hipStream_t>(stream), p, g);
}

extern "C" int64_t mrx_column_product_workspace(int64_t rows, int64_t D)
{
    return rows > 0 && D > 0 && mrx::slabs_of(rows) > 1 ? mrx::slabs_of(rows) * D : 0;
}

extern "C" int mrx_column_product(void *stream, const float *a, const float *b, float *out, float *workspace, int64_t rows, int64_t D)
{
    using namespace mrx;
    if (!a || !b || !out || rows <= 0 || D <= 0 || D >= (1ll << 31) || rows >= (1ll << 40)) return MRX_ERR_INVALID_ARG;
    const int slabs = slabs_of(rows);
    if (slabs > 1 && !workspace) return MRX_ERR_INVALID_ARG;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    float *const parts = slabs > 1 ? workspace : out;
    const int64_t slab = (rows + slabs - 1) / slabs;
    const int rc = launch_kernel(column_product_kernel, dim3((unsigned)((D + 63) / 64), (unsigned)slabs), dim3(64 * CP_ROWS), 0, st, a, b, parts, rows, slab, (int)D);
    return rc != MRX_OK || slabs == 1 ? rc : launch_column_sum(st, parts, out, nullptr, slabs, (int)D);
}
