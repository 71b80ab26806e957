// Dense layers on few rows, as acting calls them: one row per environment, a few hundred features each way.
//
//     y_l = norm(x) W_l^T + b_l      for up to MRX_ROW_DENSE_LAYERS layers l that read the same rows,
//     y   = x_res + y_0              where the block's residual branch follows (float32)
//
// The library's products take such a call apart into a kernel per layer, a kernel per cast of a weight or an input, the norm
// before them and the addition behind them -- a dozen launches of 2-5 us each for a few microseconds of reading weights.
// Here one launch does all of it: a workgroup of four waves owns MT rows and 64 columns, normalises the rows on their way into
// LDS (every workgroup needs whole rows for the product anyway), and each wave multiplies them with its sixteen weight rows,
// which it reads from memory as they are (float32 or bfloat16; L2-resident: all row tiles read the same ones) and requests
// before it touches x, so that both trips to memory overlap.
//
// Rounding follows the composition it stands for: with bfloat16 products the normalised rows, the weights and the biases are
// rounded to bfloat16, sums are float32, and a result is rounded to bfloat16 before the residual is added.
#include <type_traits>

#include "chunk_common.h"

namespace mrx {
namespace {

constexpr int RD_WAVES = 4, RD_THREADS = 64 * RD_WAVES, RD_COLS = 16 * RD_WAVES;
constexpr int RD_MAX_K = 2048;
constexpr int RD_AHEAD = 8;   // k steps whose weight fragments are requested at once

struct RowDenseArgs {
    const void *x;
    const float *scale, *nbias, *residual;
    const void *w[MRX_ROW_DENSE_LAYERS], *b[MRX_ROW_DENSE_LAYERS];
    void *y[MRX_ROW_DENSE_LAYERS];
    int n[MRX_ROW_DENSE_LAYERS], first_tile[MRX_ROW_DENSE_LAYERS + 1];   // columns of a layer, its first 64-column tile
    int layers, K, norm;          // norm: 0 none, 1 RMS, 2 layer norm
    int64_t rows;
    float eps, inv_K;
    bool x_bf16, w_bf16, b_bf16, y_bf16, round_norm;   // round_norm: the normalised rows pass through bfloat16 (float32 products)
};

struct Quad {
    float v[4];
};
template <bool BF> __device__ __forceinline__ Quad quad_of(const void *p, int64_t at)
{
    Quad q;
    if (BF) {
        const bf16x4 x = *reinterpret_cast<const bf16x4 *>(static_cast<const __bf16 *>(p) + at);
#pragma unroll
        for (int e = 0; e < 4; ++e) q.v[e] = (float)x[e];
    } else {
        const f32x4 x = *reinterpret_cast<const f32x4 *>(static_cast<const float *>(p) + at);
#pragma unroll
        for (int e = 0; e < 4; ++e) q.v[e] = x[e];
    }
    return q;
}

__device__ __forceinline__ float wave_total(float x)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
    return x;
}

// A weight fragment as it waits in registers: KP consecutive k of one row, stored bits.
template <typename T, bool WBF> struct RawFrag {
    static constexpr int WORDS = TT<T>::KP * (WBF ? 2 : 4) / 8;   // 8-byte words
    uint64_t w[WORDS];
};
template <typename T, bool WBF> __device__ __forceinline__ RawFrag<T, WBF> weight_raw(const void *w, int64_t at)
{
    RawFrag<T, WBF> r;
    const char *p = static_cast<const char *>(w) + at * (WBF ? 2 : 4);
#pragma unroll
    for (int i = 0; i < RawFrag<T, WBF>::WORDS; ++i) r.w[i] = reinterpret_cast<const uint64_t *>(p)[i];
    return r;
}
template <typename T, bool WBF> __device__ __forceinline__ typename TT<T>::frag weight_frag(const RawFrag<T, WBF> &r)
{
    typename TT<T>::frag f;
    if constexpr (std::is_same<T, __bf16>::value && WBF) {
        f = __builtin_bit_cast(bf16x8, r);
    } else if constexpr (std::is_same<T, __bf16>::value) {
        struct F8 {
            float v[8];
        };
        const F8 x = __builtin_bit_cast(F8, r);
        const bf16x4 lo = TT<__bf16>::pack(x.v[0], x.v[1], x.v[2], x.v[3]), hi = TT<__bf16>::pack(x.v[4], x.v[5], x.v[6], x.v[7]);
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = lo[e], f[4 + e] = hi[e];
    } else if constexpr (WBF) {
        const bf16x4 x = __builtin_bit_cast(bf16x4, r);
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = (float)x[e];
    } else {
        f = __builtin_bit_cast(f32x4, r);
    }
    return f;
}

// T: the products' type; MT: rows per workgroup (16 or 32); NV: 256-feature groups a lane holds of a row (K <= 256 NV).
template <typename T, bool WBF, int MT, int NV>
__global__ void __launch_bounds__(RD_THREADS) row_dense_kernel(RowDenseArgs a)
{
    using F = typename TT<T>::frag;
    constexpr int KP = TT<T>::KP, KB = TT<T>::KB, RT = MT / 16, RPW = MT / RD_WAVES;
    extern __shared__ __align__(16) unsigned char smem[];
    T *sx = reinterpret_cast<T *>(smem);
    const int kpad = (a.K + KB - 1) / KB * KB, ld = kpad + pad_of<T>(), steps = kpad / KB;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, i16 = lane & 15, g = lane >> 4;
    const int tiles = a.first_tile[a.layers];
    const int tile = (int)(blockIdx.x % (unsigned)tiles);
    const int64_t r0 = (int64_t)(blockIdx.x / (unsigned)tiles) * MT;
    int l = 0;
    while (tile >= a.first_tile[l + 1]) ++l;
    const int n0 = (tile - a.first_tile[l]) * RD_COLS + wv * 16, N = a.n[l];
    const void *w = a.w[l];
    const int wrow = n0 + i16;   // this lane's weight row as an operand of the products

    RawFrag<T, WBF> next[RD_AHEAD];
    auto fetch = [&](int s0) {
#pragma unroll
        for (int s = 0; s < RD_AHEAD; ++s) {
            const int k = (s0 + s) * KB + KP * g;
            if (wrow < N && k < a.K) next[s] = weight_raw<T, WBF>(w, (int64_t)wrow * a.K + k);   // K is a multiple of KP
            else next[s] = RawFrag<T, WBF>{};
        }
    };
    fetch(0);

    {   // rows -> norm -> LDS; a wave takes RPW rows, all of them requested before the first is used
        Quad xv[RPW][NV];
#pragma unroll
        for (int j = 0; j < RPW; ++j)
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int c = (i * 64 + lane) * 4;
                const int64_t r = r0 + wv * RPW + j;
                if (r < a.rows && c < a.K) xv[j][i] = a.x_bf16 ? quad_of<true>(a.x, r * a.K + c) : quad_of<false>(a.x, r * a.K + c);
                else xv[j][i] = Quad{{0.f, 0.f, 0.f, 0.f}};
            }
        Quad sc[NV], nb[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = (i * 64 + lane) * 4;
            const bool in = a.norm && c < a.K;
            sc[i] = in && a.scale ? quad_of<false>(a.scale, c) : Quad{{1.f, 1.f, 1.f, 1.f}};
            nb[i] = in && a.nbias ? quad_of<false>(a.nbias, c) : Quad{{0.f, 0.f, 0.f, 0.f}};
        }
#pragma unroll
        for (int j = 0; j < RPW; ++j) {
            float rstd = 1.f;
            if (a.norm) {
                if (a.norm == 2) {
                    float s = 0.f;
#pragma unroll
                    for (int i = 0; i < NV; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) s += xv[j][i].v[e];
                    const float mu = wave_total(s) * a.inv_K;
#pragma unroll
                    for (int i = 0; i < NV; ++i)
                        if ((i * 64 + lane) * 4 < a.K)
#pragma unroll
                            for (int e = 0; e < 4; ++e) xv[j][i].v[e] -= mu;
                }
                float ss = 0.f;
#pragma unroll
                for (int i = 0; i < NV; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) ss += xv[j][i].v[e] * xv[j][i].v[e];
                rstd = rsqrtf(wave_total(ss) * a.inv_K + a.eps);
            }
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int c = (i * 64 + lane) * 4;
                if (c >= kpad) continue;   // columns K .. kpad hold zeros
                Quad o = xv[j][i];
                if (a.norm && c < a.K)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        o.v[e] = o.v[e] * rstd * sc[i].v[e] + nb[i].v[e];
                        if (a.round_norm) o.v[e] = (float)(__bf16)o.v[e];
                    }
                *reinterpret_cast<typename TT<T>::pack4 *>(sx + (wv * RPW + j) * ld + c) = TT<T>::pack(o.v[0], o.v[1], o.v[2], o.v[3]);
            }
        }
    }
    __syncthreads();

    f32x4 acc[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < steps; s0 += RD_AHEAD) {
        RawFrag<T, WBF> cur[RD_AHEAD];
#pragma unroll
        for (int s = 0; s < RD_AHEAD; ++s) cur[s] = next[s];
        if (s0 + RD_AHEAD < steps) fetch(s0 + RD_AHEAD);
#pragma unroll
        for (int s = 0; s < RD_AHEAD; ++s) {
            if (s0 + s >= steps) break;
            const F wf = weight_frag<T, WBF>(cur[s]);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                acc[rt] = TT<T>::mma(wf, TT<T>::template load<ROWK>(sx, ld, rt * 16, (s0 + s) * KB, lane), acc[rt]);
        }
    }

    // lane (i16, g) holds columns n0 + 4 g + 0..3 of row i16 of each row tile
    const int c0 = n0 + 4 * g;
    float bias[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        bias[e] = 0.f;
        if (a.b[l] && c0 + e < N) {
            bias[e] = a.b_bf16 ? (float)static_cast<const __bf16 *>(a.b[l])[c0 + e] : static_cast<const float *>(a.b[l])[c0 + e];
            if (std::is_same<T, __bf16>::value) bias[e] = (float)(__bf16)bias[e];
        }
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int64_t r = r0 + rt * 16 + i16;
        if (r >= a.rows) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (c0 + e >= N) break;
            float y = acc[rt][e] + bias[e];
            if (std::is_same<T, __bf16>::value) y = (float)(__bf16)y;
            const int64_t at = r * N + c0 + e;
            if (a.residual) static_cast<float *>(a.y[l])[at] = a.residual[at] + y;
            else if (a.y_bf16) static_cast<__bf16 *>(a.y[l])[at] = (__bf16)y;
            else static_cast<float *>(a.y[l])[at] = y;
        }
    }
}

template <typename T, bool WBF, int MT> int launch_rows(hipStream_t st, const RowDenseArgs &a)
{
    constexpr int KB = TT<T>::KB;
    const size_t lds = (size_t)MT * ((a.K + KB - 1) / KB * KB + pad_of<T>()) * sizeof(T);
    const int64_t grid = (a.rows + MT - 1) / MT * a.first_tile[a.layers];
    if (grid >= (1ll << 31)) return MRX_ERR_INVALID_ARG;
    auto go = [&](auto nv) {
        return launch_kernel(row_dense_kernel<T, WBF, MT, decltype(nv)::value>, dim3((unsigned)grid), dim3(RD_THREADS), lds, st, a);
    };
    if (a.K <= 256) return go(std::integral_constant<int, 1>{});
    if constexpr (MT == 16) {
        if (a.K > 1024) return go(std::integral_constant<int, 8>{});
        if (a.K > 512) return go(std::integral_constant<int, 4>{});
    }
    return go(std::integral_constant<int, 2>{});
}

// Dynamic LDS beyond the default limit of 64 KB: float32 rows of more than 500 (32 rows) or 1 000 features (16 rows).
constexpr int RD_MAX_LDS = 16 * (RD_MAX_K + 4) * 4;
const KernelRegistrar registrars[] = {
    {reinterpret_cast<const void *>(row_dense_kernel<float, false, 16, 8>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<float, true, 16, 8>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<float, false, 16, 4>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<float, true, 16, 4>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<float, false, 32, 2>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<float, true, 32, 2>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<__bf16, false, 16, 8>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<__bf16, true, 16, 8>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<__bf16, false, 16, 4>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<__bf16, true, 16, 4>), RD_MAX_LDS},
};

}  // namespace
}  // namespace mrx

extern "C" int mrx_row_dense(void *stream, const void *x, const float *scale, const float *norm_bias, int norm, int round_norm,
                             const void *const *weights, const void *const *biases, void *const *outs, const int64_t *n_out, int layers,
                             const float *residual, int64_t rows, int64_t K, int x_dtype, int w_dtype, int b_dtype, int y_dtype,
                             int product_dtype, float eps)
{
    using namespace mrx;
    auto known = [](int dt) { return dt == MRX_F32 || dt == MRX_BF16; };
    if (!x || !weights || !biases || !outs || !n_out || layers < 1 || layers > MRX_ROW_DENSE_LAYERS || rows <= 0 || K <= 0)
        return MRX_ERR_INVALID_ARG;
    if (norm < 0 || norm > 2 || !known(x_dtype) || !known(w_dtype) || !known(b_dtype) || !known(y_dtype) || !known(product_dtype))
        return MRX_ERR_INVALID_ARG;
    if (residual && (layers != 1 || y_dtype != MRX_F32)) return MRX_ERR_INVALID_ARG;
    if (K % 8 != 0 || K > RD_MAX_K) return MRX_ERR_UNSUPPORTED;
    RowDenseArgs a{};
    a.x = x, a.scale = scale, a.nbias = norm_bias, a.residual = residual;
    a.layers = layers, a.K = (int)K, a.norm = norm, a.rows = rows, a.eps = eps, a.inv_K = 1.f / (float)K;
    a.x_bf16 = x_dtype == MRX_BF16, a.w_bf16 = w_dtype == MRX_BF16, a.b_bf16 = b_dtype == MRX_BF16, a.y_bf16 = y_dtype == MRX_BF16;
    a.round_norm = round_norm != 0;
    if (!aligned(x, 16) || !aligned(scale, 16) || !aligned(norm_bias, 16) || !aligned(residual, 4)) return MRX_ERR_INVALID_ARG;
    for (int l = 0; l < layers; ++l) {
        if (!weights[l] || !outs[l] || !aligned(weights[l], 16) || !aligned(outs[l], 4)) return MRX_ERR_INVALID_ARG;
        if (n_out[l] <= 0 || n_out[l] > (1 << 24)) return MRX_ERR_INVALID_ARG;
        a.w[l] = weights[l], a.b[l] = biases[l], a.y[l] = outs[l], a.n[l] = (int)n_out[l];
        a.first_tile[l + 1] = a.first_tile[l] + (int)((n_out[l] + RD_COLS - 1) / RD_COLS);
    }
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool bf = product_dtype == MRX_BF16;
    // 32 rows per workgroup read every weight half as often; 16 where that leaves workgroups for the compute units, and where
    // a row is so wide that its registers (eight rows per wave) or its LDS would not fit
    const bool wide = K <= 512 && (rows + 31) / 32 * a.first_tile[layers] >= 256;
    if (bf) {
        if (a.w_bf16) return wide ? launch_rows<__bf16, true, 32>(st, a) : launch_rows<__bf16, true, 16>(st, a);
        return wide ? launch_rows<__bf16, false, 32>(st, a) : launch_rows<__bf16, false, 16>(st, a);
    }
    if (a.w_bf16) return wide ? launch_rows<float, true, 32>(st, a) : launch_rows<float, true, 16>(st, a);
    return wide ? launch_rows<float, false, 32>(st, a) : launch_rows<float, false, 16>(st, a);
}
