// Dense layers on few rows, as acting calls them: one row per environment, a few hundred features each way.
//
//     y_l = norm(x) W_l^T + b_l      for up to MRX_ROW_DENSE_LAYERS layers l that read the same rows,
//     y   = x_res + y_0              where the block's residual branch follows (float32)
//
// The library's products take such a call apart into a kernel per layer, a kernel per cast of a weight or an input, the norm
// before them and the addition behind them -- a dozen launches of 2-5 us each for a few microseconds of reading weights.
// Here one launch does all of it: a workgroup of four waves owns MT rows and 64 CT columns, normalises the rows on their way into
// LDS (every workgroup needs whole rows for the product anyway), and each wave multiplies them with its 16 or 32 weight rows,
// which it reads from memory as they are (float32 or bfloat16; L2-resident: all row tiles read the same ones) and requests
// before it touches x, so that both trips to memory overlap.
//
// Rounding follows the composition it stands for: with bfloat16 products the normalised rows, the weights and the biases are
// rounded to bfloat16, sums are float32, and a result is rounded to bfloat16 before the residual is added.
#include <type_traits>

#include "chunk_common.h"

namespace mrx {
namespace {

constexpr int RD_WAVES = 4, RD_THREADS = 64 * RD_WAVES;
constexpr int RD_MAX_K = 2048;

struct RowDenseArgs {
    const void *x;
    const float *scale, *nbias, *residual;
    const float *skip;      // K factors: skip_out = x + skip * norm(x), for the residual branch of a cell with a feed-through term
    float *skip_out;
    const void *w2;         // a single layer whose weights lie in two arrays: columns k1 .. K
    int k1;
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

// Sum over a wave, in every lane: within rows of sixteen lanes by DPP moves (one instruction each, where a shuffle is a trip to
// LDS), the four rows by shuffles.
__device__ __forceinline__ float wave_total(float x)
{
    auto add = [&](auto ctrl) {
        const int moved = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, true);
        x += __builtin_bit_cast(float, moved);
    };
    add(std::integral_constant<int, 0xB1>{});    // quad_perm [1,0,3,2]
    add(std::integral_constant<int, 0x4E>{});    // quad_perm [2,3,0,1]
    add(std::integral_constant<int, 0x141>{});   // row_half_mirror
    add(std::integral_constant<int, 0x140>{});   // row_mirror
    x += __shfl_xor(x, 16);
    x += __shfl_xor(x, 32);
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

// T: the products' type; MT: rows per workgroup (16 or 32); NV: 256-feature groups a lane holds of a row (K <= 256 NV);
// CT: 16-column tiles per wave.
template <typename T, bool WBF, int MT, int NV, int CT>
__global__ void __launch_bounds__(RD_THREADS) row_dense_kernel(RowDenseArgs a)
{
    using F = typename TT<T>::frag;
    constexpr int KP = TT<T>::KP, KB = TT<T>::KB, RT = MT / 16, RPW = MT / RD_WAVES;
    constexpr int AHEAD = 8 / CT;   // k steps whose weight fragments are requested at once
    extern __shared__ __align__(16) unsigned char smem[];
    T *sx = reinterpret_cast<T *>(smem);
    const int kpad = (a.K + KB - 1) / KB * KB, ld = kpad + pad_of<T>(), steps = kpad / KB;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, i16 = lane & 15, g = lane >> 4;
    const int tiles = a.first_tile[a.layers];
    const int tile = (int)(blockIdx.x % (unsigned)tiles);
    const int64_t r0 = (int64_t)(blockIdx.x / (unsigned)tiles) * MT;
    int l = 0;
    while (tile >= a.first_tile[l + 1]) ++l;
    const int n0 = ((tile - a.first_tile[l]) * RD_WAVES + wv) * 16 * CT, N = a.n[l];
    const void *w = a.w[l];

    RawFrag<T, WBF> next[AHEAD][CT];
    auto fetch = [&](int s0) {
#pragma unroll
        for (int s = 0; s < AHEAD; ++s)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const int k = (s0 + s) * KB + KP * g, row = n0 + ct * 16 + i16;   // K is a multiple of KP
                if (row < N && k < a.K) {
                    const bool second = a.w2 && k >= a.k1;
                    const int wide = a.w2 ? (second ? a.K - a.k1 : a.k1) : a.K;
                    next[s][ct] = weight_raw<T, WBF>(second ? a.w2 : w, (int64_t)row * wide + (second ? k - a.k1 : k));
                }
                else next[s][ct] = RawFrag<T, WBF>{};
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
                if (a.skip_out && tile == 0 && r0 + wv * RPW + j < a.rows && c < a.K) {
                    const int64_t at = (r0 + wv * RPW + j) * a.K + c;
                    const Quad x = a.x_bf16 ? quad_of<true>(a.x, at) : quad_of<false>(a.x, at), d = quad_of<false>(a.skip, c);
                    *reinterpret_cast<f32x4 *>(a.skip_out + at) =
                        f32x4{x.v[0] + d.v[0] * o.v[0], x.v[1] + d.v[1] * o.v[1], x.v[2] + d.v[2] * o.v[2], x.v[3] + d.v[3] * o.v[3]};
                }
                *reinterpret_cast<typename TT<T>::pack4 *>(sx + (wv * RPW + j) * ld + c) = TT<T>::pack(o.v[0], o.v[1], o.v[2], o.v[3]);
            }
        }
    }
    __syncthreads();

    f32x4 acc[RT][CT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < steps; s0 += AHEAD) {
        RawFrag<T, WBF> cur[AHEAD][CT];
#pragma unroll
        for (int s = 0; s < AHEAD; ++s)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) cur[s][ct] = next[s][ct];
        if (s0 + AHEAD < steps) fetch(s0 + AHEAD);
#pragma unroll
        for (int s = 0; s < AHEAD; ++s) {
            if (s0 + s >= steps) break;
            F wf[CT];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) wf[ct] = weight_frag<T, WBF>(cur[s][ct]);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const F xf = TT<T>::template load<ROWK>(sx, ld, rt * 16, (s0 + s) * KB, lane);
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = TT<T>::mma(wf[ct], xf, acc[rt][ct]);
            }
        }
    }

    // lane (i16, g) holds columns c0 .. c0 + 3 of row i16 of each row tile: one store where rows are whole quads
    const bool quads = N % 4 == 0;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int c0 = n0 + ct * 16 + 4 * g;
        if (c0 >= N) continue;
        float bias[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (a.b[l] && c0 + e < N) {
                bias[e] = a.b_bf16 ? (float)static_cast<const __bf16 *>(a.b[l])[c0 + e] : static_cast<const float *>(a.b[l])[c0 + e];
                if (std::is_same<T, __bf16>::value) bias[e] = (float)(__bf16)bias[e];
            }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const int64_t r = r0 + rt * 16 + i16, at = r * N + c0;
            if (r >= a.rows) continue;
            f32x4 y;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                y[e] = acc[rt][ct][e] + bias[e];
                if (std::is_same<T, __bf16>::value) y[e] = (float)(__bf16)y[e];
            }
            float *yf = static_cast<float *>(a.y[l]) + at;
            __bf16 *yb = static_cast<__bf16 *>(a.y[l]) + at;
            if (quads) {
                if (a.residual) y += *reinterpret_cast<const f32x4 *>(a.residual + at);
                if (a.y_bf16) *reinterpret_cast<bf16x4 *>(yb) = TT<__bf16>::pack(y[0], y[1], y[2], y[3]);
                else *reinterpret_cast<f32x4 *>(yf) = y;
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (c0 + e >= N) break;
                if (a.residual) y[e] += a.residual[at + e];
                if (a.y_bf16) yb[e] = (__bf16)y[e];
                else yf[e] = y[e];
            }
        }
    }
}

template <typename T, bool WBF, int MT, int CT> int launch_rows(hipStream_t st, RowDenseArgs &a)
{
    constexpr int KB = TT<T>::KB, COLS = 16 * CT * RD_WAVES;
    for (int l = 0; l < a.layers; ++l) a.first_tile[l + 1] = a.first_tile[l] + (a.n[l] + COLS - 1) / COLS;
    const size_t lds = (size_t)MT * ((a.K + KB - 1) / KB * KB + pad_of<T>()) * sizeof(T);
    const int64_t grid = (a.rows + MT - 1) / MT * a.first_tile[a.layers];
    if (grid >= (1ll << 31)) return MRX_ERR_INVALID_ARG;
    auto go = [&](auto nv) {
        return launch_kernel(row_dense_kernel<T, WBF, MT, decltype(nv)::value, CT>, dim3((unsigned)grid), dim3(RD_THREADS), lds, st, a);
    };
    if (a.K <= 256) return go(std::integral_constant<int, 1>{});
    if constexpr (MT == 16) {
        if (a.K > 1024) return go(std::integral_constant<int, 8>{});
        if (a.K > 512) return go(std::integral_constant<int, 4>{});
    }
    return go(std::integral_constant<int, 2>{});
}
// Rows and columns per workgroup.  Few workgroups finish soonest small (16 rows x 64 columns: the call is one trip to memory and
// back); once they outnumber the compute units a few times over, larger ones read every weight and every row less often.
// Measured inside a HIP graph, 256 features (us): q, k, v and beta of 1 024 environments 8.1 / 7.7 / 7.7 at 16 x 64 / 32 x 64 /
// 32 x 128, of 2 048 12.0 / 10.9 / 9.6, of 4 096 19.4 / 17.4 / 14.2; a single 256-column layer 5.3 / 7.3 / 9.0 at 1 024 rows,
// 6.3 / 7.5 / 9.3 at 2 048, 9.2 / 8.8 / 9.4 at 4 096.  (The library's products alone, without the norm: 14.8, 15.8, 19.7 for the
// first three.)  Wide rows stay at 16: their registers and LDS would not fit otherwise.
template <typename T, bool WBF> int by_shape(hipStream_t st, RowDenseArgs &a)
{
    int64_t small = 0;
    for (int l = 0; l < a.layers; ++l) small += (a.n[l] + 63) / 64;
    small *= (a.rows + 15) / 16;
    if (small <= 512 || a.K > 512) return launch_rows<T, WBF, 16, 1>(st, a);
    if (small <= 1024) return launch_rows<T, WBF, 32, 1>(st, a);
    return launch_rows<T, WBF, 32, 2>(st, a);
}

// Dynamic LDS beyond the default limit of 64 KB: float32 rows of more than 500 (32 rows) or 1 000 features (16 rows).
constexpr int RD_MAX_LDS = 16 * (RD_MAX_K + 4) * 4;
const KernelRegistrar registrars[] = {
    {reinterpret_cast<const void *>(row_dense_kernel<float, false, 16, 8, 1>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<float, true, 16, 8, 1>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<float, false, 16, 4, 1>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<float, true, 16, 4, 1>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<float, false, 32, 2, 1>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<float, true, 32, 2, 1>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<float, false, 32, 2, 2>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<float, true, 32, 2, 2>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<__bf16, false, 16, 8, 1>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<__bf16, true, 16, 8, 1>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<__bf16, false, 16, 4, 1>), RD_MAX_LDS},
    {reinterpret_cast<const void *>(row_dense_kernel<__bf16, true, 16, 4, 1>), RD_MAX_LDS},
};

}  // namespace
}  // namespace mrx

extern "C" int mrx_row_dense(void *stream, const void *x, const float *scale, const float *norm_bias, int norm, int round_norm,
                             const void *const *weights, const void *const *biases, void *const *outs, const int64_t *n_out, int layers,
                             const float *residual, int64_t rows, int64_t K, int x_dtype, int w_dtype, int b_dtype, int y_dtype,
                             int product_dtype, float eps, const void *weights2, int64_t k1, const float *skip, float *skip_out)
{
    using namespace mrx;
    auto known = [](int dt) { return dt == MRX_F32 || dt == MRX_BF16; };
    if (!x || !weights || !biases || !outs || !n_out || layers < 1 || layers > MRX_ROW_DENSE_LAYERS || rows <= 0 || K <= 0)
        return MRX_ERR_INVALID_ARG;
    if (norm < 0 || norm > 2 || !known(x_dtype) || !known(w_dtype) || !known(b_dtype) || !known(y_dtype) || !known(product_dtype))
        return MRX_ERR_INVALID_ARG;
    if (residual && (layers != 1 || y_dtype != MRX_F32)) return MRX_ERR_INVALID_ARG;
    if (K % 8 != 0 || K > RD_MAX_K) return MRX_ERR_UNSUPPORTED;
    if (weights2 && (layers != 1 || k1 <= 0 || k1 >= K || k1 % 8 != 0 || !aligned(weights2, 16))) return MRX_ERR_INVALID_ARG;
    if ((skip == nullptr) != (skip_out == nullptr) || !aligned(skip, 16) || !aligned(skip_out, 16)) return MRX_ERR_INVALID_ARG;
    RowDenseArgs a{};
    a.w2 = weights2, a.k1 = (int)k1, a.skip = skip, a.skip_out = skip_out;
    a.x = x, a.scale = scale, a.nbias = norm_bias, a.residual = residual;
    a.layers = layers, a.K = (int)K, a.norm = norm, a.rows = rows, a.eps = eps, a.inv_K = 1.f / (float)K;
    a.x_bf16 = x_dtype == MRX_BF16, a.w_bf16 = w_dtype == MRX_BF16, a.b_bf16 = b_dtype == MRX_BF16, a.y_bf16 = y_dtype == MRX_BF16;
    a.round_norm = round_norm != 0;
    if (!aligned(x, 16) || !aligned(scale, 16) || !aligned(norm_bias, 16) || !aligned(residual, 4)) return MRX_ERR_INVALID_ARG;
    for (int l = 0; l < layers; ++l) {
        if (!weights[l] || !outs[l] || !aligned(weights[l], 16) || !aligned(outs[l], 4)) return MRX_ERR_INVALID_ARG;
        if (n_out[l] <= 0 || n_out[l] > (1 << 24)) return MRX_ERR_INVALID_ARG;
        a.w[l] = weights[l], a.b[l] = biases[l], a.y[l] = outs[l], a.n[l] = (int)n_out[l];
    }
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool bf = product_dtype == MRX_BF16;
    if (bf) return a.w_bf16 ? by_shape<__bf16, true>(st, a) : by_shape<__bf16, false>(st, a);
    return a.w_bf16 ? by_shape<float, true>(st, a) : by_shape<float, false>(st, a);
}
