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
#include "row_parts.h"

namespace mrx {
namespace {

constexpr int RD_WAVES = 4, RD_THREADS = 64 * RD_WAVES;
constexpr int RD_MAX_K = 2048;

struct RowDenseArgs {
    RowInput in;
    const float *residual;
    const float *skip;      // K factors: skip_out = x + skip * norm(x), for the residual branch of a cell with a feed-through term
    float *skip_out;
    const void *w2;         // a single layer whose weights lie in two arrays: columns k1 .. K
    int k1;
    const void *w[MRX_ROW_DENSE_LAYERS], *b[MRX_ROW_DENSE_LAYERS];
    void *y[MRX_ROW_DENSE_LAYERS];
    int n[MRX_ROW_DENSE_LAYERS], first_tile[MRX_ROW_DENSE_LAYERS + 1];   // columns of a layer, its first 64-column tile
    int layers;
    bool x_bf16, w_bf16, b_bf16, y_bf16;
};

// T: the products' type; WBF, XBF: bfloat16 weights, rows; MT: rows per workgroup (16 or 32); NV: 256-feature groups a lane holds of a row
// (K <= 256 NV); CT: 16-column tiles per wave; EXTRA: weights in two arrays, the feed-through term.
template <typename T, bool WBF, bool XBF, int MT, int NV, int CT, bool EXTRA>
__global__ void __launch_bounds__(RD_THREADS) row_dense_kernel(RowDenseArgs a)
{
    using F = typename TT<T>::frag;
    constexpr int KP = TT<T>::KP, KB = TT<T>::KB, RT = MT / 16, RPW = MT / RD_WAVES;
    constexpr int AHEAD = 8 / CT;   // k steps whose weight fragments are requested at once
    extern __shared__ __align__(16) unsigned char smem[];
    T *sx = reinterpret_cast<T *>(smem);
    const int K = a.in.K, kpad = (K + KB - 1) / KB * KB, ld = kpad + pad_of<T>(), steps = kpad / KB;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i16 = lane & 15, g = lane >> 4;
    const int tiles = a.first_tile[a.layers];
    const int tile = (int)(blockIdx.x % (unsigned)tiles);
    const int64_t r0 = (int64_t)(blockIdx.x / (unsigned)tiles) * MT, rows = a.in.rows;
    int l = 0;
#pragma unroll
    for (int j = 1; j < MRX_ROW_DENSE_LAYERS; ++j) l += j < a.layers && tile >= a.first_tile[j];
    const int n0 = ((tile - a.first_tile[l]) * RD_WAVES + wv) * 16 * CT, N = a.n[l];
    const void *w = a.w[l], *b = a.b[l], *out = a.y[l];

    RowPanel<XBF, RPW, NV> panel;
    panel.load(a.in, r0 + wv * RPW, lane);
    RawFrag<T, WBF> next[AHEAD][CT];
    auto fetch = [&](int s0) {
#pragma unroll
        for (int s = 0; s < AHEAD; ++s)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const int k = weight_k<T>((s0 + s) * KB + KP * g, K), c = n0 + ct * 16 + i16, row = c < N ? c : N - 1;
                const bool second = EXTRA && a.w2 && k >= a.k1;
                const int wide = EXTRA && a.w2 ? (second ? K - a.k1 : a.k1) : K;
                next[s][ct] = weight_raw<T, WBF>(second ? a.w2 : w, (int64_t)row * wide + (second ? k - a.k1 : k));
            }
    };
    fetch(0);
    panel.load_norm(a.in, lane);
    // lane (i16, g) ends up with columns c0 .. c0 + 3 of row i16 of each row tile: one load or store where rows are whole quads
    const bool quads = N % 4 == 0;
    uint32_t bias_raw[CT][4];
    f32x4 res[RT][CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int c0 = n0 + ct * 16 + 4 * g;
#pragma unroll
        for (int e = 0; e < 4; ++e) bias_raw[ct][e] = 0u;
        if (b) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int c = c0 + e < N ? c0 + e : N - 1;
                if (a.b_bf16) bias_raw[ct][e] = static_cast<const uint16_t *>(b)[c];
                else bias_raw[ct][e] = static_cast<const uint32_t *>(b)[c];
            }
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            res[rt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
            const int64_t r = r0 + rt * 16 + i16 < rows ? r0 + rt * 16 + i16 : rows - 1;
            if (a.residual && quads) res[rt][ct] = *reinterpret_cast<const f32x4 *>(a.residual + r * N + (c0 < N ? c0 : 0));
        }
    }

    panel.template finish<T>(a.in, sx + wv * RPW * ld, ld, kpad, lane, [&](int j, int i, int c, const f32x4 &y) {
        const int64_t r = r0 + wv * RPW + j;
        if (EXTRA && a.skip_out && tile == 0 && r < rows && c < K)
            *reinterpret_cast<f32x4 *>(a.skip_out + r * K + c) = panel.floats(panel.x[j][i]) + *reinterpret_cast<const f32x4 *>(a.skip + c) * y;
    });
    sync_lds();   // (the weights may still be on their way)

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
            for (int ct = 0; ct < CT; ++ct) {
                wf[ct] = weight_frag<T, WBF>(cur[s][ct]);
                if (kpad != K && (s0 + s) * KB + KP * g >= K) wf[ct] = F{};
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const F xf = TT<T>::template load<ROWK>(sx, ld, rt * 16, (s0 + s) * KB, lane);
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = TT<T>::mma(wf[ct], xf, acc[rt][ct]);
            }
        }
    }

#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int c0 = n0 + ct * 16 + 4 * g;
        if (c0 >= N) continue;
        float bias[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            bias[e] = a.b_bf16 ? raw_to_float<__bf16>(bias_raw[ct][e]) : raw_to_float<float>(bias_raw[ct][e]);
            if (std::is_same<T, __bf16>::value) bias[e] = (float)(__bf16)bias[e];
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const int64_t r = r0 + rt * 16 + i16, at = r * N + c0;
            if (r >= rows) continue;
            f32x4 y;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                y[e] = acc[rt][ct][e] + bias[e];
                if (std::is_same<T, __bf16>::value) y[e] = (float)(__bf16)y[e];
            }
            float *yf = static_cast<float *>(const_cast<void *>(out)) + at;
            __bf16 *yb = static_cast<__bf16 *>(const_cast<void *>(out)) + at;
            if (quads) {
                y += res[rt][ct];
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

// A kernel that needs more than the default 64 KB of dynamic LDS (float32 rows of more than 500 features at 32 rows, 1 000 at 16)
// announces it.
template <typename T, bool WBF, bool XBF, int MT, int NV, int CT, bool EXTRA> struct RowKernel {
    static constexpr auto fn = row_dense_kernel<T, WBF, XBF, MT, NV, CT, EXTRA>;
    static constexpr int most_lds = MT * (256 * NV + pad_of<T>()) * (int)sizeof(T);
    static inline const KernelRegistrar registrar{reinterpret_cast<const void *>(fn), most_lds};
    static auto get()
    {
        if constexpr (most_lds > 64 * 1024) (void)&registrar;
        return fn;
    }
};
template <typename T, bool WBF, bool XBF, int MT, int CT, bool EXTRA = false> int launch_rows(hipStream_t st, RowDenseArgs &a)
{
    constexpr int KB = TT<T>::KB, COLS = 16 * CT * RD_WAVES;
    for (int l = 0; l < a.layers; ++l) a.first_tile[l + 1] = a.first_tile[l] + (a.n[l] + COLS - 1) / COLS;
    const size_t lds = (size_t)MT * ((a.in.K + KB - 1) / KB * KB + pad_of<T>()) * sizeof(T);
    const int64_t grid = (a.in.rows + MT - 1) / MT * a.first_tile[a.layers];
    if (grid >= (1ll << 31)) return MRX_ERR_INVALID_ARG;
    auto go = [&](auto nv) {
        return launch_kernel(RowKernel<T, WBF, XBF, MT, decltype(nv)::value, CT, EXTRA>::get(), dim3((unsigned)grid), dim3(RD_THREADS), lds, st, a);
    };
    if (a.in.K <= 256) return go(std::integral_constant<int, 1>{});
    if constexpr (MT == 16) {
        if (a.in.K > 1024) return go(std::integral_constant<int, 8>{});
        if (a.in.K > 512) return go(std::integral_constant<int, 4>{});
    }
    return go(std::integral_constant<int, 2>{});
}
// Rows and columns per workgroup.  Few workgroups finish soonest small (16 rows x 64 columns: the call is one trip to memory and
// back); once they outnumber the compute units a few times over, larger ones read every weight and every row less often.
// Measured inside a HIP graph, 256 features (us): q, k, v and beta of 1 024 environments 8.1 / 7.7 / 7.7 at 16 x 64 / 32 x 64 /
// 32 x 128, of 2 048 12.0 / 10.9 / 9.6, of 4 096 19.4 / 17.4 / 14.2; a single 256-column layer 5.3 / 7.3 / 9.0 at 1 024 rows,
// 6.3 / 7.5 / 9.3 at 2 048, 9.2 / 8.8 / 9.4 at 4 096.  (The library's products alone, without the norm: 14.8, 15.8, 19.7 for the
// first three.)  Wide rows stay at 16: their registers and LDS would not fit otherwise.
template <typename T, bool WBF, bool XBF> int by_shape(hipStream_t st, RowDenseArgs &a)
{
    if (a.w2 || a.skip_out) return launch_rows<T, WBF, XBF, 16, 1, true>(st, a);
    int64_t small = 0;
    for (int l = 0; l < a.layers; ++l) small += (a.n[l] + 63) / 64;
    small *= (a.in.rows + 15) / 16;
    if (small <= 512 || a.in.K > 512) return launch_rows<T, WBF, XBF, 16, 1>(st, a);
    if (small <= 1024) return launch_rows<T, WBF, XBF, 32, 1>(st, a);
    return launch_rows<T, WBF, XBF, 32, 2>(st, a);
}
template <typename T> int by_type(hipStream_t st, RowDenseArgs &a)
{
    if (a.x_bf16) return a.w_bf16 ? by_shape<T, true, true>(st, a) : by_shape<T, false, true>(st, a);
    return a.w_bf16 ? by_shape<T, true, false>(st, a) : by_shape<T, false, false>(st, a);
}

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
    a.in = RowInput{x, scale, norm_bias, rows, (int)K, norm, eps, 1.f / (float)K, round_norm != 0};
    a.residual = residual, a.layers = layers;
    a.x_bf16 = x_dtype == MRX_BF16, a.w_bf16 = w_dtype == MRX_BF16, a.b_bf16 = b_dtype == MRX_BF16, a.y_bf16 = y_dtype == MRX_BF16;
    if (!aligned(x, 16) || !aligned(scale, 16) || !aligned(norm_bias, 16) || !aligned(residual, 4)) return MRX_ERR_INVALID_ARG;
    for (int l = 0; l < layers; ++l) {
        if (!weights[l] || !outs[l] || !aligned(weights[l], 16) || !aligned(outs[l], 4)) return MRX_ERR_INVALID_ARG;
        if (n_out[l] <= 0 || n_out[l] > (1 << 24)) return MRX_ERR_INVALID_ARG;
        a.w[l] = weights[l], a.b[l] = biases[l], a.y[l] = outs[l], a.n[l] = (int)n_out[l];
    }
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    return product_dtype == MRX_BF16 ? by_type<__bf16>(st, a) : by_type<float>(st, a);
}
