// Gradients of dense layers that read the same rows, for a whole group of them:
//
//     dW_l = dy_l^T x      db_l = sum over the rows of dy_l      dx = sum_l dy_l W_l
//
// A rollout batch has a hundred thousand rows and a few hundred features.  The first two are products with a tiny result and an
// enormous inner dimension, the third is one whose operands are read once; all are bound by reading dy and x.  The array
// library runs them as a product per layer and direction -- with the rows cut into slices by hand, a reduction per layer over
// those, a reduction per bias, and the sum of the input gradients rounded and read back between the layers -- most of them at a
// fraction of the bandwidth (131072 rows, three layers of 256 x 256 and one of 256 x 4 in bfloat16: 330 us for the parameters and 150 us
// for the input; 11455 rows, three of 128 x 256: 225 and 23 us).  Here they are two launches and one reduction: 134 and 118 us, 24 and
// 16 us.  At 256 features a compute unit is short of loads in flight rather than of bandwidth: LDS holds two steps of two workgroups.
//
// Weight gradients: a workgroup of four waves owns a TN x TK tile of one layer's result and a slice of the rows, 64 (float32: 32)
// of which wait in LDS while the next are on their way; both operands are contracted over their rows, which the transposing
// LDS reads serve without a copy.  The slices' partial results are summed in a fixed order (col_sum.h).
// Input gradient: a workgroup owns TM rows and TK features and walks the layers' outputs, two steps ahead in registers (one step: 120
// -> 115 us at 131072 rows, 19.9 -> 17.3 us at 11455 rows of the sizes above.  The weight gradients are bound by the transposing reads
// of both operands instead: a second step there costs the registers those need, 123 -> 147 us).
#include "chunk_common.h"
#include "col_sum.h"

#include <type_traits>

namespace mrx {
namespace {

constexpr int DG_WAVES = 4, DG_THREADS = 64 * DG_WAVES;

struct DenseGradArgs {
    const void *x, *dy[MRX_DENSE_LAYERS], *w[MRX_DENSE_LAYERS];
    void *dx;
    float *out;                                                   // (slices, total)
    int64_t w_at[MRX_DENSE_LAYERS], b_at[MRX_DENSE_LAYERS];       // where a layer's gradients start in a row of `out`; b_at < 0: no bias
    int n[MRX_DENSE_LAYERS], first_tile[MRX_DENSE_LAYERS + 1];
    int layers, K, ktiles, slices;
    int64_t rows, slice_rows, total;
    bool dx_bf16;
};

typedef uint32_t W4 __attribute__((ext_vector_type(4)));
typedef W4 W4a2 __attribute__((aligned(2)));
typedef W4 W4a4 __attribute__((aligned(4)));

// R rows x W columns of a row-major array, on their way to LDS: columns from col0 (what lies beyond N reads as zero), rows up to
// row_end.  A lane takes 16 bytes whatever the rows' alignment; where they reach into the next row (a layer of few outputs, one
// gate per head), to_lds drops the rest -- anything done to a value right after its load, or several narrower loads put together,
// would wait for it, and a workgroup that waits holds up the launch (beside three layers of 256, one of 4 outputs cost 95 us).
template <typename T, int R, int W, OpMode MODE> struct RowTile {
    static constexpr int KP = TT<T>::KP, SEGS = W / KP, PASSES = R * SEGS / DG_THREADS, PER_WORD = 4 / (int)sizeof(T);
    using W4u = typename std::conditional<sizeof(T) == 2, W4a2, W4a4>::type;
    static_assert(R * SEGS % DG_THREADS == 0, "whole passes");
    // rows of 128 bfloat16 that are read transposed: four of them at once, eight banks each, must not meet in the 64 banks
    static constexpr int LD = W + (MODE == KROW && sizeof(T) == 2 ? 16 : pad_of<T>());
    W4 v[PASSES];
    int cols;   // of the tile that exist
    __device__ __forceinline__ void load(const T *base, int64_t row0, int64_t row_end, int64_t rows, int col0, int N, int tid)
    {
        cols = N - col0;
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            const int idx = tid + p * DG_THREADS, c = idx % SEGS * KP;
            const int64_t row = row0 + idx / SEGS, at = row * N + col0 + c;
            v[p] = W4{0u, 0u, 0u, 0u};
            if (row >= row_end || c >= cols) continue;
            if (at + KP <= rows * N) {
                v[p] = *reinterpret_cast<const W4u *>(base + at);
            } else {   // the array's last elements
#pragma unroll
                for (int e = 0; e < KP; ++e) {
                    if (c + e >= cols) break;
                    if constexpr (sizeof(T) == 2) v[p][e / 2] |= (uint32_t)reinterpret_cast<const uint16_t *>(base)[at + e] << 16 * (e % 2);
                    else v[p][e] = reinterpret_cast<const uint32_t *>(base)[at + e];
                }
            }
        }
    }
    __device__ __forceinline__ void to_lds(T *dst, int tid)
    {
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            const int idx = tid + p * DG_THREADS, have = cols - idx % SEGS * KP;
            if (have < KP) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (q * PER_WORD >= have) v[p][q] = 0u;
                    else if (PER_WORD == 2 && q * PER_WORD + 1 >= have) v[p][q] &= 0xffffu;
                }
            }
            *reinterpret_cast<W4 *>(dst + idx / SEGS * LD + idx % SEGS * KP) = v[p];
        }
    }
};

template <typename T> constexpr int dg_rows() { return sizeof(T) == 2 ? 64 : 32; }   // rows (weight gradients) or outputs (dx) per step

// Workgroups are dealt to the eight dies in turn, and tasks that read the same rows follow each other: each die takes a contiguous
// share of them, and its L2 serves the second reader.  -1: none left.
__device__ __forceinline__ int64_t task_of(int64_t tasks)
{
    const int64_t t = (blockIdx.x & 7) * ((tasks + 7) / 8) + (blockIdx.x >> 3);
    return (int64_t)(blockIdx.x >> 3) < (tasks + 7) / 8 && t < tasks ? t : -1;
}
inline unsigned grid_of(int64_t tasks) { return (unsigned)((tasks + 7) / 8 * 8); }

template <typename T, int TN, int TK>
__global__ void __launch_bounds__(DG_THREADS, 2) dense_weight_grad_kernel(DenseGradArgs a)
{
    constexpr int RC = dg_rows<T>(), MBW = TK / 32, NBW = TN / 32;
    using TileX = RowTile<T, RC, TK, KROW>;
    using TileY = RowTile<T, RC, TN, KROW>;
    using TM = TileMap<TK, TN, DG_WAVES, MBW>;
    constexpr int BUF = RC * (TileX::LD + TileY::LD);
    extern __shared__ __align__(16) unsigned char smem[];
    T *const lds = reinterpret_cast<T *>(smem);
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), i16 = lane & 15, g = lane >> 4;
    const int tiles = a.first_tile[a.layers] * a.ktiles;
    const int64_t task = task_of((int64_t)tiles * a.slices);
    if (task < 0) return;
    const int slice = (int)(task / tiles), tile = (int)(task % tiles);
    const int kt = tile % a.ktiles, nt = tile / a.ktiles;
    int l = 0;
    while (nt >= a.first_tile[l + 1]) ++l;
    const int N = a.n[l], n0 = (nt - a.first_tile[l]) * TN, k0 = kt * TK;
    const int64_t r0 = slice * a.slice_rows, r1 = r0 + a.slice_rows < a.rows ? r0 + a.slice_rows : a.rows;
    const T *x = static_cast<const T *>(a.x), *dy = static_cast<const T *>(a.dy[l]);
    const bool bias = a.b_at[l] >= 0 && kt == 0 && w % TM::WM == 0;

    f32x4 acc[TM::TPW], accb[NBW];
    zero_acc<TM::TPW>(acc);
    zero_acc<NBW>(accb);
    // the bias gradient, in float32 a step's sum at a time with what its additions round off (131072 x 4: 1.6e-7 -> 4e-8)
    float bias_sum[NBW], bias_low[NBW];
#pragma unroll
    for (int j = 0; j < NBW; ++j) bias_sum[j] = bias_low[j] = 0.f;
    TileX tx;
    TileY ty;
    tx.load(x, r0, r1, a.rows, k0, a.K, tid);
    ty.load(dy, r0, r1, a.rows, n0, N, tid);
    int buf = 0;
    auto sum_bias = [&]() {
#pragma unroll
        for (int j = 0; j < NBW; ++j) {
            const float y = accb[j][0] - bias_low[j], s = bias_sum[j] + y;
            bias_low[j] = (s - bias_sum[j]) - y;
            bias_sum[j] = s;
        }
        zero_acc<NBW>(accb);
    };
    for (int64_t r = r0; r < r1; r += RC, buf ^= 1) {
        T *const sx = lds + buf * BUF, *const sy = sx + RC * TileX::LD;
        tx.to_lds(sx, tid);
        ty.to_lds(sy, tid);
        if (r + RC < r1) {
            tx.load(x, r + RC, r1, a.rows, k0, a.K, tid);
            ty.load(dy, r + RC, r1, a.rows, n0, N, tid);
        }
        if (sizeof(T) == 4 && bias) sum_bias();   // of the step before: its products are done
        sync_lds();   // the buffer two steps back has been read by every wave that reaches the barrier
        gemm<T, TK, TN, RC, KROW, KROW, DG_WAVES, MBW>(acc, sx, TileX::LD, sy, TileY::LD, w, lane, NoHook(),
                                                       [&](int ni, int, typename TT<T>::frag &f) {
                                                           if (bias) accb[ni] = TT<T>::mma(TT<T>::ones(), f, accb[ni]);
                                                       });
    }
    float *const out = a.out + slice * a.total;
#pragma unroll
    for (int j = 0; j < TM::TPW; ++j) {
        const int k = k0 + TM::mt(w, j) * 16 + 4 * g, n = n0 + TM::nt(w, j) * 16 + i16;
        if (k < a.K && n < N) *reinterpret_cast<f32x4 *>(out + a.w_at[l] + (int64_t)n * a.K + k) = acc[j];
    }
    if (bias) sum_bias();
    if (bias && g == 0) {
#pragma unroll
        for (int j = 0; j < NBW; ++j) {
            const int n = n0 + TM::nt(w, j) * 16 + i16;
            if (n < N) out[a.b_at[l] + n] = bias_sum[j];
        }
    }
}

template <typename T, int TM_, int TK>
__global__ void __launch_bounds__(DG_THREADS, 2) dense_input_grad_kernel(DenseGradArgs a)
{
    constexpr int NC = dg_rows<T>(), MBW = TK / 32;
    using TileW = RowTile<T, NC, TK, KROW>;
    using TileY = RowTile<T, TM_, NC, ROWK>;
    using TM = TileMap<TK, TM_, DG_WAVES, MBW>;
    constexpr int BUF = NC * TileW::LD + TM_ * TileY::LD;
    extern __shared__ __align__(16) unsigned char smem[];
    T *const lds = reinterpret_cast<T *>(smem);
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), i16 = lane & 15, g = lane >> 4;
    const int64_t task = task_of((a.rows + TM_ - 1) / TM_ * a.ktiles);
    if (task < 0) return;
    const int64_t r0 = task / a.ktiles * TM_;
    const int k0 = (int)(task % a.ktiles) * TK;
    // float32: a layer's share is summed by itself, as products one after another would sum it (three layers of 128: 3.5e-7 -> 2.1e-7, the
    // array library's error; 131072 x 128 138 -> 142 us).  bfloat16 operands hide the difference.
    constexpr bool BY_LAYER = sizeof(T) == 4;
    f32x4 acc[TM::TPW], total[BY_LAYER ? TM::TPW : 1];
    zero_acc<TM::TPW>(acc);
    zero_acc<(BY_LAYER ? TM::TPW : 1)>(total);
    bool last[2] = {false, false};   // of its layer
    TileW tw[2];   // the steps on their way: two, so that a trip to memory spans two products
    TileY ty[2];
    int l = 0, n0 = 0, steps = 0;   // where the next fetch reads; steps fetched and not yet multiplied
    auto fetch = [&](int i) {
        if (l >= a.layers) return;
        tw[i].load(static_cast<const T *>(a.w[l]), n0, a.n[l], a.n[l], k0, a.K, tid);
        ty[i].load(static_cast<const T *>(a.dy[l]), r0, a.rows, a.rows, n0, a.n[l], tid);
        n0 += NC;
        last[i] = n0 >= a.n[l];
        if (last[i]) ++l, n0 = 0;
        ++steps;
    };
    fetch(0);
    fetch(1);
    auto step = [&](int i) {
        T *const sw = lds + i * BUF, *const sy = sw + NC * TileW::LD;
        tw[i].to_lds(sw, tid);
        ty[i].to_lds(sy, tid);
        --steps;
        const bool ends = last[i];
        fetch(i);
        sync_lds();
        gemm<T, TK, TM_, NC, KROW, ROWK, DG_WAVES, MBW>(acc, sw, TileW::LD, sy, TileY::LD, w, lane);
        if (BY_LAYER && ends) {
#pragma unroll
            for (int j = 0; j < TM::TPW; ++j) total[j] += acc[j];
            zero_acc<TM::TPW>(acc);
        }
    };
    while (steps > 0) {
        step(0);
        if (steps > 0) step(1);
    }
#pragma unroll
    for (int j = 0; j < TM::TPW; ++j) {
        const int k = k0 + TM::mt(w, j) * 16 + 4 * g;
        const int64_t r = r0 + TM::nt(w, j) * 16 + i16;
        if (k >= a.K || r >= a.rows) continue;
        const int64_t at = r * a.K + k;
        const f32x4 y = BY_LAYER ? total[BY_LAYER ? j : 0] : acc[j];
        if (a.dx_bf16) *reinterpret_cast<bf16x4 *>(static_cast<__bf16 *>(a.dx) + at) = TT<__bf16>::pack(y[0], y[1], y[2], y[3]);
        else *reinterpret_cast<f32x4 *>(static_cast<float *>(a.dx) + at) = y;
    }
}

template <typename T, int R1, int W1, int R2, int W2, OpMode M2> constexpr size_t dg_lds()
{
    return 2 * sizeof(T) * (R1 * RowTile<T, R1, W1, KROW>::LD + R2 * RowTile<T, R2, W2, M2>::LD);
}

struct WeightPlan {
    int tn, tk, tiles, slices;
    int64_t slice_rows, total;
};
// 128 x 128 tiles, 64 where the layers are narrower; the rows cut so that five hundred workgroups run (two per compute unit), but no
// shorter than four steps of a workgroup, and a whole number of such rounds where a slice would have more than CHAIN rows: a running
// sum in float32 errs in proportion to its length.  131072 rows, three layers of 256 x 256 and one of 256 x 4, error of the weights against
// float64: bfloat16 (3648 rows a slice) 8.4e-8 -> 4.5e-8, where the array library's slices have 5.2e-8, 132 -> 134 us; float32 1.6e-7 -> 4.4e-8
// (library 9.3e-8), 576 -> 618 us.
constexpr int64_t CHAIN_BF16 = 2048, CHAIN_F32 = 512;
WeightPlan plan_weights(int64_t rows, int64_t K, const int64_t *n, int layers, bool bf16, unsigned bias_mask)
{
    WeightPlan p{};
    int64_t widest = 0;
    for (int l = 0; l < layers; ++l) widest = n[l] > widest ? n[l] : widest;
    p.tn = widest <= 64 ? 64 : 128, p.tk = K <= 64 ? 64 : 128;
    const int64_t rc = bf16 ? 64 : 32, ktiles = (K + p.tk - 1) / p.tk;
    int64_t tiles = 0;
    for (int l = 0; l < layers; ++l) {
        tiles += (n[l] + p.tn - 1) / p.tn * ktiles;
        p.total += n[l] * K;
    }
    for (int l = 0; l < layers; ++l)
        if (bias_mask >> l & 1) p.total += n[l];
    p.total = (p.total + 3) / 4 * 4;   // rows of partial results start on 16-byte boundaries
    const int64_t most = (rows + 4 * rc - 1) / (4 * rc);
    int64_t s = tiles >= 512 ? 1 : 512 / tiles;
    s = s > most ? most : s;
    const int64_t chain = bf16 ? CHAIN_BF16 : CHAIN_F32;
    if (tiles < 512 && rows > s * chain) s = (rows + s * chain - 1) / (s * chain) * 512 / tiles;
    p.slice_rows = ((rows + s - 1) / s + rc - 1) / rc * rc;
    p.slices = (int)((rows + p.slice_rows - 1) / p.slice_rows);
    p.tiles = (int)tiles;
    return p;
}

template <typename T, int TN, int TK> int launch_weight_grads(hipStream_t st, DenseGradArgs &a, const WeightPlan &p)
{
    for (int l = 0; l < a.layers; ++l) a.first_tile[l + 1] = a.first_tile[l] + (a.n[l] + TN - 1) / TN;
    a.ktiles = (a.K + TK - 1) / TK;
    return launch_kernel(dense_weight_grad_kernel<T, TN, TK>, dim3(grid_of((int64_t)p.tiles * p.slices)), dim3(DG_THREADS),
                         dg_lds<T, dg_rows<T>(), TK, dg_rows<T>(), TN, KROW>(), st, a);
}
template <typename T, int TM, int TK> int launch_input_grad(hipStream_t st, DenseGradArgs &a)
{
    a.ktiles = (a.K + TK - 1) / TK;
    return launch_kernel(dense_input_grad_kernel<T, TM, TK>, dim3(grid_of((a.rows + TM - 1) / TM * a.ktiles)), dim3(DG_THREADS),
                         dg_lds<T, dg_rows<T>(), TK, TM, dg_rows<T>(), ROWK>(), st, a);
}

template <typename T> int launch_grads(hipStream_t st, DenseGradArgs &a, const WeightPlan &p, float *params, float *workspace)
{
    if (a.dx) {
        // rows and features per workgroup: large tiles read dy and the weights less often, small ones fill the device
        const int64_t large = (a.rows + 127) / 128 * ((a.K + 127) / 128);
        const int rc = a.K <= 64 ? (a.rows >= 128 * 512 ? launch_input_grad<T, 128, 64>(st, a) : launch_input_grad<T, 64, 64>(st, a))
                       : large >= 512 ? launch_input_grad<T, 128, 128>(st, a)
                                      : launch_input_grad<T, 64, 64>(st, a);
        if (rc != MRX_OK) return rc;
    }
    if (!params) return MRX_OK;
    a.slices = p.slices, a.slice_rows = p.slice_rows, a.total = p.total;
    a.out = p.slices == 1 ? params : workspace;
    const int rc = p.tn == 64 ? (p.tk == 64 ? launch_weight_grads<T, 64, 64>(st, a, p) : launch_weight_grads<T, 64, 128>(st, a, p))
                              : (p.tk == 64 ? launch_weight_grads<T, 128, 64>(st, a, p) : launch_weight_grads<T, 128, 128>(st, a, p));
    if (rc != MRX_OK || p.slices == 1) return rc;
    return launch_column_sum(st, workspace, params, nullptr, p.slices, (int)p.total);
}

template <typename T> constexpr int big_lds = (int)dg_lds<T, 128, 128, 128, 128, KROW>();
const KernelRegistrar registrars[] = {
    {reinterpret_cast<const void *>(dense_weight_grad_kernel<__bf16, 128, 128>), big_lds<__bf16>},
    {reinterpret_cast<const void *>(dense_weight_grad_kernel<float, 128, 128>), big_lds<__bf16>},
    {reinterpret_cast<const void *>(dense_input_grad_kernel<__bf16, 128, 128>), big_lds<__bf16>},
    {reinterpret_cast<const void *>(dense_input_grad_kernel<float, 128, 128>), big_lds<__bf16>},
};

bool dense_shape_ok(int64_t rows, int64_t K, const int64_t *n, int layers)
{
    if (!n || layers < 1 || layers > MRX_DENSE_LAYERS || rows <= 0 || rows >= (1ll << 31) || K <= 0 || K % 8 != 0 || K > (1 << 16)) return false;
    for (int l = 0; l < layers; ++l)
        if (n[l] <= 0 || n[l] > (1 << 16)) return false;
    return true;
}

}  // namespace
}  // namespace mrx

extern "C" int64_t mrx_dense_grads_workspace(int64_t rows, int64_t K, const int64_t *n_out, int layers, int dtype, unsigned bias_mask)
{
    using namespace mrx;
    if (!dense_shape_ok(rows, K, n_out, layers)) return 0;
    const WeightPlan p = plan_weights(rows, K, n_out, layers, dtype == MRX_BF16, bias_mask);
    return p.slices == 1 ? 0 : p.slices * p.total;
}

extern "C" int mrx_dense_grads(void *stream, const void *x, const void *const *dys, const void *const *weights, const int64_t *n_out,
                               int layers, void *dx, float *params, float *workspace, int64_t rows, int64_t K, int dtype, int dx_dtype,
                               unsigned bias_mask)
{
    using namespace mrx;
    if (!dys || !dense_shape_ok(rows, K, n_out, layers) || (!dx && !params)) return MRX_ERR_INVALID_ARG;
    if ((dtype != MRX_F32 && dtype != MRX_BF16) || (dx_dtype != MRX_F32 && dx_dtype != MRX_BF16)) return MRX_ERR_INVALID_ARG;
    const bool bf = dtype == MRX_BF16;
    const size_t esize = bf ? 2 : 4;
    DenseGradArgs a{};
    a.x = x, a.dx = dx, a.dx_bf16 = dx_dtype == MRX_BF16, a.layers = layers, a.K = (int)K, a.rows = rows;
    if (params && (!x || !aligned(x, 16) || !aligned(params, 16))) return MRX_ERR_INVALID_ARG;
    if (dx && (!weights || !aligned(dx, 16))) return MRX_ERR_INVALID_ARG;
    int64_t at = 0;
    for (int l = 0; l < layers; ++l) {
        if (!dys[l] || !aligned(dys[l], esize) || (dx && (!weights[l] || !aligned(weights[l], 16)))) return MRX_ERR_INVALID_ARG;
        a.dy[l] = dys[l], a.w[l] = dx ? weights[l] : nullptr, a.n[l] = (int)n_out[l];
        a.w_at[l] = at, at += n_out[l] * K;
    }
    for (int l = 0; l < layers; ++l) {
        a.b_at[l] = -1;
        if (bias_mask >> l & 1) a.b_at[l] = at, at += n_out[l];
    }
    const WeightPlan p = plan_weights(rows, K, n_out, layers, bf, bias_mask);
    if (params && p.slices > 1 && (!workspace || !aligned(workspace, 16))) return MRX_ERR_INVALID_ARG;
    if ((int64_t)p.tiles * p.slices >= (1ll << 31) || p.total >= (1ll << 31) || (rows + 63) / 64 * ((K + 63) / 64) >= (1ll << 31))
        return MRX_ERR_INVALID_ARG;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    return bf ? launch_grads<__bf16>(st, a, p, params, workspace) : launch_grads<float>(st, a, p, params, workspace);
}
