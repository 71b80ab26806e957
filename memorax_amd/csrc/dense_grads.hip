// Gradients of dense layers that read the same rows, for a whole group of them:
//
//     dW_l = dy_l^T x      db_l = sum over the rows of dy_l      dx = sum_l dy_l W_l
//
// A rollout batch has a hundred thousand rows and a few hundred features.  The first two are products with a tiny result and an
// enormous inner dimension, the third is one whose operands are read once; all are bound by reading dy and x.  The array
// library runs them as a product per layer and direction -- with the rows cut into slices by hand, a reduction per layer over
// those, a reduction per bias, and the sum of the input gradients rounded and read back between the layers -- most of them at a
// fraction of the bandwidth (131072 rows, three layers of 256 x 256 and one of 256 x 4 in bfloat16: 330 us for the parameters and 150 us
// for the input; 11455 rows, three of 128 x 256: 225 and 23 us).  Here they are two launches and one reduction: 104 (on wide tiles, below; 134 on the others) and
// 118 us, 24 and 16 us; the input's gradient in bfloat16 over wide rows is dense_rows.hip's (60 us), in float32 dense_split.hip's, the kernel here serves the rest.  At 256 features a compute unit is short of loads in flight rather than of bandwidth: LDS holds two steps of two workgroups.
//
// Weight gradients: a workgroup of four waves owns a TN x TK tile of one layer's result and a slice of the rows, 64 (float32: 32, below)
// of which wait in LDS while the next are on their way; both operands are contracted over their rows, which the transposing
// LDS reads serve without a copy.  The slices' partial results are summed in a fixed order (col_sum.h).
// Input gradient: a workgroup owns TM rows and TK features and walks the layers' outputs, two steps ahead in registers (one step: 120
// -> 115 us at 131072 rows, 19.9 -> 17.3 us at 11455 rows of the sizes above.  The weight gradients are bound by the transposing reads
// of both operands instead: a second step there costs the registers those need, 123 -> 147 us).
#include "chunk_common.h"
#include "col_sum.h"
#include "dense_split.h"
#include "row_dma.h"
#include "split_bf16.h"

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

constexpr int DG_STEP = 64, SG_STEP = 32;   // rows (weight gradients) or outputs (dx) of a step, in bfloat16 and in float32

// Workgroups are dealt to the eight dies in turn, and tasks that read the same rows follow each other: each die takes a contiguous
// share of them, and its L2 serves the second reader.  -1: none left.
__device__ __forceinline__ int64_t task_of(int64_t tasks)
{
    const int64_t t = (blockIdx.x & 7) * ((tasks + 7) / 8) + (blockIdx.x >> 3);
    return (int64_t)(blockIdx.x >> 3) < (tasks + 7) / 8 && t < tasks ? t : -1;
}
inline unsigned grid_of(int64_t tasks) { return (unsigned)((tasks + 7) / 8 * 8); }

template <int TN, int TK>
__global__ void __launch_bounds__(DG_THREADS, 2) dense_weight_grad_kernel(DenseGradArgs a)
{
    using T = __bf16;
    constexpr int RC = DG_STEP, MBW = TK / 32, NBW = TN / 32;
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
    TileX tx;
    TileY ty;
    tx.load(x, r0, r1, a.rows, k0, a.K, tid);
    ty.load(dy, r0, r1, a.rows, n0, N, tid);
    int buf = 0;
    for (int64_t r = r0; r < r1; r += RC, buf ^= 1) {
        T *const sx = lds + buf * BUF, *const sy = sx + RC * TileX::LD;
        tx.to_lds(sx, tid);
        ty.to_lds(sy, tid);
        if (r + RC < r1) {
            tx.load(x, r + RC, r1, a.rows, k0, a.K, tid);
            ty.load(dy, r + RC, r1, a.rows, n0, N, tid);
        }
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
    if (bias && g == 0) {
#pragma unroll
        for (int j = 0; j < NBW; ++j) {
            const int n = n0 + TM::nt(w, j) * 16 + i16;
            if (n < N) out[a.b_at[l] + n] = accb[j][0];
        }
    }
}

// ---- weight gradients in float32 on the bfloat16 matrix units (split_bf16.h)
// The same tiles and slices; a step's 32 rows are split into three bfloat16 tiles an operand on their way into LDS, 55 KB of them, one step at a time: two
// workgroups of a compute unit take turns, one on its way to memory and splitting while the other multiplies (two buffers leave room for one workgroup: 365 us).
// us, here / the array library: 32768 x 256 -> 1024 + 512 + 512 + 8 259 / 289, 131072 x 256 -> 3 x 256 + 4 412 / 414, 131072 x 128 -> 3 x 128 104 / 125, 4096 x 256
// -> 3 x 256 36 / 79.  Of the first's cycles the matrix units are busy 36 %, the vector ALU 39 % (splitting, addresses, the sums of small products) and LDS
// 27 %, in two workgroups' turns.
template <int W> __device__ __forceinline__ bf16x8 split_fragment(const __bf16 *tile, int c0, int lane)
{
    return TT<__bf16>::template load<KROW>(tile, W + 16, c0, 0, lane);   // (as RowTile::LD)
}

// One operand's step: 32 rows x W columns in registers.
template <int W> struct SplitTile {
    using Rows = RowTile<float, 32, W, KROW>;
    static constexpr int LD = W + 16, PART = 32 * LD;   // bfloat16 between rows; of one part
    static constexpr int COLS = W / 4;                  // threads across
    Rows rows;
    // columns past the last count nothing
    __device__ __forceinline__ void mask(int tid)
    {
        const int have = rows.cols - tid % COLS * 4;
        if (have < 4)
#pragma unroll
            for (int p = 0; p < Rows::PASSES; ++p)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (q >= have) rows.v[p][q] = 0u;
    }
    // the largest of this thread's values; in three tiles
    __device__ __forceinline__ float to_lds(__bf16 *dst, int tid)
    {
        float most = 0.f;
#pragma unroll
        for (int p = 0; p < Rows::PASSES; ++p) {
            const f32x4 x = __builtin_bit_cast(f32x4, rows.v[p]);
            most = max4(most, x);
            Words<2>::type parts[PARTS];
            split_parts<2>(&x, parts);
            const int at = (tid / COLS + p * (DG_THREADS / COLS)) * LD + tid % COLS * 4;
#pragma unroll
            for (int h = 0; h < PARTS; ++h) *reinterpret_cast<Words<2>::type *>(dst + h * PART + at) = parts[h];
        }
        return most;
    }
};

template <int TN, int TK> constexpr size_t split_lds() { return PARTS * (SplitTile<TN>::PART + SplitTile<TK>::PART) * sizeof(__bf16); }

template <int TN, int TK> __global__ void __launch_bounds__(DG_THREADS, 2) split_weight_grad_kernel(DenseGradArgs a)
{
    constexpr int RC = SG_STEP, MBW = TK / 32, NBW = TN / 32;
    using TM = TileMap<TK, TN, DG_WAVES, MBW>;
    static_assert(RC == 32, "one block of the contraction a step");
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int beyond;   // a value without parts is among the operands
    __bf16 *const sx = reinterpret_cast<__bf16 *>(smem), *const sy = sx + PARTS * SplitTile<TK>::PART;
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
    const float *x = static_cast<const float *>(a.x), *dy = static_cast<const float *>(a.dy[l]);
    const bool bias = a.b_at[l] >= 0 && kt == 0;
    if (tid == 0) beyond = 0;
    sync_lds();   // before any wave sets it

    f32x4 acc[TM::TPW];
    zero_acc<TM::TPW>(acc);
    // the bias gradient, a step's sum at a time with what its additions round off
    f32x4 bias_sum = {0.f, 0.f, 0.f, 0.f}, bias_low = bias_sum;
    SplitTile<TK> tx;
    SplitTile<TN> ty;
    auto load = [&](int64_t r) {
        tx.rows.load(x, r, r1, a.rows, k0, a.K, tid);
        ty.rows.load(dy, r, r1, a.rows, n0, N, tid);
    };
    load(r0);
    float most = 0.f;
    for (int64_t r = r0; r < r1; r += RC) {
        tx.mask(tid);
        ty.mask(tid);
        if (bias) {
            f32x4 part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int p = 0; p < SplitTile<TN>::Rows::PASSES; ++p) part += __builtin_bit_cast(f32x4, ty.rows.v[p]);
            const f32x4 y = part - bias_low, s = bias_sum + y;
#pragma unroll
            for (int q = 0; q < 4; ++q) bias_low[q] = fabsf(s[q]) <= 3.402823466e38f ? (s[q] - bias_sum[q]) - y[q] : 0.f;   // an infinite sum rounds nothing off
            bias_sum = s;
        }
        if (r > r0) sync_lds();   // the step before has been read
        most = fmaxf(most, fmaxf(tx.to_lds(sx, tid), ty.to_lds(sy, tid)));
        if (r + RC < r1) load(r + RC);
        sync_lds();
        bf16x8 fx[MBW][PARTS];
#pragma unroll
        for (int m = 0; m < MBW; ++m)
#pragma unroll
            for (int h = 0; h < PARTS; ++h) fx[m][h] = split_fragment<TK>(sx + h * SplitTile<TK>::PART, TM::mt(w, m * TM::NBW) * 16, lane);
#pragma unroll
        for (int n = 0; n < NBW; ++n) {
            bf16x8 fy[PARTS];
#pragma unroll
            for (int h = 0; h < PARTS; ++h) fy[h] = split_fragment<TN>(sy + h * SplitTile<TN>::PART, TM::nt(w, n) * 16, lane);
            // the small products by themselves first: two roundings of the running sum a step
            f32x4 low[MBW];
#pragma unroll
            for (int q = 0; q < PRODUCTS; ++q)
#pragma unroll
                for (int m = 0; m < MBW; ++m) {
                    if (q + 1 < PRODUCTS) low[m] = mma_bf16(fx[m][PART_A[q]], fy[PART_B[q]], q ? low[m] : f32x4{0.f, 0.f, 0.f, 0.f});
                    else acc[m * TM::NBW + n] = mma_bf16(fx[m][0], fy[0], acc[m * TM::NBW + n]);
                }
#pragma unroll
            for (int m = 0; m < MBW; ++m) acc[m * TM::NBW + n] += low[m];
        }
    }
    if (most > BF16_MOST) beyond = 1;
    sync_lds();
    float *const out = a.out + slice * a.total;
    if (beyond) {   // sums one by one: what an infinity makes of them is float32's
        for (int e = tid; e < TN * TK; e += DG_THREADS) {
            const int n = n0 + e / TK, k = k0 + e % TK;
            if (n >= N || k >= a.K) continue;
            float sum = 0.f;
            for (int64_t r = r0; r < r1; ++r) sum = fmaf(dy[r * N + n], x[r * a.K + k], sum);
            out[a.w_at[l] + (int64_t)n * a.K + k] = sum;
        }
    } else {
#pragma unroll
        for (int j = 0; j < TM::TPW; ++j) {
            const int ki = TM::mt(w, j) * 16 + 4 * g, ni = TM::nt(w, j) * 16 + i16;
            if (k0 + ki >= a.K || n0 + ni >= N) continue;
            *reinterpret_cast<f32x4 *>(out + a.w_at[l] + (int64_t)(n0 + ni) * a.K + k0 + ki) = acc[j];
        }
    }
    if (bias) {   // the threads' shares of a column, in pairs
        constexpr int SHARES = DG_THREADS / SplitTile<TN>::COLS;
        float *const part = reinterpret_cast<float *>(smem);
        sync_lds();
        *reinterpret_cast<f32x4 *>(part + tid / SplitTile<TN>::COLS * TN + tid % SplitTile<TN>::COLS * 4) = bias_sum;
        sync_lds();
        if (tid < TN && n0 + tid < N) {
            float t[SHARES];
#pragma unroll
            for (int s = 0; s < SHARES; ++s) t[s] = part[s * TN + tid];
#pragma unroll
            for (int half = SHARES / 2; half > 0; half /= 2)
#pragma unroll
                for (int s = 0; s < half; ++s) t[s] += t[s + half];
            out[a.b_at[l] + n0 + tid] = t[0];
        }
    }
}

// ---- weight gradients in bfloat16 on tiles of 256 x 256
// Four times the tile of the kernel above reads the rows half as often, and a ring of row tiles that go from memory to LDS directly
// (row_dma.h) keeps three or four steps on their way where registers held one: one workgroup of eight waves on a compute unit, one
// barrier a step of 32 rows.  Granules of 32 bytes are exchanged within a row (`granule`), so that the transposing reads, which take 32
// bytes of sixteen rows at once, spread over the banks.  131072 rows x 256, with the partial results' sum, us: three layers of 256
// 131 -> 98-103, with one of 4 beside them 146 -> 109.
constexpr int WT_WAVES = 8, WT_THREADS = 64 * WT_WAVES, WT_ROWS = 32, WT_NARROW = 8, WT_SLOTS = 256;

struct WideGradArgs {
    const __bf16 *x, *dy[MRX_DENSE_LAYERS], *dyn;   // dyn: of a layer of nn outputs beside the wide ones
    float *out;                                     // (slices, total)
    int64_t w_at[MRX_DENSE_LAYERS], b_at[MRX_DENSE_LAYERS], wn_at, bn_at;
    int n[MRX_DENSE_LAYERS], first_tile[MRX_DENSE_LAYERS + 1];
    int layers, nn, K, ktiles, tiles, slices;
    int64_t rows, slice_rows, total;
};

// Granule c of row r of a tile lies at c ^ granule(r): the rows that one transposing read takes (four and, eight further on, four more, by
// each half wave) in eight different places.
__device__ __forceinline__ int granule(int r) { return (r & 3) | (r >> 3 & 1) << 2; }
__device__ __forceinline__ bf16x8 transposed_fragment(const unsigned char *p, int four_rows)
{
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    union {
        s16x4 h[2];
        bf16x8 f;
    } u;
    u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)p);
    u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(p + four_rows));
    return u.f;
}

template <bool NARROW> struct WideTile {
    static constexpr int W = 256, WN = 2, WK = WT_WAVES / WN;        // outputs and features; waves across the outputs, across the features
    static constexpr int NT = W / 16 / WN, KT = W / 16 / WK;         // 16 x 16 tiles of a wave
    static constexpr int XB = WT_ROWS * W * 2, YB = XB, NB = NARROW ? WT_ROWS * WT_NARROW * 2 : 0, STAGE = XB + YB + NB;
    static constexpr int OPS = (XB + YB) / 1024 / WT_WAVES, STAGES = 160 * 1024 / STAGE;
    static_assert((XB + YB) % (1024 * WT_WAVES) == 0 && NT % WK == 0 && KT % WN == 0, "whole requests and tiles");
};

template <bool NARROW>   // a layer of nn outputs beside the wide ones
__global__ void __launch_bounds__(WT_THREADS, 1) wide_weight_grad_kernel(WideGradArgs a)
{
    using T = WideTile<NARROW>;
    constexpr int RBX = T::W * 2, RBY = RBX, NT = T::NT, KT = T::KT, STAGES = T::STAGES;
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 15, g = lane >> 4;
    const int64_t task = task_of((int64_t)a.tiles * a.slices);
    if (task < 0) return;
    const int slice = (int)(task / a.tiles), tile = (int)(task % a.tiles);
    const int kt = tile % a.ktiles, nt = tile / a.ktiles;
    int l = 0;
    while (nt >= a.first_tile[l + 1]) ++l;
    const int n0 = (nt - a.first_tile[l]) * T::W, k0 = kt * T::W, N = a.n[l];
    const int64_t r0 = slice * a.slice_rows, r1 = r0 + a.slice_rows < a.rows ? r0 + a.slice_rows : a.rows;
    const int steps = (int)((r1 - r0 + WT_ROWS - 1) / WT_ROWS);
    const bool narrow = NARROW && nt == 0;                        // the narrow layer's gradient is these workgroups' too
    const bool bias = a.b_at[l] >= 0 && kt == 0, bias_n = narrow && a.bn_at >= 0 && kt == 0 && wv == 0;
    const bool requests_n = narrow && wv < T::NB / 256;
    const uint32_t lds0 = lds_address(smem);

    // every request of a step is made whatever exists of it: rows past the last are the last one, steps past the last are the last one
    auto request = [&](int step, int stage) {
        if (step >= steps) step = steps - 1;
        const int64_t r = r0 + (int64_t)step * WT_ROWS;
        const int last = (int)(a.rows - 1 - r < WT_ROWS - 1 ? a.rows - 1 - r : WT_ROWS - 1);
        const uint32_t at = lds0 + stage * T::STAGE;
#pragma unroll
        for (int p = 0; p < T::OPS; ++p) {
            const int op = wv * T::OPS + p;
            const bool of_x = op < T::XB / 1024;
            const int o = of_x ? op : op - T::XB / 1024, row = o * 2 + lane / 32, q = lane % 32 ^ granule(row) << 1;
            const uint32_t wide = of_x ? a.K : N;
            const __bf16 *base = of_x ? a.x + r * a.K + k0 : a.dy[l] + r * N + n0;
            dma16(base, (uint32_t)(row < last ? row : last) * wide * 2 + q * 16, at + op * 1024);
        }
        if (requests_n) {
            const uint32_t off = wv * 256 + lane * 4, end = (uint32_t)((last + 1) * a.nn * 2 - 4);
            dma4(a.dyn + r * a.nn, off < end ? off : end, at + T::XB + T::YB + wv * 256);
        }
    };
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s) request(s, s);

    const int wn = wv / T::WK, wk = wv % T::WK;
    constexpr int BT = NT / T::WK, ST = KT / T::WN;   // of the bias and of the narrow layer: each wave its share
    f32x4 acc[KT][NT], accb[BT], accn[ST], accbn = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KT; ++k) zero_acc<NT>(acc[k]);
    zero_acc<BT>(accb);
    zero_acc<ST>(accn);
    const int row = 8 * g + (i >> 2), sw = granule(row);
    int stage = 0;
    for (int step = 0; step < steps; ++step) {
        if (requests_n) wait_vm<(STAGES - 2) * (T::OPS + 1)>();
        else wait_vm<(STAGES - 2) * T::OPS>();
        sync_lds();   // every wave has its part, and is done with the step before, whose place the next request takes
        request(step + STAGES - 1, stage == 0 ? STAGES - 1 : stage - 1);
        unsigned char *const sx = smem + stage * T::STAGE, *const sy = sx + T::XB, *const sn = sy + T::YB;
        const int have = (int)(r1 - r0 - (int64_t)step * WT_ROWS);
        if (have < WT_ROWS) {   // of the last step: rows that are not there count nothing
            for (int e = tid; e < (WT_ROWS - have) * (RBX / 4); e += WT_THREADS) reinterpret_cast<uint32_t *>(sx + have * RBX)[e] = 0u;
            for (int e = tid; e < (WT_ROWS - have) * (RBY / 4); e += WT_THREADS) reinterpret_cast<uint32_t *>(sy + have * RBY)[e] = 0u;
            if (narrow)
                for (int e = tid; e < (WT_ROWS - have) * a.nn / 2; e += WT_THREADS) reinterpret_cast<uint32_t *>(sn + have * a.nn * 2)[e] = 0u;
            sync_lds();
        }
        const unsigned char *px = sx + row * RBX + (i & 3) * 8, *py = sy + row * RBY + (i & 3) * 8;
        bf16x8 fx[KT];
#pragma unroll
        for (int k = 0; k < KT; ++k) fx[k] = transposed_fragment(px + ((wk * KT + k) ^ sw) * 32, 4 * RBX);
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const bf16x8 fy = transposed_fragment(py + ((wn * NT + n) ^ sw) * 32, 4 * RBY);
#pragma unroll
            for (int k = 0; k < KT; ++k) acc[k][n] = TT<__bf16>::mma(fx[k], fy, acc[k][n]);
        }
        if (bias)
#pragma unroll
            for (int j = 0; j < BT; ++j)
                accb[j] = TT<__bf16>::mma(TT<__bf16>::ones(), transposed_fragment(py + ((wn * NT + wk * BT + j) ^ sw) * 32, 4 * RBY), accb[j]);
        if (narrow) {
            bf16x8 fy = {};
            if (i < a.nn)
#pragma unroll
                for (int e = 0; e < 8; ++e) fy[e] = reinterpret_cast<const __bf16 *>(sn)[(8 * g + e) * a.nn + i];
#pragma unroll
            for (int j = 0; j < ST; ++j)
                accn[j] = TT<__bf16>::mma(transposed_fragment(px + ((wk * KT + wn * ST + j) ^ sw) * 32, 4 * RBX), fy, accn[j]);
            if (bias_n) accbn = TT<__bf16>::mma(TT<__bf16>::ones(), fy, accbn);
        }
        stage = stage == STAGES - 1 ? 0 : stage + 1;
    }
    wait_vm<0>();
    float *const out = a.out + slice * a.total;
#pragma unroll
    for (int k = 0; k < KT; ++k)
#pragma unroll
        for (int n = 0; n < NT; ++n)
            *reinterpret_cast<f32x4 *>(out + a.w_at[l] + (int64_t)(n0 + (wn * NT + n) * 16 + i) * a.K + k0 + (wk * KT + k) * 16 + 4 * g) = acc[k][n];
    if (bias && g == 0)
#pragma unroll
        for (int j = 0; j < BT; ++j) out[a.b_at[l] + n0 + (wn * NT + wk * BT + j) * 16 + i] = accb[j][0];
    if (narrow && i < a.nn) {
#pragma unroll
        for (int j = 0; j < ST; ++j)
            *reinterpret_cast<f32x4 *>(out + a.wn_at + (int64_t)i * a.K + k0 + (wk * KT + wn * ST + j) * 16 + 4 * g) = accn[j];
        if (bias_n && g == 0) out[a.bn_at + i] = accbn[0];
    }
}

template <int TM_, int TK>
__global__ void __launch_bounds__(DG_THREADS, 2) dense_input_grad_kernel(DenseGradArgs a)
{
    using T = __bf16;
    constexpr int NC = DG_STEP, MBW = TK / 32;
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
    f32x4 acc[TM::TPW];
    zero_acc<TM::TPW>(acc);
    TileW tw[2];   // the steps on their way: two, so that a trip to memory spans two products
    TileY ty[2];
    int l = 0, n0 = 0, steps = 0;   // where the next fetch reads; steps fetched and not yet multiplied
    auto fetch = [&](int i) {
        if (l >= a.layers) return;
        tw[i].load(static_cast<const T *>(a.w[l]), n0, a.n[l], a.n[l], k0, a.K, tid);
        ty[i].load(static_cast<const T *>(a.dy[l]), r0, a.rows, a.rows, n0, a.n[l], tid);
        n0 += NC;
        if (n0 >= a.n[l]) ++l, n0 = 0;
        ++steps;
    };
    fetch(0);
    fetch(1);
    auto step = [&](int i) {
        T *const sw = lds + i * BUF, *const sy = sw + NC * TileW::LD;
        tw[i].to_lds(sw, tid);
        ty[i].to_lds(sy, tid);
        --steps;
        fetch(i);
        sync_lds();
        gemm<T, TK, TM_, NC, KROW, ROWK, DG_WAVES, MBW>(acc, sw, TileW::LD, sy, TileY::LD, w, lane);
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
        const f32x4 y = acc[j];
        if (a.dx_bf16) *reinterpret_cast<bf16x4 *>(static_cast<__bf16 *>(a.dx) + at) = TT<__bf16>::pack(y[0], y[1], y[2], y[3]);
        else *reinterpret_cast<f32x4 *>(static_cast<float *>(a.dx) + at) = y;
    }
}

template <int R1, int W1, int R2, int W2, OpMode M2> constexpr size_t dg_lds()
{
    return 2 * sizeof(__bf16) * (R1 * RowTile<__bf16, R1, W1, KROW>::LD + R2 * RowTile<__bf16, R2, W2, M2>::LD);
}

struct WeightPlan {
    int tn, tk, tiles, slices, narrow;   // narrow: the layer that rides along, -1
    int64_t slice_rows, total;
    bool wide;                           // wide_weight_grad_kernel
};
// 128 x 128 tiles, 64 where the layers are narrower; the rows cut so that five hundred workgroups run (two per compute unit), but no
// shorter than four steps of a workgroup, and a whole number of such rounds where a slice would have more than CHAIN rows: a running
// sum in float32 errs in proportion to its length.  131072 rows, three layers of 256 x 256 and one of 256 x 4, error of the weights against
// float64: bfloat16 (3648 rows a slice) 8.4e-8 -> 4.5e-8, where the array library's slices have 5.2e-8, 132 -> 134 us.  A float32 slice may be longer
// than on float32 products (512 rows, 3.9e-7), with a quarter of their roundings: 32768 x 256 -> 2056 outputs 512 rows a slice 1.5e-7 and 280 us, 1152 2.3e-7 and
// 259 us; the array library 8.1e-7.
constexpr int64_t CHAIN_BF16 = 2048, CHAIN_F32 = 1152;

constexpr int64_t WIDE_WORK = 3 << 16;
// The plan on wide tiles, for bfloat16 layers whose sizes are whole tiles (one of two, four, six or eight outputs may ride along): one round of
// workgroups, or whole rounds where a slice would be longer than CHAIN.  Its partial results are 64 MB whatever the rows, so it needs rows
// times tiles (us, here / the plan below): three layers of 256 x 256 16384 rows 35 / 31, 49152 53 / 53, 65536 61 / 63, 100000 80 / 101,
// 131072 98-103 / 131 and with one of 4 beside them 109 / 146; one of 512 x 512 32768 rows 48 / 47, 65536 68 / 77, 131072 118 / 151; two
// of 256 x 256 65536 rows 49 / 46, 100000 63 / 64, 131072 72 / 77.  Tiles of half the size gained 8 % at 131072 rows and lost below 65536.
bool plan_wide(WeightPlan &p, int64_t rows, int64_t K, const int64_t *n, int layers)
{
    if (K % 256 != 0) return false;
    p.narrow = -1;
    int64_t columns = 0;
    for (int l = 0; l < layers; ++l) {
        if (n[l] <= WT_NARROW && n[l] % 2 == 0 && p.narrow < 0) {
            p.narrow = l;
            continue;
        }
        if (n[l] % 256 != 0) return false;
        columns += n[l];
    }
    const int64_t tiles = columns / 256 * (K / 256);
    if (tiles < 2 || tiles > WT_SLOTS || rows * tiles < WIDE_WORK) return false;
    const int64_t s = WT_SLOTS / tiles, rounds = (rows + s * CHAIN_BF16 - 1) / (s * CHAIN_BF16);
    p.tiles = (int)tiles;
    p.slice_rows = ((rows + rounds * s - 1) / (rounds * s) + WT_ROWS - 1) / WT_ROWS * WT_ROWS;
    p.slices = (int)((rows + p.slice_rows - 1) / p.slice_rows);
    return true;
}
WeightPlan plan_weights(int64_t rows, int64_t K, const int64_t *n, int layers, bool bf16, unsigned bias_mask, bool wide)
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
    if (wide && bf16 && plan_wide(p, rows, K, n, layers)) {
        p.wide = true;
        return p;
    }
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

template <int TN, int TK> int launch_weight_grads(hipStream_t st, DenseGradArgs &a, const WeightPlan &p, bool bf16)
{
    for (int l = 0; l < a.layers; ++l) a.first_tile[l + 1] = a.first_tile[l] + (a.n[l] + TN - 1) / TN;
    a.ktiles = (a.K + TK - 1) / TK;
    const dim3 grid(grid_of((int64_t)p.tiles * p.slices));
    return bf16 ? launch_kernel(dense_weight_grad_kernel<TN, TK>, grid, dim3(DG_THREADS), dg_lds<DG_STEP, TK, DG_STEP, TN, KROW>(), st, a)
                : launch_kernel(split_weight_grad_kernel<TN, TK>, grid, dim3(DG_THREADS), split_lds<TN, TK>(), st, a);
}
template <int TM, int TK> int launch_input_grad(hipStream_t st, DenseGradArgs &a)
{
    a.ktiles = (a.K + TK - 1) / TK;
    return launch_kernel(dense_input_grad_kernel<TM, TK>, dim3(grid_of((a.rows + TM - 1) / TM * a.ktiles)), dim3(DG_THREADS),
                         dg_lds<DG_STEP, TK, TM, DG_STEP, ROWK>(), st, a);
}

template <bool NARROW> int launch_wide(hipStream_t st, const DenseGradArgs &a, const WeightPlan &p)
{
    using T = WideTile<NARROW>;
    WideGradArgs w{};
    w.x = static_cast<const __bf16 *>(a.x), w.out = a.out, w.K = a.K, w.ktiles = a.K / T::W, w.tiles = p.tiles, w.slices = p.slices, w.rows = a.rows;
    w.slice_rows = p.slice_rows, w.total = p.total;
    for (int l = 0; l < a.layers; ++l) {
        if (l == p.narrow) {
            w.dyn = static_cast<const __bf16 *>(a.dy[l]), w.nn = a.n[l], w.wn_at = a.w_at[l], w.bn_at = a.b_at[l];
            continue;
        }
        const int j = w.layers++;
        w.dy[j] = static_cast<const __bf16 *>(a.dy[l]), w.n[j] = a.n[l], w.w_at[j] = a.w_at[l], w.b_at[j] = a.b_at[l];
        w.first_tile[j + 1] = w.first_tile[j] + a.n[l] / T::W;
    }
    return launch_kernel(wide_weight_grad_kernel<NARROW>, dim3(grid_of((int64_t)p.tiles * p.slices)), dim3(WT_THREADS), T::STAGES * T::STAGE, st, w);
}

int launch_grads(hipStream_t st, DenseGradArgs &a, const WeightPlan &p, bool bf16, float *params, float *workspace)
{
    if (a.dx && bf16) {
        // rows and features per workgroup: large tiles read dy and the weights less often, small ones fill the device
        const int64_t large = (a.rows + 127) / 128 * ((a.K + 127) / 128);
        const int rc = a.K <= 64 ? (a.rows >= 128 * 512 ? launch_input_grad<128, 64>(st, a) : launch_input_grad<64, 64>(st, a))
                       : large >= 512 ? launch_input_grad<128, 128>(st, a)
                                      : launch_input_grad<64, 64>(st, a);
        if (rc != MRX_OK) return rc;
    }
    if (!params) return MRX_OK;
    a.slices = p.slices, a.slice_rows = p.slice_rows, a.total = p.total;
    a.out = p.slices == 1 ? params : workspace;
    const int rc = p.wide ? (p.narrow >= 0 ? launch_wide<true>(st, a, p) : launch_wide<false>(st, a, p))
                   : p.tn == 64 ? (p.tk == 64 ? launch_weight_grads<64, 64>(st, a, p, bf16) : launch_weight_grads<64, 128>(st, a, p, bf16))
                                : (p.tk == 64 ? launch_weight_grads<128, 64>(st, a, p, bf16) : launch_weight_grads<128, 128>(st, a, p, bf16));
    if (rc != MRX_OK || p.slices == 1) return rc;
    return launch_column_sum(st, workspace, params, nullptr, p.slices, (int)p.total);
}

constexpr int big_lds = (int)dg_lds<128, 128, 128, 128, KROW>();
const KernelRegistrar registrars[] = {
    {reinterpret_cast<const void *>(dense_weight_grad_kernel<128, 128>), big_lds},
    {reinterpret_cast<const void *>(split_weight_grad_kernel<128, 128>), (int)split_lds<128, 128>()},
    {reinterpret_cast<const void *>(dense_input_grad_kernel<128, 128>), big_lds},
    {reinterpret_cast<const void *>(wide_weight_grad_kernel<false>), WideTile<false>::STAGES *WideTile<false>::STAGE},
    {reinterpret_cast<const void *>(wide_weight_grad_kernel<true>), WideTile<true>::STAGES *WideTile<true>::STAGE},
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
    int64_t floats = 0;   // enough for either plan: which of them it is depends on where the rows lie
    for (bool wide : {false, true}) {
        const WeightPlan p = plan_weights(rows, K, n_out, layers, dtype == MRX_BF16, bias_mask, wide);
        if (p.slices > 1) floats = p.slices * p.total > floats ? p.slices * p.total : floats;
    }
    return floats + (dtype == MRX_F32 ? split_pack_floats(n_out, layers, K, true) : 0);   // and the weights behind them
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
    bool wide = true;   // rows on the boundaries of whole requests
    for (int l = 0; l < layers; ++l) wide = wide && aligned(dys[l], n_out[l] <= WT_NARROW ? 4 : 16);
    const WeightPlan p = plan_weights(rows, K, n_out, layers, bf, bias_mask, wide);
    if (((params && p.slices > 1) || (dx && !bf)) && (!workspace || !aligned(workspace, 16))) return MRX_ERR_INVALID_ARG;
    if ((int64_t)p.tiles * p.slices >= (1ll << 31) || p.total >= (1ll << 31) || (rows + 63) / 64 * ((K + 63) / 64) >= (1ll << 31))
        return MRX_ERR_INVALID_ARG;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (dx && !bf) {
        SplitCall c;
        c.dys = dys, c.weights = weights, c.n_out = n_out, c.layers = layers, c.dx = dx, c.dx_bf16 = a.dx_bf16, c.rows = rows, c.K = K;
        c.workspace = workspace + (p.slices > 1 ? p.slices * p.total : 0);
        if (const int rc = split_rows(st, c); rc != MRX_OK) return rc;
    }
    return launch_grads(st, a, p, bf, params, workspace);
}
