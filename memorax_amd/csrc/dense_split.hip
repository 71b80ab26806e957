// Dense layers over rows in float32, forward and with respect to their input, on the float16 matrix units (split_f16.h):
//
//     y_l = x W_l^T + b_l      a group of layers that read the same rows;  y = residual + (x W^T + b + skip z) for one
//     dx  = sum_l dy_l W_l     of such a group, + skip z
//
// In float32 these are bound by the matrix units -- 154 TFLOP/s dense where float16 has sixteen times that -- and the array library runs
// one product per layer and direction, at three quarters of the float32 rate over many rows, for 20 us of the host each.  Here a group is two
// launches: the weights are split once (`split_pack_kernel`) into the fragments that the products read, and a workgroup of eight waves splits 64
// rows on their way into LDS and takes them past the weights, each wave its own columns, the weights straight from L2 into registers.  Up to
// 256 features of a row lie in LDS at a time (64 KB, two workgroups on a compute unit, so that one multiplies while the other stages or stores);
// longer contractions go on in steps of 256, the layers of an input gradient one after the other.  Every row of a step and every
// column of the weights has a power of two of its own; the running sums are brought to the next step's when it comes.
// us, here / the array library: 32768 x 256 -> 1024 + 512 + 512 + 8 forward 155 / 325 (224 TFLOP/s of float32 products, 0.67 PFLOP/s of float16 ones),
// their input gradient 148 / 295; 131072 x 256 -> 3 x 256 + 4 256 / 485 and 261 / 520; 4096 x 256 -> 3 x 256 28 / 36 and 30 / 33.  The forward's
// results take 35 us of the 155 to write (75 before they were stored past the caches); the products by themselves
// run at half the float16 rate, where an 8192^3 product of the array library is too.  Four more waves that only fetched and split for the
// others (180 us) and four waves of 64 x 64 results each (187) were not faster.
#include "dense_split.h"
#include <type_traits>

#include "chunk_common.h"
#include "split_f16.h"

namespace mrx {
namespace {

constexpr int SP_ROWS = 64, SP_WAVES = 8, SP_THREADS = 64 * SP_WAVES, SP_PACK = 256, SP_K = 256, SP_MT = SP_ROWS / 16;
constexpr int SP_TOP = 14;          // the largest of a row or column lies in [2^14, 2^15)
constexpr int SP_FLOOR_ROW = 20;    // a later step's row scale is at most this far above the largest so far: the running sums stay finite
constexpr int SP_LOW = -24, SP_HIGH = 40, SP_WILD = 1 << 12;   // columns of weights below 2^-24 share its scale, from 2^40 on they are summed one by one

struct SplitIn {
    const float *x;        // (rows, n)
    const float *w;        // input gradient: the layer's weights (n, K)
    int n, step, block;    // features; its first step of SP_K and first block of 32 among all
    bool whole;            // rows of whole 16-byte pieces, on their boundaries
};
struct SplitOut {
    const float *w, *b;    // w: forward, (n, K)
    void *y;
    int n, tile;           // outputs; first 16-column tile
};
struct SplitArgs {
    SplitIn in[MRX_DENSE_LAYERS];    // what the contraction runs over: the rows (forward), or the layers' gradients
    SplitOut out[MRX_DENSE_LAYERS];  // what the columns belong to: the layers, or the input
    const f16x8 *packed;
    const int *exps;       // (steps, 16 tiles): exponent of each column
    const float *residual, *skip, *skip_x;
    int64_t rows;
    int ins, outs, steps, tiles, passes, groups, K;
    bool y_bf16;
};
// One step of the contraction: up to SP_K features of one input.
struct SplitStep {
    const float *x, *w;
    int n, len, blocks, first, k0;   // floats between rows; features, blocks of 32; blocks before it; where it starts
    bool whole;
};
__device__ __forceinline__ SplitStep step_of(const SplitArgs &a, int s)
{
    int l = 0;
    while (l + 1 < a.ins && s >= a.in[l + 1].step) ++l;
    const SplitIn &in = a.in[l];
    const int k0 = (s - in.step) * SP_K, len = in.n - k0 < SP_K ? in.n - k0 : SP_K;
    return {in.x + k0, in.w + (int64_t)k0 * a.K, in.n, len, (len + 31) / 32, in.block + k0 / 32, k0, in.whole};
}
__device__ __forceinline__ int out_of(const SplitArgs &a, int ct)
{
    int l = 0;
    while (l + 1 < a.outs && ct >= a.out[l + 1].tile) ++l;
    return l;
}

// The 64-lane fragments of a step lie one after the other; lane (i, g) of fragment k at slot 16 g + (i ^ (4 k + g)): the lanes that write a row and
// the lanes that read a fragment spread over the banks.
__device__ __forceinline__ int slot_of(int i, int k8) { return (k8 & 3) * 16 + (i ^ (k8 & 15)); }

// The largest over the half of a wave that holds a row.
__device__ __forceinline__ float half_wave_max(float x)
{
    auto with = [&](auto ctrl) {
        x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, true)));
    };
    with(std::integral_constant<int, 0xB1>{});
    with(std::integral_constant<int, 0x4E>{});
    with(std::integral_constant<int, 0x141>{});
    with(std::integral_constant<int, 0x140>{});
    return fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, x), 0x401f)));   // lane ^ 16
}

// Eight features of a row from k on; what lies at len and beyond is zero.
__device__ __forceinline__ void load8(const float *row, int k, int len, bool whole, sf32x4 (&v)[2])
{
    v[0] = v[1] = sf32x4{0.f, 0.f, 0.f, 0.f};
    if (k >= len) return;
    if (whole) {
        v[0] = *reinterpret_cast<const sf32x4 *>(row + k);
        if (k + 4 < len) v[1] = *reinterpret_cast<const sf32x4 *>(row + k + 4);
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (k + e < len) v[e / 4][e % 4] = row[k + e];
    }
}

// ---- the weights: 16 columns of a step a workgroup
template <bool ACROSS> __global__ void __launch_bounds__(SP_PACK) split_pack_kernel(SplitArgs a, f16x8 *packed, int *exps)
{
    __shared__ int top[16];
    const int ct = blockIdx.x, tid = threadIdx.x;
    const SplitStep st = step_of(a, blockIdx.y);
    const int l = out_of(a, ct);
    const int c0 = (ct - a.out[l].tile) * 16, n = a.out[l].n;
    if (tid < 16) top[tid] = 0;
    __syncthreads();
    sf32x4 v[2][2];
    int col[2], k8[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int u = tid + p * SP_PACK;
        float m;
        if constexpr (ACROSS) {   // the weights' rows lie along the contraction: sixteen columns of one a quarter wave
            col[p] = u & 15, k8[p] = u >> 4;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v[p][e / 4][e % 4] = c0 + col[p] < n && k8[p] * 8 + e < st.len ? st.w[(int64_t)(k8[p] * 8 + e) * a.K + c0 + col[p]] : 0.f;
            m = max4(max4(0.f, v[p][0]), v[p][1]);
        } else {
            col[p] = u >> 5, k8[p] = u & 31;
            load8(a.out[l].w + (int64_t)(c0 + col[p] < n ? c0 + col[p] : 0) * a.K + st.k0, k8[p] * 8, c0 + col[p] < n ? st.len : 0, true, v[p]);
            m = max4(max4(0.f, v[p][0]), v[p][1]);
        }
        atomicMax(&top[col[p]], (int)(__float_as_uint(m) & 0x7fffffffu));
    }
    __syncthreads();
    const int64_t at = ((int64_t)st.first * a.tiles + (int64_t)ct * st.blocks) * 128;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int e = exponent(__uint_as_float((uint32_t)top[col[p]]));
        const int ex = e < SP_LOW ? SP_LOW : e >= SP_HIGH ? SP_WILD : e;
        if (k8[p] < 4 * st.blocks) {
            const float s = ex == SP_WILD ? 0.f : power_of_two(SP_TOP - ex);
            const Split4 a4 = split4(v[p][0], s), b4 = split4(v[p][1], s);
            f16x8 *dst = packed + at + (int64_t)(k8[p] >> 2) * 128 + (k8[p] & 3) * 16 + col[p];
            dst[0] = join(a4.hi, b4.hi), dst[64] = join(a4.lo, b4.lo);
        }
        if (k8[p] == 0) exps[(int64_t)blockIdx.y * a.tiles * 16 + ct * 16 + col[p]] = ex;
    }
}

// ---- rows
// The same sums one by one, where an infinity (or weights of 2^40 and more) is among the operands: NT 16-column tiles of a wave.
template <int NT, bool ACROSS, typename Store>
__device__ __forceinline__ void plain_tiles(const SplitArgs &a, int64_t r0, int ct0, int lane, Store store)
{
    const int i = lane & 15, g = lane >> 4;
#pragma unroll 1
    for (int e = 0; e < SP_MT * NT * 4; ++e) {
        const int m = e / (NT * 4), j = e / 4 % NT, v = e % 4, ct = ct0 + j;
        const int64_t r = r0 + 16 * m + i;
        if (ct >= a.tiles || r >= a.rows) continue;
        const int l = out_of(a, ct), c = (ct - a.out[l].tile) * 16 + 4 * g + v;
        if (c >= a.out[l].n) continue;
        float sum = 0.f;
        for (int s = 0; s < a.ins; ++s) {
            const SplitIn &in = a.in[s];
            for (int k = 0; k < in.n; ++k) sum = fmaf(in.x[r * in.n + k], ACROSS ? in.w[(int64_t)k * a.K + c] : a.out[l].w[(int64_t)c * a.K + k], sum);
        }
        store(l, r, c, sum);
    }
}

template <int NT, bool ACROSS> __global__ void __launch_bounds__(SP_THREADS, NT == 1 ? 2 : 4) split_rows_kernel(SplitArgs a)
{
    constexpr bool FEW = NT == 1;
    constexpr int AHEAD = FEW ? 8 : 1;   // blocks of weights in registers, one in use: a step's where few workgroups share a compute unit
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int row_exp[2][SP_ROWS], row_peak[SP_ROWS];   // of this step and the one before; the largest so far
    __shared__ int infinite;
    f16x8 *const tile = reinterpret_cast<f16x8 *>(smem);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 15, g = lane >> 4;
    // workgroups are dealt to the eight dies in turn: each takes a contiguous share of the row tiles, the column groups of a tile side by side
    const int64_t tasks = (a.rows + SP_ROWS - 1) / SP_ROWS * a.groups, share = (tasks + 7) / 8;
    const int64_t task = (blockIdx.x & 7) * share + (blockIdx.x >> 3);
    if ((int64_t)(blockIdx.x >> 3) >= share || task >= tasks) return;
    const int64_t r0 = task / a.groups * SP_ROWS;
    const int group = (int)(task % a.groups);
    const int first = (int)((int64_t)a.passes * group / a.groups), last = (int)((int64_t)a.passes * (group + 1) / a.groups);
    const int row = tid >> 5, k8 = tid & 31;
    if (tid == 0) infinite = 0;
    sync_lds();   // before any wave sets it

    constexpr int UNITS = SP_ROWS * 32 / SP_THREADS, APART = SP_THREADS / 32;
    sf32x4 v[UNITS][2];
    auto load = [&](const SplitStep &st) {
#pragma unroll
        for (int p = 0; p < UNITS; ++p) {
            const int64_t r = r0 + row + APART * p;
            load8(st.x + (r < a.rows ? r : a.rows - 1) * st.n, k8 * 8, st.len, st.whole, v[p]);
        }
    };
    auto stage = [&](int s, int blocks) {
#pragma unroll
        for (int p = 0; p < UNITS; ++p) {
            const float m = half_wave_max(max4(max4(0.f, v[p][0]), v[p][1]));
            int e = exponent(m);
            if (e == 128) infinite = 1;
            e = e < -98 ? -98 : e;
            if (a.steps > 1) {
                const int peak = s > 0 ? row_peak[row + APART * p] : e;
                e = e < peak - SP_FLOOR_ROW ? peak - SP_FLOOR_ROW : e;
                if (k8 == 0) row_peak[row + APART * p] = peak > e ? peak : e;
            }
            const float scale = power_of_two(SP_TOP - e);
            if (k8 == 0) row_exp[s & 1][row + APART * p] = e;
            if (k8 >= 4 * blocks) continue;
            const Split4 lo4 = split4(v[p][0], scale), hi4 = split4(v[p][1], scale);
            const int rr = row + APART * p;
            f16x8 *const dst = tile + ((rr >> 4) * blocks + (k8 >> 2)) * 128 + slot_of(rr & 15, k8);
            dst[0] = join(lo4.hi, hi4.hi), dst[64] = join(lo4.lo, hi4.lo);
        }
    };

    auto store = [&](int l, int64_t r, int c, float y) {
        const SplitOut &o = a.out[l];
        if (o.b) y += o.b[c];
        if (a.skip) y = fmaf(a.skip[c], a.skip_x[r * o.n + c], y);
        if (a.residual) y += a.residual[r * o.n + c];
        if (ACROSS && a.y_bf16) static_cast<__bf16 *>(o.y)[r * o.n + c] = (__bf16)y;
        else static_cast<float *>(o.y)[r * o.n + c] = y;
    };

    for (int pass = first; pass < last; ++pass) {
        const int ct0 = (pass * SP_WAVES + wv) * NT;
        sf32x4 acc[SP_MT][NT];
#pragma unroll
        for (int m = 0; m < SP_MT; ++m)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[m][j] = sf32x4{0.f, 0.f, 0.f, 0.f};
        int ex[NT][4];          // of this lane's columns
        bool wild = false;
        for (int s = 0; s < a.steps; ++s) {
            const SplitStep st = step_of(a, s);
            const int blocks = st.blocks;
            // tiles past the last are the last one; their results are dropped
            const f16x8 *w[NT];
            int4 exps[NT];
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const int ct = ct0 + j < a.tiles ? ct0 + j : a.tiles - 1;
                w[j] = a.packed + ((int64_t)st.first * a.tiles + (int64_t)ct * blocks) * 128 + lane;
                exps[j] = *reinterpret_cast<const int4 *>(a.exps + ((int64_t)s * a.tiles + ct) * 16 + 4 * g);
            }
            f16x8 b[AHEAD][NT][2];
            auto weights = [&]() {
#pragma unroll
                for (int k = 0; k < AHEAD - 1; ++k)
                    if (k < blocks)
#pragma unroll
                        for (int j = 0; j < NT; ++j) b[k][j][0] = w[j][k * 128], b[k][j][1] = w[j][k * 128 + 64];
            };
            if (FEW) weights();
            if (a.steps > 1 || pass == first) {
                if (!FEW || (s == 0 && pass == first)) load(st);
                if (s > 0 || pass > first) sync_lds();   // the step before has been read
                stage(s, blocks);
                sync_lds();
                if (FEW && a.steps > 1 && (s + 1 < a.steps || pass + 1 < last)) load(step_of(a, s + 1 < a.steps ? s + 1 : 0));
            }
            if (!FEW) weights();
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const int e[4] = {exps[j].x, exps[j].y, exps[j].z, exps[j].w};
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    wild = wild || e[u] == SP_WILD;
                    if (s > 0)
#pragma unroll
                        for (int m = 0; m < SP_MT; ++m)
                            acc[m][j][u] = __builtin_ldexpf(acc[m][j][u], row_exp[(s + 1) & 1][16 * m + i] - row_exp[s & 1][16 * m + i] + ex[j][u] - e[u]);
                    ex[j][u] = e[u];
                }
            }
            if (ct0 >= a.tiles) continue;
            for (int k0 = 0; k0 < blocks; k0 += AHEAD) {
#pragma unroll
                for (int p = 0; p < AHEAD; ++p) {
                    const int k = k0 + p, then = k + AHEAD - 1;
                    if (k >= blocks) break;
                    if (then < blocks)
#pragma unroll
                        for (int j = 0; j < NT; ++j)
                            b[(p + AHEAD - 1) % AHEAD][j][0] = w[j][then * 128], b[(p + AHEAD - 1) % AHEAD][j][1] = w[j][then * 128 + 64];
                    const f16x8 *f = tile + k * 128 + slot_of(i, 4 * k + g);
                    // the small products by themselves first: two roundings of the running sum a block instead of three
                    constexpr int MB = FEW ? SP_MT : 1;   // row tiles whose products take turns
#pragma unroll
                    for (int m0 = 0; m0 < SP_MT; m0 += MB) {
                        f16x8 hi[MB], lo[MB];
                        sf32x4 low[MB][NT];
#pragma unroll
                        for (int m = 0; m < MB; ++m) hi[m] = f[(m0 + m) * blocks * 128], lo[m] = f[(m0 + m) * blocks * 128 + 64];
#pragma unroll
                        for (int m = 0; m < MB; ++m)
#pragma unroll
                            for (int j = 0; j < NT; ++j) low[m][j] = mma_f16(b[p][j][0], lo[m], sf32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                        for (int m = 0; m < MB; ++m)
#pragma unroll
                            for (int j = 0; j < NT; ++j) low[m][j] = mma_f16(b[p][j][1], hi[m], low[m][j]);
#pragma unroll
                        for (int m = 0; m < MB; ++m)
#pragma unroll
                            for (int j = 0; j < NT; ++j) acc[m0 + m][j] = mma_f16(b[p][j][0], hi[m], acc[m0 + m][j]);
#pragma unroll
                        for (int m = 0; m < MB; ++m)
#pragma unroll
                            for (int j = 0; j < NT; ++j) acc[m0 + m][j] += low[m][j];
                    }
                }
            }
        }
        if (infinite || __any(wild)) {
            plain_tiles<NT, ACROSS>(a, r0, ct0, lane, store);
            continue;
        }
        const int (&re)[SP_ROWS] = row_exp[(a.steps - 1) & 1];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int ct = ct0 + j;
            if (ct >= a.tiles) break;
            const int l = out_of(a, ct);
            const SplitOut &o = a.out[l];
            const int c = (ct - o.tile) * 16 + 4 * g;
#pragma unroll
            for (int m = 0; m < SP_MT; ++m) {
                const int64_t r = r0 + 16 * m + i;
                if (r >= a.rows) continue;
                sf32x4 y;
#pragma unroll
                for (int u = 0; u < 4; ++u) y[u] = __builtin_ldexpf(acc[m][j][u], re[16 * m + i] + ex[j][u] - 2 * SP_TOP);
                if (o.n % 4 == 0) {   // rows of whole 16-byte pieces, on their boundaries
                    if (c >= o.n) continue;
                    if (o.b) y += sf32x4{o.b[c], o.b[c + 1], o.b[c + 2], o.b[c + 3]};
                    const int64_t at = r * o.n + c;
                    if (a.skip) y += *reinterpret_cast<const sf32x4 *>(a.skip + c) * *reinterpret_cast<const sf32x4 *>(a.skip_x + at);
                    if (a.residual) y += *reinterpret_cast<const sf32x4 *>(a.residual + at);
                    if (ACROSS && a.y_bf16) {
                        typedef __bf16 b4 __attribute__((ext_vector_type(4)));
                        *reinterpret_cast<b4 *>(static_cast<__bf16 *>(o.y) + at) = __builtin_convertvector(y, b4);
                    } else {
                        __builtin_nontemporal_store(y, reinterpret_cast<sf32x4 *>(static_cast<float *>(o.y) + at));
                    }
                } else {
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (c + u < o.n) store(l, r, c + u, y[u]);
                }
            }
        }
    }
}

template <int NT, bool ACROSS> struct LaunchRows {
    static constexpr auto kernel = split_rows_kernel<NT, ACROSS>;
    static inline const KernelRegistrar registrar{reinterpret_cast<const void *>(kernel), SP_ROWS * SP_K * 4};
    static int go(hipStream_t st, SplitArgs &a, int most)
    {
        (void)&registrar;
        const int64_t row_tiles = (a.rows + SP_ROWS - 1) / SP_ROWS;
        a.passes = (a.tiles + SP_WAVES * NT - 1) / (SP_WAVES * NT);
        // two workgroups for every compute unit, where the columns give that many
        int64_t groups = (512 + row_tiles - 1) / row_tiles;
        a.groups = (int)(groups < a.passes ? groups : a.passes);
        const int64_t blocks = (row_tiles * a.groups + 7) / 8 * 8;
        if (blocks >= (1ll << 31)) return MRX_ERR_INVALID_ARG;
        return launch_kernel(kernel, dim3((unsigned)blocks), dim3(SP_THREADS), SP_MT * most * 2048, st, a);
    }
};

struct Sizes {
    int64_t steps = 0, tiles = 0, blocks = 0;   // of the contraction; 16-column tiles; 32-feature blocks of all steps
    bool ok = true;
};
Sizes sizes_of(const int64_t *n, int layers, int64_t K, bool across)
{
    Sizes r;
    r.ok = n && layers >= 1 && layers <= MRX_DENSE_LAYERS && K > 0 && K % 8 == 0 && K <= (1 << 16);
    for (int l = 0; r.ok && l < layers; ++l) {
        r.ok = n[l] > 0 && n[l] <= (1 << 16);
        if (across) r.steps += (n[l] + SP_K - 1) / SP_K, r.blocks += (n[l] + 31) / 32;
        else r.tiles += (n[l] + 15) / 16;
    }
    if (across) r.tiles = (K + 15) / 16;
    else r.steps = (K + SP_K - 1) / SP_K, r.blocks = (K + 31) / 32;
    return r;
}

}  // namespace

int64_t split_pack_floats(const int64_t *n_out, int layers, int64_t K, bool across)
{
    const Sizes z = sizes_of(n_out, layers, K, across);
    return z.ok ? z.blocks * z.tiles * 512 + z.steps * z.tiles * 16 : 0;
}

int split_rows(hipStream_t st, const SplitCall &c)
{
    const bool across = c.dys != nullptr;
    const Sizes z = sizes_of(c.n_out, c.layers, c.K, across);
    if (!z.ok || !c.workspace || !aligned(c.workspace, 16) || c.rows <= 0 || c.rows >= (1ll << 31)) return MRX_ERR_INVALID_ARG;
    SplitArgs a{};
    a.rows = c.rows, a.K = (int)c.K, a.steps = (int)z.steps, a.tiles = (int)z.tiles, a.residual = c.residual, a.skip = c.skip, a.skip_x = c.skip_x, a.y_bf16 = c.dx_bf16;
    int64_t widest = 0;
    int step = 0, block = 0, tile = 0;
    auto in = [&](const float *x, const float *w, int64_t n) {
        a.in[a.ins++] = {x, w, (int)n, step, block, n % 4 == 0 && aligned(x, 16)};
        step += (int)((n + SP_K - 1) / SP_K), block += (int)((n + 31) / 32), widest = n > widest ? n : widest;
    };
    auto out = [&](const float *w, const float *b, void *y, int64_t n) {
        a.out[a.outs++] = {w, b, y, (int)n, tile};
        tile += (int)((n + 15) / 16);
    };
    if (across) out(nullptr, nullptr, c.dx, c.K);
    else in(c.x, nullptr, c.K);
    for (int l = 0; l < c.layers; ++l) {
        const float *w = static_cast<const float *>(c.weights[l]);
        if (across) in(static_cast<const float *>(c.dys[l]), w, c.n_out[l]);
        else out(w, static_cast<const float *>(c.biases[l]), c.outs[l], c.n_out[l]);
    }
    const int most = (int)((widest < SP_K ? widest : SP_K) + 31) / 32;
    f16x8 *const packed = reinterpret_cast<f16x8 *>(c.workspace);
    int *const exps = reinterpret_cast<int *>(c.workspace + z.blocks * z.tiles * 512);
    a.packed = packed, a.exps = exps;
    const dim3 grid((unsigned)z.tiles, (unsigned)z.steps);
    const int rc = across ? launch_kernel(split_pack_kernel<true>, grid, dim3(SP_PACK), 0, st, a, packed, exps)
                    : launch_kernel(split_pack_kernel<false>, grid, dim3(SP_PACK), 0, st, a, packed, exps);
    if (rc != MRX_OK) return rc;
    // columns of a wave: 64 read the rows from LDS least often, fewer make more workgroups of few rows
    const int64_t row_tiles = (c.rows + SP_ROWS - 1) / SP_ROWS;
    auto enough = [&](int nt) { return row_tiles * ((z.tiles + SP_WAVES * nt - 1) / (SP_WAVES * nt)) >= 256 && z.tiles > SP_WAVES * nt / 2; };
    if (across) return enough(2) ? LaunchRows<2, true>::go(st, a, most) : LaunchRows<1, true>::go(st, a, most);
    return enough(2) ? LaunchRows<2, false>::go(st, a, most) : LaunchRows<1, false>::go(st, a, most);
}

}  // namespace mrx

extern "C" int64_t mrx_dense_f32_workspace(const int64_t *n_out, int layers, int64_t K) { return mrx::split_pack_floats(n_out, layers, K, false); }

extern "C" int mrx_dense_f32(void *stream, const float *x, const void *const *weights, const void *const *biases, void *const *outs,
                             const int64_t *n_out, int layers, const float *residual, const float *skip, const float *skip_x, int64_t rows, int64_t K,
                             float *workspace)
{
    using namespace mrx;
    if (!skip != !skip_x || (skip && layers != 1) || !aligned(skip, 16) || !aligned(skip_x, 16)) return MRX_ERR_INVALID_ARG;
    if (!x || !weights || !biases || !outs || !n_out || layers < 1 || layers > MRX_DENSE_LAYERS || !aligned(x, 16) || !aligned(residual, 16) || (residual && layers != 1))
        return MRX_ERR_INVALID_ARG;
    for (int l = 0; l < layers; ++l)
        if (!weights[l] || !outs[l] || !aligned(weights[l], 16) || !aligned(outs[l], 16) || !aligned(biases[l], 4)) return MRX_ERR_INVALID_ARG;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    SplitCall c;
    c.x = x, c.weights = weights, c.biases = biases, c.outs = outs, c.residual = residual, c.skip = skip, c.skip_x = skip_x, c.n_out = n_out, c.layers = layers, c.rows = rows, c.K = K;
    c.workspace = workspace;
    return split_rows(static_cast<hipStream_t>(stream), c);
}

extern "C" int64_t mrx_dense_f32_input_grad_workspace(const int64_t *n_out, int layers, int64_t K) { return mrx::split_pack_floats(n_out, layers, K, true); }

extern "C" int mrx_dense_f32_input_grad(void *stream, const void *const *dys, const void *const *weights, const int64_t *n_out, int layers, const float *skip,
                                        const float *skip_x, float *dx, int64_t rows, int64_t K, float *workspace)
{
    using namespace mrx;
    if (!dys || !weights || !n_out || !dx || layers < 1 || layers > MRX_DENSE_LAYERS || !aligned(dx, 16) || !skip != !skip_x || !aligned(skip, 16) || !aligned(skip_x, 16))
        return MRX_ERR_INVALID_ARG;
    for (int l = 0; l < layers; ++l)
        if (!dys[l] || !weights[l] || !aligned(dys[l], 4) || !aligned(weights[l], 16)) return MRX_ERR_INVALID_ARG;
    SplitCall c;
    c.dys = dys, c.weights = weights, c.dx = dx, c.skip = skip, c.skip_x = skip_x, c.n_out = n_out, c.layers = layers, c.rows = rows, c.K = K;
    c.workspace = workspace;
    return split_rows(static_cast<hipStream_t>(stream), c);
}
