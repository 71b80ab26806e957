// Dense layers over rows in float32, forward and with respect to their input, on the bfloat16 matrix units (split_bf16.h):
//
//     y_l = x W_l^T + b_l      a group of layers that read the same rows;  y = residual + (x W^T + b + skip z) for one
//     dx  = sum_l dy_l W_l     of such a group, + skip z
//
// In float32 these are bound by the matrix units -- 154 TFLOP/s dense where bfloat16 has sixteen times that -- and the array library runs
// one product per layer and direction, at three quarters of the float32 rate over many rows, for 20 us of the host each.  Here a group is two
// launches: the weights are split once (`split_pack_kernel`) into the fragments that the products read, and a workgroup splits up to 64
// rows on their way into LDS and takes them past the weights, each wave its own columns, the weights straight from L2 into registers.
// Forward, up to 256 features of a row lie in LDS at a time, 96 KB of 64 rows: one workgroup of sixteen waves on a compute unit, two of eight where the
// rows are narrower.  Along the layers' outputs a step is 128 features, so that two workgroups share a compute unit and one multiplies while the other stages
// (32768 rows, below: 256 features 211 us, 128 185).  Longer contractions go on in steps, the layers of an input gradient one after the other.
// us, here / the array library: 32768 x 256 -> 1024 + 512 + 512 + 8 forward 184 / 297 (188 TFLOP/s of float32 products, 1.1 PFLOP/s of bfloat16 ones),
// their input gradient 180 / 280; 131072 x 256 -> 3 x 256 + 4 290 / 448 and 303 / 504; 4096 x 256 -> 3 x 256 31 / 34 and 29 / 32.  The matrix units are
// busy 58 % of the first's cycles and 52 % of its input gradient's, the vector ALU 18 and 24 %, LDS 15 and 17.
#include "dense_split.h"

#include "chunk_common.h"
#include "split_bf16.h"

namespace mrx {
namespace {

constexpr int SP_PACK = 256;
constexpr int SP_LANES = 64 * PARTS;   // 16-byte pieces of a fragment, its parts one behind the other
// Features of a step.
constexpr int step_features(bool across) { return across ? 128 : 256; }

struct SplitIn {
    const float *x;        // (rows, n)
    const float *w;        // input gradient: the layer's weights (n, K)
    int n, step, block;    // features; its first step and first block of 32 among all
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
    const bf16x8 *packed;
    const int *wild;       // (steps, tiles): whether a value among them has no parts
    const float *residual, *skip, *skip_x;
    int64_t rows;
    int ins, outs, steps, tiles, passes, groups, K;
    bool y_bf16;
};
// One step of the contraction: features of one input.
struct SplitStep {
    const float *x, *w;
    int n, len, blocks, first, k0;   // floats between rows; features, blocks of 32; blocks before it; where it starts
    bool whole;
};
template <bool ACROSS> __device__ __forceinline__ SplitStep step_of(const SplitArgs &a, int s)
{
    constexpr int SP_K = step_features(ACROSS);
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

// Eight features of a row from k on; what lies at len and beyond is zero.
__device__ __forceinline__ void load8(const float *row, int k, int len, bool whole, f32x4 (&v)[2])
{
    v[0] = v[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (k >= len) return;
    if (whole) {
        v[0] = *reinterpret_cast<const f32x4 *>(row + k);
        if (k + 4 < len) v[1] = *reinterpret_cast<const f32x4 *>(row + k + 4);
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (k + e < len) v[e / 4][e % 4] = row[k + e];
    }
}

// ---- the weights: 16 columns of a step a workgroup
template <bool ACROSS> __global__ void __launch_bounds__(SP_PACK) split_pack_kernel(SplitArgs a, bf16x8 *packed, int *wild)
{
    constexpr int SP_K = step_features(ACROSS), K8 = SP_K / 8, UNITS = 16 * K8 / SP_PACK;
    __shared__ int beyond;
    const int ct = blockIdx.x, tid = threadIdx.x;
    const SplitStep st = step_of<ACROSS>(a, blockIdx.y);
    const int l = out_of(a, ct);
    const int c0 = (ct - a.out[l].tile) * 16, n = a.out[l].n;
    if (tid == 0) beyond = 0;
    __syncthreads();
    float most = 0.f;
    const int64_t at = ((int64_t)st.first * a.tiles + (int64_t)ct * st.blocks) * SP_LANES;
#pragma unroll
    for (int p = 0; p < UNITS; ++p) {
        const int u = tid + p * SP_PACK;
        const int col = ACROSS ? u & 15 : u / K8, k8 = ACROSS ? u >> 4 : u % K8;
        f32x4 v[2];
        if constexpr (ACROSS) {   // the weights' rows lie along the contraction: sixteen columns of one a quarter wave
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v[e / 4][e % 4] = c0 + col < n && k8 * 8 + e < st.len ? st.w[(int64_t)(k8 * 8 + e) * a.K + c0 + col] : 0.f;
        } else {
            load8(a.out[l].w + (int64_t)(c0 + col < n ? c0 + col : 0) * a.K + st.k0, k8 * 8, c0 + col < n ? st.len : 0, true, v);
        }
        most = max4(max4(most, v[0]), v[1]);
        if (k8 < 4 * st.blocks) {
            Words<4>::type parts[PARTS];
            split_parts<4>(v, parts);
            bf16x8 *dst = packed + at + (int64_t)(k8 >> 2) * SP_LANES + (k8 & 3) * 16 + col;
#pragma unroll
            for (int h = 0; h < PARTS; ++h) dst[64 * h] = __builtin_bit_cast(bf16x8, parts[h]);
        }
    }
    if (most > BF16_MOST) beyond = 1;
    __syncthreads();
    if (tid == 0) wild[(int64_t)blockIdx.y * a.tiles + ct] = beyond;
}

// ---- rows
// The same sums one by one, where a value without parts is among the operands: NT 16-column tiles of a wave.
template <int MT, int NT, bool ACROSS, typename Store>
__device__ __forceinline__ void plain_tiles(const SplitArgs &a, int64_t r0, int ct0, int lane, Store store)
{
    const int i = lane & 15, g = lane >> 4;
#pragma unroll 1
    for (int e = 0; e < MT * NT * 4; ++e) {
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

template <int MT, int NT, bool ACROSS, bool FEW, int WAVES> __global__ void __launch_bounds__(64 * WAVES, FEW ? 2 : 4) split_rows_kernel(SplitArgs a)
{
    constexpr int SP_K = step_features(ACROSS), K8 = SP_K / 8, SP_ROWS = 16 * MT, SP_THREADS = 64 * WAVES;
    // blocks of weights in registers, one in use: a step's where few workgroups share a compute unit, along the layers' outputs the next step's too
    constexpr int AHEAD = FEW ? SP_K / 32 : 1;
    constexpr bool NEXT = FEW && ACROSS;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int beyond;   // a value without parts is among the rows
    bf16x8 *const tile = reinterpret_cast<bf16x8 *>(smem);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 15, g = lane >> 4;
    // workgroups are dealt to the eight dies in turn: each takes a contiguous share of the row tiles, the column groups of a tile side by side
    const int64_t tasks = (a.rows + SP_ROWS - 1) / SP_ROWS * a.groups, share = (tasks + 7) / 8;
    const int64_t task = (blockIdx.x & 7) * share + (blockIdx.x >> 3);
    if ((int64_t)(blockIdx.x >> 3) >= share || task >= tasks) return;
    const int64_t r0 = task / a.groups * SP_ROWS;
    const int group = (int)(task % a.groups);
    const int first = (int)((int64_t)a.passes * group / a.groups), last = (int)((int64_t)a.passes * (group + 1) / a.groups);
    const int row = tid / K8, k8 = tid % K8;
    if (tid == 0) beyond = 0;
    sync_lds();   // before any wave sets it

    constexpr int UNITS = (SP_ROWS * K8 + SP_THREADS - 1) / SP_THREADS, APART = SP_THREADS / K8;
    const bool stages = SP_ROWS * K8 % SP_THREADS == 0 || row < SP_ROWS;
    f32x4 v[UNITS][2];
    auto load = [&](const SplitStep &st) {
#pragma unroll
        for (int p = 0; p < UNITS; ++p) {
            const int64_t r = r0 + row + APART * p;
            load8(st.x + (r < a.rows ? r : a.rows - 1) * st.n, k8 * 8, st.len, st.whole, v[p]);
        }
    };
    auto stage = [&](int blocks) {
        float most = 0.f;
#pragma unroll
        for (int p = 0; p < UNITS; ++p) {
            if (k8 >= 4 * blocks || !stages) continue;
            most = max4(max4(most, v[p][0]), v[p][1]);
            Words<4>::type parts[PARTS];
            split_parts<4>(v[p], parts);
            const int rr = row + APART * p;
            bf16x8 *const dst = tile + ((rr >> 4) * blocks + (k8 >> 2)) * SP_LANES + slot_of(rr & 15, k8);
#pragma unroll
            for (int h = 0; h < PARTS; ++h) dst[64 * h] = __builtin_bit_cast(bf16x8, parts[h]);
        }
        if (most > BF16_MOST) beyond = 1;
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
        const int ct0 = (pass * WAVES + wv) * NT;
        f32x4 acc[MT][NT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[m][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        bool wild = false;
        // tiles past the last are the last one; their results are dropped
        auto tile_of = [&](int j) { return ct0 + j < a.tiles ? ct0 + j : a.tiles - 1; };
        auto fetch = [&](bf16x8 (&b)[NT][PARTS], const SplitStep &st, int k) {
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const bf16x8 *const w = a.packed + ((int64_t)st.first * a.tiles + (int64_t)tile_of(j) * st.blocks + k) * SP_LANES + lane;
#pragma unroll
                for (int h = 0; h < PARTS; ++h) b[j][h] = w[64 * h];
            }
        };
        bf16x8 b[AHEAD][NT][PARTS], then[NEXT ? AHEAD : 1][NT][PARTS];
        auto fetch_step = [&](bf16x8 (&b)[NEXT ? AHEAD : 1][NT][PARTS], const SplitStep &st) {
#pragma unroll
            for (int k = 0; k < (NEXT ? AHEAD : 1); ++k)
                if (k < st.blocks) fetch(b[k], st, k);
        };
        if (NEXT) fetch_step(then, step_of<ACROSS>(a, 0));
        for (int s = 0; s < a.steps; ++s) {
            const SplitStep st = step_of<ACROSS>(a, s), after = step_of<ACROSS>(a, s + 1 < a.steps ? s + 1 : 0);
            const int blocks = st.blocks;
#pragma unroll
            for (int j = 0; j < NT; ++j) wild = wild || a.wild[(int64_t)s * a.tiles + tile_of(j)] != 0;
            if constexpr (NEXT) {
#pragma unroll
                for (int k = 0; k < AHEAD; ++k)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
#pragma unroll
                        for (int h = 0; h < PARTS; ++h) b[k][j][h] = then[k][j][h];
                if (s + 1 < a.steps) fetch_step(then, after);
            } else {
#pragma unroll
                for (int k = 0; k < AHEAD - 1; ++k)
                    if (k < blocks) fetch(b[k], st, k);
            }
            if (a.steps > 1 || pass == first) {
                if (!FEW || (s == 0 && pass == first)) load(st);
                if (s > 0 || pass > first) sync_lds();   // the step before has been read
                stage(blocks);
                sync_lds();
                if (FEW && a.steps > 1 && (s + 1 < a.steps || pass + 1 < last)) load(after);
            }
            if (ct0 >= a.tiles) continue;
            for (int k0 = 0; k0 < blocks; k0 += AHEAD) {
#pragma unroll
                for (int p = 0; p < AHEAD; ++p) {
                    const int k = k0 + p;
                    if (k >= blocks) break;
                    if (!NEXT && k + AHEAD - 1 < blocks) fetch(b[(p + AHEAD - 1) % AHEAD], st, k + AHEAD - 1);
                    const bf16x8 *f = tile + k * SP_LANES + slot_of(i, 4 * k + g);
                    // the small products by themselves first: two roundings of the running sum a block
                    constexpr int MB = FEW ? MT : 1;   // row tiles whose products take turns
#pragma unroll
                    for (int m0 = 0; m0 < MT; m0 += MB) {
                        bf16x8 x[MB][PARTS];
                        f32x4 low[MB][NT];
#pragma unroll
                        for (int m = 0; m < MB; ++m)
#pragma unroll
                            for (int h = 0; h < PARTS; ++h) x[m][h] = f[(m0 + m) * blocks * SP_LANES + 64 * h];
#pragma unroll
                        for (int q = 0; q < PRODUCTS; ++q)
#pragma unroll
                            for (int m = 0; m < MB; ++m)
#pragma unroll
                                for (int j = 0; j < NT; ++j) {
                                    if (q + 1 < PRODUCTS)
                                        low[m][j] = mma_bf16(b[p][j][PART_A[q]], x[m][PART_B[q]], q ? low[m][j] : f32x4{0.f, 0.f, 0.f, 0.f});
                                    else
                                        acc[m0 + m][j] = mma_bf16(b[p][j][0], x[m][0], acc[m0 + m][j]);
                                }
#pragma unroll
                        for (int m = 0; m < MB; ++m)
#pragma unroll
                            for (int j = 0; j < NT; ++j) acc[m0 + m][j] += low[m][j];
                    }
                }
            }
        }
        if (beyond || wild) {
            plain_tiles<MT, NT, ACROSS>(a, r0, ct0, lane, store);
            continue;
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int ct = ct0 + j;
            if (ct >= a.tiles) break;
            const int l = out_of(a, ct);
            const SplitOut &o = a.out[l];
            const int c = (ct - o.tile) * 16 + 4 * g;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const int64_t r = r0 + 16 * m + i;
                if (r >= a.rows) continue;
                f32x4 y = acc[m][j];
                if (o.n % 4 == 0) {   // rows of whole 16-byte pieces, on their boundaries
                    if (c >= o.n) continue;
                    if (o.b) y += f32x4{o.b[c], o.b[c + 1], o.b[c + 2], o.b[c + 3]};
                    const int64_t at = r * o.n + c;
                    if (a.skip) y += *reinterpret_cast<const f32x4 *>(a.skip + c) * *reinterpret_cast<const f32x4 *>(a.skip_x + at);
                    if (a.residual) y += *reinterpret_cast<const f32x4 *>(a.residual + at);
                    if (ACROSS && a.y_bf16) {
                        typedef __bf16 b4 __attribute__((ext_vector_type(4)));
                        *reinterpret_cast<b4 *>(static_cast<__bf16 *>(o.y) + at) = __builtin_convertvector(y, b4);
                    } else {
                        __builtin_nontemporal_store(y, reinterpret_cast<f32x4 *>(static_cast<float *>(o.y) + at));
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

template <int MT, int NT, bool ACROSS, bool FEW, int WAVES = 8> struct LaunchRows {
    static constexpr int SP_ROWS = 16 * MT;
    static constexpr auto kernel = split_rows_kernel<MT, NT, ACROSS, FEW, WAVES>;
    static inline const KernelRegistrar registrar{reinterpret_cast<const void *>(kernel), MT * (step_features(ACROSS) / 32) * SP_LANES * 16};
    static int go(hipStream_t st, SplitArgs &a, int most)
    {
        (void)&registrar;
        const int64_t row_tiles = (a.rows + SP_ROWS - 1) / SP_ROWS;
        a.passes = (a.tiles + WAVES * NT - 1) / (WAVES * NT);
        // two workgroups for every compute unit, where the columns give that many
        int64_t groups = (512 + row_tiles - 1) / row_tiles;
        a.groups = (int)(groups < a.passes ? groups : a.passes);
        const int64_t blocks = (row_tiles * a.groups + 7) / 8 * 8;
        if (blocks >= (1ll << 31)) return MRX_ERR_INVALID_ARG;
        return launch_kernel(kernel, dim3((unsigned)blocks), dim3(64 * WAVES), MT * most * SP_LANES * 16, st, a);
    }
};

// Columns of a wave: 32 read the rows from LDS half as often as 16 and are taken where they leave a workgroup for every compute unit.  Few rows: the
// fewest of a workgroup, 16, 32 or 64, that are no more than one workgroup for each (us, input gradient, 16 / 32 / 64: 1024 x 256 -> 3 x 256 26 / 29 / 37,
// 4096 x 256 40 / 30 / 37, 10620 x 128 -> 4 x 128 41 / 36 / 30; 1024 x 1024 -> 1024 54 / 38 / 49).
template <bool ACROSS> int launch_rows(hipStream_t st, SplitArgs &a, int most)
{
    auto workgroups = [&](int rows, int columns) { return (a.rows + rows - 1) / rows * ((a.tiles * 16 + columns - 1) / columns); };
    if (workgroups(64, 256) >= 256 && a.tiles > 8) {
        // rows of which one workgroup's fill a compute unit's LDS: sixteen waves of it, if they have columns (32768 x 256 -> 2056 217 -> 190 us)
        if constexpr (!ACROSS)
            if (most > 5 && workgroups(64, 512) >= 192 && a.tiles > 16) return LaunchRows<4, 2, ACROSS, false, 16>::go(st, a, most);
        return LaunchRows<4, 2, ACROSS, false>::go(st, a, most);
    }
    if (workgroups(16, 128) <= 256) return LaunchRows<1, 1, ACROSS, true>::go(st, a, most);
    if (workgroups(32, 128) <= 256) return LaunchRows<2, 1, ACROSS, true>::go(st, a, most);
    return workgroups(64, 128) <= 512 ? LaunchRows<4, 1, ACROSS, true>::go(st, a, most) : LaunchRows<4, 1, ACROSS, false>::go(st, a, most);
}

struct Sizes {
    int64_t steps = 0, tiles = 0, blocks = 0;   // of the contraction; 16-column tiles; 32-feature blocks of all steps
    bool ok = true;
};
Sizes sizes_of(const int64_t *n, int layers, int64_t K, bool across)
{
    const int SP_K = step_features(across);
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
    return z.ok ? z.blocks * z.tiles * 4 * SP_LANES + (z.steps * z.tiles + 3) / 4 * 4 : 0;
}

int split_rows(hipStream_t st, const SplitCall &c)
{
    const bool across = c.dys != nullptr;
    const Sizes z = sizes_of(c.n_out, c.layers, c.K, across);
    if (!z.ok || !c.workspace || !aligned(c.workspace, 16) || c.rows <= 0 || c.rows >= (1ll << 31)) return MRX_ERR_INVALID_ARG;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    SplitArgs a{};
    a.rows = c.rows, a.K = (int)c.K, a.steps = (int)z.steps, a.tiles = (int)z.tiles, a.residual = c.residual, a.skip = c.skip, a.skip_x = c.skip_x, a.y_bf16 = c.dx_bf16;
    const int SP_K = step_features(across);
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
    bf16x8 *const packed = reinterpret_cast<bf16x8 *>(c.workspace);
    int *const wild = reinterpret_cast<int *>(c.workspace + z.blocks * z.tiles * 4 * SP_LANES);
    a.packed = packed, a.wild = wild;
    const dim3 grid((unsigned)z.tiles, (unsigned)z.steps);
    const int rc = across ? launch_kernel(split_pack_kernel<true>, grid, dim3(SP_PACK), 0, st, a, packed, wild)
                    : launch_kernel(split_pack_kernel<false>, grid, dim3(SP_PACK), 0, st, a, packed, wild);
    if (rc != MRX_OK) return rc;
    return across ? launch_rows<true>(st, a, most) : launch_rows<false>(st, a, most);
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
