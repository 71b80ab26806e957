// What lies between two state updates of an acting step, as one launch: the closing layer of one block and the opening of the next.
//
//     x' = x + norm_c(rows) W_c^T + b_c                         (closing; left out where a chain of blocks begins)
//     y_l = norm(x') W_l^T + b_l  for a group of layers         (a matrix state's q, k, v, beta: mrx_closed_row_dense), or
//     z, h~, gate = norm(x') W^T -> MinGRU step -> gated state  (a gated recurrence: mrx_gated_recurrence_act)
//
// Few rows, one per environment.  A workgroup of eight waves owns 16 rows and 64 (gated: of each of its three layers) or 256 columns of
// the opening layers, and computes the closing layer for its rows whole: what that costs is reading W_c once more for each
// workgroup of a row tile.  Bound by its trips to memory -- a matrix state's traffic has pushed the weights out of L2 -- and
// by the 64 bytes a clock that a compute unit takes in.  So the rows and the weights of either product are requested in the order
// they are needed and go to LDS without passing through registers, in steps through slots of each wave's own: 128 bytes of k of the wave's
// 16 (up to 3) weight rows, fetched as whole lines of eight lanes (read as the matrix instruction wants them, 16 lanes on 16 lines, 128 KB take
// 2.9 us instead of 1.0).  Only the wave that requested a slot reads it, after a wait of its own; the workgroup meets at the barriers of the norms.
//
// In a graph behind 512 MB of other traffic, 256 features, bfloat16 (us; the closing layer in a launch of its own and then the opening / one launch):
//     gated recurrence     32 rows 12.2 / 11.8, 1024 14.2 / 13.8, 2048 18.4 / 19.3
//     q, k, v and beta     32 rows 9.4 / 10.7, 1024 14.0 / 11.8, 2048 18.1 / 16.2
// Which of the two is the callers' rule (host_ops.cpp, chain_pays).
// (A matrix state's projections and its step in one launch, the states on their way meanwhile, gain nothing: whole rows of states are 256 KB a
// workgroup, one workgroup a compute unit, and the slowest of them ends 40 % after the mean: 31 us, as two launches 31; few rows 9.2 / 7.7.)
//
// Rounding follows the launches it stands for (row_dense.hip, mingru_step_kernel).  The rows of x' that the second norm takes are still in
// float32 registers; sums are in another order than those launches take.
#include "mingru.h"
#include "row_dma.h"
#include "row_parts.h"

namespace mrx {
namespace {

typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

constexpr int AC_WAVES = 8, AC_THREADS = 64 * AC_WAVES, AC_ROWS = 16, AC_RPW = AC_ROWS / AC_WAVES, AC_SLOTS = 4;
constexpr int AC_PIECE = 16 * 128;            // bytes: 128 of k of 16 weight rows
constexpr int AC_REGION = 8 * AC_PIECE;       // of a wave's steps on their way, at most
constexpr int AC_MOST_X = 256;                // features of x' behind a closing layer
constexpr int AC_MOST_K = 512;                // features of a normalised row
constexpr int AC_MOST_LDS = 160 * 1024, AC_UNITS = 256;

// Where things lie in LDS.
struct ChainLds {
    int region, slots1, slots2;               // bytes of a wave's slots, and how many of each product's steps they hold
    int raw, raw_wave, scale, nbias, sums, tile, ld, bytes;
};

struct ChainArgs {
    RowInput in;                              // closing: the rows it reads, and their norm; else x and the opening's norm
    const void *wc, *bc;
    const float *residual;                    // (rows, F)
    float *x_out;                             // (rows, F)
    const float *scale, *nbias;               // closing: the opening's norm
    float eps, inv_F;
    int norm, F;                              // features of x'
    bool x_bf16, bc_bf16;
    // the opening
    const void *w[MRX_ROW_DENSE_LAYERS], *b[MRX_ROW_DENSE_LAYERS];
    void *y[MRX_ROW_DENSE_LAYERS];
    int n[MRX_ROW_DENSE_LAYERS], first[MRX_ROW_DENSE_LAYERS + 1];   // columns of a layer, its first 16-column tile
    int layers, tiles;                        // workgroups of a row tile
    bool b_bf16, y_bf16;
    const void *done;                         // gated
    const float *log_state, *log_decay;       // (rows, n[0]); may be updated in place
    float *log_state_out, *log_decay_out;
    void *z;                                  // (rows, n[0]) in the products' type; y[0]: the gated state
    int done_f32;
    ChainLds at;
};

__host__ __device__ inline int up(int x, int to) { return (x + to - 1) / to * to; }

// `bytes` from a base the wave shares to LDS, lane by lane, at most `most` of them there to read (the rest stays as it was).
__device__ __forceinline__ void dma_block(const void *base, int64_t most, int bytes, uint32_t lds, int lane)
{
    for (int at = 0; at < bytes; at += 1024)
        if (at + lane * 16 < bytes && at + lane * 16 < most) dma16(base, at + lane * 16, lds + at);
}

// All but the last n steps of C requests each have arrived.
template <int C> __device__ __forceinline__ void wait_steps(int n)
{
    static_assert(AC_SLOTS == 4);
    if (n <= 0) wait_vm<0>();
    else if (n == 1) wait_vm<C>();
    else if (n == 2) wait_vm<2 * C>();
    else if (n == 3) wait_vm<3 * C>();
    else wait_vm<4 * C>();
}

__device__ __forceinline__ f32x4 wide(const bf16x4 &b) { return f32x4{(float)b[0], (float)b[1], (float)b[2], (float)b[3]}; }

// log(1 + e) for 0 <= e <= 1 as 2 artanh(e / (2 + e)): eight terms of its series in (e / (2 + e))^2 <= 1/9 (1, 1/3 .. 1/15) leave 2^-29 of the result, a
// quarter of the library routine's instructions.
__device__ __forceinline__ float log1p_unit(float e)
{
    const float s = e / (2.f + e), q = s * s;
    float p = 1.f / 15.f;
    p = fmaf(p, q, 1.f / 13.f);
    p = fmaf(p, q, 1.f / 11.f);
    p = fmaf(p, q, 1.f / 9.f);
    p = fmaf(p, q, 1.f / 7.f);
    p = fmaf(p, q, 1.f / 5.f);
    p = fmaf(p, q, 1.f / 3.f);
    const float t = s + s;
    return fmaf(p * q, t, t);
}

// The weight rows of up to CT tiles of 16 columns, as they go through a wave's slots.
template <typename T, bool WBF, int CT> struct WeightStream {
    static constexpr int ES = WBF ? 2 : 4, KPIECE = 128 / ES, KB = TT<T>::KB, KS = KPIECE / KB;   // k of a piece, products in it
    static constexpr int PARTS = sizeof(RawFrag<T, WBF>) / 16;   // of 16 bytes in a fragment: two for weights that are rounded on their way
    const char *w[CT];
    uint32_t row[CT][2];   // where a lane's weight row starts, and which 16 of its 128 bytes the lane fetches, for each half of a piece:
    uint32_t chunk[2];     // stored rows are turned so that the reads below meet no bank twice
    uint32_t width;        // bytes of a row

    __device__ __forceinline__ void start(int K, int lane)
    {
        width = K * ES;
#pragma unroll
        for (int j = 0; j < 2; ++j) chunk[j] = ((lane % 8) ^ (j * 4 + lane / 16)) * 16;
    }
    __device__ __forceinline__ void place(int ct, const void *base, int n0, int N, int lane)
    {
        const int first = n0 < N ? n0 : N - 1, last = N - 1 - n0;
        w[ct] = static_cast<const char *>(base) + (int64_t)first * width;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int r = j * 8 + lane / 8, most = last < 15 ? (last < 0 ? 0 : last) : 15;
            row[ct][j] = __umul24(r < most ? r : most, width) + chunk[j];
        }
    }
    __device__ __forceinline__ void fetch(int step, uint32_t slot) const
    {
        const uint32_t k0 = step * 128;
        if (k0 + 128 <= width) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int j = 0; j < 2; ++j) dma16(w[ct] + k0, row[ct][j], slot + ct * AC_PIECE + j * 1024);
            return;
        }
        // the last of a row that is no whole number of steps: what lies past it is its end once more
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t k = k0 + chunk[j];
                dma16(w[ct], row[ct][j] - chunk[j] + (k < width ? k : width - 16), slot + ct * AC_PIECE + j * 1024);
            }
    }
    // acc += tile (rows x k) times the weights of this step: all that is read of LDS at once
    template <bool WHOLE> __device__ __forceinline__ void multiply(int step, const unsigned char *slot, const T *tile, int ld, int K, int lane, f32x4 *acc) const
    {
        using F = typename TT<T>::frag;
        const int i16 = lane & 15, g = lane >> 4, turn = i16 >> 1;
        const unsigned char *p = slot + i16 * 128;
        F xf[KS], wf[KS][CT];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int k = step * KPIECE + s * KB;
            if (!WHOLE && k >= K) break;
            xf[s] = TT<T>::template load<ROWK>(tile, ld, 0, k, lane);
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                struct {
                    f32x4 part[PARTS];
                } raw;
#pragma unroll
                for (int i = 0; i < PARTS; ++i)
                    raw.part[i] = *reinterpret_cast<const f32x4 *>(p + ((((s * 4 + g) * PARTS + i) ^ turn) * 16) + ct * AC_PIECE);
                wf[s][ct] = weight_frag<T, WBF>(__builtin_bit_cast(RawFrag<T, WBF>, raw));
                if (!WHOLE && k + TT<T>::KP * g >= K) wf[s][ct] = F{};
            }
        }
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            if (!WHOLE && step * KPIECE + s * KB >= K) break;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) acc[ct] = TT<T>::mma(wf[s][ct], xf[s], acc[ct]);
        }
    }
    // Two waves that share a contraction take every other 64 of it (whatever the weights' type: the same sums) -- or one takes all.
    static constexpr int BLOCK = 64 / KPIECE;
    template <bool SHARED> static __device__ __forceinline__ int step_of(int i, int half)
    {
        return SHARED ? i / BLOCK * (2 * BLOCK) + half * BLOCK + i % BLOCK : i;
    }
    template <bool SHARED> static __host__ __device__ __forceinline__ int steps_of(int K, int half)
    {
        const int all = (K + KPIECE - 1) / KPIECE, pairs = all / (2 * BLOCK), rest = all - pairs * 2 * BLOCK - half * BLOCK;
        return SHARED ? pairs * BLOCK + (rest < 0 ? 0 : rest < BLOCK ? rest : BLOCK) : all;
    }
    // A wave's steps through its slots: the requests of the first ones, and then the walk.
    template <bool SHARED> __device__ __forceinline__ void request(int half, int steps, int slots, uint32_t region) const
    {
        for (int i = 0; i < slots && i < steps; ++i) fetch(step_of<SHARED>(i, half), region + i * (CT * AC_PIECE));
    }
    template <bool SHARED>
    __device__ __forceinline__ void walk(int half, int steps, int slots, uint32_t region, const unsigned char *smem_region, const T *tile, int ld, int K,
                                         int lane, f32x4 *acc) const
    {
        for (int i = 0, slot = 0; i < steps; ++i) {
            const int left = steps - 1 - i, s = step_of<SHARED>(i, half);
            wait_steps<2 * CT>(left < slots - 1 ? left : slots - 1);
            const unsigned char *here = smem_region + slot * (CT * AC_PIECE);
            if ((s + 1) * KPIECE <= K) multiply<true>(s, here, tile, ld, K, lane, acc);
            else multiply<false>(s, here, tile, ld, K, lane, acc);
            if (i + slots < steps) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // read before it is fetched over
                fetch(step_of<SHARED>(i + slots, half), region + slot * (CT * AC_PIECE));
            }
            slot = slot + 1 == slots ? 0 : slot + 1;
        }
    }
};

// T: the products' type; WBF: bfloat16 weights; CT1: 16-column tiles of the closing layer a wave owns (F <= 128 CT1; 0: there is none);
// GATED: the opening is a gated recurrence's: two waves share 16 columns of its three layers, half of the contraction and then half of the
// results each.
template <typename T, bool WBF, int CT1, bool GATED> __global__ void __launch_bounds__(AC_THREADS) act_chain_kernel(ChainArgs a)
{
    using P = typename TT<T>::pack4;
    constexpr bool CLOSING = CT1 > 0;
    constexpr int C1 = CLOSING ? CT1 : 1, CT2 = GATED ? 3 : 2;
    extern __shared__ __align__(16) unsigned char smem[];
    touch(a);
    const ChainLds &at = a.at;
    const int K = a.in.K, F = a.F, lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i16 = lane & 15, g = lane >> 4;
    const uint32_t lds = lds_address(smem), region = lds + wv * at.region;
    const unsigned char *smem_region = smem + wv * at.region;
    T *tile = reinterpret_cast<T *>(smem + at.tile);
    const int64_t rows = a.in.rows, r0 = (int64_t)(blockIdx.x / (unsigned)a.tiles) * AC_ROWS, rw = r0 + wv * AC_RPW;
    const int column = (int)(blockIdx.x % (unsigned)a.tiles), half = GATED ? wv / 4 : 0;

    // ---- requests: rows and what their norm takes, what the closing layer's results meet, the first steps of the weights
    const int x_row = K * (a.x_bf16 ? 2 : 4);
    auto left = [&](int64_t row_bytes) { return rw < rows ? (rows - rw) * row_bytes : 0; };
    const int64_t rs = rw < rows ? rw : 0;   // a wave without rows asks for none
    dma_block(static_cast<const char *>(a.in.x) + rs * x_row, left(x_row), AC_RPW * x_row, lds + at.raw + wv * at.raw_wave, lane);
    if (wv == 0 && a.in.norm && a.in.scale) dma_block(a.in.scale, K * 4, K * 4, lds + at.scale, lane);
    if (!CLOSING && wv == 1 && a.in.norm && a.in.nbias) dma_block(a.in.nbias, K * 4, K * 4, lds + at.nbias, lane);
    WeightStream<T, WBF, C1> closing;
    WeightStream<T, WBF, CT2> opening;
    const int steps1 = closing.template steps_of<false>(K, 0), steps2 = opening.template steps_of<GATED>(F, half);
    // a lane's features 16 (wv CT1 + ct) + 4 g .. + 3 of x', row i16: what the closing layer's result meets waits in registers
    const int64_t r = r0 + i16, rin = r < rows ? r : rows - 1;
    auto feature = [&](int ct) { return (wv * C1 + ct) * 16 + 4 * g; };
    f32x4 add[C1], scale1[C1], nbias1[C1];
    u32x2 bias1[C1][2];   // four float32, or twice four bfloat16
    const bool scaled = a.norm && a.scale, shifted = a.norm && a.nbias;
    if constexpr (CLOSING) {
        // no branches: where there is nothing to load, something is, and dropped later
        const float *sc = scaled ? a.scale : a.residual, *nb = shifted ? a.nbias : a.residual;
        const char *bc = a.bc ? static_cast<const char *>(a.bc) : reinterpret_cast<const char *>(a.residual);
#pragma unroll
        for (int ct = 0; ct < C1; ++ct) {
            const int c = feature(ct) < F ? feature(ct) : 0;
            add[ct] = *reinterpret_cast<const f32x4 *>(a.residual + rin * F + c);
            scale1[ct] = *reinterpret_cast<const f32x4 *>(sc + c);
            nbias1[ct] = *reinterpret_cast<const f32x4 *>(nb + c);
            bias1[ct][0] = *reinterpret_cast<const u32x2 *>(bc + c * (a.bc_bf16 ? 2 : 4));
            bias1[ct][1] = *reinterpret_cast<const u32x2 *>(bc + c * (a.bc_bf16 ? 2 : 4) + (a.bc_bf16 ? 0 : 8));
        }
        closing.start(K, lane);
#pragma unroll
        for (int ct = 0; ct < C1; ++ct) closing.place(ct, a.wc, (wv * C1 + ct) * 16, F, lane);
        closing.template request<false>(0, steps1, at.slots1, region);
    }
    int n0[CT2], layer[CT2];
    opening.start(F, lane);
#pragma unroll
    for (int ct = 0; ct < CT2; ++ct) {
        if (GATED) {
            layer[ct] = ct, n0[ct] = (column * 4 + wv % 4) * 16;
        } else {
            const int t = (column * AC_WAVES + wv) * CT2 + ct;
            int l = 0;
#pragma unroll
            for (int j = 1; j < MRX_ROW_DENSE_LAYERS; ++j) l += j < a.layers && t >= a.first[j];
            layer[ct] = l, n0[ct] = (t - a.first[l]) * 16;   // past the last layer's columns: nothing of it is kept
        }
        opening.place(ct, a.w[layer[ct]], n0[ct], a.n[layer[ct]], lane);
    }
    if (!CLOSING) opening.template request<GATED>(half, steps2, at.slots2, region);
    // what the lanes need in the end waits in registers; gated: features 4 g + 2 half, + 1 of the wave's columns
    f32x2 ls = {}, ldc = {};
    uint32_t flag = 0, bias_raw[CT2][4] = {};
    const int cg = n0[0] + 4 * g + 2 * half;
    if (GATED) {
        ls = *reinterpret_cast<const f32x2 *>(a.log_state + rin * a.n[0] + (cg < a.n[0] ? cg : 0));   // a multiple of 4 columns
        ldc = *reinterpret_cast<const f32x2 *>(a.log_decay + rin * a.n[0] + (cg < a.n[0] ? cg : 0));
        flag = done_raw(a.done, a.done_f32, rin);
    } else {
#pragma unroll
        for (int ct = 0; ct < CT2; ++ct)
            if (const void *b = a.b[layer[ct]]) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int c = n0[ct] + 4 * g + e < a.n[layer[ct]] ? n0[ct] + 4 * g + e : a.n[layer[ct]] - 1;
                    bias_raw[ct][e] = a.b_bf16 ? static_cast<const uint16_t *>(b)[c] : static_cast<const uint32_t *>(b)[c];
                }
            }
    }

    // ---- the rows, normalised
    if (CLOSING) wait_steps<2 * C1>(steps1 < at.slots1 ? steps1 : at.slots1);
    else wait_steps<2 * CT2>(steps2 < at.slots2 ? steps2 : at.slots2);
    sync_lds();
    auto rows_in = [&](auto xbf, auto nv) {
        RowPanel<decltype(xbf)::value, AC_RPW, decltype(nv)::value> panel;
        using Raw = typename decltype(panel)::Raw;
        const unsigned char *raw = smem + at.raw + wv * at.raw_wave;
#pragma unroll
        for (int i = 0; i < decltype(nv)::value; ++i) {
            const int c = (i * 64 + lane) * 4 < K ? (i * 64 + lane) * 4 : 0;
            panel.scale[i] = f32x4{1.f, 1.f, 1.f, 1.f};
            panel.nbias[i] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (a.in.norm && a.in.scale) panel.scale[i] = *reinterpret_cast<const f32x4 *>(smem + at.scale + c * 4);
            if (!CLOSING && a.in.norm && a.in.nbias) panel.nbias[i] = *reinterpret_cast<const f32x4 *>(smem + at.nbias + c * 4);
#pragma unroll
            for (int j = 0; j < AC_RPW; ++j) {   // rows past the last: zeros, what lies in LDS is not theirs
                const Raw x = *reinterpret_cast<const Raw *>(raw + j * x_row + c * (decltype(xbf)::value ? 2 : 4));
                panel.x[j][i] = rw + j < rows ? x : Raw{};
            }
        }
        panel.template finish<T>(a.in, tile + wv * AC_RPW * at.ld, at.ld, up(K, 32), lane, [](int, int, int, const f32x4 &) {});
    };
    auto by_type = [&](auto nv) {
        if (a.x_bf16) rows_in(std::true_type{}, nv);
        else rows_in(std::false_type{}, nv);
    };
    if (K <= 256) by_type(std::integral_constant<int, 1>{});
    else by_type(std::integral_constant<int, 2>{});
    sync_lds();

    // ---- the closing layer, its residual, and the norm of what comes out: a lane has features 16 (wv CT1 + ct) + 4 g .. + 3 of row i16
    if constexpr (CLOSING) {
        f32x4 x[C1];
        zero_acc<C1>(x);
        closing.template walk<false>(0, steps1, at.slots1, region, smem_region, tile, at.ld, K, lane, x);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slots are read
        // (waited for now, where every request has arrived, and not behind the next ones)
#pragma unroll
        for (int ct = 0; ct < C1; ++ct) asm volatile("" : "+v"(add[ct]), "+v"(scale1[ct]), "+v"(nbias1[ct]), "+v"(bias1[ct][0]), "+v"(bias1[ct][1]));
        opening.template request<GATED>(half, steps2, at.slots2, region);
#pragma unroll
        for (int ct = 0; ct < C1; ++ct) {
            f32x4 bias = {0.f, 0.f, 0.f, 0.f};
            if (a.bc && a.bc_bf16) bias = wide(__builtin_bit_cast(bf16x4, bias1[ct][0]));
            else if (a.bc) bias = __builtin_shufflevector(__builtin_bit_cast(f32x2, bias1[ct][0]), __builtin_bit_cast(f32x2, bias1[ct][1]), 0, 1, 2, 3);
            if constexpr (std::is_same<T, __bf16>::value) {
                x[ct] += wide(TT<__bf16>::pack(bias[0], bias[1], bias[2], bias[3]));
                x[ct] = wide(TT<__bf16>::pack(x[ct][0], x[ct][1], x[ct][2], x[ct][3]));
            } else {
                x[ct] += bias;
            }
            x[ct] += add[ct];
            const int c = feature(ct);
            if (c >= F || r >= rows) x[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
            else if (column == 0) *reinterpret_cast<f32x4 *>(a.x_out + r * F + c) = x[ct];
        }
        float *sums = reinterpret_cast<float *>(smem + at.sums);
        auto total = [&](float s, float *to) {   // over a row's features: four lane groups, eight waves
            s = add_across<32>(add_across<16>(s));
            if (g == 0) to[i16 * AC_WAVES + wv] = s;
            sync_lds();
            const f32x4 t = *reinterpret_cast<const f32x4 *>(to + i16 * AC_WAVES), u = *reinterpret_cast<const f32x4 *>(to + i16 * AC_WAVES + 4);
            return (t[0] + t[1] + t[2] + t[3]) + (u[0] + u[1] + u[2] + u[3]);
        };
        if (a.norm == 2) {
            float s = 0.f;
#pragma unroll
            for (int ct = 0; ct < C1; ++ct) s += x[ct][0] + x[ct][1] + x[ct][2] + x[ct][3];
            const float mean = total(s, sums + AC_ROWS * AC_WAVES) * a.inv_F;
#pragma unroll
            for (int ct = 0; ct < C1; ++ct)
                if (feature(ct) < F)
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[ct][e] -= mean;
        }
        float s = 0.f;
#pragma unroll
        for (int ct = 0; ct < C1; ++ct)
#pragma unroll
            for (int e = 0; e < 4; ++e) s += x[ct][e] * x[ct][e];
        const float squares = total(s, sums);   // (behind its barrier every wave is done with the tile)
        const float rstd = a.norm ? rsqrtf(squares * a.inv_F + a.eps) : 1.f;
#pragma unroll
        for (int ct = 0; ct < C1; ++ct) {
            const int c = feature(ct);
            if (c >= up(F, 32)) continue;
            x[ct] = x[ct] * rstd;
            if (scaled) x[ct] *= scale1[ct];
            if (shifted) x[ct] += nbias1[ct];
            if (c >= F) x[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
            *reinterpret_cast<P *>(tile + i16 * at.ld + c) = TT<T>::pack(x[ct][0], x[ct][1], x[ct][2], x[ct][3]);
        }
        sync_lds();
    }

    // ---- the opening
    f32x4 acc[CT2];
    zero_acc<CT2>(acc);
    opening.template walk<GATED>(half, steps2, at.slots2, region, smem_region, tile, at.ld, F, lane, acc);
    wait_vm<0>();   // (a wave without a step of its own)
    if constexpr (GATED) {
        // each of the two waves gets the other's part of its half of the results, through the other's slots
        float *give = reinterpret_cast<float *>(smem + wv * at.region) + lane, *take = reinterpret_cast<float *>(smem + (wv ^ 4) * at.region) + lane;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int l = 0; l < 3; ++l)
#pragma unroll
            for (int e = 0; e < 2; ++e) give[(l * 2 + e) * 64] = half ? acc[l][e] : acc[l][2 + e];
        sync_lds();
        f32x2 mine[3];
#pragma unroll
        for (int l = 0; l < 3; ++l)
#pragma unroll
            for (int e = 0; e < 2; ++e) mine[l][e] = (half ? acc[l][2 + e] : acc[l][e]) + take[(l * 2 + e) * 64];
        if (r >= rows || cg >= a.n[0]) return;
        const int64_t to = r * a.n[0] + cg;
        const bool reset = done_test(flag, a.done_f32);
        typedef T Pair __attribute__((ext_vector_type(2)));
        Pair zs, ys;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            zs[e] = (T)mine[0][e];
            const float z = (float)zs[e];
            float za = z, xb = (float)(T)mine[1][e];
            const float log_a = -(fmaxf(z, 0.f) + log1p_unit(expf(-fabsf(z))));   // log sigma(-z)
            MinGru::coeffs(za, xb);
            const float h = reset ? xb : za * expf(ls[e]) + xb, gate = (float)(T)mine[2][e];
            ls[e] = logf(h);
            ldc[e] = reset ? log_a : ldc[e] + log_a;
            ys[e] = (T)((float)(T)h * gate / (1.f + __expf(-gate)));   // the state as the cell hands it on
        }
        *reinterpret_cast<f32x2 *>(a.log_state_out + to) = ls;
        *reinterpret_cast<f32x2 *>(a.log_decay_out + to) = ldc;
        *reinterpret_cast<Pair *>(static_cast<T *>(a.z) + to) = zs;
        *reinterpret_cast<Pair *>(static_cast<T *>(a.y[0]) + to) = ys;
    } else {
#pragma unroll
        for (int ct = 0; ct < CT2; ++ct) {
            const int N = a.n[layer[ct]], c = n0[ct] + 4 * g;
            if (r >= rows || c >= N) continue;
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float bias = a.b_bf16 ? raw_to_float<__bf16>(bias_raw[ct][e]) : raw_to_float<float>(bias_raw[ct][e]);
                if (std::is_same<T, __bf16>::value) bias = (float)(__bf16)bias;
                y[e] = acc[ct][e] + bias;
                if (std::is_same<T, __bf16>::value) y[e] = (float)(__bf16)y[e];
            }
            float *yf = static_cast<float *>(a.y[layer[ct]]) + r * N + c;
            __bf16 *yb = static_cast<__bf16 *>(a.y[layer[ct]]) + r * N + c;
            if (N % 4 == 0) {
                if (a.y_bf16) *reinterpret_cast<bf16x4 *>(yb) = TT<__bf16>::pack(y[0], y[1], y[2], y[3]);
                else *reinterpret_cast<f32x4 *>(yf) = f32x4{y[0], y[1], y[2], y[3]};
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (c + e >= N) break;
                if (a.y_bf16) yb[e] = (__bf16)y[e];
                else yf[e] = y[e];
            }
        }
    }
}

template <typename T, bool WBF, int CT1, bool GATED> struct ChainKernel {
    static constexpr auto fn = act_chain_kernel<T, WBF, CT1, GATED>;
    static inline const KernelRegistrar registrar{reinterpret_cast<const void *>(fn), AC_MOST_LDS};
    static auto get()
    {
        (void)&registrar;
        return fn;
    }
};

// The workgroup's LDS with `region` bytes of weights on their way for each wave; false: more than there is.
bool lay_out(ChainArgs &a, bool closing, int ct1, int ct2, int t_bytes, int region)
{
    ChainLds &s = a.at;
    const int K = a.in.K, F = a.F;
    auto slots = [&](int ct) { return region / (ct * AC_PIECE) < AC_SLOTS ? region / (ct * AC_PIECE) : AC_SLOTS; };
    s.region = region, s.slots1 = closing ? slots(ct1) : 0, s.slots2 = slots(ct2);
    int at = AC_WAVES * region;
    auto take = [&](int n) {
        const int p = at;
        at += up(n, 16);
        return p;
    };
    s.raw_wave = up(AC_RPW * K * (a.x_bf16 ? 2 : 4), 16);
    s.raw = take(AC_WAVES * s.raw_wave), s.scale = take(K * 4), s.nbias = closing ? 0 : take(K * 4);
    s.sums = closing ? take(AC_ROWS * AC_WAVES * 2 * 4) : 0;
    s.ld = up(K > F ? K : F, 32) + 16 / t_bytes;
    s.tile = take(AC_ROWS * s.ld * t_bytes);
    s.bytes = at;
    return at <= AC_MOST_LDS && s.slots2 > 0 && (!closing || s.slots1 > 0);
}
template <typename T, bool WBF, bool GATED> int launch_chain(hipStream_t st, ChainArgs &a, bool closing)
{
    const int64_t grid = (a.in.rows + AC_ROWS - 1) / AC_ROWS * a.tiles;
    if (grid >= (1ll << 31)) return MRX_ERR_INVALID_ARG;
    auto go = [&](auto ct1) -> int {
        constexpr int CT1 = decltype(ct1)::value, CT2 = GATED ? 3 : 2;
        // No more than the steps there are; and room for a second workgroup on the compute unit where there are workgroups for it and the rows leave it: with
        // one of 160 KB a grid of more than the compute units loses to smaller workgroups.  A gated recurrence alone, bfloat16, us, four waves with
        // their weights in registers / one workgroup a unit / two: 256 features and columns 4096 rows 24.7 / 26.4 / 20.2, 16 384 74 / 90 / 62; 256 by 1024 columns
        // 2048 rows 41 / 48 / 34; float32 128 by 256 columns 8192 rows 49 / 56 / 41.  (Rows of 320 to 500 features leave none: 384, 8192 rows 79 / 82.)
        using Closing = WeightStream<T, WBF, CT1 ? CT1 : 1>;
        using Opening = WeightStream<T, WBF, CT2>;
        const int need1 = CT1 * Closing::template steps_of<false>(a.in.K, 0), need2 = CT2 * Opening::template steps_of<GATED>(a.F, 0), need = need1 > need2 ? need1 : need2;
        int region = need * AC_PIECE < AC_REGION ? need * AC_PIECE : AC_REGION;
        while (region > 0 && !lay_out(a, closing, CT1, CT2, sizeof(T), region)) region -= AC_PIECE;
        if (region <= 0) return MRX_ERR_UNSUPPORTED;
        if (grid > AC_UNITS) {
            int less = region;
            while (less > 0 && !(lay_out(a, closing, CT1, CT2, sizeof(T), less) && a.at.bytes <= AC_MOST_LDS / 2)) less -= AC_PIECE;
            if (less <= 0) lay_out(a, closing, CT1, CT2, sizeof(T), region);
        }
        return launch_kernel(ChainKernel<T, WBF, CT1, GATED>::get(), dim3((unsigned)grid), dim3(AC_THREADS), a.at.bytes, st, a);
    };
    if constexpr (GATED)
        if (!closing) return go(std::integral_constant<int, 0>{});
    if (a.F <= 128) return go(std::integral_constant<int, 1>{});
    return go(std::integral_constant<int, 2>{});
}
template <bool GATED> int by_type(hipStream_t st, ChainArgs &a, bool closing, int w_dtype, int product_dtype)
{
    if (product_dtype == MRX_F32) return launch_chain<float, false, GATED>(st, a, closing);
    return w_dtype == MRX_BF16 ? launch_chain<__bf16, true, GATED>(st, a, closing) : launch_chain<__bf16, false, GATED>(st, a, closing);
}

bool known(int dt) { return dt == MRX_F32 || dt == MRX_BF16; }

// The rows that come in, and what is done to them before the opening's products.
int chain_input(ChainArgs &a, const mrx_closing *c, const float *x, const float *scale, const float *norm_bias, int norm, int64_t rows, int64_t K,
                int w_dtype, int product_dtype, float eps)
{
    if (!known(w_dtype) || !known(product_dtype) || norm < 0 || norm > 2 || rows <= 0 || rows >= (1ll << 31) || K <= 0) return MRX_ERR_INVALID_ARG;
    if (!aligned(scale, 16) || !aligned(norm_bias, 16)) return MRX_ERR_INVALID_ARG;
    if (K > AC_MOST_K || (product_dtype == MRX_F32 && w_dtype != MRX_F32)) return MRX_ERR_UNSUPPORTED;
    if (K % 8 != 0) return MRX_ERR_INVALID_ARG;
    a.F = (int)K, a.inv_F = 1.f / (float)K, a.eps = eps, a.norm = norm;
    if (!c) {
        if (!x || !aligned(x, 16)) return MRX_ERR_INVALID_ARG;
        a.in = RowInput{x, scale, norm_bias, rows, (int)K, norm, eps, 1.f / (float)K, false};
        return MRX_OK;
    }
    if (!c->rows || !c->weight || !c->residual || !c->out || !known(c->row_dtype) || c->K <= 0 || (c->bias && !known(c->bias_dtype))) return MRX_ERR_INVALID_ARG;
    const void *arrays[] = {c->rows, c->scale, c->weight, c->bias, c->residual, c->out};
    for (const void *p : arrays)
        if (!aligned(p, 16)) return MRX_ERR_INVALID_ARG;
    if (K > AC_MOST_X || c->K > AC_MOST_K) return MRX_ERR_UNSUPPORTED;
    if (c->K % 8 != 0) return MRX_ERR_INVALID_ARG;
    // the first workgroup of a row tile writes `out` while the others still read what it comes from
    auto apart = [&](const void *p, int64_t bytes) {
        const uintptr_t from = reinterpret_cast<uintptr_t>(p), out = reinterpret_cast<uintptr_t>(c->out);
        return from + bytes <= out || out + rows * K * 4 <= from;
    };
    if (!apart(c->residual, rows * K * 4) || !apart(c->rows, rows * c->K * (c->row_dtype == MRX_BF16 ? 2 : 4))) return MRX_ERR_INVALID_ARG;
    a.in = RowInput{c->rows, c->scale, nullptr, rows, (int)c->K, c->norm ? 1 : 0, c->eps, 1.f / (float)c->K, c->round_norm != 0};
    a.wc = c->weight, a.bc = c->bias, a.residual = c->residual, a.x_out = c->out, a.scale = scale, a.nbias = norm_bias;
    a.x_bf16 = c->row_dtype == MRX_BF16, a.bc_bf16 = c->bias_dtype == MRX_BF16;
    return MRX_OK;
}

}  // namespace
}  // namespace mrx

extern "C" int mrx_closed_row_dense(void *stream, const mrx_closing *closing, const float *scale, const float *norm_bias, int norm,
                                    const void *const *weights, const void *const *biases, void *const *outs, const int64_t *n_out, int layers,
                                    int64_t rows, int64_t K, int w_dtype, int b_dtype, int y_dtype, int product_dtype, float eps)
{
    using namespace mrx;
    ChainArgs a{};
    if (!closing) return MRX_ERR_INVALID_ARG;
    if (const int rc = chain_input(a, closing, nullptr, scale, norm_bias, norm, rows, K, w_dtype, product_dtype, eps); rc != MRX_OK) return rc;
    if (!weights || !biases || !outs || !n_out || layers < 1 || layers > MRX_ROW_DENSE_LAYERS || !known(b_dtype) || !known(y_dtype)) return MRX_ERR_INVALID_ARG;
    int tiles = 0;
    for (int l = 0; l < layers; ++l) {
        if (!weights[l] || !outs[l] || !aligned(weights[l], 16) || !aligned(outs[l], 16) || n_out[l] <= 0) return MRX_ERR_INVALID_ARG;
        if (n_out[l] > (1 << 24)) return MRX_ERR_UNSUPPORTED;
        a.w[l] = weights[l], a.b[l] = biases[l], a.y[l] = outs[l], a.n[l] = (int)n_out[l], a.first[l] = tiles;
        tiles += (int)(n_out[l] + 15) / 16;
    }
    a.layers = layers, a.b_bf16 = b_dtype == MRX_BF16, a.y_bf16 = y_dtype == MRX_BF16;
    a.tiles = (tiles + 2 * AC_WAVES - 1) / (2 * AC_WAVES);
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    return by_type<false>(static_cast<hipStream_t>(stream), a, true, w_dtype, product_dtype);
}

extern "C" int mrx_closed_gated_recurrence_act(void *stream, const mrx_closing *closing, const float *x, const float *scale,
                                               const float *norm_bias, int norm, const void *w_z, const void *w_h, const void *w_gate, const void *done,
                                               const float *log_state, const float *log_decay, void *z, void *y, float *log_state_out,
                                               float *log_decay_out, int64_t rows, int64_t K, int64_t N, int w_dtype, int product_dtype, int done_dtype,
                                               float eps)
{
    using namespace mrx;
    ChainArgs a{};
    const void *arrays[] = {w_z, w_h, w_gate, log_state, log_decay, z, y, log_state_out, log_decay_out};
    for (const void *p : arrays)
        if (!p || !aligned(p, 16)) return MRX_ERR_INVALID_ARG;
    if (!done || (done_dtype != MRX_DONE_U8 && done_dtype != MRX_DONE_F32)) return MRX_ERR_INVALID_ARG;
    if (const int rc = chain_input(a, closing, x, scale, norm_bias, norm, rows, K, w_dtype, product_dtype, eps); rc != MRX_OK) return rc;
    if (N <= 0 || N % 4 != 0 || N > (1 << 24)) return MRX_ERR_UNSUPPORTED;
    a.w[0] = w_z, a.w[1] = w_h, a.w[2] = w_gate, a.done = done, a.done_f32 = done_dtype == MRX_DONE_F32, a.layers = 3;
    for (int l = 0; l < 3; ++l) a.n[l] = (int)N;
    a.log_state = log_state, a.log_decay = log_decay, a.log_state_out = log_state_out, a.log_decay_out = log_decay_out, a.z = z, a.y[0] = y;
    a.tiles = (int)((N + 63) / 64);
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    return by_type<true>(static_cast<hipStream_t>(stream), a, closing != nullptr, w_dtype, product_dtype);
}

extern "C" int mrx_gated_recurrence_act(void *stream, const float *x, const float *scale, const float *norm_bias, int norm, const void *w_z,
                                        const void *w_h, const void *w_gate, const void *done, const float *log_state,
                                        const float *log_decay, void *z, void *y, float *log_state_out, float *log_decay_out,
                                        int64_t rows, int64_t K, int64_t N, int w_dtype, int product_dtype, int done_dtype, float eps)
{
    return mrx_closed_gated_recurrence_act(stream, nullptr, x, scale, norm_bias, norm, w_z, w_h, w_gate, done, log_state, log_decay, z, y,
                                           log_state_out, log_decay_out, rows, K, N, w_dtype, product_dtype, done_dtype, eps);
}
