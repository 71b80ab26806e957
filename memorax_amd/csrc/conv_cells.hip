// What the Mamba and mLSTM cells do around their recurrence (mamba.py:88-144, mlstm.py:88-187), as passes that read
// their operands once: the causal depthwise convolution over time with silu behind it, the elements made of it, and
// the gated read-out.  As array operations (a transpose, a padding, the library's grouped convolution, slices, products)
// these took twenty times what the cell's products and its recurrence take together.
//
//   conv      s_t = bias + sum_j w_j x_{t-K+1+j}  (x = 0 before the call's first step: the reference's convolution
//             restarts at every call, resets or not),   y_t = silu(s_t)
//   elements  v = y of the hidden channels,  k = y of B's channels * dt,  q = y of C's channels,
//             dt = softplus(dt_in + dt_bias),  g = -dt exp(A_log)
//   read-out  y = rms_norm(o + D hidden) * scale * silu(z)
//
// Layout: a wave is 64 lanes x 4 consecutive channels of one time tile and walks its steps with the last K inputs in registers, so a row of an
// array is read once per tile (plus K - 1 rows that the neighbouring tile of the same workgroup has just brought in), four rows requested ahead
// of their use.  256 x 128 steps x 1536 channels: the elements 84 us forward and 143 backward (402 and 670 MB: 63 and 105 us at what a copy
// reaches), bound by HBM and the exponentials' arithmetic about alike; with a branch at every load, a division per sigmoid and a head's gate formed
// by each of its lanes at each step they took 93 and 184.  Two channels per lane -- twice the waves in flight -- read the same (86 and 143).
#include <initializer_list>
#include <type_traits>

#include "col_sum.h"
#include "common.h"

namespace mrx {
namespace {

constexpr int CV_WAVES = 4, CV_THREADS = 64 * CV_WAVES;
constexpr int CV_AHEAD = 4;       // rows requested ahead
constexpr int CV_MAX_K = 4;       // widest convolution

struct alignas(16) F4 {
    float v[4];
};
constexpr F4 F4_ZERO{{0.f, 0.f, 0.f, 0.f}};
__device__ __forceinline__ F4 load4(const float *p) { return *reinterpret_cast<const F4 *>(p); }
__device__ __forceinline__ void store4(float *p, const F4 &x) { *reinterpret_cast<F4 *>(p) = x; }

// The library exponential: the hardware's errs by |x| / 2 ulp, which silu keeps as a relative error, and the passes are bound by HBM.
// The quotient by one Newton step on the hardware's reciprocal (the remainder formed exactly: as good as a division's own steps, a third as many;
// the fix-up restores 0 and NaN).
__device__ __forceinline__ float sigmoidf(float x)
{
    const float d = 1.f + expf(-x), r = __builtin_amdgcn_rcpf(d);
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, r, 1.f), r, r), d, 1.f);
}
__device__ __forceinline__ float softplusf(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// One run of channels of a convolution: where its rows lie and what becomes of them.
struct Segment {
    const float *x;       // inputs, rows ld apart
    int64_t ld;
    float *y;             // forward: results, rows C apart
    const float *dy;      // backward: their gradients, rows C apart
    const float *skip;    // backward: a second gradient of y, read as skip * skip_scale[channel / P] (the D-skip of the read-out)
    float *dx;            // backward: rows ld_dx apart
    int64_t ld_dx;
    int C, w0;            // channels; the first one's index among the convolution's channels
    bool gated;           // y is multiplied by dt[head], head = channel / N
};
struct ConvArgs {
    Segment seg[3];
    int nseg, tiles[3];   // 256-channel tiles of each segment
    const float *w, *bias;            // (C_total, K), (C_total)
    const float *dt_in, *dt_bias, *A_log, *D;   // (B,T,H), (H), (H), (H): the elements' gates (null: a plain convolution)
    float *g;                         // forward: log-decay (B,T,H)
    const float *dg;                  // backward: its gradient
    float *ddt_in;                    // backward: (B,T,H)
    float *parts;                     // backward: (nparts, columns) partial sums of the parameters' gradients
    int nparts;
    int columns;                      // C_total * K + C_total + 2 H + C_seg0 / 4
    int T, H, P, N, C_total, tile_t, tiles_t;
    int64_t items;                    // B * tiles_t
};

// Which segment, and which of its tiles, a workgroup column serves.
__device__ __forceinline__ int segment_of(const ConvArgs &a, int &tile)
{
    int s = 0;
    while (s + 1 < a.nseg && tile >= a.tiles[s]) tile -= a.tiles[s++];
    return s;
}

template <int K> __device__ __forceinline__ void load_taps(const ConvArgs &a, const Segment &sg, int c, bool act, F4 (&w)[K], F4 &bias)
{
    bias = F4_ZERO;
#pragma unroll
    for (int j = 0; j < K; ++j) w[j] = F4_ZERO;
    if (!act) return;
    bias = load4(a.bias + sg.w0 + c);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < K; ++j) w[j].v[e] = a.w[(int64_t)(sg.w0 + c + e) * K + j];
}

// A value of lane I of the lane's group of four, and that of the lane whose number differs in the bits of M.
template <int I> __device__ __forceinline__ float of_lane(float x)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), I * 0x55, 0xf, 0xf, true));
}
template <int M> __device__ __forceinline__ float other_lane(float x)
{
    constexpr int ctrl = (0 ^ M) | (1 ^ M) << 2 | (2 ^ M) << 4 | (3 ^ M) << 6;
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), ctrl, 0xf, 0xf, true));
}
// Four values of every lane, added up over the lane's group of four: lane l is left with the sum of the value l & 3.
__device__ __forceinline__ float sum_of_four(const float (&x)[4], int lane)
{
    const bool odd = lane & 1, high = lane & 2;
    const float s01 = (odd ? x[1] : x[0]) + other_lane<1>(odd ? x[0] : x[1]), s23 = (odd ? x[3] : x[2]) + other_lane<1>(odd ? x[2] : x[3]);
    return (high ? s23 : s01) + other_lane<2>(high ? s01 : s23);
}

// What the kinds of channels differ in: PLAIN, GATED (y times dt of the head), SKIP (a second gradient, backward only).
enum Kind { PLAIN, GATED, SKIP };

// Rows are requested four at a time and four ahead of their use, without a branch: rows past the sequence read its last one, lanes past the
// channels the first ones.  A head's gate at the four steps is formed once, by the four lanes of each group of four (a head of sixteen features
// is four lanes; narrower ones form all four in every lane).
template <int K, int KIND> __device__ __forceinline__ void conv_fwd_walk(const ConvArgs &a, const Segment &sg, int c, bool act, int64_t item)
{
    const int lane = threadIdx.x & 63, cc = act ? c : 0;
    const int64_t b = item / a.tiles_t;
    const int t0 = (int)(item % a.tiles_t) * a.tile_t, t1 = min(a.T, t0 + a.tile_t);
    const int64_t row0 = b * a.T;
    F4 w[K], bias, win[K];
    load_taps<K>(a, sg, c, act, w, bias);
    const float *x = sg.x + row0 * sg.ld;
    float *y = sg.y + row0 * sg.C;
    const int h = KIND == GATED ? cc / a.N : 0;
    const bool four = a.N >= 16;
    const float dtb = KIND == GATED ? a.dt_bias[h] : 0.f;
    auto row = [&](int t) { return t < a.T ? t : a.T - 1; };
#pragma unroll
    for (int j = 0; j < K - 1; ++j) {
        const int t = t0 - (K - 1) + j;
        win[j + 1] = load4(x + (t < 0 ? 0 : t) * sg.ld + cc);
        if (t < 0) win[j + 1] = F4_ZERO;
    }
    F4 next[CV_AHEAD];
    float dt_next = 0.f;
    auto fetch = [&](int t) {
#pragma unroll
        for (int i = 0; i < CV_AHEAD; ++i) next[i] = load4(x + row(t + i) * sg.ld + cc);
        if (KIND == GATED && four) dt_next = a.dt_in[(row0 + row(t + (lane & 3))) * a.H + h];
    };
    fetch(t0);
    for (int t = t0; t < t1; t += CV_AHEAD) {
        F4 cur[CV_AHEAD];
#pragma unroll
        for (int i = 0; i < CV_AHEAD; ++i) cur[i] = next[i];
        float gate[CV_AHEAD] = {1.f, 1.f, 1.f, 1.f};
        const float dt = dt_next;
        if (t + CV_AHEAD < t1) fetch(t + CV_AHEAD);
        if (KIND == GATED) {
            if (four) {
                const float g = softplusf(dt + dtb);
                gate[0] = of_lane<0>(g), gate[1] = of_lane<1>(g), gate[2] = of_lane<2>(g), gate[3] = of_lane<3>(g);
            } else {
#pragma unroll
                for (int i = 0; i < CV_AHEAD; ++i) gate[i] = softplusf(a.dt_in[(row0 + row(t + i)) * a.H + h] + dtb);
            }
        }
#pragma unroll
        for (int i = 0; i < CV_AHEAD; ++i) {
#pragma unroll
            for (int j = 0; j + 1 < K; ++j) win[j] = win[j + 1];
            win[K - 1] = cur[i];
            F4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float s = bias.v[e];
#pragma unroll
                for (int j = 0; j < K; ++j) s += w[j].v[e] * win[j].v[e];
                o.v[e] = s * sigmoidf(s);
                if (KIND == GATED) o.v[e] *= gate[i];
            }
            if (act && t + i < t1) store4(y + (int64_t)(t + i) * sg.C + c, o);
        }
    }
}

template <int K> __global__ void __launch_bounds__(CV_THREADS) conv_fwd_kernel(ConvArgs a)
{
    int ntiles = 0;
    for (int s = 0; s < a.nseg; ++s) ntiles += a.tiles[s];
    int tile = (int)(blockIdx.x % (unsigned)ntiles);
    const int64_t item = (int64_t)(blockIdx.x / (unsigned)ntiles) * CV_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (item >= a.items) return;
    const int lane = threadIdx.x & 63;
    if (tile == 0 && a.g) {   // the log-decay, beside the first tile's work
        const int t0 = (int)(item % a.tiles_t) * a.tile_t, n = (min(a.T, t0 + a.tile_t) - t0) * a.H;
        const int64_t first = (item / a.tiles_t * a.T + t0) * a.H;
        for (int i = lane; i < n; i += 64) {
            const int h = i % a.H;
            a.g[first + i] = softplusf(a.dt_in[first + i] + a.dt_bias[h]) * -expf(a.A_log[h]);
        }
    }
    const Segment &sg = a.seg[segment_of(a, tile)];
    const int c = (tile * 64 + lane) * 4;
    if (sg.gated) conv_fwd_walk<K, GATED>(a, sg, c, c < sg.C, item);
    else conv_fwd_walk<K, PLAIN>(a, sg, c, c < sg.C, item);
}

// A wave's share of the parameters' gradients.
template <int K> struct ConvSums {
    F4 dw[K], dbias;
    float dtb, A, D;
};

// Backward: the pre-activations are formed again from the inputs; a step's gradient ds_t = dy_t silu'(s_t) reaches the inputs
// t-K+1 .. t, so dx_{t-K+1} is complete once ds_t is known, and a tile walks K - 1 steps past its end for its last rows.
// The parameters' gradients stay in registers over all tiles of a wave (workgroup column p takes the items p, p + nparts, ...)
// and leave as one row of partial sums per workgroup.
template <int K, int KIND> __device__ __forceinline__ void conv_bwd_walk(const ConvArgs &a, const Segment &sg, int c, bool act, int64_t first, ConvSums<K> &sum)
{
    const int lane = threadIdx.x & 63, cc = act ? c : 0;
    F4 w[K], bias;
    load_taps<K>(a, sg, c, act, w, bias);
    const int h = KIND == GATED ? cc / a.N : KIND == SKIP ? cc / a.P : 0;
    const bool four = a.N >= 16;
    const float dtb = KIND == GATED ? a.dt_bias[h] : 0.f, A = KIND == GATED ? -expf(a.A_log[h]) : 0.f;
    const float skip_scale = KIND == SKIP ? a.D[h] : 0.f;
    const bool heads_lane = KIND == GATED && act && cc % a.N < (four ? 16 : 4);   // the lanes that write what is one number per head and step

    for (int64_t item = first; item < a.items; item += (int64_t)a.nparts * CV_WAVES) {
        const int64_t b = item / a.tiles_t;
        const int t0 = (int)(item % a.tiles_t) * a.tile_t, t1 = min(a.T, t0 + a.tile_t);
        const int64_t row0 = b * a.T;
        const float *x = sg.x + row0 * sg.ld, *dy = sg.dy + row0 * sg.C, *skip = KIND == SKIP ? sg.skip + row0 * sg.C : nullptr;
        float *dx = sg.dx + row0 * sg.ld_dx;
        auto row = [&](int t) { return t < a.T ? t : a.T - 1; };
        F4 win[K], dwin[K];
#pragma unroll
        for (int j = 0; j < K; ++j) dwin[j] = F4_ZERO;
#pragma unroll
        for (int j = 0; j < K - 1; ++j) {
            const int t = t0 - (K - 1) + j;
            win[j + 1] = load4(x + (t < 0 ? 0 : t) * sg.ld + cc);
            if (t < 0) win[j + 1] = F4_ZERO;
        }
        F4 xn[CV_AHEAD], yn[CV_AHEAD], kn[KIND == SKIP ? CV_AHEAD : 1];
        float dtn = 0.f, dgn = 0.f;
        auto fetch = [&](int t) {
#pragma unroll
            for (int i = 0; i < CV_AHEAD; ++i) {
                const int64_t r = row(t + i);
                xn[i] = load4(x + r * sg.ld + cc);
                yn[i] = load4(dy + r * sg.C + cc);
                if constexpr (KIND == SKIP) kn[i] = load4(skip + r * sg.C + cc);
            }
            if (KIND == GATED && four) {
                const int64_t at = (row0 + row(t + (lane & 3))) * a.H + h;
                dtn = a.dt_in[at], dgn = a.dg[at];
            }
        };
        // Four steps; whole: all of them in the tile.
        auto steps = [&](int t, auto whole) {
            F4 xc[CV_AHEAD], yc[CV_AHEAD], kc[KIND == SKIP ? CV_AHEAD : 1];
#pragma unroll
            for (int i = 0; i < CV_AHEAD; ++i) {
                xc[i] = xn[i], yc[i] = yn[i];
                if constexpr (KIND == SKIP) kc[i] = kn[i];
                if (!decltype(whole)::value && t + i >= a.T) {   // rows past the sequence hold zeros
                    xc[i] = yc[i] = F4_ZERO;
                    if constexpr (KIND == SKIP) kc[i] = F4_ZERO;
                }
            }
            const float dt = dtn, dg = dgn;
            if (t + CV_AHEAD < t1 + K - 1) fetch(t + CV_AHEAD);
            float gate[CV_AHEAD], ddt[CV_AHEAD] = {0.f, 0.f, 0.f, 0.f};
            const float pre = dt + dtb, gate4 = KIND == GATED ? softplusf(pre) : 1.f;
            if (KIND == GATED) {
                if (four) {
                    gate[0] = of_lane<0>(gate4), gate[1] = of_lane<1>(gate4), gate[2] = of_lane<2>(gate4), gate[3] = of_lane<3>(gate4);
                } else {
#pragma unroll
                    for (int i = 0; i < CV_AHEAD; ++i) gate[i] = softplusf(a.dt_in[(row0 + row(t + i)) * a.H + h] + dtb);
                }
            }
#pragma unroll
            for (int i = 0; i < CV_AHEAD; ++i) {
                const int ti = t + i;
                const bool own = decltype(whole)::value || ti < t1;   // counts towards the parameters here; later steps count in their own tile
#pragma unroll
                for (int j = 0; j + 1 < K; ++j) win[j] = win[j + 1], dwin[j] = dwin[j + 1];
                win[K - 1] = xc[i];
                dwin[K - 1] = F4_ZERO;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float s = bias.v[e];
#pragma unroll
                    for (int j = 0; j < K; ++j) s += w[j].v[e] * win[j].v[e];
                    const float sg1 = sigmoidf(s), y = s * sg1;
                    float up = yc[i].v[e];   // gradient of y
                    if (KIND == GATED) up *= gate[i], ddt[i] += yc[i].v[e] * y;
                    if constexpr (KIND == SKIP) up += kc[i].v[e] * skip_scale;
                    const float ds = up * sg1 * (1.f + s * (1.f - sg1));
                    if (own) {
                        if constexpr (KIND == SKIP) sum.D += kc[i].v[e] * y;
                        sum.dbias.v[e] += ds;
#pragma unroll
                        for (int j = 0; j < K; ++j) sum.dw[j].v[e] += ds * win[j].v[e];
                    }
#pragma unroll
                    for (int j = 0; j < K; ++j) dwin[j].v[e] += w[j].v[e] * ds;
                }
                const int tx = ti - (K - 1);
                if (act && tx >= t0 && tx < t1) store4(dx + tx * sg.ld_dx + c, dwin[0]);
            }
            if (KIND != GATED) return;
            auto leaves = [&](int ti, float total, float pre_t, float gate_t, float dg_t) {   // a head's gradient at one step
                if (!heads_lane || ti >= t1) return;
                const float dpre = (total + dg_t * A) * (pre_t > 20.f ? 1.f : sigmoidf(pre_t));
                a.ddt_in[(row0 + ti) * a.H + h] = dpre;
                sum.dtb += dpre;
                sum.A += dg_t * gate_t * A;   // dg/dA_log = g
            };
            if (four) {   // lane l sees to step l & 3
                float total = sum_of_four(ddt, lane);
                for (int off = 4; off < a.N / 4; off <<= 1) total += __shfl_xor(total, off);
                leaves(t + (lane & 3), total, pre, gate4, dg);
            } else {
                for (int i = 0; i < CV_AHEAD; ++i) {
                    float total = i == 0 ? ddt[0] : i == 1 ? ddt[1] : i == 2 ? ddt[2] : ddt[3];
                    if (a.N == 8) total += __shfl_xor(total, 1);
                    const int64_t at = (row0 + row(t + i)) * a.H + h;
                    const float p = a.dt_in[at] + dtb;
                    leaves(t + i, total, p, softplusf(p), a.dg[at]);
                }
            }
        };
        fetch(t0);
        int t = t0;
        for (; t + CV_AHEAD <= t1; t += CV_AHEAD) steps(t, std::true_type{});
        for (; t < t1 + K - 1; t += CV_AHEAD) steps(t, std::false_type{});
    }
}

template <int K> __global__ void __launch_bounds__(CV_THREADS) conv_bwd_kernel(ConvArgs a)
{
    __shared__ F4 red[CV_WAVES][K + 1][64];
    __shared__ float red_h[CV_WAVES][3][64];
    int ntiles = 0;
    for (int s = 0; s < a.nseg; ++s) ntiles += a.tiles[s];
    int tile = (int)(blockIdx.x % (unsigned)ntiles);
    const int part = (int)(blockIdx.x / (unsigned)ntiles);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int si = segment_of(a, tile);
    const Segment &sg = a.seg[si];
    const int c = (tile * 64 + lane) * 4;
    const bool act = c < sg.C;
    ConvSums<K> sum{};
    const int64_t first = (int64_t)part * CV_WAVES + wv;
    if (sg.gated) conv_bwd_walk<K, GATED>(a, sg, c, act, first, sum);
    else if (sg.skip) conv_bwd_walk<K, SKIP>(a, sg, c, act, first, sum);
    else conv_bwd_walk<K, PLAIN>(a, sg, c, act, first, sum);
    // the workgroup's share of the parameters' gradients
#pragma unroll
    for (int j = 0; j < K; ++j) red[wv][j][lane] = sum.dw[j];
    red[wv][K][lane] = sum.dbias;
    red_h[wv][0][lane] = sum.dtb;
    red_h[wv][1][lane] = sum.A;
    red_h[wv][2][lane] = sum.D;
    __syncthreads();
    if (wv != 0 || !act) return;
    float *out = a.parts + (int64_t)part * a.columns;
#pragma unroll
    for (int j = 0; j <= K; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float s = 0.f;
            for (int u = 0; u < CV_WAVES; ++u) s += red[u][j][lane].v[e];
            const int ch = sg.w0 + c + e;
            out[j < K ? ch * K + j : a.C_total * K + ch] = s;
        }
    if (!a.dt_in) return;
    float s[3] = {0.f, 0.f, 0.f};
    float *out_h = out + a.C_total * (K + 1);
    if (sg.gated && c % a.N == 0) {
        const int lanes = a.N >= 16 ? 4 : 1;   // of a head that saw to steps
        for (int u = 0; u < CV_WAVES; ++u)
            for (int l = lane; l < lane + lanes; ++l)
                for (int m = 0; m < 2; ++m) s[m] += red_h[u][m][l];
        out_h[c / a.N] = s[0];
        out_h[a.H + c / a.N] = s[1];
    }
    for (int u = 0; u < CV_WAVES; ++u) s[2] += red_h[u][2][lane];
    if (si == 0) out_h[2 * a.H + c / 4] = s[2];
}

// Sum of g over a sequence from its last reset on (the step of the reset included), on top of the carried decay where
// there is none: decay_last = (no reset ? decay0 : 1) * exp(sum).  One wave per (b, h), lanes along time.
__global__ void __launch_bounds__(CV_THREADS) decay_last_kernel(const float *__restrict__ g, const void *__restrict__ done, int done_f32,
                                                                const float *__restrict__ decay0, float *__restrict__ out, int64_t BH, int T,
                                                                int H)
{
    const int64_t bh = (int64_t)blockIdx.x * CV_WAVES + (threadIdx.x >> 6);
    if (bh >= BH) return;
    const int lane = threadIdx.x & 63, h = (int)(bh % H);
    const int64_t row0 = bh / H * T;
    float sum = 0.f;
    bool reset = false;
    for (int hi = T; hi > 0 && !reset; hi -= 64) {   // from the end, until a reset is met
        const int t = hi - 1 - lane;
        const unsigned long long resets = __ballot(t >= 0 && done_at(done, done_f32, row0 + t));
        const int last = resets ? __builtin_ctzll(resets) : 63;   // lanes up to it lie behind the last reset
        if (t >= 0 && lane <= last) sum += g[(row0 + t) * H + h];
        reset = resets != 0;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    if (lane == 0) out[bh] = (reset ? 1.f : decay0[bh]) * expf(sum);
}

__device__ __forceinline__ float wave_sum(float x)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
    return x;
}

struct ReadoutArgs {
    const float *o, *hid, *z, *D, *scale, *dy;
    int64_t ld_z, ld_dz, rows;
    float *y, *d_o, *dz, *parts;
    int W, P;       // row width H * P
    float eps, inv_W;
};

// One wave per row of W <= 256 NV features: y = rms_norm(o + D hidden) * scale * silu(z).
template <int NV> __global__ void __launch_bounds__(CV_THREADS) readout_fwd_kernel(ReadoutArgs a)
{
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t)blockIdx.x * CV_WAVES + (threadIdx.x >> 6), nwaves = (int64_t)gridDim.x * CV_WAVES;
    F4 sc[NV];
    float D[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int col = (i * 64 + lane) * 4;
        sc[i] = col < a.W ? load4(a.scale + col) : F4_ZERO;
        D[i] = col < a.W ? a.D[col / a.P] : 0.f;
    }
    for (int64_t r = wave; r < a.rows; r += nwaves) {
        F4 y[NV], z[NV];
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int col = (i * 64 + lane) * 4;
            const bool in = col < a.W;
            const F4 o = in ? load4(a.o + r * a.W + col) : F4_ZERO, hd = in ? load4(a.hid + r * a.W + col) : F4_ZERO;
            z[i] = in ? load4(a.z + r * a.ld_z + col) : F4_ZERO;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                y[i].v[e] = o.v[e] + D[i] * hd.v[e];
                ss += y[i].v[e] * y[i].v[e];
            }
        }
        const float rstd = rsqrtf(wave_sum(ss) * a.inv_W + a.eps);
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int col = (i * 64 + lane) * 4;
            if (col >= a.W) continue;
            F4 out;
#pragma unroll
            for (int e = 0; e < 4; ++e) out.v[e] = y[i].v[e] * rstd * sc[i].v[e] * z[i].v[e] * sigmoidf(z[i].v[e]);
            store4(a.y + r * a.W + col, out);
        }
    }
}

// With s = o + D hidden, r = rsqrt(mean(s^2) + eps), n = s r scale: dn = dy silu(z), dz = dy n silu'(z),
// ds = r dn scale - s r^3 mean(dn scale s) (= do; hidden's share D ds is taken where hidden's gradient is, conv_bwd_kernel),
// dscale = sum of dn s r as per-workgroup partial sums.
template <int NV> __global__ void __launch_bounds__(CV_THREADS) readout_bwd_kernel(ReadoutArgs a)
{
    __shared__ F4 red[CV_WAVES][NV * 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t wave = (int64_t)blockIdx.x * CV_WAVES + wv, nwaves = (int64_t)gridDim.x * CV_WAVES;
    F4 sc[NV], ds[NV];
    float D[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int col = (i * 64 + lane) * 4;
        sc[i] = col < a.W ? load4(a.scale + col) : F4_ZERO;
        D[i] = col < a.W ? a.D[col / a.P] : 0.f;
        ds[i] = F4_ZERO;
    }
    for (int64_t r = wave; r < a.rows; r += nwaves) {
        F4 s[NV], z[NV], dy[NV], dn[NV];
        float ss = 0.f, dot = 0.f;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int col = (i * 64 + lane) * 4;
            const bool in = col < a.W;
            const F4 o = in ? load4(a.o + r * a.W + col) : F4_ZERO, hd = in ? load4(a.hid + r * a.W + col) : F4_ZERO;
            z[i] = in ? load4(a.z + r * a.ld_z + col) : F4_ZERO;
            dy[i] = in ? load4(a.dy + r * a.W + col) : F4_ZERO;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s[i].v[e] = o.v[e] + D[i] * hd.v[e];
                ss += s[i].v[e] * s[i].v[e];
                dn[i].v[e] = dy[i].v[e] * z[i].v[e] * sigmoidf(z[i].v[e]);
                dot += dn[i].v[e] * sc[i].v[e] * s[i].v[e];
            }
        }
        const float rstd = rsqrtf(wave_sum(ss) * a.inv_W + a.eps);
        const float cc = wave_sum(dot) * a.inv_W * rstd * rstd * rstd;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int col = (i * 64 + lane) * 4;
            if (col >= a.W) continue;
            F4 d_o, dz;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float zz = z[i].v[e], sg = sigmoidf(zz), n = s[i].v[e] * rstd;
                d_o.v[e] = dn[i].v[e] * sc[i].v[e] * rstd - s[i].v[e] * cc;
                dz.v[e] = dy[i].v[e] * n * sc[i].v[e] * sg * (1.f + zz * (1.f - sg));
                ds[i].v[e] += dn[i].v[e] * n;
            }
            store4(a.d_o + r * a.W + col, d_o);
            store4(a.dz + r * a.ld_dz + col, dz);
        }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) red[wv][i * 64 + lane] = ds[i];
    __syncthreads();
    for (int i = threadIdx.x; i < a.W / 4; i += CV_THREADS) {
        F4 t = F4_ZERO;
#pragma unroll
        for (int u = 0; u < CV_WAVES; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) t.v[e] += red[u][i].v[e];
        store4(a.parts + (int64_t)blockIdx.x * a.W + 4 * i, t);
    }
}

// Steps a wave walks: long tiles read few rows twice, short ones give enough waves where there is little to do.
// Measured on 256 x 128 x 1536 channels (f32): see the launch functions.
int tile_steps(int64_t B, int64_t T, int64_t tiles)
{
    int t = 32;
    while (t > 8 && B * ((T + t - 1) / t) * tiles < 4096) t >>= 1;
    return t;
}

bool sizes_ok(std::initializer_list<int64_t> positive)
{
    for (const int64_t n : positive)
        if (n <= 0 || n >= (1ll << 30)) return false;
    return true;
}
bool pointers_ok(std::initializer_list<const void *> ps)
{
    for (const void *p : ps)
        if (!p || !aligned(p, 16)) return false;
    return true;
}

template <template <int> class F, typename... A> int by_width(int64_t K, A &&...args)
{
    switch (K) {
    case 1: return F<1>::go(args...);
    case 2: return F<2>::go(args...);
    case 3: return F<3>::go(args...);
    case 4: return F<4>::go(args...);
    default: return MRX_ERR_UNSUPPORTED;
    }
}
template <int K> struct ConvFwd {
    static int go(hipStream_t st, unsigned grid, const ConvArgs &a) { return launch_kernel(conv_fwd_kernel<K>, dim3(grid), dim3(CV_THREADS), 0, st, a); }
};
template <int K> struct ConvBwd {
    static int go(hipStream_t st, unsigned grid, const ConvArgs &a) { return launch_kernel(conv_bwd_kernel<K>, dim3(grid), dim3(CV_THREADS), 0, st, a); }
};

int finish_args(ConvArgs &a, int64_t B)
{
    int tiles = 0;
    for (int s = 0; s < a.nseg; ++s) tiles += a.tiles[s] = (a.seg[s].C + 255) / 256;
    a.tile_t = tile_steps(B, a.T, tiles);
    a.tiles_t = (a.T + a.tile_t - 1) / a.tile_t;
    a.items = B * a.tiles_t;
    return tiles;
}
int run_fwd(hipStream_t st, ConvArgs &a, int64_t B, int64_t K)
{
    const int tiles = finish_args(a, B);
    const int64_t grid = (a.items + CV_WAVES - 1) / CV_WAVES * tiles;
    if (grid >= (1ll << 31)) return MRX_ERR_INVALID_ARG;
    return by_width<ConvFwd>(K, st, (unsigned)grid, a);
}
int run_bwd(hipStream_t st, ConvArgs &a, int64_t B, int64_t K, float *param_grads)
{
    const int tiles = finish_args(a, B);
    const int64_t wgs = (a.items + CV_WAVES - 1) / CV_WAVES;
    a.nparts = (int)(wgs < MRX_CONV_PARTS ? wgs : MRX_CONV_PARTS);
    if (const int rc = by_width<ConvBwd>(K, st, (unsigned)(a.nparts * tiles), a); rc != MRX_OK) return rc;
    return launch_column_sum(st, a.parts, param_grads, nullptr, a.nparts, a.columns);
}

int mamba_args(ConvArgs &a, int64_t B, int64_t T, int64_t H, int64_t P, int64_t N, int64_t K, int64_t ld_up)
{
    if (!sizes_ok({B, T, H, P, N, K, H * P, H * N, ld_up})) return MRX_ERR_INVALID_ARG;
    // four channels per lane inside one head; the lanes of a head's N features are summed by shuffles
    if (P % 4 != 0 || N % 4 != 0 || N > 256 || (N & (N - 1)) != 0 || K > CV_MAX_K) return MRX_ERR_UNSUPPORTED;
    if (ld_up % 4 != 0 || ld_up < H * P) return MRX_ERR_INVALID_ARG;
    a.nseg = 3;
    a.T = (int)T, a.H = (int)H, a.P = (int)P, a.N = (int)N;
    a.C_total = (int)(H * P + 2 * H * N);
    a.columns = (int)(a.C_total * (K + 1) + 2 * H + H * P / 4);
    const int C[3] = {(int)(H * P), (int)(H * N), (int)(H * N)};
    for (int s = 0, w0 = 0; s < 3; w0 += C[s++]) a.seg[s].C = C[s], a.seg[s].w0 = w0, a.seg[s].ld = s ? C[s] : ld_up, a.seg[s].gated = s == 1;
    return MRX_OK;
}

template <int NV> int launch_readout(hipStream_t st, const ReadoutArgs &a, unsigned grid, bool bwd)
{
    return bwd ? launch_kernel(readout_bwd_kernel<NV>, dim3(grid), dim3(CV_THREADS), 0, st, a)
               : launch_kernel(readout_fwd_kernel<NV>, dim3(grid), dim3(CV_THREADS), 0, st, a);
}
int run_readout(hipStream_t st, ReadoutArgs &a, int64_t rows, int64_t H, int64_t P, float eps, bool bwd, float *dscale)
{
    if (!sizes_ok({H, P, H * P}) || rows <= 0) return MRX_ERR_INVALID_ARG;
    if (P % 4 != 0 || H * P > 2048) return MRX_ERR_UNSUPPORTED;
    if (a.ld_z % 4 != 0 || a.ld_z < H * P || (bwd && (a.ld_dz % 4 != 0 || a.ld_dz < H * P))) return MRX_ERR_INVALID_ARG;
    a.rows = rows, a.W = (int)(H * P), a.P = (int)P, a.eps = eps, a.inv_W = 1.f / (float)a.W;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    const int64_t wgs = (rows + CV_WAVES - 1) / CV_WAVES;
    const unsigned grid = (unsigned)(wgs < (bwd ? MRX_RMS_NORM_PARTS : 4096) ? wgs : (bwd ? MRX_RMS_NORM_PARTS : 4096));
    const int rc = a.W <= 256    ? launch_readout<1>(st, a, grid, bwd)
                   : a.W <= 512  ? launch_readout<2>(st, a, grid, bwd)
                   : a.W <= 1024 ? launch_readout<4>(st, a, grid, bwd)
                                 : launch_readout<8>(st, a, grid, bwd);
    if (rc != MRX_OK || !bwd) return rc;
    return launch_column_sum(st, a.parts, dscale, nullptr, (int)grid, a.W);
}

}  // namespace
}  // namespace mrx

extern "C" int mrx_causal_conv_silu_fwd(void *stream, const float *x, int64_t ld_x, const float *w, const float *bias, float *y, int64_t B,
                                        int64_t T, int64_t C, int64_t K)
{
    using namespace mrx;
    if (!sizes_ok({B, T, C, K, ld_x}) || !pointers_ok({x, bias, y}) || !w || ld_x % 4 != 0 || ld_x < C) return MRX_ERR_INVALID_ARG;
    if (C % 4 != 0 || K > CV_MAX_K) return MRX_ERR_UNSUPPORTED;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    ConvArgs a{};
    a.nseg = 1, a.T = (int)T, a.C_total = (int)C, a.w = w, a.bias = bias;
    a.seg[0].x = x, a.seg[0].ld = ld_x, a.seg[0].y = y, a.seg[0].C = (int)C;
    return run_fwd(static_cast<hipStream_t>(stream), a, B, K);
}

extern "C" int mrx_causal_conv_silu_bwd(void *stream, const float *x, int64_t ld_x, const float *w, const float *bias, const float *dy,
                                        float *dx, int64_t ld_dx, float *param_grads, float *workspace, int64_t B, int64_t T, int64_t C,
                                        int64_t K)
{
    using namespace mrx;
    if (!sizes_ok({B, T, C, K, ld_x, ld_dx}) || !pointers_ok({x, bias, dy, dx, param_grads, workspace}) || !w) return MRX_ERR_INVALID_ARG;
    if (ld_x % 4 != 0 || ld_x < C || ld_dx % 4 != 0 || ld_dx < C) return MRX_ERR_INVALID_ARG;
    if (C % 4 != 0 || K > CV_MAX_K) return MRX_ERR_UNSUPPORTED;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    ConvArgs a{};
    a.nseg = 1, a.T = (int)T, a.C_total = (int)C, a.w = w, a.bias = bias, a.parts = workspace, a.columns = (int)(C * (K + 1));
    a.seg[0].x = x, a.seg[0].ld = ld_x, a.seg[0].dy = dy, a.seg[0].dx = dx, a.seg[0].ld_dx = ld_dx, a.seg[0].C = (int)C;
    return run_bwd(static_cast<hipStream_t>(stream), a, B, K, param_grads);
}

extern "C" int mrx_mamba_elements_fwd(void *stream, const float *up, int64_t ld_up, const float *b_in, const float *c_in, const float *dt_in,
                                      const float *conv_w, const float *conv_b, const float *dt_bias, const float *A_log, float *v, float *k,
                                      float *q, float *g, int64_t B, int64_t T, int64_t H, int64_t P, int64_t N, int64_t K)
{
    using namespace mrx;
    ConvArgs a{};
    if (const int rc = mamba_args(a, B, T, H, P, N, K, ld_up); rc != MRX_OK) return rc;
    if (!pointers_ok({up, b_in, c_in, conv_b, v, k, q}) || !dt_in || !conv_w || !dt_bias || !A_log || !g) return MRX_ERR_INVALID_ARG;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    const float *x[3] = {up, b_in, c_in};
    float *y[3] = {v, k, q};
    for (int s = 0; s < 3; ++s) a.seg[s].x = x[s], a.seg[s].y = y[s];
    a.w = conv_w, a.bias = conv_b, a.dt_in = dt_in, a.dt_bias = dt_bias, a.A_log = A_log, a.g = g;
    return run_fwd(static_cast<hipStream_t>(stream), a, B, K);
}

extern "C" int mrx_mamba_elements_bwd(void *stream, const float *up, int64_t ld_up, const float *b_in, const float *c_in, const float *dt_in,
                                      const float *conv_w, const float *conv_b, const float *dt_bias, const float *A_log, const float *D,
                                      const float *dv, const float *dk, const float *dq, const float *dg, const float *d_o, float *d_up,
                                      int64_t ld_dup, float *db_in, float *dc_in, float *ddt_in, float *param_grads, float *workspace, int64_t B,
                                      int64_t T, int64_t H, int64_t P, int64_t N, int64_t K)
{
    using namespace mrx;
    ConvArgs a{};
    if (const int rc = mamba_args(a, B, T, H, P, N, K, ld_up); rc != MRX_OK) return rc;
    if (!pointers_ok({up, b_in, c_in, conv_b, dv, dk, dq, d_o, d_up, db_in, dc_in, param_grads, workspace}) || !dt_in || !conv_w || !dt_bias ||
        !A_log || !D || !dg || !ddt_in)
        return MRX_ERR_INVALID_ARG;
    if (ld_dup % 4 != 0 || ld_dup < H * P) return MRX_ERR_INVALID_ARG;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    const float *x[3] = {up, b_in, c_in}, *dy[3] = {dv, dk, dq};
    float *dx[3] = {d_up, db_in, dc_in};
    for (int s = 0; s < 3; ++s) a.seg[s].x = x[s], a.seg[s].dy = dy[s], a.seg[s].dx = dx[s], a.seg[s].ld_dx = s ? a.seg[s].C : ld_dup;
    a.seg[0].skip = d_o;
    a.w = conv_w, a.bias = conv_b, a.dt_in = dt_in, a.dt_bias = dt_bias, a.A_log = A_log, a.D = D, a.dg = dg, a.ddt_in = ddt_in;
    a.parts = workspace;
    return run_bwd(static_cast<hipStream_t>(stream), a, B, K, param_grads);
}

extern "C" int mrx_decay_last(void *stream, const float *g, const void *done, const float *decay0, float *decay_last, int64_t B, int64_t T,
                              int64_t H, int done_dtype)
{
    using namespace mrx;
    if (!g || !done || !decay0 || !decay_last || !sizes_ok({B, T, H})) return MRX_ERR_INVALID_ARG;
    if (done_dtype != MRX_DONE_U8 && done_dtype != MRX_DONE_F32) return MRX_ERR_INVALID_ARG;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    return launch_kernel(decay_last_kernel, dim3((unsigned)((B * H + CV_WAVES - 1) / CV_WAVES)), dim3(CV_THREADS), 0,
                         static_cast<hipStream_t>(stream), g, done, int(done_dtype == MRX_DONE_F32), decay0, decay_last, B * H, (int)T, (int)H);
}

extern "C" int mrx_mamba_readout_fwd(void *stream, const float *o, const float *hidden, const float *z, int64_t ld_z, const float *D,
                                     const float *scale, float *y, int64_t rows, int64_t H, int64_t P, float eps)
{
    using namespace mrx;
    if (!pointers_ok({o, hidden, z, scale, y}) || !D) return MRX_ERR_INVALID_ARG;
    ReadoutArgs a{};
    a.o = o, a.hid = hidden, a.z = z, a.ld_z = ld_z, a.D = D, a.scale = scale, a.y = y;
    return run_readout(static_cast<hipStream_t>(stream), a, rows, H, P, eps, false, nullptr);
}

extern "C" int mrx_mamba_readout_bwd(void *stream, const float *o, const float *hidden, const float *z, int64_t ld_z, const float *D,
                                     const float *scale, const float *dy, float *d_o, float *dz, int64_t ld_dz, float *dscale,
                                     float *workspace, int64_t rows, int64_t H, int64_t P, float eps)
{
    using namespace mrx;
    if (!pointers_ok({o, hidden, z, scale, dy, d_o, dz, dscale, workspace}) || !D) return MRX_ERR_INVALID_ARG;
    ReadoutArgs a{};
    a.o = o, a.hid = hidden, a.z = z, a.ld_z = ld_z, a.D = D, a.scale = scale, a.dy = dy, a.d_o = d_o, a.dz = dz, a.ld_dz = ld_dz;
    a.parts = workspace;
    return run_readout(static_cast<hipStream_t>(stream), a, rows, H, P, eps, true, dscale);
}
