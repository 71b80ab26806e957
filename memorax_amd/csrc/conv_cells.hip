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
// All are bound by HBM.  Layout: a wave is 64 lanes x 4 consecutive channels of one time tile and walks its steps with the
// last K inputs in registers, so a row of an array is read once per tile (plus K - 1 rows that the neighbouring tile of the
// same workgroup has just brought in), four rows requested ahead of their use.
#include <initializer_list>

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
__device__ __forceinline__ float sigmoidf(float x) { return 1.f / (1.f + expf(-x)); }
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

template <int K> __global__ void __launch_bounds__(CV_THREADS) conv_fwd_kernel(ConvArgs a)
{
    int ntiles = 0;
    for (int s = 0; s < a.nseg; ++s) ntiles += a.tiles[s];
    int tile = (int)(blockIdx.x % (unsigned)ntiles);
    const int64_t item = (int64_t)(blockIdx.x / (unsigned)ntiles) * CV_WAVES + (threadIdx.x >> 6);
    if (item >= a.items) return;
    const bool first = tile == 0;
    const int lane = threadIdx.x & 63;
    const Segment &sg = a.seg[segment_of(a, tile)];
    const int c = (tile * 64 + lane) * 4;
    const bool act = c < sg.C;
    const int64_t b = item / a.tiles_t;
    const int t0 = (int)(item % a.tiles_t) * a.tile_t, t1 = min(a.T, t0 + a.tile_t);
    const int64_t row0 = b * a.T;

    if (first && a.g) {   // the log-decay, beside the first tile's work
        const int n = (t1 - t0) * a.H;
        for (int i = lane; i < n; i += 64) {
            const int h = i % a.H;
            const int64_t at = (row0 + t0) * a.H + i;
            a.g[at] = softplusf(a.dt_in[at] + a.dt_bias[h]) * -expf(a.A_log[h]);
        }
    }
    F4 w[K], bias, win[K];
    load_taps<K>(a, sg, c, act, w, bias);
    const float *x = sg.x + row0 * sg.ld + c;
    float *y = sg.y + row0 * sg.C + c;
    const int h = sg.gated && act ? c / a.N : 0;
    const float dtb = sg.gated ? a.dt_bias[h] : 0.f;
#pragma unroll
    for (int j = 0; j < K - 1; ++j) {
        const int t = t0 - (K - 1) + j;
        win[j + 1] = act && t >= 0 ? load4(x + t * sg.ld) : F4_ZERO;
    }
    F4 next[CV_AHEAD];
    float dt_next[CV_AHEAD];
    auto fetch = [&](int t) {
#pragma unroll
        for (int i = 0; i < CV_AHEAD; ++i) {
            const bool in = act && t + i < t1;
            next[i] = in ? load4(x + (t + i) * sg.ld) : F4_ZERO;
            dt_next[i] = in && sg.gated ? a.dt_in[(row0 + t + i) * a.H + h] : 0.f;
        }
    };
    fetch(t0);
    for (int t = t0; t < t1; t += CV_AHEAD) {
        F4 cur[CV_AHEAD];
        float dt[CV_AHEAD];
#pragma unroll
        for (int i = 0; i < CV_AHEAD; ++i) cur[i] = next[i], dt[i] = dt_next[i];
        fetch(t + CV_AHEAD);
#pragma unroll
        for (int i = 0; i < CV_AHEAD; ++i) {
#pragma unroll
            for (int j = 0; j + 1 < K; ++j) win[j] = win[j + 1];
            win[K - 1] = cur[i];
            const float gate = sg.gated ? softplusf(dt[i] + dtb) : 1.f;
            F4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float s = bias.v[e];
#pragma unroll
                for (int j = 0; j < K; ++j) s += w[j].v[e] * win[j].v[e];
                o.v[e] = s * sigmoidf(s) * gate;
            }
            if (act && t + i < t1) store4(y + (int64_t)(t + i) * sg.C, o);
        }
    }
}

// Backward: the pre-activations are formed again from the inputs; a step's gradient ds_t = dy_t silu'(s_t) reaches the inputs
// t-K+1 .. t, so dx_{t-K+1} is complete once ds_t is known, and a tile walks K - 1 steps past its end for its last rows.
// The parameters' gradients stay in registers over all tiles of a wave (workgroup column p takes the items p, p + nparts, ...)
// and leave as one row of partial sums per workgroup.
template <int K> __global__ void __launch_bounds__(CV_THREADS) conv_bwd_kernel(ConvArgs a)
{
    __shared__ F4 red[CV_WAVES][K + 1][64];
    __shared__ float red_h[CV_WAVES][3][64];
    int ntiles = 0;
    for (int s = 0; s < a.nseg; ++s) ntiles += a.tiles[s];
    int tile = (int)(blockIdx.x % (unsigned)ntiles);
    const int part = (int)(blockIdx.x / (unsigned)ntiles);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int si = segment_of(a, tile);
    const Segment &sg = a.seg[si];
    const int c = (tile * 64 + lane) * 4;
    const bool act = c < sg.C;
    F4 w[K], bias, dw[K], dbias = F4_ZERO;
    load_taps<K>(a, sg, c, act, w, bias);
#pragma unroll
    for (int j = 0; j < K; ++j) dw[j] = F4_ZERO;
    const int h = act ? (sg.gated ? c / a.N : sg.skip ? c / a.P : 0) : 0;
    const float dtb = sg.gated ? a.dt_bias[h] : 0.f, A = sg.gated ? -expf(a.A_log[h]) : 0.f;
    const float skip_scale = sg.skip ? a.D[h] : 0.f;
    float acc_dtb = 0.f, acc_A = 0.f, acc_D = 0.f;

    for (int64_t item = (int64_t)part * CV_WAVES + wv; item < a.items; item += (int64_t)a.nparts * CV_WAVES) {
        const int64_t b = item / a.tiles_t;
        const int t0 = (int)(item % a.tiles_t) * a.tile_t, t1 = min(a.T, t0 + a.tile_t);
        const int t2 = min(a.T, t1 + K - 1);   // steps whose ds reaches a row of this tile
        const int64_t row0 = b * a.T;
        const float *x = sg.x + row0 * sg.ld + c, *dy = sg.dy + row0 * sg.C + c;
        const float *skip = sg.skip ? sg.skip + row0 * sg.C + c : nullptr;
        float *dx = sg.dx + row0 * sg.ld_dx + c;
        F4 win[K], dwin[K];
#pragma unroll
        for (int j = 0; j < K; ++j) dwin[j] = F4_ZERO;
#pragma unroll
        for (int j = 0; j < K - 1; ++j) {
            const int t = t0 - (K - 1) + j;
            win[j + 1] = act && t >= 0 ? load4(x + t * sg.ld) : F4_ZERO;
        }
        F4 xn[CV_AHEAD], yn[CV_AHEAD], kn[CV_AHEAD];
        float dtn[CV_AHEAD], dgn[CV_AHEAD];
        auto fetch = [&](int t) {
#pragma unroll
            for (int i = 0; i < CV_AHEAD; ++i) {
                const bool in = act && t + i < t2;
                xn[i] = in ? load4(x + (t + i) * sg.ld) : F4_ZERO;
                yn[i] = in ? load4(dy + (int64_t)(t + i) * sg.C) : F4_ZERO;
                kn[i] = in && skip ? load4(skip + (int64_t)(t + i) * sg.C) : F4_ZERO;
                const int64_t at = (row0 + t + i) * a.H + h;
                dtn[i] = in && sg.gated ? a.dt_in[at] : 0.f;
                dgn[i] = in && sg.gated ? a.dg[at] : 0.f;
            }
        };
        fetch(t0);
        for (int t = t0; t < t1 + K - 1; t += CV_AHEAD) {
            F4 xc[CV_AHEAD], yc[CV_AHEAD], kc[CV_AHEAD];
            float dtc[CV_AHEAD], dgc[CV_AHEAD];
#pragma unroll
            for (int i = 0; i < CV_AHEAD; ++i) xc[i] = xn[i], yc[i] = yn[i], kc[i] = kn[i], dtc[i] = dtn[i], dgc[i] = dgn[i];
            fetch(t + CV_AHEAD);
#pragma unroll
            for (int i = 0; i < CV_AHEAD; ++i) {
                const int ti = t + i;
                const bool own = ti < t1;   // counts towards the parameters here; later steps count in their own tile
#pragma unroll
                for (int j = 0; j + 1 < K; ++j) win[j] = win[j + 1], dwin[j] = dwin[j + 1];
                win[K - 1] = xc[i];
                dwin[K - 1] = F4_ZERO;
                const float pre = dtc[i] + dtb, gate = sg.gated ? softplusf(pre) : 1.f;
                float ddt = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float s = bias.v[e];
#pragma unroll
                    for (int j = 0; j < K; ++j) s += w[j].v[e] * win[j].v[e];
                    const float sg1 = sigmoidf(s), y = s * sg1;
                    const float up = yc[i].v[e] * gate + kc[i].v[e] * skip_scale;   // gradient of y (rows past the sequence hold zeros)
                    const float ds = up * sg1 * (1.f + s * (1.f - sg1));
                    ddt += yc[i].v[e] * y;
                    if (own) {
                        acc_D += kc[i].v[e] * y;
                        dbias.v[e] += ds;
#pragma unroll
                        for (int j = 0; j < K; ++j) dw[j].v[e] += ds * win[j].v[e];
                    }
#pragma unroll
                    for (int j = 0; j < K; ++j) dwin[j].v[e] += w[j].v[e] * ds;
                }
                if (sg.gated) {   // one head = N / 4 neighbouring lanes
                    for (int off = a.N / 8; off > 0; off >>= 1) ddt += __shfl_xor(ddt, off);
                    const float dpre = (ddt + dgc[i] * A) * (pre > 20.f ? 1.f : sigmoidf(pre));
                    if (own && act && (c % a.N) == 0) {
                        a.ddt_in[(row0 + ti) * a.H + h] = dpre;
                        acc_dtb += dpre;
                        acc_A += dgc[i] * gate * A;   // dg/dA_log = g
                    }
                }
                const int tx = ti - (K - 1);
                if (act && tx >= t0 && tx < t1) store4(dx + tx * sg.ld_dx, dwin[0]);
            }
        }
    }
    // the workgroup's share of the parameters' gradients
#pragma unroll
    for (int j = 0; j < K; ++j) red[wv][j][lane] = dw[j];
    red[wv][K][lane] = dbias;
    red_h[wv][0][lane] = acc_dtb;
    red_h[wv][1][lane] = acc_A;
    red_h[wv][2][lane] = acc_D;
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
    for (int u = 0; u < CV_WAVES; ++u)
        for (int m = 0; m < 3; ++m) s[m] += red_h[u][m][lane];
    float *out_h = out + a.C_total * (K + 1);
    if (sg.gated && (c % a.N) == 0) {
        out_h[h] = s[0];
        out_h[a.H + h] = s[1];
    }
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
