// One acting step (one time step per environment, no gradients) of the cells whose step is more than a recurrence: what lies
// between the dense layers of a block (row_dense.hip) as one kernel.  All float32.
//
// As array-library operations on a few kilobytes to a few megabytes, an LRU step was seventeen launches and an mLSTM step
// forty-eight; a step of an agent is bound by their number, on the host as on the device.
#include <math.h>

#include <type_traits>

#include "common.h"

namespace mrx {
namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ---- LRU: lambda = exp(-exp(nu) + i exp(theta)), h' = (done ? 0 : lambda h) + exp(gamma) (u_re + i u_im), P' = (done ? 1 : P) lambda.
// The state leaves once as the carry and once as the row [Re h' | -Im h'] that the read-out multiplies with [C_re | C_im].
struct LruArgs {
    const float *u_re, *u_im, *nu, *theta, *gamma;
    const f32x2 *h, *P;
    const void *done;
    f32x2 *h_out, *P_out;
    float *row;
    int64_t count;
    int N, done_f32;
};
__global__ void __launch_bounds__(256) lru_step_kernel(LruArgs a)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= a.count) return;
    const int64_t b = i / a.N;
    const int n = (int)(i % a.N);
    const bool reset = done_at(a.done, a.done_f32, b);
    const f32x2 h = a.h[i], P = a.P[i];
    const float radius = expf(-expf(a.nu[n])), angle = expf(a.theta[n]), scale = expf(a.gamma[n]);
    float s, c;
    sincosf(angle, &s, &c);
    const float lr = radius * c, li = radius * s;
    f32x2 hn = {a.u_re[i] * scale, a.u_im[i] * scale}, Pn = {lr, li};
    if (!reset) {
        hn[0] += lr * h[0] - li * h[1];
        hn[1] += lr * h[1] + li * h[0];
        Pn = f32x2{lr * P[0] - li * P[1], lr * P[1] + li * P[0]};
    }
    a.h_out[i] = hn;
    a.P_out[i] = Pn;
    a.row[b * 2 * a.N + n] = hn[0];
    a.row[b * 2 * a.N + a.N + n] = -hn[1];
}

// ---- mLSTM: a workgroup per environment.  The matrix state is what the step moves (16 KB in and out per head of 64): its loads
// are issued first and wait in registers while the projections, the gates and the normaliser are formed from a few hundred
// values in LDS.
struct MlstmStepArgs {
    const float *up, *conv_w, *conv_b, *wq, *wk, *wv, *wi, *bi, *wf, *bf, *norm_w, *skip;
    const float *C, *lf, *n, *m;
    const void *done;
    float *C_out, *lf_out, *n_out, *m_out, *y;
    int conv_k, H, done_f32;
    float g_floor;
};
__device__ __forceinline__ float silu(float x) { return x / (1.f + expf(-x)); }
// Sum over groups of 4, 8 or 16 lanes, in every one of them: DPP moves.
template <int LANES> __device__ __forceinline__ float lanes_total(float x)
{
    auto add = [&](auto ctrl) {
        const int moved = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, true);
        x += __builtin_bit_cast(float, moved);
    };
    add(std::integral_constant<int, 0xB1>{});    // quad_perm [1,0,3,2]
    add(std::integral_constant<int, 0x4E>{});    // quad_perm [2,3,0,1]
    if constexpr (LANES >= 8) add(std::integral_constant<int, 0x141>{});    // row_half_mirror
    if constexpr (LANES >= 16) add(std::integral_constant<int, 0x140>{});   // row_mirror
    return x;
}
template <int D> __device__ __forceinline__ float head_total(float x)   // over the D lanes that hold a head's values
{
#pragma unroll
    for (int off = 1; off < D; off <<= 1) x += __shfl_xor(x, off);
    return x;
}

constexpr int MS_HEADS = 8, MS_WIDTH = 256;
template <int D> __global__ void __launch_bounds__(256) mlstm_step_kernel(MlstmStepArgs a)
{
    constexpr int HEAD4 = D * D / 4, MAXP = MS_WIDTH * D / 1024 > MS_HEADS * HEAD4 / 256 ? MS_HEADS * HEAD4 / 256 : MS_WIDTH * D / 1024;
    __shared__ __align__(16) float su[MS_WIDTH], sx[MS_WIDTH], sq[MS_WIDTH], sk[MS_WIDTH], sv[MS_WIDTH], red[4][MS_WIDTH];
    __shared__ float gates[4][2 * MS_HEADS], decay[MS_HEADS], weight[MS_HEADS], floor_m[MS_HEADS];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, H = a.H, W = H * D;
    const int64_t b = blockIdx.x;
    const bool reset = done_at(a.done, a.done_f32, b);
    const f32x4 *C = reinterpret_cast<const f32x4 *>(a.C) + b * (H * HEAD4);
    f32x4 *C_out = reinterpret_cast<f32x4 *>(a.C_out) + b * (H * HEAD4);
    f32x4 state[MAXP];
#pragma unroll
    for (int p = 0; p < MAXP; ++p) {
        state[p] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (!reset && p * 256 + t < H * HEAD4) state[p] = C[p * 256 + t];
    }
    const int h = t / D, o = t % D;
    const bool own = t < W;   // this thread's channel
    float z = 0.f, n_prev = 0.f, u = 0.f;
    if (own) {
        const float x = a.up[b * 2 * W + t];
        z = a.up[b * 2 * W + W + t];
        n_prev = a.n[b * W + t];
        u = silu(a.conv_w[t * a.conv_k + a.conv_k - 1] * x + a.conv_b[t]);   // one step: the convolution sees no other
        sx[t] = x;
        su[t] = u;
    }
    __syncthreads();
    // the block-diagonal maps: D / 4 lanes read a row together and sum over themselves (a row per lane touches a cache line per
    // lane and load: 877 environments with four heads of 64 65 -> 32 us, where the state's way in and out is 19)
    {
        constexpr int LPR = D / 4, RPI = 64 / LPR;
        const int j = lane % LPR;
#pragma unroll
        for (int p = 0; p < LPR; ++p) {
            const int r = w * 64 + p * RPI + lane / LPR, at = r / D * D + 4 * j;
            if (w * 64 + p * RPI >= W) break;   // W is a multiple of the rows of an instruction
            const f32x4 uj = *reinterpret_cast<const f32x4 *>(su + at), xj = *reinterpret_cast<const f32x4 *>(sx + at);
            const f32x4 a0 = reinterpret_cast<const f32x4 *>(a.wq)[r * LPR + j], a1 = reinterpret_cast<const f32x4 *>(a.wk)[r * LPR + j],
                        a2 = reinterpret_cast<const f32x4 *>(a.wv)[r * LPR + j];
            float q = 0.f, k = 0.f, v = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) q += a0[e] * uj[e], k += a1[e] * uj[e], v += a2[e] * xj[e];
            q = lanes_total<LPR>(q), k = lanes_total<LPR>(k), v = lanes_total<LPR>(v);
            if (j == 0) sq[r] = q, sk[r] = k, sv[r] = v;
        }
    }
    __syncthreads();
    float q = 0.f, k = 0.f, v = 0.f;
    if (own) q = sq[t], k = sk[t], v = sv[t];
    // the gates of every head read all of (q | k | v), head by head
    for (int g = 0; g < 2 * H; ++g) {
        const float *row = (g < H ? a.wi + (int64_t)g * 3 * W : a.wf + (int64_t)(g - H) * 3 * W) + h * 3 * D + o;
        float s = own ? row[0] * q + row[D] * k + row[2 * D] * v : 0.f;
        s = head_total<64>(s);
        if (lane == 0) gates[w][g] = s;
    }
    __syncthreads();
    if (t < H) {
        const float li = gates[0][t] + gates[1][t] + gates[2][t] + gates[3][t] + a.bi[t];
        const float f = gates[0][H + t] + gates[1][H + t] + gates[2][H + t] + gates[3][H + t] + a.bf[t];
        const float lf = fminf(f, 0.f) - log1pf(expf(-fabsf(f)));
        const float mp = a.m[b * H + t], m = reset ? li : fmaxf(mp + lf, li);
        decay[t] = expf(fminf(fmaxf(lf + mp - m, a.g_floor), 0.f));   // not used at a reset
        weight[t] = expf(li - m) * (1.f / sqrtf((float)D));
        floor_m[t] = expf(-m);
        a.m_out[b * H + t] = m;
        a.lf_out[b * H + t] = reset ? lf : a.lf[b * H + t] + lf;
    }
    __syncthreads();
    float den = 1.f;
    {
        float n = 0.f;
        if (own) {
            k *= weight[h];
            n = reset ? k : decay[h] * n_prev + k;
            a.n_out[b * W + t] = n;
            sk[t] = k;
        }
        const float qn = head_total<D>(own ? q * n : 0.f);
        if (own) den = fmaxf(fabsf(qn), floor_m[h]) + 1e-6f;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) red[r][t] = 0.f;
    __syncthreads();
    f32x4 part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < MAXP; ++p) {
        const int idx = p * 256 + t;
        constexpr int PER_HEAD = HEAD4 >= 256 ? HEAD4 / 256 : 1;   // consecutive p of one head
        if (p * 256 < H * HEAD4 && idx < H * HEAD4) {
            const int hh = idx / HEAD4, i = idx % HEAD4 / (D / 4), j4 = idx % (D / 4);
            const f32x4 vj = *reinterpret_cast<const f32x4 *>(sv + hh * D + 4 * j4);
            const float ki = sk[hh * D + i], qi = sq[hh * D + i];
            f32x4 s;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s[e] = reset ? ki * vj[e] : decay[hh] * state[p][e] + ki * vj[e];
                part[e] += qi * s[e];
            }
            C_out[idx] = s;
            if (p % PER_HEAD == PER_HEAD - 1) {   // the rows of this head that the wave holds: over the lanes of one column
#pragma unroll
                for (int e = 0; e < 4; ++e) {
#pragma unroll
                    for (int off = D / 4; off < 64; off <<= 1) part[e] += __shfl_xor(part[e], off);
                }
                if (lane < D / 4) *reinterpret_cast<f32x4 *>(&red[w][hh * D + 4 * j4]) = part;
                part = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
    }
    __syncthreads();
    float y = own ? (red[0][t] + red[1][t] + red[2][t] + red[3][t]) / den : 0.f;
    const float mean = head_total<D>(y) * (1.f / D);
    const float c = y - mean, var = head_total<D>(c * c) * (1.f / D);
    if (own) {
        y = c * rsqrtf(var + 1e-5f) * (1.f + a.norm_w[t]) + a.skip[t] * u;
        a.y[b * W + t] = y * silu(z);
    }
}

}  // namespace
}  // namespace mrx

extern "C" int mrx_lru_step(void *stream, const float *u_re, const float *u_im, const float *nu_log, const float *theta_log,
                            const float *gamma_log, const void *done, const void *h, const void *P, void *h_out, void *P_out, float *row,
                            int64_t B, int64_t N, int done_dtype)
{
    using namespace mrx;
    if (!u_re || !u_im || !nu_log || !theta_log || !gamma_log || !done || !h || !P || !h_out || !P_out || !row || B <= 0 || N <= 0)
        return MRX_ERR_INVALID_ARG;
    if (done_dtype != MRX_DONE_U8 && done_dtype != MRX_DONE_F32) return MRX_ERR_INVALID_ARG;
    if (N >= (1ll << 30) || B >= (1ll << 31) || B * N >= (1ll << 38)) return MRX_ERR_INVALID_ARG;
    for (const void *p : {h, P, (const void *)h_out, (const void *)P_out})
        if (!aligned(p, 8)) return MRX_ERR_INVALID_ARG;
    LruArgs a{u_re, u_im, nu_log, theta_log, gamma_log, (const f32x2 *)h, (const f32x2 *)P, done, (f32x2 *)h_out, (f32x2 *)P_out, row, B * N,
              (int)N, done_dtype == MRX_DONE_F32};
    return launch_kernel(lru_step_kernel, dim3((unsigned)((B * N + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream), a);
}

extern "C" int mrx_mlstm_step(void *stream, const float *up, const float *conv_w, const float *conv_b, const float *wq, const float *wk,
                              const float *wv, const float *wi, const float *bi, const float *wf, const float *bf, const float *norm_w,
                              const float *skip, const void *done, const float *C, const float *lf, const float *n, const float *m,
                              float *C_out, float *lf_out, float *n_out, float *m_out, float *y, int64_t B, int64_t H, int64_t D,
                              int64_t conv_k, int done_dtype, float g_floor)
{
    using namespace mrx;
    for (const void *p : {(const void *)up, (const void *)conv_w, (const void *)conv_b, (const void *)wq, (const void *)wk, (const void *)wv,
                          (const void *)wi, (const void *)bi, (const void *)wf, (const void *)bf, (const void *)norm_w, (const void *)skip, done,
                          (const void *)C, (const void *)lf, (const void *)n, (const void *)m, (const void *)C_out, (const void *)lf_out,
                          (const void *)n_out, (const void *)m_out, (const void *)y})
        if (!p) return MRX_ERR_INVALID_ARG;
    if (done_dtype != MRX_DONE_U8 && done_dtype != MRX_DONE_F32) return MRX_ERR_INVALID_ARG;
    if (B <= 0 || B >= (1ll << 31) || H <= 0 || conv_k <= 0 || conv_k > 64) return MRX_ERR_INVALID_ARG;
    if (H > MS_HEADS || H * D > MS_WIDTH || (D != 16 && D != 32 && D != 64)) return MRX_ERR_UNSUPPORTED;
    for (const float *p : {wq, wk, wv, C, (const float *)C_out})
        if (!aligned(p, 16)) return MRX_ERR_INVALID_ARG;
    MlstmStepArgs a{up, conv_w, conv_b, wq, wk, wv, wi, bi, wf, bf, norm_w, skip, C, lf, n, m, done, C_out, lf_out, n_out, m_out, y,
                    (int)conv_k, (int)H, done_dtype == MRX_DONE_F32, g_floor};
    hipStream_t st = static_cast<hipStream_t>(stream);
    const dim3 grid((unsigned)B), block(256);
    if (D == 64) return launch_kernel(mlstm_step_kernel<64>, grid, block, 0, st, a);
    if (D == 32) return launch_kernel(mlstm_step_kernel<32>, grid, block, 0, st, a);
    return launch_kernel(mlstm_step_kernel<16>, grid, block, 0, st, a);
}
