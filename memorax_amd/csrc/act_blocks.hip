// Acting steps of whole recurrences, from the block's input to what its closing layer reads, as one launch: norm, the dense layers that read
// its result, and the recurrence's step on their outputs, which never leave the workgroup.  As launches of their own the step waits for
// memory twice more -- for the projections that have just been written, and for the weights, behind which the carried states could
// already be on their way.
//
// gated_step_kernel: norm -> z, h~, gate -> MinGRU step -> gated state.  A workgroup of four waves owns 16 rows and 64 features of all
// three layers, so that a lane ends up with the three values of four features of a row.
// state_act_kernel: norm -> q, k, v (, beta) of one head -> step of the head's matrix state (step.hip) -> read-out.  A workgroup of eight
// waves owns R rows and a head; its states (R x D x D floats: 256 KB at 16 x 64 x 64, half a compute unit's registers) are requested
// before the rows are normalised and arrive while the products run.  Few rows are cut finer (R = 4), for the states of a row are what one
// workgroup moves slowly.
// Rounding follows the launches they stand for (row_dense.hip, step.hip, mingru_step_kernel).
#include "mingru.h"
#include "row_parts.h"

namespace mrx {
namespace {

// ---- gated recurrence
struct GatedStepArgs {
    RowInput in;
    const void *w[3], *done;
    const float *log_state, *log_decay;   // (rows, N); may be updated in place
    float *log_state_out, *log_decay_out;
    void *z, *y;                          // (rows, N) in the products' type
    int N, done_f32;
};

constexpr int GS_WAVES = 4, GS_THREADS = 64 * GS_WAVES, GS_ROWS = 16;

template <typename T, bool WBF, int NV> __global__ void __launch_bounds__(GS_THREADS) gated_step_kernel(GatedStepArgs a)
{
    using F = typename TT<T>::frag;
    using P = typename TT<T>::pack4;
    constexpr int KP = TT<T>::KP, KB = TT<T>::KB, RPW = GS_ROWS / GS_WAVES, AHEAD = 8;
    extern __shared__ __align__(16) unsigned char smem[];
    T *sx = reinterpret_cast<T *>(smem);
    const int K = a.in.K, N = a.N, kpad = (K + KB - 1) / KB * KB, ld = kpad + pad_of<T>(), steps = kpad / KB;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i16 = lane & 15, g = lane >> 4;
    const unsigned tiles = (unsigned)(N + 63) / 64, tile = blockIdx.x % tiles;
    const int64_t r0 = (int64_t)(blockIdx.x / tiles) * GS_ROWS, rows = a.in.rows;
    const int n0 = (tile * GS_WAVES + wv) * 16;

    RowPanel<false, RPW, NV> panel;
    panel.load(a.in, r0 + wv * RPW, lane);
    RawFrag<T, WBF> ahead[AHEAD][3];   // of the next k steps: each is requested again as soon as it has been used
    const int64_t column = (int64_t)(n0 + i16 < N ? n0 + i16 : N - 1) * K;
#pragma unroll
    for (int s = 0; s < AHEAD; ++s)
#pragma unroll
        for (int l = 0; l < 3; ++l) ahead[s][l] = weight_raw<T, WBF>(a.w[l], column + weight_k<T>(s * KB + KP * g, K));
    panel.load_norm(a.in, lane);
    const int c0 = n0 + 4 * g;
    const int64_t r = r0 + i16 < rows ? r0 + i16 : rows - 1, at = r * N + (c0 < N ? c0 : 0);   // N is a multiple of 4
    f32x4 ls = *reinterpret_cast<const f32x4 *>(a.log_state + at), ldc = *reinterpret_cast<const f32x4 *>(a.log_decay + at);
    const uint32_t flag = done_raw(a.done, a.done_f32, r);

    panel.template finish<T>(a.in, sx + wv * RPW * ld, ld, kpad, lane, [](int, int, int, const f32x4 &) {});
    sync_lds();
    f32x4 acc[3];
    zero_acc<3>(acc);
    for (int s0 = 0; s0 < steps; s0 += AHEAD) {
#pragma unroll
        for (int s = 0; s < AHEAD; ++s) {
            if (s0 + s >= steps) break;
            const int k = (s0 + s) * KB + KP * g;
            const F xf = TT<T>::template load<ROWK>(sx, ld, 0, (s0 + s) * KB, lane);
#pragma unroll
            for (int l = 0; l < 3; ++l) {
                F wf = weight_frag<T, WBF>(ahead[s][l]);
                if (kpad != K && k >= K) wf = F{};
                if (s0 + s + AHEAD < steps) ahead[s][l] = weight_raw<T, WBF>(a.w[l], column + weight_k<T>(k + AHEAD * KB, K));
                acc[l] = TT<T>::mma(wf, xf, acc[l]);
            }
        }
    }
    if (r0 + i16 >= rows || c0 >= N) return;
    const bool reset = done_test(flag, a.done_f32);
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float z = (float)(T)acc[0][e];
        float za = z, xb = (float)(T)acc[1][e];
        const float log_a = -(fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))));   // log sigma(-z)
        MinGru::coeffs(za, xb);
        const float h = reset ? xb : za * expf(ls[e]) + xb, gate = (float)(T)acc[2][e];
        ls[e] = logf(h);
        ldc[e] = reset ? log_a : ldc[e] + log_a;
        y[e] = (float)(T)h * gate / (1.f + __expf(-gate));   // the state as the cell hands it on
    }
    *reinterpret_cast<f32x4 *>(a.log_state_out + at) = ls;
    *reinterpret_cast<f32x4 *>(a.log_decay_out + at) = ldc;
    *reinterpret_cast<P *>(static_cast<T *>(a.z) + at) = TT<T>::pack(acc[0][0], acc[0][1], acc[0][2], acc[0][3]);
    *reinterpret_cast<P *>(static_cast<T *>(a.y) + at) = TT<T>::pack(y[0], y[1], y[2], y[3]);
}

// ---- matrix states
struct StateActArgs {
    RowInput in;
    const void *w[4], *done;        // query, key, value (H D, K), beta (H, K)
    const float *S_in, *z_in;       // (rows, H, D, D) and (rows, H, D); may be updated in place
    float *S_out, *z_out;
    void *o;                        // (rows, H D)
    float eps;
    int H, done_f32;
    bool s_bf16;                    // the type that projections and read-out are handed on in
};

constexpr int SA_WAVES = 8, SA_THREADS = 64 * SA_WAVES, SA_MAX_K = 256;

// T: the products' type; D: head dim; R: rows per workgroup; DELTA: the delta rule with its prologue, otherwise linear attention with the
// elu + 1 map and the normalised read-out.
template <typename T, bool WBF, int D, int R, bool DELTA> __global__ void __launch_bounds__(SA_THREADS) state_act_kernel(StateActArgs a)
{
    using F = typename TT<T>::frag;
    constexpr int KP = TT<T>::KP, KB = TT<T>::KB, AHEAD = 8, MOST_STEPS = SA_MAX_K / KB, RPW = R > SA_WAVES ? R / SA_WAVES : 1;
    constexpr int NQ = D / 16, TILES = 3 * NQ + DELTA, MT = (TILES + SA_WAVES - 1) / SA_WAVES;   // 16-column tiles: of a layer, in all, of a wave
    // the threads of a state: four columns each, RPP rows at a time; SG states at once
    constexpr int TG = D * D / 4 < SA_THREADS ? D * D / 4 : SA_THREADS, SG = SA_THREADS / TG, LPR = D / 4, RPP = TG / LPR, NP = D / RPP,
                  RPG = (R + SG - 1) / SG;
    extern __shared__ __align__(16) unsigned char smem[];
    float *const sp = reinterpret_cast<float *>(smem);               // q, k, v: [3][16][D]
    float *const so = sp + 3 * 16 * D, *const sz = so + R * D;       // read-out, normaliser: [R][D]
    float *const sb = sz + R * D;                                    // beta [16], flags [16]
    T *const sx = reinterpret_cast<T *>(sb + 32);
    const int K = a.in.K, kpad = (K + KB - 1) / KB * KB, ld = kpad + pad_of<T>(), steps = kpad / KB;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), i16 = lane & 15, g = lane >> 4;
    const int h = (int)(blockIdx.x % (unsigned)a.H);
    const int64_t r0 = (int64_t)(blockIdx.x / (unsigned)a.H) * R, rows = a.in.rows;
    auto row_at = [&](int j) { return r0 + j < rows ? r0 + j : rows - 1; };   // rows that are not there read another's

    RowPanel<false, RPW, 1> panel;
    panel.load(a.in, r0 + wv * RPW, lane);
    const void *w[MT];
    int first[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int t = wv + SA_WAVES * m < TILES ? wv + SA_WAVES * m : TILES - 1, l = t / NQ;
        w[m] = a.w[l];
        first[m] = l < 3 ? h * D + t % NQ * 16 + i16 : h;
    }
    RawFrag<T, WBF> ahead[AHEAD][MT];   // of the next k steps: each is requested again as soon as it has been used
#pragma unroll
    for (int t = 0; t < AHEAD; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) ahead[t][m] = weight_raw<T, WBF>(w[m], (int64_t)first[m] * K + weight_k<T>(t * KB + KP * g, K));
    panel.load_norm(a.in, lane);
    f32x4 z4 = {0.f, 0.f, 0.f, 0.f};
    const bool has_z = !DELTA && tid < R * LPR;   // thread (row, four columns) owns them of the normaliser
    const int64_t zat = (row_at(tid / LPR % R) * a.H + h) * D + tid % LPR * 4;
    if (has_z) z4 = *reinterpret_cast<const f32x4 *>(a.z_in + zat);
    const uint32_t flag = done_raw(a.done, a.done_f32, row_at(tid % R));
    const int sg = tid / TG, c4 = tid % LPR, ir = tid % TG / LPR;
    f32x4 s[RPG][NP];
#pragma unroll
    for (int j = 0; j < RPG; ++j) {
        const float *S = a.S_in + (row_at(sg + j * SG) * a.H + h) * (D * D) + ir * D + 4 * c4;
#pragma unroll
        for (int p = 0; p < NP; ++p) s[j][p] = *reinterpret_cast<const f32x4 *>(S + p * RPP * D);
    }

    if (wv * RPW < 16) panel.template finish<T>(a.in, sx + wv * RPW * ld, ld, kpad, lane, [](int, int, int, const f32x4 &) {});
    if (tid < R) sb[16 + tid] = done_test(flag, a.done_f32) ? 1.f : 0.f;
    if (has_z) *reinterpret_cast<f32x4 *>(sz + tid * 4) = z4;
    sync_lds();
    f32x4 acc[MT];
    zero_acc<MT>(acc);
    for (int s0 = 0; s0 < steps; s0 += AHEAD) {
#pragma unroll
        for (int t = 0; t < AHEAD; ++t) {
            if (s0 + t >= steps) break;
            const int k = (s0 + t) * KB + KP * g;
            const F xf = TT<T>::template load<ROWK>(sx, ld, 0, (s0 + t) * KB, lane);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                F wf = weight_frag<T, WBF>(ahead[t][m]);
                if (kpad != K && k >= K) wf = F{};
                if (MOST_STEPS > AHEAD && s0 + t + AHEAD < steps) ahead[t][m] = weight_raw<T, WBF>(w[m], (int64_t)first[m] * K + weight_k<T>(k + AHEAD * KB, K));
                acc[m] = TT<T>::mma(wf, xf, acc[m]);
            }
        }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int t = wv + SA_WAVES * m, l = t / NQ;
        f32x4 y = acc[m];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            y[e] = (float)(T)y[e];
            if (a.s_bf16) y[e] = (float)(__bf16)y[e];
        }
        if (t >= TILES) continue;
        if (l < 3) *reinterpret_cast<f32x4 *>(sp + (l * 16 + i16) * D + t % NQ * 16 + 4 * g) = y;
        else if (g == 0) sb[i16] = y[0];
    }
    sync_lds();

#pragma unroll
    for (int j = 0; j < RPG; ++j) {
        const int row = sg + j * SG;
        if (R < SG && row >= R) continue;
        const float *const qr = sp + row * D, *const kr = sp + (16 + row) * D, *const vr = sp + (32 + row) * D;
        f32x4 q4 = *reinterpret_cast<const f32x4 *>(qr + 4 * c4), k4 = *reinterpret_cast<const f32x4 *>(kr + 4 * c4);
        const bool reset = sb[16 + row] != 0.f, there = r0 + row < rows;
        auto dot = [](const f32x4 &x, const f32x4 &y) { return seg_sum<LPR>(x[0] * y[0] + x[1] * y[1] + x[2] * y[2] + x[3] * y[3]); };
        float u[NP], den = 1.f;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            if (reset) s[j][p] = f32x4{0.f, 0.f, 0.f, 0.f};
            u[p] = vr[ir + p * RPP];
        }
        if (DELTA) {
            const float norm = fmaxf(sqrtf(dot(k4, k4)), 1e-12f), inv = 1.f / norm;
#pragma unroll
            for (int e = 0; e < 4; ++e) k4[e] = a.s_bf16 ? (float)(__bf16)(k4[e] * inv) : k4[e] / norm;
            float beta = 1.f / (1.f + expf(-sb[row]));
            if (a.s_bf16) beta = (float)(__bf16)beta;
#pragma unroll
            for (int p = 0; p < NP; ++p) u[p] = beta * (u[p] - dot(s[j][p], k4));
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) k4[e] = elu1(k4[e]), q4[e] = elu1(q4[e]);
            f32x4 z = *reinterpret_cast<const f32x4 *>(sz + row * D + 4 * c4);
            if (reset) z = f32x4{0.f, 0.f, 0.f, 0.f};
            z += k4;
            if (ir == 0 && there) *reinterpret_cast<f32x4 *>(a.z_out + ((r0 + row) * a.H + h) * D + 4 * c4) = z;
            den = fmaxf(dot(z, q4), a.eps);
        }
        float *const S = a.S_out + ((r0 + row) * a.H + h) * (D * D) + ir * D + 4 * c4;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            s[j][p] += k4 * u[p];
            if (there) *reinterpret_cast<f32x4 *>(S + p * RPP * D) = s[j][p];
            const float x = dot(s[j][p], q4);
            if (c4 == 0) so[row * D + ir + p * RPP] = x / den;
        }
    }
    sync_lds();
    for (int e = tid; e < R * D / 4; e += SA_THREADS) {
        const int row = e / (D / 4), c = e % (D / 4) * 4;
        if (r0 + row >= rows) break;
        const f32x4 x = *reinterpret_cast<const f32x4 *>(so + row * D + c);
        const int64_t at = ((r0 + row) * a.H + h) * D + c;
        if (a.s_bf16) *reinterpret_cast<bf16x4 *>(static_cast<__bf16 *>(a.o) + at) = TT<__bf16>::pack(x[0], x[1], x[2], x[3]);
        else *reinterpret_cast<f32x4 *>(static_cast<float *>(a.o) + at) = x;
    }
}

template <typename T, bool WBF, int D, bool DELTA> int launch_state(hipStream_t st, const StateActArgs &a, int cus)
{
    constexpr int KB = TT<T>::KB, MOST = D < 64 || (DELTA && (WBF || sizeof(T) == 4)) ? 16 : 8;   // as the registers have room for
    auto go = [&](auto rows) {
        constexpr int R = decltype(rows)::value;
        const int64_t grid = (a.in.rows + R - 1) / R * a.H;
        const size_t lds = (3 * 16 * D + 2 * R * D + 32) * 4 + 16 * ((a.in.K + KB - 1) / KB * KB + pad_of<T>()) * sizeof(T);
        return launch_kernel(state_act_kernel<T, WBF, D, R, DELTA>, dim3((unsigned)grid), dim3(SA_THREADS), lds, st, a);
    };
    // as many rows as fill the device once, for they share the weights
    if (a.in.rows * a.H >= (int64_t)MOST * cus) return go(std::integral_constant<int, MOST>{});
    return go(std::integral_constant<int, 4>{});
}
template <int D, bool DELTA> int launch_state_types(hipStream_t st, const StateActArgs &a, bool bf, bool wbf, int cus)
{
    if (bf) return wbf ? launch_state<__bf16, true, D, DELTA>(st, a, cus) : launch_state<__bf16, false, D, DELTA>(st, a, cus);
    return launch_state<float, false, D, DELTA>(st, a, cus);
}

bool input_ok(const RowInput &in, int most)
{
    return in.x && in.rows > 0 && in.rows < (1ll << 31) && in.K > 0 && in.K % 8 == 0 && in.K <= most && in.norm >= 0 && in.norm <= 2 && aligned(in.x, 16) &&
           aligned(in.scale, 16) && aligned(in.nbias, 16);
}

}  // namespace
}  // namespace mrx

extern "C" int mrx_gated_recurrence_act(void *stream, const float *x, const float *scale, const float *norm_bias, int norm, const void *w_z,
                                        const void *w_h, const void *w_gate, const void *done, const float *log_state,
                                        const float *log_decay, void *z, void *y, float *log_state_out, float *log_decay_out,
                                        int64_t rows, int64_t K, int64_t N, int w_dtype, int product_dtype, int done_dtype, float eps)
{
    using namespace mrx;
    GatedStepArgs a{};
    a.in = RowInput{x, scale, norm_bias, rows, (int)K, norm, eps, 1.f / (float)K, false};
    const void *arrays[] = {w_z, w_h, w_gate, log_state, log_decay, z, y, log_state_out, log_decay_out};
    for (const void *p : arrays)
        if (!p || !aligned(p, 16)) return MRX_ERR_INVALID_ARG;
    if (!done || (done_dtype != MRX_DONE_U8 && done_dtype != MRX_DONE_F32)) return MRX_ERR_INVALID_ARG;
    if (K > 512 || N <= 0 || N % 4 != 0 || N > (1 << 24) || (product_dtype == MRX_F32 && w_dtype != MRX_F32)) return MRX_ERR_UNSUPPORTED;
    if (!input_ok(a.in, 512) || (w_dtype != MRX_F32 && w_dtype != MRX_BF16) || (product_dtype != MRX_F32 && product_dtype != MRX_BF16)) return MRX_ERR_INVALID_ARG;
    a.w[0] = w_z, a.w[1] = w_h, a.w[2] = w_gate, a.done = done, a.done_f32 = done_dtype == MRX_DONE_F32;
    a.log_state = log_state, a.log_decay = log_decay, a.log_state_out = log_state_out, a.log_decay_out = log_decay_out, a.z = z, a.y = y, a.N = (int)N;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    const int64_t grid = (rows + GS_ROWS - 1) / GS_ROWS * ((N + 63) / 64);
    if (grid >= (1ll << 31)) return MRX_ERR_INVALID_ARG;
    auto go = [&](auto t, auto wbf, auto nv) {
        using T = decltype(t);
        constexpr int KB = TT<T>::KB;
        const size_t lds = GS_ROWS * ((K + KB - 1) / KB * KB + pad_of<T>()) * sizeof(T);
        return launch_kernel(gated_step_kernel<T, decltype(wbf)::value, decltype(nv)::value>, dim3((unsigned)grid), dim3(GS_THREADS), lds,
                             static_cast<hipStream_t>(stream), a);
    };
    auto by_width = [&](auto t, auto wbf) { return K <= 256 ? go(t, wbf, std::integral_constant<int, 1>{}) : go(t, wbf, std::integral_constant<int, 2>{}); };
    if (product_dtype == MRX_BF16) return w_dtype == MRX_BF16 ? by_width(__bf16(), std::true_type{}) : by_width(__bf16(), std::false_type{});
    return by_width(float(), std::false_type{});
}

extern "C" int mrx_state_act(void *stream, const float *x, const float *scale, const float *norm_bias, int norm, const void *w_q,
                             const void *w_k, const void *w_v, const void *w_beta, const void *done, const float *S_in, const float *z_in,
                             void *o, float *S_out, float *z_out, int64_t rows, int64_t K, int64_t H, int64_t D, int w_dtype,
                             int product_dtype, int o_dtype, int done_dtype, float eps, float den_eps)
{
    using namespace mrx;
    StateActArgs a{};
    a.in = RowInput{x, scale, norm_bias, rows, (int)K, norm, eps, 1.f / (float)K, false};
    const void *arrays[] = {w_q, w_k, w_v, S_in, S_out, o};
    for (const void *p : arrays)
        if (!p || !aligned(p, 16)) return MRX_ERR_INVALID_ARG;
    if (!done || (done_dtype != MRX_DONE_U8 && done_dtype != MRX_DONE_F32) || (!w_beta && (!z_in || !z_out))) return MRX_ERR_INVALID_ARG;
    if (!aligned(w_beta, 16) || !aligned(z_in, 16) || !aligned(z_out, 16)) return MRX_ERR_INVALID_ARG;
    if (K > SA_MAX_K || (D != 16 && D != 32 && D != 64) || (product_dtype == MRX_F32 && w_dtype != MRX_F32)) return MRX_ERR_UNSUPPORTED;
    if (!input_ok(a.in, SA_MAX_K) || H <= 0 || rows * H >= (1ll << 29)) return MRX_ERR_INVALID_ARG;
    for (int dt : {w_dtype, product_dtype, o_dtype})
        if (dt != MRX_F32 && dt != MRX_BF16) return MRX_ERR_INVALID_ARG;
    a.w[0] = w_q, a.w[1] = w_k, a.w[2] = w_v, a.w[3] = w_beta, a.done = done, a.done_f32 = done_dtype == MRX_DONE_F32;
    a.S_in = S_in, a.z_in = z_in, a.S_out = S_out, a.z_out = z_out, a.o = o, a.eps = den_eps, a.H = (int)H, a.s_bf16 = o_dtype == MRX_BF16;
    int cus = 0;
    if (const int rc = prepare_device(&cus); rc != MRX_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool bf = product_dtype == MRX_BF16, wbf = w_dtype == MRX_BF16;
    if (w_beta)
        return D == 64 ? launch_state_types<64, true>(st, a, bf, wbf, cus) : D == 32 ? launch_state_types<32, true>(st, a, bf, wbf, cus)
                                                                                     : launch_state_types<16, true>(st, a, bf, wbf, cus);
    return D == 64 ? launch_state_types<64, false>(st, a, bf, wbf, cus) : D == 32 ? launch_state_types<32, false>(st, a, bf, wbf, cus)
                                                                                  : launch_state_types<16, false>(st, a, bf, wbf, cus);
}
