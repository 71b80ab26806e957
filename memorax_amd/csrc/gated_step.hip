// The acting step of a gated recurrence, from the block's input to what its closing layer reads, as one launch: norm -> z, h~, gate ->
// MinGRU step -> gated state.  A workgroup of four waves owns 16 rows and 64 features of all three layers, so that a lane ends up with the
// three values of four features of a row and nothing leaves the workgroup in between.  Bound by its trips to memory, of which there
// is one: rows, weights, carries and flags are requested together.  1024 rows x 256 within the torso's graph, where the matrix
// states have pushed the weights out of L2: 10.2 us, as two launches 9.0 + 5.4.  (The same for a matrix state -- projections of a head and
// its step in one launch, the states on their way meanwhile -- gains nothing: whole rows of states are 256 KB a workgroup, one
// workgroup a compute unit, and the slowest of them ends 40 % after the mean: 31 us, as two launches 31; few rows 9.2 / 7.7.)
// Rounding follows the launches it stands for (row_dense.hip, mingru_step_kernel); 1024 rows x 256 come out with the same bits.
#include "mingru.h"
#include "row_parts.h"

namespace mrx {
namespace {

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
