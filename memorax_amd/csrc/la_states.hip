// The kernels declared in la_states.h.
#include "la_states.h"

#include <type_traits>

#include "chunk_common.h"

namespace mrx {
inline namespace MRX_HD_NS {

namespace {

// One workgroup = one chunk of one sequence: slot <- sum over the kept rows r of y_r phi(x_r)^T,
// kept = the chunk's last episode (forward: what the chunk adds to the state that leaves it) or its
// first episode (backward: what it adds to the gradient of the state that enters it).
// NARROW: narrow heads -- x rows are dka wide in memory, y rows dva, a slot is [dva][dka]; the tiles keep the
// build's width with zeros beyond (after the feature map).
// GATED, NORM: as in the chunk kernels; kept rows are weighted in fp32 before they are rounded to the tiles' type.
template <typename T, int C, bool FMAP, bool BWD, bool NARROW, bool GATED, bool NORM>
__global__ void __launch_bounds__(256)
la_chunk_state_kernel(const T *__restrict__ x, const T *__restrict__ y, const void *__restrict__ done, int done_f32,
                      float *__restrict__ slots, int Tlen, int H, int NC, int dka, int dva, LaStateArgs a)
{
    constexpr int NW = 4, NTHR = 64 * NW, LDD = HD + pad_of<T>();
    using IO = TileIO<T, C, NTHR>;
    using TMS = TileMap<HD, HD, NW>;
    __shared__ __align__(16) T sX[C * LDD];
    __shared__ __align__(16) T sY[C * LDD];
    __shared__ float sDd[NORM && BWD ? C : 1];           // dden of the kept rows
    __shared__ float sPart[NORM ? NTHR : 1];             // partial column sums
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int bh = blockIdx.x, c = blockIdx.y, b = bh / H, h = bh % H;
    const int t0 = c * C;
    const int dkw = NARROW ? dka : HD, dvw = NARROW ? dva : HD;
    const bool segx = !NARROW || (tid % IO::SEGS) * IO::KP < dkw, segy = !NARROW || (tid % IO::SEGS) * IO::KP < dvw;

    typename IO::Regs rx, ry;
    IO::zero(rx);
    IO::zero(ry);
    if (segx) IO::load(rx, x + ((int64_t)b * Tlen * H + h) * dkw, (int64_t)H * dkw, t0, Tlen, tid);
    if (segy) IO::load(ry, y + ((int64_t)b * Tlen * H + h) * dvw, (int64_t)H * dvw, t0, Tlen, tid);
    typename IO::Regs ro;
    if (NORM && BWD) {
        IO::zero(ro);
        if (segy) IO::load(ro, static_cast<const T *>(a.o) + ((int64_t)b * Tlen * H + h) * dvw, (int64_t)H * dvw, t0, Tlen, tid);
    }
    float rg = 0.f;
    if (GATED && lane < C && t0 + lane < Tlen) rg = a.glog[((int64_t)b * Tlen + t0 + lane) * H + h];
    const bool dn = lane < C && t0 + lane < Tlen && done_at(done, done_f32, (int64_t)b * Tlen + t0 + lane);
    const unsigned long long dmask = __ballot(dn);
    const int nres = __popcll(dmask);
    if (segx) IO::template fmap<FMAP>(rx);  // columns beyond a narrow head's width stay zero
    const int ep = BWD ? 0 : nres;
    auto keep = [&](int r) { return nres == 0 || episode_of(dmask, r) == ep; };
    if (nres != 0) {  // rows of other episodes leave by select: what they hold must not meet a zero in a product
        IO::mask_rows(rx, tid, keep);
        IO::mask_rows(ry, tid, keep);
        if (NORM && BWD) IO::mask_rows(ro, tid, keep);
    }
    if (GATED) {
        // G_i = sum of the log-decays of the kept episode up to row i, without its first step's (chunk kernels)
        float G = lane < C && keep(lane) && !((dmask >> lane) & 1ull) ? rg : 0.f;
#pragma unroll
        for (int off = 1; off < C; off <<= 1) {
            const float up = __shfl_up(G, off);
            if (lane >= off) G += up;
        }
        const float Glast = __shfl(G, C - 1);
        const float E = __expf(BWD ? G : Glast - G);
        float f[IO::PASSES];
#pragma unroll
        for (int p = 0; p < IO::PASSES; ++p) f[p] = __shfl(E, IO::row_of(tid, p) % C);
        IO::scale_rows(rx, f);
        if (tid == 0) a.dec[(int64_t)bh * NC + c] = __expf(Glast);
    }
    if (NORM && !BWD && t0 + C > Tlen) IO::mask_rows(rx, tid, [&](int r) { return t0 + r < Tlen; });  // phi(0) = 1 must not count towards z
    if (NORM && BWD) {
        // dnum_i = dout_i / den_i in the place of dout_i, dden_i = -(dout_i . o_i) / den_i (chunk kernels)
        float inv[IO::PASSES];
#pragma unroll
        for (int p = 0; p < IO::PASSES; ++p) {
            const int r = IO::row_of(tid, p);
            const bool on = (IO::FULL || r < C) && t0 + r < Tlen && keep(r);
            const int64_t at = (int64_t)bh * Tlen + t0 + r;
            const float den = on ? a.den[at] : 1.f;
            if (a.d_ss) {  // dout_i + 2 d_ss_i o_i takes the place of dout_i
                const float two = on ? 2.f * a.d_ss[at] : 0.f;
                float dot = 0.f, oo = 0.f;
#pragma unroll
                for (int e = 0; e < IO::KP; ++e) {
                    const float of = (float)ro.v[p][e], yf = (float)ry.v[p][e];
                    dot += yf * of, oo += of * of;
                    ry.v[p][e] = (T)((yf + two * of) / den);
                }
                inv[p] = seg_sum<IO::SEGS>(dot) + two * seg_sum<IO::SEGS>(oo);
            } else {
                float dot = 0.f;
#pragma unroll
                for (int e = 0; e < IO::KP; ++e) dot += (float)ry.v[p][e] * (float)ro.v[p][e];
                inv[p] = seg_sum<IO::SEGS>(dot);
            }
            if (tid % IO::SEGS == 0 && (IO::FULL || r < C)) sDd[r] = on && den > a.eps ? -inv[p] / den : 0.f;
            inv[p] = 1.f / den;
        }
        if (!a.d_ss) IO::scale_rows(ry, inv);
    }
    // rows past the end of the sequence: y is zero there, and phi(0) = 1 in x is finite
    IO::to_lds(rx, sX, LDD, tid);
    IO::to_lds(ry, sY, LDD, tid);
    sync_lds();
    if (NORM) {  // column sums of the keys (of the queries, weighted by dden): the chunk's part of z (of its gradient)
        constexpr int G = NTHR / HD;
        const int col = tid % HD;
        float part = 0.f;
#pragma unroll
        for (int i = 0; i < C / G; ++i) {
            const int r = i * G + tid / HD;
            part += (float)sX[r * LDD + col] * (BWD ? sDd[BWD ? r : 0] : 1.f);
        }
        sPart[tid] = part;
        sync_lds();
        if (tid < HD && tid < dkw) {
            float z = 0.f;
#pragma unroll
            for (int i = 0; i < G; ++i) z += sPart[i * HD + tid];
            a.z[((int64_t)bh * NC + c) * dkw + tid] = z;
        }
    }
    f32x4 acc[TMS::TPW];  // S^T: m = dk, n = dv
    zero_acc<TMS::TPW>(acc);
    gemm<T, HD, HD, C, KROW, KROW, NW>(acc, sX, LDD, sY, LDD, w, lane);
    float *slot = slots + ((int64_t)bh * NC + c) * (dvw * dkw);
#pragma unroll
    for (int j = 0; j < TMS::TPW; ++j) {
        const int dk0 = TMS::mt(w, j) * 16 + 4 * lg, dv = TMS::nt(w, j) * 16 + li;
        if (!NARROW || (dv < dvw && dk0 < dkw)) *reinterpret_cast<f32x4 *>(slot + dv * dkw + dk0) = acc[j];
    }
}

// grid (B * H, d * d / 1024, plus one where z is scanned too): each thread carries four of the d x d state elements through the chunks.  Only the
// additions are sequential, so all there is to it is trips to memory: up to 32 slots are on their way at once, each requested as the one 32 before
// it has been used, and resets and decays of 64 chunks are fetched together -- the flags by all threads, a row each, and kept as one bit per chunk.
// (32 sequences of 24 chunks of 32 x 32: 7.6 us a scan with groups of eight slots and their flags on their way, 5.5 now; 4 of 512 chunks 62 and 32;
// 64 of 64 chunks of 64 x 64 26 and 24.)
// NARROW: narrow heads, the state's size is a run-time value.
// DECAY: the sum so far enters a chunk without resets times dec[chunk].  Z: the last block of the grid's second axis
// carries the dk elements of z instead.
// SLOTS: on their way at once, 32 or, where the workgroups already fill the device, 8 (launch_la_state_scan).
template <bool NARROW, bool DECAY, bool Z, int SLOTS>
__global__ void __launch_bounds__(256)
la_state_scan_kernel(float *__restrict__ slots, const float *__restrict__ init, float *__restrict__ fin,
                     const void *__restrict__ done, int done_f32, int Tlen, int H, int NC, int C, int backward, int Qn,
                     const float *__restrict__ dec, float *__restrict__ zslots, const float *__restrict__ zinit, float *__restrict__ zfin, int zq)
{
    const bool zpart = Z && blockIdx.y == gridDim.y - 1;
    const int Q = zpart ? zq : NARROW ? Qn : HD * HD / 4;  // f32x4 per state (d_v * d_k / 4)
    if (zpart) slots = zslots, init = zinit, fin = zfin;
    constexpr int G = SLOTS, WINDOW = 64;   // (WINDOW: chunks whose flags are fetched together)
    __shared__ int sCut[WINDOW];
    const int tid = threadIdx.x, lane = tid & 63;
    const int bh = blockIdx.x, b = bh / H;
    const int idx = (zpart ? 0 : blockIdx.y * 256) + tid;
    const bool act = !(NARROW || Z) || idx < Q;  // a narrow state has fewer elements than the workgroup has threads; the idle lanes
                                       // still see to their share of the flags
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 *p = reinterpret_cast<f32x4 *>(slots) + (int64_t)bh * NC * Q + (act ? idx : 0);
    auto chunk_of = [&](int s) { return backward ? NC - 1 - s : s; };
    f32x4 t[G];
    auto fetch = [&](int u, int s) { t[u] = p[(int64_t)chunk_of(s) * Q]; };
#pragma unroll
    for (int u = 0; u < G; ++u)
        if (u < NC) fetch(u, u);
    f32x4 S = init && act ? reinterpret_cast<const f32x4 *>(init)[(int64_t)bh * Q + idx] : zero;
    const int shift = 31 - __builtin_clz(C);   // (chunks are powers of two)
    uint64_t cuts = 0;   // of the window's chunks, by the order they are walked in
    float decays = 0.f;  // lane l: that of the window's chunk l
    for (int s0 = 0; s0 < NC; s0 += G) {
        if (s0 % WINDOW == 0) {
            const int n = NC - s0 < WINDOW ? NC - s0 : WINDOW;   // chunks of the window, from its first row on
            const int row0 = (backward ? NC - s0 - n : s0) * C, row1 = row0 + n * C < Tlen ? row0 + n * C : Tlen;
            if constexpr (DECAY) decays = dec[(int64_t)bh * NC + chunk_of(s0 + (lane < n ? lane : n - 1))];
            if (s0) __syncthreads();   // (the window before has been read)
            if (tid < WINDOW) sCut[tid] = 0;
            __syncthreads();
            for (int r0 = row0 + tid; r0 < row1; r0 += 8 * 256) {
                uint32_t flag[8];
                if (done_f32) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) flag[i] = done_raw(done, 1, (int64_t)b * Tlen + (r0 + i * 256 < row1 ? r0 + i * 256 : r0));
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i) flag[i] = done_raw(done, 0, (int64_t)b * Tlen + (r0 + i * 256 < row1 ? r0 + i * 256 : r0));
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int r = r0 + i * 256 < row1 ? r0 + i * 256 : r0, c = (r - row0) >> shift;
                    if (done_test(flag[i], done_f32)) sCut[backward ? n - 1 - c : c] = 1;
                }
            }
            __syncthreads();
            cuts = __ballot(sCut[lane] != 0);
        }
        auto step = [&](int u) {
            const int s = s0 + u;
            if (act) p[(int64_t)chunk_of(s) * Q] = S;
            float e = 1.f;
            if constexpr (DECAY) e = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, decays), s % WINDOW));
            const uint32_t cut = -(uint32_t)(cuts >> (s % WINDOW) & 1);
            S = DECAY ? e * S + t[u] : S + t[u];
#pragma unroll
            for (int i = 0; i < 4; ++i)   // (selected by bits: a branch per chunk costs more than the sum)
                S[i] = __builtin_bit_cast(float, (__builtin_bit_cast(uint32_t, (float)t[u][i]) & cut) | (__builtin_bit_cast(uint32_t, (float)S[i]) & ~cut));
        };
        if (s0 + G <= NC) {
#pragma unroll
            for (int u = 0; u < G; ++u) {
                step(u);
                fetch(u, s0 + G + u < NC ? s0 + G + u : NC - 1);
            }
        } else {
#pragma unroll
            for (int u = 0; u < G; ++u)
                if (s0 + u < NC) step(u);
        }
    }
    if (fin && act) reinterpret_cast<f32x4 *>(fin)[(int64_t)bh * Q + idx] = S;
}

template <typename T, int C>
int launch_states(hipStream_t st, const void *x, const void *y, const void *done, int done_f32, float *slots, int64_t B,
                  int64_t Tlen, int64_t H, bool fmap, bool backward, int64_t dk, int64_t dv, const LaStateArgs &a)
{
    const int64_t NC = (Tlen + C - 1) / C;
    if (B * H > 0x7fffffffLL || NC > 65535) return MRX_ERR_INVALID_ARG;
    auto go = [&](auto fm, auto bw, auto narrow, auto gated, auto norm) {
        return launch_kernel(la_chunk_state_kernel<T, C, decltype(fm)::value, decltype(bw)::value, decltype(narrow)::value,
                                                   decltype(gated)::value, decltype(norm)::value>,
                             dim3((unsigned)(B * H), (unsigned)NC), dim3(256), 0, st, (const T *)x, (const T *)y, done, done_f32, slots,
                             (int)Tlen, (int)H, (int)NC, (int)dk, (int)dv, a);
    };
    using Y = std::true_type;
    using N = std::false_type;
    auto variant = [&](auto fm, auto bw, auto narrow) {
        if (a.glog) return go(fm, bw, narrow, Y{}, N{});
        if (a.z) return go(fm, bw, narrow, N{}, Y{});
        return go(fm, bw, narrow, N{}, N{});
    };
    auto sized = [&](auto fm, auto bw) { return dk != HD || dv != HD ? variant(fm, bw, Y{}) : variant(fm, bw, N{}); };
    if (fmap) return backward ? sized(Y{}, Y{}) : sized(Y{}, N{});
    return backward ? sized(N{}, Y{}) : sized(N{}, N{});
}

}  // namespace

int launch_la_chunk_states(hipStream_t st, const void *x, const void *y, const void *done, int done_f32, float *slots,
                           int64_t B, int64_t Tlen, int64_t H, int dtype, bool fmap, bool backward, int64_t dk, int64_t dv,
                           const LaStateArgs &a)
{
    if (dtype == MRX_BF16)
        return launch_states<__bf16, LA_BF16_CHUNK>(st, x, y, done, done_f32, slots, B, Tlen, H, fmap, backward, dk, dv, a);
    return launch_states<float, 32>(st, x, y, done, done_f32, slots, B, Tlen, H, fmap, backward, dk, dv, a);
}

// 32 slots on their way take a compute unit's registers for one workgroup: up to one of those per compute unit (16 sequences x 8 heads x 16 chunks
// of 64 x 64, 512 workgroups: 14 us with 32, 11 with 8), and from 16 chunks on (10 chunks: 4.5 and 4.3 us).
constexpr int64_t SCAN_FEW = 256, SCAN_LONG = 16;
int launch_la_state_scan(hipStream_t st, float *slots, const float *init, float *fin, const void *done, int done_f32,
                         int64_t B, int64_t Tlen, int64_t H, int C, bool backward, int64_t dk, int64_t dv, const LaStateArgs &a)
{
    const int64_t NC = (Tlen + C - 1) / C;
    if (B * H > 0x7fffffffLL) return MRX_ERR_INVALID_ARG;
    const int Q = (int)(dk * dv / 4);
    const dim3 grid((unsigned)(B * H), (unsigned)((Q + 255) / 256 + (a.z ? 1 : 0)));
    auto scan = [&](auto narrow, auto decay, auto z, auto slots_ahead) {
        return launch_kernel(la_state_scan_kernel<decltype(narrow)::value, decltype(decay)::value, decltype(z)::value, decltype(slots_ahead)::value>,
                             grid, dim3(256), 0, st, slots, init, fin, done, done_f32, (int)Tlen, (int)H, (int)NC, C, backward ? 1 : 0, Q,
                             (const float *)a.dec, a.z, a.z_init, a.z_fin, (int)(dk / 4));
    };
    auto go = [&](auto narrow, auto decay, auto z) {
        return (int64_t)grid.x * grid.y <= SCAN_FEW && NC >= SCAN_LONG ? scan(narrow, decay, z, std::integral_constant<int, 32>{})
                                                    : scan(narrow, decay, z, std::integral_constant<int, 8>{});
    };
    auto variant = [&](auto narrow) {
        if (a.dec) return go(narrow, std::true_type{}, std::false_type{});
        if (a.z) return go(narrow, std::false_type{}, std::true_type{});
        return go(narrow, std::false_type{}, std::false_type{});
    };
    return dk != HD || dv != HD ? variant(std::true_type{}) : variant(std::false_type{});
}

}  // namespace MRX_HD_NS
}  // namespace mrx
