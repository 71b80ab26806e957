// Parts of the kernels that act: few rows, one per environment, normalised on their way into LDS and multiplied with weights that are
// read from memory as they lie there.  Whatever a kernel reads it requests before it uses any of it, and in one stretch without
// branches: a use, or the merge of a branch's values, waits for everything requested so far, and a launch of a few microseconds is
// as long as it has trips to memory one after another.
#pragma once
#include <type_traits>

#include "chunk_common.h"

namespace mrx {
namespace {

// Sums over a wave, in every lane: within rows of sixteen lanes by DPP moves (one instruction each, where a shuffle is a trip to
// LDS), the four rows by shuffles.
template <int N> __device__ __forceinline__ void wave_totals(float (&x)[N])
{
    auto add = [&](auto ctrl) {
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const int moved = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x[j]), decltype(ctrl)::value, 0xf, 0xf, true);
            x[j] += __builtin_bit_cast(float, moved);
        }
    };
    add(std::integral_constant<int, 0xB1>{});    // quad_perm [1,0,3,2]
    add(std::integral_constant<int, 0x4E>{});    // quad_perm [2,3,0,1]
    add(std::integral_constant<int, 0x141>{});   // row_half_mirror
    add(std::integral_constant<int, 0x140>{});   // row_mirror
#pragma unroll
    for (int by = 16; by <= 32; by *= 2) {
        float other[N];
#pragma unroll
        for (int j = 0; j < N; ++j) other[j] = __shfl_xor(x[j], by);
#pragma unroll
        for (int j = 0; j < N; ++j) x[j] += other[j];
    }
}

// A weight fragment as it waits in registers: KP consecutive k of one row, stored bits.
template <typename T, bool WBF> struct RawFrag {
    static constexpr int WORDS = TT<T>::KP * (WBF ? 2 : 4) / 8;   // 8-byte words
    uint64_t w[WORDS];
};
template <typename T, bool WBF> __device__ __forceinline__ RawFrag<T, WBF> weight_raw(const void *w, int64_t at)
{
    RawFrag<T, WBF> r;
    const char *p = static_cast<const char *>(w) + at * (WBF ? 2 : 4);
#pragma unroll
    for (int i = 0; i < RawFrag<T, WBF>::WORDS; ++i) r.w[i] = reinterpret_cast<const uint64_t *>(p)[i];
    return r;
}
template <typename T, bool WBF> __device__ __forceinline__ typename TT<T>::frag weight_frag(const RawFrag<T, WBF> &r)
{
    typename TT<T>::frag f;
    if constexpr (std::is_same<T, __bf16>::value && WBF) {
        f = __builtin_bit_cast(bf16x8, r);
    } else if constexpr (std::is_same<T, __bf16>::value) {
        struct F8 {
            float v[8];
        };
        const F8 x = __builtin_bit_cast(F8, r);
        const bf16x4 lo = TT<__bf16>::pack(x.v[0], x.v[1], x.v[2], x.v[3]), hi = TT<__bf16>::pack(x.v[4], x.v[5], x.v[6], x.v[7]);
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = lo[e], f[4 + e] = hi[e];
    } else if constexpr (WBF) {
        const bf16x4 x = __builtin_bit_cast(bf16x4, r);
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = (float)x[e];
    } else {
        f = __builtin_bit_cast(f32x4, r);
    }
    return f;
}

// Where a weight fragment's k starts, kept inside the row; `in` says whether it is the row's at all (columns K .. of a padded row count
// as zero on both sides: what was read there is dropped when it is used).
template <typename T> __device__ __forceinline__ int weight_k(int k, int K) { return k < K ? k : K - TT<T>::KP; }

// The rows a workgroup multiplies, and their norm: 0 none, 1 RMS, 2 layer norm (rows centred first).
struct RowInput {
    const void *x;
    const float *scale, *nbias;
    int64_t rows;
    int K, norm;
    float eps, inv_K;
    bool round_norm;   // the normalised rows pass through bfloat16
};

// RPW rows of a wave, up to 256 NV features: lane l holds features 4 l .. 4 l + 3 of each group of 256.
template <bool XBF, int RPW, int NV> struct RowPanel {
    using Raw = typename std::conditional<XBF, bf16x4, f32x4>::type;
    Raw x[RPW][NV];
    f32x4 scale[NV], nbias[NV];

    static __device__ __forceinline__ f32x4 floats(const Raw &r) { return f32x4{(float)r[0], (float)r[1], (float)r[2], (float)r[3]}; }
    // rows from r0 on; what lies past the last row or feature is some other, and dropped later
    __device__ __forceinline__ void load(const RowInput &a, int64_t r0, int lane)
    {
        using E = typename std::conditional<XBF, __bf16, float>::type;
#pragma unroll
        for (int j = 0; j < RPW; ++j) {
            const int64_t r = r0 + j < a.rows ? r0 + j : a.rows - 1;
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int c = (i * 64 + lane) * 4;
                x[j][i] = *reinterpret_cast<const Raw *>(static_cast<const E *>(a.x) + r * a.K + (c < a.K ? c : 0));
            }
        }
    }
    __device__ __forceinline__ void load_norm(const RowInput &a, int lane)
    {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = (i * 64 + lane) * 4 < a.K ? (i * 64 + lane) * 4 : 0;
            scale[i] = f32x4{1.f, 1.f, 1.f, 1.f};
            nbias[i] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (a.norm && a.scale) scale[i] = *reinterpret_cast<const f32x4 *>(a.scale + c);
            if (a.norm && a.nbias) nbias[i] = *reinterpret_cast<const f32x4 *>(a.nbias + c);
        }
    }
    // norm(rows) to LDS as T, columns up to kpad (those past K as zero); seen(j, i, c, y): the normalised features.  The rows go through
    // every stage together: their sums over the wave, each a chain of six moves, overlap.
    template <typename T, typename F> __device__ __forceinline__ void finish(const RowInput &a, T *dst, int ld, int kpad, int lane, F seen)
    {
        f32x4 y[RPW][NV];
        auto in = [&](int i) { return (i * 64 + lane) * 4 < a.K; };
#pragma unroll
        for (int j = 0; j < RPW; ++j)
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                y[j][i] = floats(x[j][i]);
                if (!in(i)) y[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        if (a.norm) {
            float s[RPW];
            if (a.norm == 2) {
#pragma unroll
                for (int j = 0; j < RPW; ++j) {
                    s[j] = 0.f;
#pragma unroll
                    for (int i = 0; i < NV; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) s[j] += y[j][i][e];
                }
                wave_totals(s);
#pragma unroll
                for (int j = 0; j < RPW; ++j)
#pragma unroll
                    for (int i = 0; i < NV; ++i)
                        if (in(i))
#pragma unroll
                            for (int e = 0; e < 4; ++e) y[j][i][e] -= s[j] * a.inv_K;
            }
#pragma unroll
            for (int j = 0; j < RPW; ++j) {
                s[j] = 0.f;
#pragma unroll
                for (int i = 0; i < NV; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[j] += y[j][i][e] * y[j][i][e];
            }
            wave_totals(s);
#pragma unroll
            for (int j = 0; j < RPW; ++j) {
                const float rstd = rsqrtf(s[j] * a.inv_K + a.eps);
#pragma unroll
                for (int i = 0; i < NV; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) y[j][i][e] = in(i) ? y[j][i][e] * rstd * scale[i][e] + nbias[i][e] : 0.f;
            }
            if (a.round_norm)
#pragma unroll
                for (int j = 0; j < RPW; ++j)
#pragma unroll
                    for (int i = 0; i < NV; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) y[j][i][e] = (float)(__bf16)y[j][i][e];
        }
#pragma unroll
        for (int j = 0; j < RPW; ++j)
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int c = (i * 64 + lane) * 4;
                if (c >= kpad) continue;
                seen(j, i, c, y[j][i]);
                *reinterpret_cast<typename TT<T>::pack4 *>(dst + j * ld + c) = TT<T>::pack(y[j][i][0], y[j][i][1], y[j][i][2], y[j][i][3]);
            }
    }
};

}  // namespace
}  // namespace mrx
