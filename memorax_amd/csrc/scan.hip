// Diagonal linear-recurrence scan for gfx950:  h_t = done_t ? b_t : a_t h_{t-1} + b_t.
//
// The op is pure streaming (2 loads + 1 store per element forward, 3 + 2 backward),
// so the design is about HBM: lanes lie along the contiguous feature axis
// (one wave row = 64 lanes x 16 B), each lane walks time in registers, and when
// the (batch x feature) extent alone cannot fill 256 CUs the time axis is split
// over the waves of a workgroup: every wave scans its slice from the identity,
// per-wave summaries (P, h, reset-seen) meet in LDS, each wave folds the
// summaries to its left into a carry-in and fixes its slice up by *select*
// (a reset inside the slice wins over the carry, so NaN/Inf never cross a reset).
// One pass over HBM in either case.
// With MG set the kernels take the MinGRU cell's two projections and form a_t, b_t in registers.
#include <initializer_list>
#include <type_traits>

#include "col_sum.h"
#include "common.h"
#include "mingru.h"

namespace {

using namespace mrx;

struct c64 {
    float re, im;
};

template <typename E> struct Ops;
template <> struct Ops<float> {
    static __device__ __forceinline__ float zero() { return 0.0f; }
    static __device__ __forceinline__ float one() { return 1.0f; }
    static __device__ __forceinline__ float conj(float a) { return a; }
    // a * x + y
    static __device__ __forceinline__ float madd(float a, float x, float y) { return a * x + y; }
    static __device__ __forceinline__ float mul(float a, float x) { return a * x; }
};
template <> struct Ops<c64> {
    static __device__ __forceinline__ c64 zero() { return {0.0f, 0.0f}; }
    static __device__ __forceinline__ c64 one() { return {1.0f, 0.0f}; }
    static __device__ __forceinline__ c64 conj(c64 a) { return {a.re, -a.im}; }
    static __device__ __forceinline__ c64 madd(c64 a, c64 x, c64 y)
    {
        return {a.re * x.re - a.im * x.im + y.re, a.re * x.im + a.im * x.re + y.im};
    }
    static __device__ __forceinline__ c64 mul(c64 a, c64 x)
    {
        return {a.re * x.re - a.im * x.im, a.re * x.im + a.im * x.re};
    }
};

// VEC consecutive channels.  Only as aligned as one of them: rows of any width take vectors (see first_col), and the
// device's vector accesses need no more than that.
template <typename E, int VEC> struct Vec {
    E v[VEC];
};

// The same in LDS, where a whole vector moves at once.
template <typename E, int VEC> struct alignas(sizeof(E) * VEC) LdsVec {
    Vec<E, VEC> x;
};

// First of the VEC channels a thread owns when threads are laid along a row: the last thread of a row whose width is no
// multiple of VEC moves back to end with it, i.e. it shares channels with its neighbour -- both compute and write the same
// values.  (One channel per lane instead, the earlier answer to odd widths, halves what a load instruction brings in: bfloat16
// MinGRU forward + backward at 2367 x 36 x 645 494 us, a third of the rate of an even width.)
template <int VEC> __device__ __forceinline__ int64_t first_col(int64_t vec_index, int64_t D)
{
    const int64_t c = vec_index * VEC;
    return c + VEC <= D ? c : D - VEC;
}

template <typename E, int VEC> __device__ __forceinline__ Vec<E, VEC> vfill(E x)
{
    Vec<E, VEC> r;
#pragma unroll
    for (int i = 0; i < VEC; ++i) r.v[i] = x;
    return r;
}

// Every (B,T,D) array is read or written once per launch and not again before the next kernel: its loads and
// stores are non-temporal, so that the stream does not sit in the caches at the expense of itself (measured at
// 512 x 1024 x 1024 float32: forward 5.77 -> 6.05 TB/s, backward 5.74 -> 6.27 TB/s).  The built-ins take
// scalars and vectors of the language, so a Vec or a raw word group goes through a word type of its size.
// AL: the alignment of one element.
template <int BYTES, int AL> struct StreamWord;
#define MRX_STREAM_WORD(AL)                                                                                          \
    template <> struct StreamWord<4, AL> { typedef uint32_t type __attribute__((aligned(AL))); };                      \
    template <> struct StreamWord<8, AL> { typedef uint32_t type __attribute__((ext_vector_type(2), aligned(AL))); };  \
    template <> struct StreamWord<16, AL> { typedef uint32_t type __attribute__((ext_vector_type(4), aligned(AL))); };
template <> struct StreamWord<2, 2> { using type = uint16_t; };
MRX_STREAM_WORD(2)
MRX_STREAM_WORD(4)
#undef MRX_STREAM_WORD
template <typename X, int AL> __device__ __forceinline__ X ld_stream(const void *p)
{
    if constexpr (sizeof(X) <= 16) {
        using W = typename StreamWord<sizeof(X), AL>::type;
        return __builtin_bit_cast(X, __builtin_nontemporal_load(reinterpret_cast<const W *>(p)));
    } else {
        return *reinterpret_cast<const X *>(p);  // wider than one instruction moves (complex64 x 4)
    }
}
template <typename X, int AL> __device__ __forceinline__ void st_stream(void *p, const X &x)
{
    if constexpr (sizeof(X) <= 16) {
        using W = typename StreamWord<sizeof(X), AL>::type;
        __builtin_nontemporal_store(__builtin_bit_cast(W, x), reinterpret_cast<W *>(p));
    } else {
        *reinterpret_cast<X *>(p) = x;
    }
}

// Storage and arithmetic types of the (B,T,D) arrays may differ: bfloat16 in memory, float in registers
// (the carries -- h0, P0, h_last, P_last, g_last, dh0 -- are always in the arithmetic type).
template <typename S, typename E, int VEC> __device__ __forceinline__ Vec<E, VEC> ldv(const S *p)
{
    if constexpr (std::is_same<S, E>::value) {
        return ld_stream<Vec<E, VEC>, alignof(E)>(p);
    } else {
        const Vec<S, VEC> raw = ld_stream<Vec<S, VEC>, alignof(S)>(p);
        Vec<E, VEC> r;
#pragma unroll
        for (int i = 0; i < VEC; ++i) r.v[i] = (E)raw.v[i];
        return r;
    }
}
// The same in two steps, for prefetched values: the load leaves the stored bits in registers and the conversion
// runs where the value is consumed -- arithmetic on a load still in flight makes the wave wait for it, and for
// every load issued before it, in the middle of issuing a group of loads.
// bfloat16 values wait as whole 32-bit words (a structure of 16-bit members would be taken apart, i.e. computed
// on, the moment it arrives); a single one is widened by its load instruction.
template <typename S, int VEC> struct RawVec {
    using type = Vec<S, VEC>;
};
template <int VEC> struct alignas(VEC >= 2 ? 2 * VEC : 4) RawBf16 {
    uint32_t w[VEC >= 2 ? VEC / 2 : 1];
};
template <int VEC> struct RawVec<__bf16, VEC> {
    using type = RawBf16<VEC>;
};
template <typename S, int VEC> using raw_t = typename RawVec<S, VEC>::type;

template <typename S, int VEC> __device__ __forceinline__ raw_t<S, VEC> ldraw(const S *p)
{
    if constexpr (std::is_same<S, __bf16>::value && VEC == 1) {
        raw_t<S, VEC> r;
        r.w[0] = *reinterpret_cast<const uint16_t *>(p);
        return r;
    } else {
        return ld_stream<raw_t<S, VEC>, alignof(S)>(p);
    }
}
template <typename S, typename E, int VEC> __device__ __forceinline__ Vec<E, VEC> cvtv(const raw_t<S, VEC> &raw)
{
    if constexpr (std::is_same<S, E>::value) {
        return raw;
    } else {
        static_assert(std::is_same<S, __bf16>::value && std::is_same<E, float>::value, "bfloat16 storage, float arithmetic");
        Vec<E, VEC> r;
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
            const uint32_t word = raw.w[i >> 1];
            r.v[i] = __builtin_bit_cast(float, (VEC == 1 || !(i & 1)) ? word << 16 : word & 0xffff0000u);
        }
        return r;
    }
}
template <typename S, typename E, int VEC> __device__ __forceinline__ void stv(S *p, const Vec<E, VEC> &x)
{
    if constexpr (std::is_same<S, E>::value) {
        st_stream<Vec<E, VEC>, alignof(E)>(p, x);
    } else {
        Vec<S, VEC> raw;
#pragma unroll
        for (int i = 0; i < VEC; ++i) raw.v[i] = (S)x.v[i];
        st_stream<Vec<S, VEC>, alignof(S)>(p, raw);
    }
}

// The carries (B,D): small, cached.
template <typename E, int VEC> __device__ __forceinline__ Vec<E, VEC> ldc(const E *p)
{
    using W = typename StreamWord<sizeof(E) * VEC, alignof(E)>::type;
    return __builtin_bit_cast(Vec<E, VEC>, W(*reinterpret_cast<const W *>(p)));
}
template <typename E, int VEC> __device__ __forceinline__ void stc(E *p, const Vec<E, VEC> &x)
{
    using W = typename StreamWord<sizeof(E) * VEC, alignof(E)>::type;
    *reinterpret_cast<W *>(p) = __builtin_bit_cast(W, x);
}

// MinGRU in linear space.  The reference scans (log h, log decay) with logaddexp
// (min_gru.py:49-78); the same recurrence is h_t = a_t h_{t-1} + b_t with, from the step's two
// projections z and x = h~:  a = sigma(-z),  b = sigma(z) g(x),  g(x) = x + 0.5 (x >= 0) | sigma(x).
// The kernels below take z and x in place of a and b when MG is set, so the coefficients never
// exist in memory; the backward kernels then emit dz and dx instead of da and db.

// Workgroup barrier that orders LDS traffic only.  __syncthreads() waits for every store of the super-step before and every load on its way,
// which nothing behind the barrier needs.
// PACED: with it, and each super-step's flags waited for before the rest is requested, one step after the other: where half a gigabyte and
// more of float32 streams past, requests that come in a burst from every wave cost the memory more than the waits did (512 x 1024 x 1024 forward
// 1025 paced, 1080 not, backward 1704 and 1744 us; 1024 x 512 x 512 501 and 522).  From 2^27 elements on, and on two or four of them a lane;
// below it costs (200 x 150 x 800 70 and 66 us, 800 x 100 x 600 133 and 127; 1024 x 128 x 256 75 and 76).
template <bool PACED> __device__ __forceinline__ void step_barrier()
{
    if constexpr (PACED) __syncthreads();
    else asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
constexpr int64_t PACED_ELEMENTS = 1ll << 27;

// A row's start, the same for the whole wave, plus a lane's place in it: what one memory instruction adds by itself (plan_scan sees to it
// that a row is less than 4 GB).
template <typename S> __device__ __forceinline__ S *at_bytes(S *row, uint32_t bytes)
{
    using C = typename std::conditional<std::is_const<S>::value, const char, char>::type;
    return reinterpret_cast<S *>(reinterpret_cast<C *>(row) + bytes);
}

constexpr int TS_MIN = 8;  // time steps a wave holds in registers per super-step (template parameter TS of the kernels), at least

// Long sequences over few columns: time is cut into n segments of `steps` steps (a multiple of a super-step), each a workgroup
// of its own.  A first launch (SEG = SUMMARISE) reads the two arrays the recurrence itself needs and leaves every segment's
// composed step -- state from zero, product of the coefficients, "holds a reset" -- in the workspace; the second (SEG = APPLY)
// composes those of the segments before its own into the state it starts from, and does the work.  Twice the reads of two
// arrays, most of them from the last-level cache, against a chain of T / 128 trips to memory that leaves most of the device
// idle.  Backward the same with time reversed.
enum Segmented { WHOLE, SUMMARISE, APPLY };
template <typename E> struct Segments {
    int n, steps;
    E *state, *product;  // (n, B, D)
    int *cut;            // (n, B)
    E *da_parts;         // (n, B, D): da_sum, a segment's share of it
};

// The summaries of the segments before `seg`, composed: each wave takes a contiguous share of them (its loads all in flight at
// once) and leaves its result where a super-step's waves leave theirs, for fold_waves to carry the state through.
template <typename E, int VEC, int MAXSEG>
__device__ __forceinline__ void compose_segments(const Segments<E> &sg, int seg, int64_t bi, int64_t B, int64_t D, int64_t col, bool act, int w,
                                                 int NW, Vec<E, VEC> &hc, Vec<E, VEC> &pc, bool &cut)
{
    using V = Vec<E, VEC>;
    using O = Ops<E>;
    constexpr int PER = MAXSEG / 8;  // NW is 8
    const int per = (seg + NW - 1) / NW, j0 = w * per;
    V hs[PER], ps[PER];
    int fs[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        hs[i] = vfill<E, VEC>(O::zero());
        ps[i] = vfill<E, VEC>(O::one());
        fs[i] = 0;
        if (i < per && j0 + i < seg && act) {
            const int64_t row = (int64_t)(j0 + i) * B + bi;
            hs[i] = ldc<E, VEC>(sg.state + row * D + col);
            ps[i] = ldc<E, VEC>(sg.product + row * D + col);
            fs[i] = sg.cut[row];
        }
    }
    hc = vfill<E, VEC>(O::zero());
    pc = vfill<E, VEC>(O::one());
    cut = false;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const bool f = fs[i] != 0;
        cut |= f;
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            const E hn = O::madd(ps[i].v[k], hc.v[k], hs[i].v[k]);
            const E pn = O::mul(ps[i].v[k], pc.v[k]);
            hc.v[k] = f ? hs[i].v[k] : hn;
            pc.v[k] = f ? ps[i].v[k] : pn;
        }
    }
}
constexpr int MAX_SEGMENTS = 64;

// GATE (MinGRU): the read-out of the block around the recurrence inside the scan, y = h silu(gate) (gate.hip's arithmetic), backward dy in the place of dh
// and the gate's gradient beside the others; and the carry in the cell's logarithms.  What that saves is a pass: forward h is not read back (six bytes an
// element of bfloat16 arrays instead of eight, besides the scan's own), backward dh is neither written nor read, nor h a second time (sixteen instead
// of twenty-two), and four launches over the carries.  1024 x 128 x 256 bfloat16, us, the launches it stands for / one: forward 43 + 31
// + 4 x 4.7 / 77, backward 76 + 55 / 105.  float32, behind 512 MB of other traffic: 157 / 125 and 255 / 189; 512 x 1024 x 512, where the scan by itself is the paced
// kernel, 1256 / 903 and 2210 / 1484.  Where it does not pay: mrx_gated_scan_pays.
// The backward reads the states before the first step and behind the last one (first, last: (B,D)) as the forward leaves them for it, not the carries
// in the caller's hands: those may be overwritten meanwhile, and a state is not what comes back from its logarithm.
template <typename S> struct Gate {
    const S *gate;
    S *y, *dgate;
    float *first, *last;
};
template <typename S, int VEC> __device__ __forceinline__ Vec<float, VEC> gated(const Vec<float, VEC> &h, const raw_t<S, VEC> &gate)
{
    const Vec<float, VEC> g = cvtv<S, float, VEC>(gate);
    Vec<float, VEC> y;
#pragma unroll
    for (int i = 0; i < VEC; ++i) y.v[i] = (float)(S)h.v[i] * g.v[i] * (1.f / (1.f + __expf(-g.v[i])));
    return y;
}
// dy -> dh in place; the gate's gradient
template <typename S, int VEC> __device__ __forceinline__ Vec<float, VEC> gate_grads(Vec<float, VEC> &dy, const Vec<float, VEC> &h, const raw_t<S, VEC> &gate)
{
    const Vec<float, VEC> g = cvtv<S, float, VEC>(gate);
    Vec<float, VEC> dg;
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
        const float sg = 1.f / (1.f + __expf(-g.v[i]));
        dg.v[i] = dy.v[i] * h.v[i] * sg * (1.f + g.v[i] * (1.f - sg));
        dy.v[i] = dy.v[i] * g.v[i] * sg;
    }
    return dg;
}
template <typename E, int VEC, typename F> __device__ __forceinline__ Vec<E, VEC> each(Vec<E, VEC> x, F f)
{
#pragma unroll
    for (int i = 0; i < VEC; ++i) x.v[i] = f(x.v[i]);
    return x;
}
// the gradient of the last state, of its logarithm's (LOG)
template <bool LOG, typename E, int VEC> __device__ __forceinline__ Vec<E, VEC> carry_grad(const E *g, [[maybe_unused]] const float *last, int64_t at)
{
    Vec<E, VEC> x = ldc<E, VEC>(g + at);
    if constexpr (LOG) {
        const Vec<E, VEC> h = ldc<E, VEC>(last + at);
#pragma unroll
        for (int i = 0; i < VEC; ++i) x.v[i] /= h.v[i];
    }
    return x;
}
template <bool LOG, typename E, int VEC> __device__ __forceinline__ Vec<E, VEC> carry_in(const E *p)
{
    const Vec<E, VEC> x = ldc<E, VEC>(p);
    if constexpr (LOG) return each<E, VEC>(x, [](float v) { return expf(v); });
    else return x;
}
template <bool LOG, typename E, int VEC> __device__ __forceinline__ void carry_out(E *p, const Vec<E, VEC> &x)
{
    if constexpr (LOG) stc<E, VEC>(p, each<E, VEC>(x, [](float v) { return logf(v); }));
    else stc<E, VEC>(p, x);
}

// Forward.  grid = B * tiles workgroups (times the segments), block = 64 * NW threads, NW <= MAXW (8, or 16 for the
// one-vector-lane instances that small shapes take: with 16 waves of 8 steps a sequence of up to 128
// steps is one super-step, every load of the workgroup in flight at once and a single barrier).
// smem: sH[2][NW][64] Vec, sP[2][NW][64] Vec, sF[2][NW] int.
template <typename E, int VEC, bool MG = false, int MAXW = 8, typename S = E, int TS = TS_MIN, int SEG = WHOLE, bool ATI = false, bool PACED = false, bool GATE = false>
__global__ void __launch_bounds__(64 * MAXW, sizeof(E) == 8 && VEC == 1 ? 4 : 1)   // (two eight-wave workgroups of single complex elements a compute unit)
diag_scan_fwd_kernel(const S *__restrict__ a, const S *__restrict__ b,
                     const void *__restrict__ done, int done_f32,
                     const E *__restrict__ h0, const E *__restrict__ P0,
                     S *__restrict__ h, E *__restrict__ h_last,
                     E *__restrict__ P_last, int T, int64_t D, int tiles, int NW,
                     int a_ti, Segments<E> sg, Gate<S> gt)
{
    using V = Vec<E, VEC>;
    using O = Ops<E>;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    using L = LdsVec<E, VEC>;
    L *sH = reinterpret_cast<L *>(smem_raw);
    L *sP = sH + 2 * NW * 64;
    int *sF = reinterpret_cast<int *>(sP + 2 * NW * 64);

    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tile = blockIdx.x % tiles;
    const int64_t bs = blockIdx.x / tiles;
    const int64_t bi = SEG == WHOLE ? bs : bs / sg.n;
    const int seg = SEG == WHOLE ? 0 : (int)(bs % sg.n);
    [[maybe_unused]] const int64_t B = SEG == WHOLE ? 0 : (int64_t)gridDim.x / ((int64_t)tiles * sg.n);
    const int t_begin = SEG == WHOLE ? 0 : seg * sg.steps, t_end = SEG == WHOLE || T - t_begin <= sg.steps ? T : t_begin + sg.steps;
    const bool act = ((int64_t)tile * 64 + lane) * VEC < D;
    const int64_t col = first_col<VEC>((int64_t)tile * 64 + lane, D);
    const int64_t row0 = bi * T;
    const uint32_t col_bytes = (uint32_t)col * (uint32_t)sizeof(S);
    constexpr bool SKIP = std::is_same<S, E>::value && (SEG == WHOLE || sizeof(E) == 8);   // (narrower storage: the branch costs a quarter more registers)

    V carry_h = vfill<E, VEC>(O::zero()), carry_p = vfill<E, VEC>(O::one());
    if (act && SEG != SUMMARISE) {
        if (h0) carry_h = carry_in<GATE, E, VEC>(h0 + bi * D + col);
        if constexpr (GATE)
            if (gt.first && w == 0) stc<E, VEC>(gt.first + bi * D + col, carry_h);
        if (P0) carry_p = carry_in<GATE, E, VEC>(P0 + bi * D + col);
    }

    int buf = 0;
    [[maybe_unused]] bool seg_cut = false;
    if constexpr (SEG == APPLY) {
        V hc, pc;
        bool cut;
        compose_segments<E, VEC, MAX_SEGMENTS>(sg, seg, bi, B, D, col, act, w, NW, hc, pc, cut);
        sH[w * 64 + lane].x = hc;
        sP[w * 64 + lane].x = pc;
        if (lane == 0) sF[w] = cut;
        step_barrier<PACED>();
        for (int j = 0; j < NW; ++j) {
            const V Hj = sH[j * 64 + lane].x, Pj = sP[j * 64 + lane].x;
            const bool fj = sF[j] != 0;
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                const E hn = O::madd(Pj.v[i], carry_h.v[i], Hj.v[i]);
                const E pn = O::mul(Pj.v[i], carry_p.v[i]);
                carry_h.v[i] = fj ? Hj.v[i] : hn;
                carry_p.v[i] = fj ? Pj.v[i] : pn;
            }
        }
        buf = 1;
    }
    [[maybe_unused]] V p_all;   // a broadcast coefficient
    if constexpr (ATI) p_all = ldv<S, E, VEC>(a + col);
    const int span = NW * TS;
    for (int t0 = t_begin; t0 < t_end; t0 += span) {
        const int ts = t0 + w * TS;
        V x[TS], p[TS];
        [[maybe_unused]] raw_t<S, VEC> rg[GATE ? TS : 1];
        // Everything is requested before anything is used, without branches: steps past the last read the last, lanes past the row its
        // last channels.  Reset flags of the wave's TS steps: lane s fetches the flag of step ts + s, one ballot makes the mask.
        uint32_t flag = 0;
        auto row_of = [&](int s) { return row0 + (ts + s < T ? ts + s : T - 1); };
        auto a_at = [&](int s) { return at_bytes(a + (a_ti ? 0 : row_of(s) * D), col_bytes); };
        auto b_at = [&](int s) { return at_bytes(b + row_of(s) * D, col_bytes); };
        unsigned rmask = 0;
        auto form_mask = [&]() { rmask = (unsigned)__ballot(lane < TS && ts + lane < T && done_test(flag, done_f32)); };
        if constexpr (PACED) {
            flag = done_raw(done, done_f32, row_of(lane & (TS - 1)));
            form_mask();
            raw_t<S, VEC> rp[TS], rx[TS];   // (loads into registers of their own: into p and x the 512 x 1024 x 1024 call took 1045 us instead of 1027)
#pragma unroll
            for (int s = 0; s < TS; ++s) {
                if (ts + s < T && act) {
                    const int64_t off = (row0 + ts + s) * D + col;
                    rp[s] = ldraw<S, VEC>(a + (a_ti ? col : off));
                    rx[s] = ldraw<S, VEC>(b + off);
                }
            }
#pragma unroll
            for (int s = 0; s < TS; ++s) {
                const bool in = ts + s < T && act;
                p[s] = in ? cvtv<S, E, VEC>(rp[s]) : vfill<E, VEC>(O::one());
                x[s] = in ? cvtv<S, E, VEC>(rx[s]) : vfill<E, VEC>(O::zero());
            }
        } else {
            if (ts < T || !SKIP) {   // (a wave past the end requests nothing)
                flag = done_raw(done, done_f32, row_of(lane));   // with those of the super-steps to come in tow
                if constexpr (std::is_same<S, E>::value) {
#pragma unroll
                    for (int s = 0; s < TS; ++s) {
                        if constexpr (ATI) p[s] = p_all;
                        else p[s] = ldv<S, E, VEC>(a_at(s));
                        x[s] = ldv<S, E, VEC>(b_at(s));
                        if constexpr (GATE) rg[s] = ldraw<S, VEC>(at_bytes(gt.gate + row_of(s) * D, col_bytes));
                    }
                } else {
                    raw_t<S, VEC> rp[TS], rx[TS];  // as stored; converted once every load of the super-step has been issued
#pragma unroll
                    for (int s = 0; s < TS; ++s) {
                        rp[s] = ldraw<S, VEC>(a_at(s));
                        rx[s] = ldraw<S, VEC>(b_at(s));
                    }
                    if constexpr (GATE)
#pragma unroll
                        for (int s = 0; s < TS; ++s) rg[s] = ldraw<S, VEC>(at_bytes(gt.gate + row_of(s) * D, col_bytes));
#pragma unroll
                    for (int s = 0; s < TS; ++s) p[s] = cvtv<S, E, VEC>(rp[s]), x[s] = cvtv<S, E, VEC>(rx[s]);
                }
            }
            form_mask();
            if (ts + TS > T) {
#pragma unroll
                for (int s = 0; s < TS; ++s)
                    if (ts + s >= T) p[s] = vfill<E, VEC>(O::one()), x[s] = vfill<E, VEC>(O::zero());
            }
        }
        if constexpr (MG) {  // after every load of the super-step has been issued
#pragma unroll
            for (int s = 0; s < TS; ++s) {
                if (ts + s < T && act) {
#pragma unroll
                    for (int i = 0; i < VEC; ++i) MinGru::coeffs(p[s].v[i], x[s].v[i]);
                }
            }
        }
        if (NW == 1) {
            // no time split: continue straight from the carry
#pragma unroll
            for (int s = 0; s < TS; ++s) {
                const bool r = (rmask >> s) & 1u;
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    const E hn = O::madd(p[s].v[i], carry_h.v[i], x[s].v[i]);
                    const E pn = O::mul(p[s].v[i], carry_p.v[i]);
                    carry_h.v[i] = r ? x[s].v[i] : hn;
                    carry_p.v[i] = r ? p[s].v[i] : pn;
                }
                if (ts + s < T && act) {
                    stv<S, E, VEC>(at_bytes(h + (row0 + ts + s) * D, col_bytes), carry_h);
                    if constexpr (GATE) stv<S, E, VEC>(at_bytes(gt.y + (row0 + ts + s) * D, col_bytes), gated<S, VEC>(carry_h, rg[s]));
                }
            }
            continue;
        }
        // local inclusive scan from the identity; x <- h_local, p <- P_local
        {
            V hc = vfill<E, VEC>(O::zero()), pc = vfill<E, VEC>(O::one());
#pragma unroll
            for (int s = 0; s < TS; ++s) {
                const bool r = (rmask >> s) & 1u;
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    const E hn = O::madd(p[s].v[i], hc.v[i], x[s].v[i]);
                    const E pn = O::mul(p[s].v[i], pc.v[i]);
                    hc.v[i] = r ? x[s].v[i] : hn;
                    pc.v[i] = r ? p[s].v[i] : pn;
                }
                x[s] = hc;
                p[s] = pc;
            }
            sH[(buf * NW + w) * 64 + lane].x = hc;
            sP[(buf * NW + w) * 64 + lane].x = pc;
            if (lane == 0) sF[buf * NW + w] = rmask != 0;
        }
        step_barrier<PACED>();
        // fold the summaries: carry-in of this wave, then the workgroup carry
        V cin_h = carry_h, cin_p = carry_p, my_h = carry_h;
        for (int j = 0; j < NW; ++j) {
            if (j == w) my_h = cin_h;
            const V Hj = sH[(buf * NW + j) * 64 + lane].x;
            const V Pj = sP[(buf * NW + j) * 64 + lane].x;
            const bool fj = sF[buf * NW + j] != 0;
            if constexpr (SEG == SUMMARISE) seg_cut |= fj;
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                const E hn = O::madd(Pj.v[i], cin_h.v[i], Hj.v[i]);
                const E pn = O::mul(Pj.v[i], cin_p.v[i]);
                cin_h.v[i] = fj ? Hj.v[i] : hn;
                cin_p.v[i] = fj ? Pj.v[i] : pn;
            }
        }
        carry_h = cin_h;
        carry_p = cin_p;
#pragma unroll
        for (int s = 0; s < TS; ++s) {
            const bool seen = (rmask & ((2u << s) - 1u)) != 0;
            V out;
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                const E fx = O::madd(p[s].v[i], my_h.v[i], x[s].v[i]);
                out.v[i] = seen ? x[s].v[i] : fx;
            }
            if (SEG != SUMMARISE && ts + s < T && act) {
                stv<S, E, VEC>(at_bytes(h + (row0 + ts + s) * D, col_bytes), out);
                if constexpr (GATE) stv<S, E, VEC>(at_bytes(gt.y + (row0 + ts + s) * D, col_bytes), gated<S, VEC>(out, rg[s]));
            }
        }
        buf ^= 1;
    }
    if constexpr (SEG == SUMMARISE) {
        if (w == 0 && act) {
            const int64_t row = (int64_t)seg * B + bi;
            stc<E, VEC>(sg.state + row * D + col, carry_h);
            stc<E, VEC>(sg.product + row * D + col, carry_p);
            if (lane == 0) sg.cut[row] = seg_cut;
        }
        return;
    }
    if (w == 0 && act && t_end == T) {
        if (h_last) carry_out<GATE, E, VEC>(h_last + bi * D + col, carry_h);
        if constexpr (GATE)
            if (gt.last) stc<E, VEC>(gt.last + bi * D + col, carry_h);
        if (P_last) carry_out<GATE, E, VEC>(P_last + bi * D + col, carry_p);
    }
}

// Backward: the same scan walked from t = T-1 down with coefficient conj(a_{t+1}),
// cut where done_{t+1}; reversed index r = T-1-t runs forward.
// MG: a holds z, hx holds x = h~; da receives dz and db receives dx.
template <typename E, int VEC, bool MG = false, int MAXW = 8, typename S = E, int TS = TS_MIN, int SEG = WHOLE, bool ATI = false, bool PACED = false, bool GATE = false>
__global__ void __launch_bounds__(64 * MAXW)
diag_scan_bwd_kernel(const S *__restrict__ a, const S *__restrict__ hx, const S *__restrict__ hfw,
                     const void *__restrict__ done, int done_f32,
                     const E *__restrict__ h0, const S *__restrict__ g,
                     const E *__restrict__ g_last, S *__restrict__ da,
                     S *__restrict__ db, E *__restrict__ dh0, int T, int64_t D,
                     int tiles, int NW, int a_ti, int da_sum, Segments<E> sg, Gate<S> gt)
{
    using V = Vec<E, VEC>;
    using O = Ops<E>;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    using L = LdsVec<E, VEC>;
    L *sH = reinterpret_cast<L *>(smem_raw);
    L *sP = sH + 2 * NW * 64;
    int *sF = reinterpret_cast<int *>(sP + 2 * NW * 64);

    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tile = blockIdx.x % tiles;
    const int64_t bs = blockIdx.x / tiles;
    const int64_t bi = SEG == WHOLE ? bs : bs / sg.n;
    const int seg = SEG == WHOLE ? 0 : (int)(bs % sg.n);
    [[maybe_unused]] const int64_t B = SEG == WHOLE ? 0 : (int64_t)gridDim.x / ((int64_t)tiles * sg.n);
    const int r_begin = SEG == WHOLE ? 0 : seg * sg.steps, r_end = SEG == WHOLE || T - r_begin <= sg.steps ? T : r_begin + sg.steps;
    const bool act = ((int64_t)tile * 64 + lane) * VEC < D;
    const int64_t col = first_col<VEC>((int64_t)tile * 64 + lane, D);
    const int64_t row0 = bi * T;
    const uint32_t col_bytes = (uint32_t)col * (uint32_t)sizeof(S);
    constexpr bool SKIP = std::is_same<S, E>::value && (SEG == WHOLE || sizeof(E) == 8);

    constexpr bool ONCE = GATE;   // z_{t+1} of a step is the z_t of the one before: read once

    V carry = vfill<E, VEC>(O::zero());  // lam_{t+1} entering from the right
    if (act && g_last && SEG != SUMMARISE) carry = carry_grad<GATE, E, VEC>(g_last, gt.last, bi * D + col);
    // da_sum (time-invariant a): da is (B,D), the sum of the per-step terms over the sequence -- what the
    // gradient of a broadcast coefficient needs -- kept in registers instead of written per step
    V dsum = vfill<E, VEC>(O::zero());

    [[maybe_unused]] V seg_p = vfill<E, VEC>(O::one());
    [[maybe_unused]] bool seg_cut = false;
    int buf = 0;
    if constexpr (SEG == APPLY) {
        V lc, pc;
        bool cut;
        compose_segments<E, VEC, MAX_SEGMENTS>(sg, seg, bi, B, D, col, act, w, NW, lc, pc, cut);
        sH[w * 64 + lane].x = lc;
        sP[w * 64 + lane].x = pc;
        if (lane == 0) sF[w] = cut;
        step_barrier<PACED>();
        for (int j = 0; j < NW; ++j) {
            const V Hj = sH[j * 64 + lane].x, Pj = sP[j * 64 + lane].x;
            const bool fj = sF[j] != 0;
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                const E ln = O::madd(Pj.v[i], carry.v[i], Hj.v[i]);
                carry.v[i] = fj ? Hj.v[i] : ln;
            }
        }
        buf = 1;
    }
    [[maybe_unused]] V h0v = vfill<E, VEC>(O::zero());   // h_{-1}: what step 0 multiplies its lam with
    if (SEG != SUMMARISE && h0) h0v = ldc<E, VEC>(h0 + bi * D + col);
    [[maybe_unused]] V p_all;                            // a broadcast coefficient
    if constexpr (ATI) {
        p_all = ldv<S, E, VEC>(a + col);
#pragma unroll
        for (int i = 0; i < VEC; ++i) p_all.v[i] = O::conj(p_all.v[i]);
    }
    const int span = NW * TS;
    for (int r0 = r_begin; r0 < r_end; r0 += span) {
        const int rs = r0 + w * TS;
        // Everything the super-step reads is requested here, before the barrier: h_{t-1} (and the
        // MinGRU projections of step t) are only needed once lam_t is known, but a load issued after the
        // barrier would be a second trip to memory on the critical path.
        V x[TS], p[TS], hp[TS];
        V zt[MG ? TS : 1], xt[MG ? TS : 1];
        [[maybe_unused]] raw_t<S, VEC> rgt[GATE ? TS : 1], rtop;   // gates, and the state of the wave's last step
        // Steps before the sequence's first read the first, as lanes past the row read its last channels: no branch between the requests.
        // Reset flags: step s of the wave is t_s = T - 1 - (rs + s); lane l fetches done at T - rs - l, i.e.
        // done_{t_0 + 1}, done_{t_0}, done_{t_1}, ..., and one ballot serves both masks (steps before the
        // sequence's first, t_s < 0, take no bit: a cut there would drop the carry on its way to dh0)
        auto t_of = [&](int s) { return T - 1 - (rs + s); };
        auto row_of = [&](int t) { return (row0 + (t < 0 ? 0 : t >= T ? T - 1 : t)) * D; };
        const int tt = T - rs - (PACED && lane > TS ? TS : lane);
        const uint32_t flag = done_raw(done, done_f32, row0 + (tt < 0 ? 0 : tt >= T ? T - 1 : tt));
        unsigned cmask = 0, dmask = 0;  // bit s: chain cut between step t_s and t_s + 1 (done_{t_s + 1}) / done_{t_s}
        auto form_masks = [&]() {
            const unsigned fl = (unsigned)__ballot(lane <= TS && tt >= 0 && tt < T && done_test(flag, done_f32));
            const int nv = T - rs < TS ? (T - rs < 0 ? 0 : T - rs) : TS;  // steps of the wave inside the sequence
            const unsigned vm = (1u << nv) - 1u;
            cmask = fl & vm;
            dmask = (fl >> 1) & vm;
        };
        if (PACED) form_masks();
        if (rs < T || !SKIP) {   // (a wave past the end requests nothing)
            if constexpr (std::is_same<S, E>::value) {
#pragma unroll
                for (int s = 0; s < TS; ++s) {
                    const int t = t_of(s);
                    if (PACED && !(t >= 0 && act)) continue;
                    x[s] = ldv<S, E, VEC>(at_bytes(g + row_of(t), col_bytes));
                    if constexpr (GATE) {
                        rgt[s] = ldraw<S, VEC>(at_bytes(gt.gate + row_of(t), col_bytes));
                        if (s == 0) rtop = ldraw<S, VEC>(at_bytes(hfw + row_of(t), col_bytes));
                    }
                    if constexpr (ATI) p[s] = p_all;
                    else if (!ONCE || !s) p[s] = ldv<S, E, VEC>(at_bytes(a + (a_ti ? 0 : row_of(t + 1)), col_bytes));
                    if constexpr (SEG != SUMMARISE) {
                        hp[s] = ldv<S, E, VEC>(at_bytes(hfw + row_of(t - 1), col_bytes));
                        if constexpr (MG) {
                            zt[s] = ldv<S, E, VEC>(at_bytes(a + row_of(t), col_bytes));
                            xt[s] = ldv<S, E, VEC>(at_bytes(hx + row_of(t), col_bytes));
                        }
                    }
                }
            } else {
                // narrower storage: the values wait as stored and are widened once every load has been issued
                raw_t<S, VEC> rg[TS], ra[TS], rh[TS], rz[MG ? TS : 1], rxt[MG ? TS : 1];
#pragma unroll
                for (int s = 0; s < TS; ++s) {
                    const int t = t_of(s);
                    rg[s] = ldraw<S, VEC>(at_bytes(g + row_of(t), col_bytes));
                    if constexpr (GATE) {
                        rgt[s] = ldraw<S, VEC>(at_bytes(gt.gate + row_of(t), col_bytes));
                        if (s == 0) rtop = ldraw<S, VEC>(at_bytes(hfw + row_of(t), col_bytes));
                    }
                    if (!ONCE || !s) ra[s] = ldraw<S, VEC>(at_bytes(a + (a_ti ? 0 : row_of(t + 1)), col_bytes));
                    if constexpr (SEG != SUMMARISE) {
                        rh[s] = ldraw<S, VEC>(at_bytes(hfw + row_of(t - 1), col_bytes));
                        if constexpr (MG) {
                            rz[s] = ldraw<S, VEC>(at_bytes(a + row_of(t), col_bytes));
                            rxt[s] = ldraw<S, VEC>(at_bytes(hx + row_of(t), col_bytes));
                        }
                    }
                }
#pragma unroll
                for (int s = 0; s < TS; ++s) {
                    x[s] = cvtv<S, E, VEC>(rg[s]);
                    if (!ONCE || !s) p[s] = cvtv<S, E, VEC>(ra[s]);
                    if constexpr (SEG != SUMMARISE) {
                        hp[s] = cvtv<S, E, VEC>(rh[s]);
                        if constexpr (MG) {
                            zt[s] = cvtv<S, E, VEC>(rz[s]);
                            xt[s] = cvtv<S, E, VEC>(rxt[s]);
                        }
                    }
                }
            }
        }
        if (!PACED) form_masks();
        if constexpr (ONCE) {
#pragma unroll
            for (int s = 1; s < TS; ++s) p[s] = zt[s - 1];
        }
        if constexpr (GATE) {   // the state of a step is what the step behind it starts from
#pragma unroll
            for (int s = 0; s < TS; ++s) {
                const V dg = gate_grads<S, VEC>(x[s], s ? hp[s ? s - 1 : 0] : cvtv<S, E, VEC>(rtop), rgt[s]);
                if (t_of(s) >= 0 && act) stv<S, E, VEC>(at_bytes(gt.dgate + row_of(t_of(s)), col_bytes), dg);
            }
        }
        if constexpr (!MG && !ATI) {
#pragma unroll
            for (int s = 0; s < TS; ++s)
#pragma unroll
                for (int i = 0; i < VEC; ++i) p[s].v[i] = O::conj(p[s].v[i]);   // MG: z_{t+1} for now
        }
        if (rs == 0) p[0] = vfill<E, VEC>(O::one());   // nothing follows the last step
        if (rs + TS >= T) {   // the sequence's first step, and what would come before it
#pragma unroll
            for (int s = 0; s < TS; ++s) {
                const int t = t_of(s);
                if (t == 0 && SEG != SUMMARISE) hp[s] = h0v;
                if (t < 0) {
                    p[s] = vfill<E, VEC>(O::one());
                    x[s] = vfill<E, VEC>(O::zero());
                    hp[s] = vfill<E, VEC>(O::zero());
                }
            }
        }
        if constexpr (MG) {  // a_{t+1} = sigma(-z_{t+1}), after every load of the super-step has been issued
#pragma unroll
            for (int s = 0; s < TS; ++s) {
                const int t = T - 1 - (rs + s);
                if (t >= 0 && t + 1 < T && act) {
#pragma unroll
                    for (int i = 0; i < VEC; ++i) {
                        float sg;
                        MinGru::gates(p[s].v[i], sg, p[s].v[i]);
                    }
                }
            }
        }
        V my = carry;
        if (NW == 1) {
#pragma unroll
            for (int s = 0; s < TS; ++s) {
                const bool c = (cmask >> s) & 1u;
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    const E ln = O::madd(p[s].v[i], carry.v[i], x[s].v[i]);
                    carry.v[i] = c ? x[s].v[i] : ln;
                }
                x[s] = carry;
            }
        } else {
            V lc = vfill<E, VEC>(O::zero()), pc = vfill<E, VEC>(O::one());
#pragma unroll
            for (int s = 0; s < TS; ++s) {
                const bool c = (cmask >> s) & 1u;
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    const E ln = O::madd(p[s].v[i], lc.v[i], x[s].v[i]);
                    const E pn = O::mul(p[s].v[i], pc.v[i]);
                    lc.v[i] = c ? x[s].v[i] : ln;
                    pc.v[i] = c ? p[s].v[i] : pn;
                }
                x[s] = lc;
                p[s] = pc;
            }
            sH[(buf * NW + w) * 64 + lane].x = lc;
            sP[(buf * NW + w) * 64 + lane].x = pc;
            if (lane == 0) sF[buf * NW + w] = cmask != 0;
            step_barrier<PACED>();
            V cin = carry;
            for (int j = 0; j < NW; ++j) {
                if (j == w) my = cin;
                const V Hj = sH[(buf * NW + j) * 64 + lane].x;
                const V Pj = sP[(buf * NW + j) * 64 + lane].x;
                const bool fj = sF[buf * NW + j] != 0;
                if constexpr (SEG == SUMMARISE) seg_cut |= fj;
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    const E ln = O::madd(Pj.v[i], cin.v[i], Hj.v[i]);
                    cin.v[i] = fj ? Hj.v[i] : ln;
                    if constexpr (SEG == SUMMARISE) {
                        const E pn = O::mul(Pj.v[i], seg_p.v[i]);
                        seg_p.v[i] = fj ? Pj.v[i] : pn;
                    }
                }
            }
            carry = cin;
#pragma unroll
            for (int s = 0; s < TS; ++s) {
                const bool seen = (cmask & ((2u << s) - 1u)) != 0;
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    const E fx = O::madd(p[s].v[i], my.v[i], x[s].v[i]);
                    x[s].v[i] = seen ? x[s].v[i] : fx;
                }
            }
            buf ^= 1;
        }
        if constexpr (SEG == SUMMARISE) continue;
        // x[s] = lam_t : emit db_t and da_t = done_t ? 0 : lam_t conj(h_{t-1})
#pragma unroll
        for (int s = 0; s < TS; ++s) {
            const int t = T - 1 - (rs + s);
            if (t >= 0 && act) {
                const int64_t off = (row0 + t) * D + col;
                const bool dn = (dmask >> s) & 1u;
                V o;
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    const E prod = O::mul(x[s].v[i], O::conj(hp[s].v[i]));
                    o.v[i] = dn ? O::zero() : prod;
                }
                if constexpr (MG) {
                    V oz, ox;
#pragma unroll
                    for (int i = 0; i < VEC; ++i) MinGru::grads(zt[s].v[i], xt[s].v[i], x[s].v[i], o.v[i], oz.v[i], ox.v[i]);
                    stv<S, E, VEC>(db + off, ox);
                    stv<S, E, VEC>(da + off, oz);
                } else {
                    stv<S, E, VEC>(db + off, x[s]);
                    if (da_sum) {
#pragma unroll
                        for (int i = 0; i < VEC; ++i) dsum.v[i] = O::madd(O::one(), dsum.v[i], o.v[i]);
                    } else {
                        stv<S, E, VEC>(da + off, o);
                    }
                }
            }
        }
    }
    if constexpr (SEG == SUMMARISE) {
        if (w == 0 && act) {
            const int64_t row = (int64_t)seg * B + bi;
            stc<E, VEC>(sg.state + row * D + col, carry);
            stc<E, VEC>(sg.product + row * D + col, seg_p);
            if (lane == 0) sg.cut[row] = seg_cut;
        }
        return;
    }
    if (!MG && da_sum) {  // uniform over the workgroup
        if (NW > 1) {
            step_barrier<PACED>();  // the last fold has read sH
            sH[w * 64 + lane].x = dsum;
            step_barrier<PACED>();
            if (w == 0) {
                for (int j = 1; j < NW; ++j) {
                    const V dj = sH[j * 64 + lane].x;
#pragma unroll
                    for (int i = 0; i < VEC; ++i) dsum.v[i] = O::madd(O::one(), dsum.v[i], dj.v[i]);
                }
            }
        }
        E *const sum = SEG == APPLY ? sg.da_parts + (int64_t)seg * B * D : reinterpret_cast<E *>(da);  // (B,D), arithmetic type
        if (w == 0 && act) stc<E, VEC>(sum + bi * D + col, dsum);
    }
    if (w == 0 && act && dh0 && r_end == T) {
        // carry = lam_0 ; dh0 = done_0 ? 0 : conj(a_0) lam_0
        const bool d0 = done_at(done, done_f32, row0);
        V a0 = ldv<S, E, VEC>(a + (a_ti ? col : row0 * D + col));
        if constexpr (MG) {
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                float sg;
                MinGru::gates(a0.v[i], sg, a0.v[i]);
            }
        }
        V o;
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
            const E prod = O::mul(O::conj(a0.v[i]), carry.v[i]);
            o.v[i] = d0 ? O::zero() : prod;
            if constexpr (GATE) o.v[i] *= h0v.v[i];   // of its logarithm
        }
        stc<E, VEC>(dh0 + bi * D + col, o);
    }
}


// ---- streaming kernels: enough (batch x feature) columns to fill the chip ------------
// No time split.  Each lane walks all of T for its VEC channels in groups of SG steps,
// with the loads of the next group issued before the current group is consumed
// (register double buffering), so a wave always has 2*SG (forward) / 3*SG (backward)
// row loads in flight.  done flags are prefetched as raw bits with the data.
template <typename E, int VEC, int SG, bool MG = false, typename S = E, bool DF = false, bool GATE = false>
__global__ void __launch_bounds__(256)
diag_scan_fwd_stream_kernel(const S *__restrict__ a, const S *__restrict__ b,
                            const void *__restrict__ done, int,
                            const E *__restrict__ h0, const E *__restrict__ P0,
                            S *__restrict__ h, E *__restrict__ h_last, E *__restrict__ P_last,
                            int64_t B, int T, int64_t D, int64_t cols_per_row, int a_ti, Gate<S> gt)
{
    using V = Vec<E, VEC>;
    using O = Ops<E>;
    // the flags' type is a template parameter here: with both kinds of load in the code the compiler reuses
    // registers of loads still in flight for the other kind's address and waits for them in mid-prefetch
    constexpr int done_f32 = DF;
    // one thread per VEC channels of one batch row
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t bi = gid / cols_per_row;
    const int64_t col = first_col<VEC>(gid % cols_per_row, D);
    if (bi >= B) return;  // padding threads of the last workgroup (this kernel has no barriers)
    const int64_t row0 = bi * T;
    V ch = vfill<E, VEC>(O::zero()), cp = vfill<E, VEC>(O::one());
    if (h0) ch = carry_in<GATE, E, VEC>(h0 + bi * D + col);
    if constexpr (GATE)
        if (gt.first) stc<E, VEC>(gt.first + bi * D + col, ch);
    if (P0) cp = carry_in<GATE, E, VEC>(P0 + bi * D + col);

    using R = raw_t<S, VEC>;  // prefetched values stay as stored until they are consumed
    R xa[SG], xb[SG], na[SG], nb[SG];
    [[maybe_unused]] R xg[GATE ? SG : 1], ng[GATE ? SG : 1];
    uint32_t xd[SG], nd[SG];
    auto load = [&](int t0, R *pa, R *pb, [[maybe_unused]] R *pg, uint32_t *pd) {
#pragma unroll
        for (int s = 0; s < SG; ++s) {
            const int t = t0 + s;
            pd[s] = 0u;
            if (t < T) {
                const int64_t off = (row0 + t) * D + col;
                pa[s] = ldraw<S, VEC>(a + (a_ti ? col : off));
                pb[s] = ldraw<S, VEC>(b + off);
                if constexpr (GATE) pg[s] = ldraw<S, VEC>(gt.gate + off);
                pd[s] = done_raw(done, done_f32, row0 + t);
            }
        }
    };
    load(0, xa, xb, xg, xd);
    for (int t0 = 0; t0 < T; t0 += SG) {
        if (t0 + SG < T) load(t0 + SG, na, nb, ng, nd);
#pragma unroll
        for (int s = 0; s < SG; ++s) {
            if (t0 + s < T) {
                const bool r = done_test(xd[s], done_f32);
                V va = cvtv<S, E, VEC>(xa[s]), vb = cvtv<S, E, VEC>(xb[s]);
                if constexpr (MG) {  // here, not at the load: the loads stay in flight
#pragma unroll
                    for (int i = 0; i < VEC; ++i) MinGru::coeffs(va.v[i], vb.v[i]);
                }
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    const E hn = O::madd(va.v[i], ch.v[i], vb.v[i]);
                    const E pn = O::mul(va.v[i], cp.v[i]);
                    ch.v[i] = r ? vb.v[i] : hn;
                    cp.v[i] = r ? va.v[i] : pn;
                }
                stv<S, E, VEC>(h + (row0 + t0 + s) * D + col, ch);
                if constexpr (GATE) stv<S, E, VEC>(gt.y + (row0 + t0 + s) * D + col, gated<S, VEC>(ch, xg[s]));
            }
        }
#pragma unroll
        for (int s = 0; s < SG; ++s) { xa[s] = na[s]; xb[s] = nb[s]; xd[s] = nd[s]; }
        if constexpr (GATE)
#pragma unroll
            for (int s = 0; s < SG; ++s) xg[s] = ng[s];
    }
    if (h_last) carry_out<GATE, E, VEC>(h_last + bi * D + col, ch);
    if constexpr (GATE)
        if (gt.last) stc<E, VEC>(gt.last + bi * D + col, ch);
    if (P_last) carry_out<GATE, E, VEC>(P_last + bi * D + col, cp);
}

// ---- final state only, decay shared by groups of channels ---------------------------
// h_T of h_t = done_t ? b_t : a_t h_{t-1} + b_t where a:(B,T,D/a_group) holds one decay per
// a_group consecutive channels.  Nothing but the last state is written, so the traffic is one
// read of b.  This is the real-time-recurrent-learning sensitivity update
// (memoroid.py:114-141: S <- last(scan(a = where(done, 0, repeat(decay, param_size)), J))),
// without materialising the repeated decay or the per-step states.
template <typename E, int VEC, int SG>
__global__ void __launch_bounds__(256)
diag_scan_last_kernel(const E *__restrict__ a, const E *__restrict__ b, const void *__restrict__ done,
                      int done_f32, const E *__restrict__ h0, E *__restrict__ h_last, int64_t B, int T,
                      int64_t D, int64_t cols_per_row, int64_t a_group)
{
    using V = Vec<E, VEC>;
    using O = Ops<E>;
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t bi = gid / cols_per_row;
    const int64_t col = (gid % cols_per_row) * VEC;
    if (bi >= B) return;  // padding threads of the last workgroup (this kernel has no barriers)
    const int64_t row0 = bi * T, Da = D / a_group, acol = col / a_group;  // VEC divides a_group
    V ch = vfill<E, VEC>(O::zero());
    if (h0) ch = ldc<E, VEC>(h0 + bi * D + col);

    E xa[SG], na[SG];
    V xb[SG], nb[SG];
    uint32_t xd[SG], nd[SG];
    auto load = [&](int t0, E *pa, V *pb, uint32_t *pd) {
#pragma unroll
        for (int s = 0; s < SG; ++s) {
            const int t = t0 + s;
            pd[s] = 0u;
            if (t < T) {
                pa[s] = a[(row0 + t) * Da + acol];
                pb[s] = ldc<E, VEC>(b + (row0 + t) * D + col);
                pd[s] = done_raw(done, done_f32, row0 + t);
            }
        }
    };
    load(0, xa, xb, xd);
    for (int t0 = 0; t0 < T; t0 += SG) {
        if (t0 + SG < T) load(t0 + SG, na, nb, nd);
#pragma unroll
        for (int s = 0; s < SG; ++s) {
            if (t0 + s < T) {
                const bool r = done_test(xd[s], done_f32);
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    const E hn = O::madd(xa[s], ch.v[i], xb[s].v[i]);
                    ch.v[i] = r ? xb[s].v[i] : hn;
                }
            }
        }
#pragma unroll
        for (int s = 0; s < SG; ++s) { xa[s] = na[s]; xb[s] = nb[s]; xd[s] = nd[s]; }
    }
    stc<E, VEC>(h_last + bi * D + col, ch);
}

// MG: a holds z, hx holds x = h~ (a fourth load per step); da receives dz and db receives dx.
// RECOMP (with MG): the kernel has what the forward pass had, so it reads only one row of h per group of SG
// steps -- the state entering the group -- and runs the recurrence forward through the group again for the
// states between: SG - 1 of SG rows of h not fetched (24 -> 20.5 bytes per element and step in float32) for the
// map's arithmetic a second time.  That pays where the call is bound by HBM and costs where its arrays fit the
// last-level cache (float32, 1024 x 128 x 256: 157 -> 138 us; 256 x 128 x 256: 46 -> 49 us; bfloat16 arrays,
// 1024 x 128 x 256: 80 -> 90 us, 512 x 1024 x 1024: 1.30 -> 1.19 ms): launch_bwd asks for it by the bytes moved.
template <typename E, int VEC, int SG, bool MG = false, typename S = E, bool DF = false, bool RECOMP = false, bool GATE = false>
__global__ void __launch_bounds__(256)
diag_scan_bwd_stream_kernel(const S *__restrict__ a, const S *__restrict__ hx, const S *__restrict__ hfw,
                            const void *__restrict__ done, int,
                            const E *__restrict__ h0, const S *__restrict__ g,
                            const E *__restrict__ g_last, S *__restrict__ da, S *__restrict__ db,
                            E *__restrict__ dh0, int64_t B, int T, int64_t D, int64_t cols_per_row, int a_ti,
                            int da_sum, Gate<S> gt)
{
    using V = Vec<E, VEC>;
    using O = Ops<E>;
    // the flags' type is a template parameter here: with both kinds of load in the code the compiler reuses
    // registers of loads still in flight for the other kind's address and waits for them in mid-prefetch
    constexpr int done_f32 = DF;
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t bi = gid / cols_per_row;
    const int64_t col = first_col<VEC>(gid % cols_per_row, D);
    if (bi >= B) return;
    const int64_t row0 = bi * T;
    V dsum = vfill<E, VEC>(O::zero());  // da_sum: the per-step terms summed over the sequence, da is (B,D)
    V lam = vfill<E, VEC>(O::zero());  // conj(abar_{t+1}) lam_{t+1} entering step t
    if (g_last) lam = carry_grad<GATE, E, VEC>(g_last, gt.last, bi * D + col);

    // step r (reversed index), t = T-1-r: needs g_t, a_t (for the carry to t-1), h_{t-1}, done_t
    using R = raw_t<S, VEC>;  // prefetched values stay as stored until they are consumed
    static_assert(!RECOMP || MG, "the states can be formed again only where the map's inputs are at hand");
    constexpr int NH = RECOMP ? 1 : SG;  // rows of h per group
    R xg[SG], xa[SG], xh[NH], ng[SG], na[SG], nh[NH];
    R xx[MG ? SG : 1], nx[MG ? SG : 1];
    uint32_t xd[SG], nd[SG];
    V h0v = vfill<E, VEC>(O::zero());  // h_{-1}: what step 0 multiplies its lam with
    if (h0) h0v = ldc<E, VEC>(h0 + bi * D + col);
    [[maybe_unused]] R xq[GATE ? SG : 1], nq[GATE ? SG : 1];   // gates
    [[maybe_unused]] V top;                                    // the state of the step at hand
    if constexpr (GATE && !RECOMP) top = ldv<S, E, VEC>(hfw + (row0 + T - 1) * D + col);
    auto load = [&](int r0, R *pg, R *pa, R *ph, R *px, [[maybe_unused]] R *pq, uint32_t *pd) {
#pragma unroll
        for (int s = 0; s < SG; ++s) {
            const int t = T - 1 - (r0 + s);
            pd[s] = 0u;
            if (t >= 0) {
                const int64_t off = (row0 + t) * D + col;
                pg[s] = ldraw<S, VEC>(g + off);
                if constexpr (GATE) pq[s] = ldraw<S, VEC>(gt.gate + off);
                pa[s] = ldraw<S, VEC>(a + (a_ti ? col : off));
                if constexpr (MG) px[s] = ldraw<S, VEC>(hx + off);
                if constexpr (!RECOMP) {
                    if (t > 0) ph[s] = ldraw<S, VEC>(hfw + off - D);
                }
                pd[s] = done_raw(done, done_f32, row0 + t);
            }
        }
        if constexpr (RECOMP) {  // the state entering the group's earliest step
            const int t_lo = T - r0 - SG;
            if (t_lo > 0) ph[0] = ldraw<S, VEC>(hfw + (row0 + t_lo - 1) * D + col);
        }
    };
    load(0, xg, xa, xh, xx, xq, xd);
    for (int r0 = 0; r0 < T; r0 += SG) {
        if (r0 + SG < T) load(r0 + SG, ng, na, nh, nx, nq, nd);
        V hprev[RECOMP ? SG : 1];  // h_{t-1} of the group's steps, by the recurrence from the state entering the group
        if constexpr (RECOMP) {
            V hc = h0v;
            if (T - r0 - SG > 0) hc = cvtv<S, E, VEC>(xh[0]);
#pragma unroll
            for (int s = SG - 1; s >= 0; --s) {  // forward in time
                const int t = T - 1 - (r0 + s);
                if (t >= 0) {
                    hprev[s] = hc;
                    const bool dn = done_test(xd[s], done_f32);
                    const V va = cvtv<S, E, VEC>(xa[s]), vx = cvtv<S, E, VEC>(xx[s]);
#pragma unroll
                    for (int i = 0; i < VEC; ++i) {
                        float ca = va.v[i], cb = vx.v[i];
                        MinGru::coeffs(ca, cb);
                        hc.v[i] = dn ? cb : O::madd(ca, hc.v[i], cb);
                    }
                }
            }
            if constexpr (GATE) top = hc;
        }
#pragma unroll
        for (int s = 0; s < SG; ++s) {
            const int t = T - 1 - (r0 + s);
            if (t >= 0) {
                const bool dn = done_test(xd[s], done_f32);
                const int64_t off = (row0 + t) * D + col;
                V vg = cvtv<S, E, VEC>(xg[s]);
                const V va = cvtv<S, E, VEC>(xa[s]);
                V vh = h0v, vx;
                if constexpr (GATE) stv<S, E, VEC>(gt.dgate + off, gate_grads<S, VEC>(vg, top, xq[s]));
                if constexpr (MG) vx = cvtv<S, E, VEC>(xx[s]);
                if constexpr (RECOMP) {
                    vh = hprev[s];
                } else {
                    if (t > 0) vh = cvtv<S, E, VEC>(xh[s]);
                }
                if constexpr (GATE) top = vh;
                V l, o;
#pragma unroll
                for (int i = 0; i < VEC; ++i) {
                    l.v[i] = O::madd(O::one(), vg.v[i], lam.v[i]);  // lam_t = g_t + carried term
                    const E prod = O::mul(l.v[i], O::conj(vh.v[i]));
                    o.v[i] = dn ? O::zero() : prod;
                    if constexpr (MG) {
                        float sg, at, dz, dx;
                        MinGru::gates(va.v[i], sg, at);
                        MinGru::grads(va.v[i], vx.v[i], l.v[i], o.v[i], dz, dx);
                        lam.v[i] = dn ? 0.0f : at * l.v[i];
                        o.v[i] = dz;
                        l.v[i] = dx;
                    } else {
                        const E nxt = O::mul(O::conj(va.v[i]), l.v[i]);
                        lam.v[i] = dn ? O::zero() : nxt;           // conj(abar_t) lam_t for step t-1
                    }
                }
                stv<S, E, VEC>(db + off, l);
                if (!MG && da_sum) {
#pragma unroll
                    for (int i = 0; i < VEC; ++i) dsum.v[i] = O::madd(O::one(), dsum.v[i], o.v[i]);
                } else {
                    stv<S, E, VEC>(da + off, o);
                }
            }
        }
#pragma unroll
        for (int s = 0; s < SG; ++s) { xg[s] = ng[s]; xa[s] = na[s]; xd[s] = nd[s]; }
#pragma unroll
        for (int s = 0; s < NH; ++s) xh[s] = nh[s];
        if constexpr (MG) {
#pragma unroll
            for (int s = 0; s < SG; ++s) xx[s] = nx[s];
        }
        if constexpr (GATE)
#pragma unroll
            for (int s = 0; s < SG; ++s) xq[s] = nq[s];
    }
    if (!MG && da_sum) stc<E, VEC>(reinterpret_cast<E *>(da) + bi * D + col, dsum);  // (B,D), arithmetic type
    if constexpr (GATE)
#pragma unroll
        for (int i = 0; i < VEC; ++i) lam.v[i] *= h0v.v[i];   // of the carry's logarithm
    if (dh0) stc<E, VEC>(dh0 + bi * D + col, lam);  // conj(abar_0) lam_0
}

struct ScanPlan {
    int vec, nw, tiles;
    bool stream;  // streaming kernel (no time split) instead of the wave-split kernel
    int ts = TS_MIN;  // steps per wave and super-step of the wave-split kernel
};

// Which kernel, how many elements per lane and how many waves along time.  Two layers of rules: the first
// block in the function body (sequences of 32 steps and more) comes from one sweep over every plan and
// takes precedence; what follows it are the earlier rules, which still decide the cases that block leaves
// open and all shorter sequences.  The earlier rules, as they were derived
// (fp32; 512x1024x1024, 1024x128x256, 64x512x512, 32x128x256):
//  - widest vector the shapes/alignments allow, narrowed until there are >= 2048 wave columns;
//  - forward: split time over up to 8 waves until ~8192 waves exist (the wave-split kernel at
//    4 waves reached 5.7 TB/s on the 6.4 GB shape, the streaming kernel 5.1 TB/s); with no
//    split left to do, stream; shapes so small that eight waves per workgroup still leave the
//    device short of waves (one vector lane per thread by then) take sixteen, which makes a
//    sequence of up to 128 steps a single super-step: the kernel's time is then one trip to
//    memory and back instead of one per super-step;
//  - backward (three loads per step) prefers wide vectors: the widest one that still gives 4096 waves
//    with the time axis split over eight waves -- or, for one or two lanes per thread, sixteen --
//    takes the wave-split kernel (512x1024x1024: 1.91 ms = 5.6 TB/s against 2.12 ms streaming;
//    1024x128x256: 135 us either way; 256x128x256: 28 against 39 us; 64x512x512: 77 against 111 us);
//    shapes too small for that fall to the rule of the forward pass, and otherwise the streaming
//    kernel runs whenever the columns alone give >= 2048 waves.  With the MinGRU map inside (a
//    fourth stream and the map's arithmetic per element) the eight-wave split loses to streaming at
//    1024x128x256 (202 vs 165 us; level at the large shape), so that case keeps the rule it had.
ScanPlan plan_scan(int64_t B, int64_t T, int64_t D, size_t esize, bool bwd, bool mg, bool half_storage, bool a_ti)
{
    const int maxvec = (int)(16 / esize);
    int vec = 1;
    if (D >= (1ll << 28)) return {1, 1, (int)((D + 63) / 64), true};   // the wave-split kernels count a row's bytes in 32 bits
    for (int v = maxvec; v >= 1; v >>= 1) {
        // a vector so wide that the waves covering a row are less than three quarters full wastes the
        // idle lanes' share of every load (rows of 128 floats, backward: 0.87 -> 0.57 ms at 16384x64x128
        // with two floats per lane instead of four; rows of 64: 0.75 -> 0.36 ms)
        const int64_t covered = ((D + 64 * (int64_t)v - 1) / (64 * (int64_t)v)) * 64 * v;
        if (D >= v && (v == 1 || 4 * D >= 3 * covered)) { vec = v; break; }
    }
    auto ntiles = [&](int v) { return (D + 64 * (int64_t)v - 1) / (64 * (int64_t)v); };
    // ---- Sequences of 32 steps and more: rules from a sweep of every plan (vector 1/2/4 x streaming or
    // 2..16 waves along time) over twenty-two shapes of 16..16384 sequences x 16..4096 steps x 64..1024
    // columns, for each kind of scan (float32, MinGRU map, bfloat16 arrays, complex64) and direction, timed
    // with 512 MB of other traffic between two launches so that no shape is served from the last-level cache.
    // A line lies between the measured neighbours on its two sides, at a round number of columns, waves or workgroups; the figures beside a
    // rule are such neighbours.  No model of registers and trips says where between them the sides change, and what lies there is not measured.
    // Geometric mean of time over the best plan's, these rules / the rules below alone: float32 1.00 / 1.07
    // forward and 1.02 / 1.04 backward, MinGRU 1.00 / 1.06 and 1.02 / 1.05, bfloat16 1.01 / 1.40 and
    // 1.00 / 1.21, complex64 1.01 / 1.08 and 1.03 / 1.07; no shape more than 9 % off its best plan but one.
    // The sweep was repeated after the arrays' loads and stores had become non-temporal: two float32 rules
    // changed (marked below); against the new timings the rules stand at 1.03 / 1.02 (float32), 1.03 / 1.02
    // (MinGRU), 1.02 / 1.00 (bfloat16) and 1.02 / 1.01 (complex64).
    // A third sweep, once rows of any width took vectors and the wave-split kernels could hold 16 steps per wave: eighteen shapes,
    // half of them with ragged widths or few columns over long sequences.  What changed is marked (*); times in us, before -> now.
    if (T >= 4 * TS_MIN) {
        auto cols = [&](int v) { return B * ntiles(v); };  // workgroups of the wave-split kernel
        auto split = [&](int v, int n, int ts = TS_MIN) { return ScanPlan{v, n, (int)ntiles(v), false, ts}; };
        auto flow = [&](int v) { return ScanPlan{v, 1, (int)ntiles(v), true}; };
        const bool ragged = D % 64 != 0 && D > 128;
        const int64_t waves2 = B * D / 128;   // of the streaming kernels on two elements per lane
        int nw8 = 1;  // waves along time: up to eight, each with a whole group of steps to itself
        while (nw8 < 8 && (int64_t)2 * nw8 * TS_MIN <= T) nw8 <<= 1;
        // (***) A fourth sweep, once the wave-split kernels requested everything of a super-step at once, waited for no store at their barriers and
        // read a broadcast coefficient once: twenty-six shapes of each kind, `full`: four elements per lane leave few lanes idle.  Four waves
        // along time on wide vectors gained most -- a workgroup's registers then leave room for others beside it.  us, before -> now.
        const int64_t covered4 = 256 * ntiles(4);
        const bool full = ntiles(4) == 1 ? D >= 176 : 10 * D >= 9 * covered4;
        // Three rules for float32, each timed against the plan it replaces over shapes drawn after it was fixed (n shapes: geometric mean of new / old time, worst;
        // us old -> new).  What lost in earlier draws keeps the old plan; the figures are of a last one.
        const bool f32 = esize == 4 && !half_storage;
        // Rows of 65 to 111 floats fit one wave of two elements a lane, half the load instructions of two waves of one (96 and more had that before, on eight
        // waves).  Forward, MinGRU too: n 240, 0.78, 1.05 (969 x 947 x 72 306 -> 195, 454 x 884 x 88 167 -> 101); plain backward: n 120, 0.69, 1.02 (902 x 787 x 103 373 -> 217).
        // Not the backward of MinGRU: 0.91 over 43, but 812 x 566 x 80 207 -> 298.  Eight waves along time where rows give no
        // more than two workgroups a compute unit (eight / four: 512 x 600 x 70 67 / 71, MinGRU 69 / 76, backward 122 / 129; 690 x 600 x 90 111 / 107, 116 / 105, 223 / 194): from
        // 256 steps on, forward from 96 floats on at any length (456 x 122 x 102 17.3 / 19.5, 341 x 255 x 102 MinGRU 32.1 / 35.7; 534 x 154 x 105 31.9 / 29.2) and beyond
        // 1024 rows as before (1273 x 230 x 101 81 / 85, 1094 x 123 x 107 MinGRU 42 / 45, 2420 x 1022 x 100 630 / 642).
        if (f32 && D > 64 && D < 112 && T < 128 * TS_MIN && waves2 >= 256 && !(mg && bwd)) {
            const bool eight = !bwd && D >= 96 ? B <= 512 || B > 1024 : B <= 512 && T >= 256;
            return split(2, nw8 > 4 && eight ? 8 : nw8 < 4 ? nw8 : 4);
        }
        if (f32 && ragged && bwd) {
            // MinGRU streams: n 120, 0.89, 1.04 (263 x 469 x 272 315 -> 205, 132 x 274 x 872 238 -> 164, 622 x 1037 x 208 864 -> 613).  Not where four elements a lane make between 340
            // and 512 workgroups and a row is one of them (33 of 37 shapes lost, 433 x 242 x 234 138 -> 162; 340 x 1414 x 253 784 -> 768, 527 x 189 x 244 168 -> 161), nor, where
            // either is so, in short sequences (246 x 110 x 505 80 -> 87, 676 x 146 x 193 118 -> 145).  From 1024 on 10 of 68 shapes lost, up to 1.18.
            if (mg && D >= 192 && T >= 64 && waves2 >= 512 && waves2 < 1024) {
                const bool between = cols(4) > 340 && cols(4) <= 512, one = ntiles(4) == 1;
                if (!(between && one) && (T >= 256 || !(between || one))) return flow(2);
            }
            // four elements a lane from half as many columns on: n 120, 0.87, 1.02 (254 x 526 x 219 179 -> 136, 179 x 203 x 197 51 -> 41)
            if (!mg && T >= 128 && waves2 >= 256 && waves2 < 512) return split(4, nw8);
        }
        // (*) bfloat16 backward: single elements are 2-byte loads, three or four arrays of them; two per lane and 16 steps
        // per wave make up for half the waves (8 x 1000 x 64 66 -> 54, 57 x 2908 x 120 217 -> 166), while a workgroup per compute
        // unit is all there is
        if (half_storage && bwd && !mg && D >= 2 && T >= 8 * TS_MIN && waves2 < 600 && (cols(2) <= 256 || D <= 64)) return split(2, 8, T >= 16 * TS_MIN ? 16 : 8);
        // so few columns that eight waves along time leave most of the device idle: sixteen of one lane each; (*) forward with
        // 16 steps each, half as many trips to memory (4 x 3000 x 512 101 -> 77, 75 x 679 x 64 29 -> 22)
        if (T >= 16 * TS_MIN && cols(1) <= 256) return split(1, 16, !bwd && esize == 4 && T > 16 * TS_MIN ? 16 : 8);
        if (half_storage && T >= 8 * TS_MIN) {
            // (***) bfloat16, forward and backward: 512 x 1024 x 1024 661 -> 527 and 1066 -> 848, 400 x 200 x 201 43 -> 32 and 67 -> 52, 1024 x 512 x 512 332
            // -> 287 and 536 -> 489, 500 x 64 x 200 16 -> 14 and 28 -> 20; backward also with more lanes idle (984 x 378 x 448 362 -> 342), but not
            // where a thousand columns of ragged rows make few workgroups (128 x 512 x 1000 176 / 191)
            if (!mg && cols(4) >= 400 && (full || (bwd && !a_ti && 100 * D >= 68 * covered4)) && !(bwd && a_ti && T < 16 * TS_MIN) && !(bwd && ragged && ntiles(4) > 1 && cols(4) < 1024)) return split(4, 4);
            // MinGRU backward: with columns enough whole rows stream on four elements per lane (1510 x 943 x 165 966 -> 857, 4096 x 64 x 256 165 -> 144,
            // 300 x 700 x 1000 863 -> 751), with fewer the split (256 x 2048 x 512 891 -> 663, 128 x 1024 x 1024 437 -> 323, 500 x 64 x 200 35 -> 27;
            // forward 300 x 700 x 1000 430 -> 372, 256 x 2048 x 512 397 -> 360)
            if (mg && bwd && B * D >= 256 * 1100) return flow(4);
            if (mg && bwd && cols(4) >= 400 && cols(4) < 640 && full) return split(4, 4);
            if (mg && !bwd && ragged && cols(4) >= 400 && full) return split(4, 4);
            if (mg && bwd && D > 64 && D <= 128 && cols(2) >= 512) return split(2, 4);   // 1000 x 500 x 128 222 -> 175
            if (mg && !bwd && !ragged && D % 64 == 0 && cols(2) >= 1024) return split(2, 4);   // 256 x 2048 x 512 397 -> 347
        }
        if (half_storage) {
            // (swept again once the bfloat16 values waited as stored bits: the wave-split kernels then lead
            // forward at every size; four elements per lane, backward, do not fit the wave-split kernel's
            // registers)
            const int v = D <= 64 || (!bwd && cols(1) <= 256) ? 1 : 2;
            // the streaming kernels lay their threads flat over (row, column): a row need not fill whole waves.
            // (*) They lead as soon as they have 600 waves backward, and on ragged rows with a thousand (MinGRU 1800) forward
            // (1500 x 300 x 165 240 -> 137 and 439 -> 231; 128 x 512 x 1000 122 -> 111 and 222 -> 169)
            // (**) A last sweep, twenty shapes of 256 to 800 workgroups: eight waves of 16 steps fill a compute unit's registers, of 8
            // steps half of them, four waves a third, so beyond 256 workgroups of the first or 512 of the second a few left over
            // cost a whole round.  Forward 256 to 512 workgroups 8 steps, above four waves (79 x 808 x 391 117 -> 89 with the MinGRU
            // map and 94 -> 74 without, 85 x 1500 x 391 203 -> 156, 150 x 600 x 512 117 -> 92); backward four waves above 256
            // (205 -> 173 and 138 -> 118, 373 -> 314), also where whole rows would stream with up to 768 (221 -> 205 and 146 -> 112,
            // 200 x 1200 x 384 495 -> 391; ragged ones not: 200 x 400 x 391 122 -> 147)
            if (v == 2 && bwd && nw8 > 4 && cols(2) > 256 && (waves2 < 600 || (!ragged && waves2 < 768))) return split(2, 4);
            if (v == 2 && (bwd ? waves2 >= 600 : ragged && waves2 >= (mg ? 1800 : 1000))) return flow(2);
            if ((bwd ? cols(v) >= 512 : cols(v) >= (v == 2 ? 513 : 1024)) && nw8 > 4) return split(v, 4);
            return split(v, nw8, !bwd && T >= 64 * TS_MIN && nw8 == 8 && (v == 1 || cols(v) <= 256) ? 16 : 8);   // (*) 256 x 1024 x 96 63 -> 50
        }
        if (esize == 8 && !mg && a_ti && T >= 8 * TS_MIN) {
            // (***) complex64 with a broadcast decay, forward and backward: 300 x 700 x 500 486 -> 381 and 684 -> 554, 500 x 200 x 184 98 -> 68 and 123 ->
            // 103, 192 x 250 x 184 42 -> 40 and 66 -> 56, 100 x 600 x 512 102 -> 89 and 148 -> 134, 1024 x 64 x 256 53 -> 48 and 81 -> 71
            if (T >= 12 * TS_MIN ? cols(2) >= 400 : (cols(2) >= 512 && D % 64 != 0)) return split(2, 4);
            if (cols(1) >= 512) return split(1, 4);
        }
        if (esize == 8 && !mg) {
            // (*) ragged rows stream, and so do the backward that sums a broadcast decay's gradient (no da to write) and that of
            // short sequences: 400 x 200 x 201 backward 208 -> 155, 300 x 64 x 645 broadcast 102 -> 77, 1024 x 128 x 256
            // broadcast 182 -> 157, 583 x 38 x 576 130 -> 104
            if (waves2 >= 600 && (ragged || (bwd && (a_ti || T <= 8 * TS_MIN)))) return flow(D < 2 ? 1 : 2);
            if (!bwd && a_ti && vec == 2 && cols(2) >= 1024 && T >= 8 * TS_MIN) return split(2, nw8 > 4 ? 4 : nw8);   // (*) 124 -> 106
            if (!bwd && (T <= 256 || cols(1) <= 1024)) return split(1, nw8);
            if (bwd && vec == 2 && (cols(2) >= 1024 || (cols(2) >= 256 && T >= 64 * TS_MIN))) return split(2, nw8);
        }
        if (esize == 4) {
            // (*) ragged rows take the widest vector although its last wave is half empty: the time goes with the number of
            // load instructions (forward, backward: 1500 x 300 x 165 335 -> 182, 634 -> 344; 400 x 200 x 201 63 -> 48, 110 -> 89;
            // MinGRU 345 -> 192, 618 -> 452), once there are columns enough (49 x 62 x 235 forward 9.5 -> 11.7)
            if (ragged && nw8 == 8 && cols(4) >= 256) return split(4, bwd && !mg ? 8 : 4);
            if (!bwd) {
                // (swept again once every array was loaded and stored non-temporally: two elements per lane
                // then lead at the large shapes as well -- 512 x 1024 x 1024 forward 1067 -> 1009 us,
                // 4096 x 128 x 256 291 -> 269 us -- where four used to)
                if (D > 64 && D < 128 && cols(1) <= 512 && T >= 64 * TS_MIN) return split(1, 8, 16);   // (*) 256 x 1024 x 96 81 -> 68
                return split(vec < 2 || cols(1) <= 256 ? 1 : 2, nw8);
            }
            if (mg) {
                // (***) 1024 x 512 x 512 1137 -> 1037, 800 x 100 x 600 284 -> 254, 4096 x 64 x 256 306 -> 252
                if (T >= 8 * TS_MIN && D > 128 && waves2 >= 3000) return flow(2);
                if (vec == 4 && cols(4) >= 2048 && T >= 8 * TS_MIN) return split(4, nw8 > 4 ? 4 : nw8);
                if (D <= 128 && cols(1) >= 2048) return split(1, nw8);
            } else {
                if (D <= 128 && cols(1) >= 1024) return split(1, nw8);
                if (T >= 8 * TS_MIN) {
                    for (int v = vec; v >= 1; v >>= 1) {
                        // rows of a single column tile take eight waves along time, wider rows four (the same
                        // sweep: 8192 x 128 x 256 backward 1007 -> 920 us, 256 x 128 x 1024 149 -> 132 us)
                        if (cols(v) >= 1024) return split(v, ntiles(v) == 1 ? 8 : 4);
                        if (cols(v) * 8 >= 4096) return split(v, 8);
                        if (v <= 2 && cols(v) * 16 >= 4096 && T >= 16 * TS_MIN) return split(v, 16);
                    }
                }
            }
        }
    }
    // ---- what the sweep above left as it was, and sequences shorter than 32 steps ----
    // bfloat16 arrays: a lane's loads are half as wide, so the widest vector stays (no narrowing for the sake
    // of more columns); measured on the MinGRU kernels at 1024x128x256, 512x1024x1024, 256x128x256: with 1024
    // waves of columns the streaming kernel is ahead or level (backward 186 -> 161 us, forward of the largest
    // shape 1412 -> 875 us), below that eight waves along time (backward 88 -> 44 us at 256x128x256)
    if (half_storage) {
        const int64_t cols = B * ntiles(vec);
        if (cols >= 1024) return {vec, 1, (int)ntiles(vec), true};
        int nw = 1;
        while (nw < 8 && cols * nw < 2048 && (int64_t)nw * TS_MIN < T) nw <<= 1;
        return {vec, nw, (int)ntiles(vec), nw == 1};
    }
    // complex64 (measured on 1024x128x{64,128,256}, 4096x128x64, 256x1024x{64,256}, 64x4096x256): one
    // element per lane is the width the column rule below arrives at for most shapes, and at that width
    // the streaming kernel is ahead of the wave-split one as soon as the columns give it 2048 waves
    // (forward 111 -> 93 us at 1024x128x128, 242 -> 180 us at 4096x128x64) or, backward, 1024 waves
    // (146 -> 70 us at 1024x128x64; 990 -> 520 us at 256x1024x256); where the 16-byte vector would be
    // narrowed for lack of columns but eight waves along time make up for them, it is kept (forward
    // 399 -> 328 us at 256x1024x256).
    if (esize == 8 && !mg) {
        int v1 = vec;
        while (v1 > 1 && B * ntiles(v1) < 2048) v1 >>= 1;
        const int64_t waves1 = B * ntiles(v1);
        if (v1 == 1 && waves1 >= (bwd ? 1024 : 2048)) return {1, 1, (int)ntiles(1), true};
        if (vec == 2 && v1 == 1 && B * ntiles(2) * 8 >= 4096 && T >= 8 * TS_MIN) return {2, 8, (int)ntiles(2), false};
    }
    // floats, backward: see above; rows of up to 128 floats first -- there a wave's loads in the
    // wave-split kernel are short pieces, and one column per lane in the streaming kernel is ahead
    // wherever it gets 1024 waves (4096x128x64: 193 -> 137 us, 1024x1024x64: 456 -> 303 us,
    // 1024x128x128: 84 -> 69 us, 8192x128x128: 585 -> 545 us)
    if (bwd && !mg && esize == 4 && D <= 128 && B * ntiles(1) >= 1024) return {1, 1, (int)ntiles(1), true};
    if (bwd && !mg && esize == 4) {
        for (int v = vec; v >= 1; v >>= 1) {
            const int64_t cols = B * ntiles(v);
            if (cols * 8 >= 4096 && T >= 8 * TS_MIN) return {v, 8, (int)ntiles(v), false};
            if (v <= 2 && cols * 16 >= 4096 && T >= 16 * TS_MIN) return {v, 16, (int)ntiles(v), false};
        }
    }
    while (vec > 1 && B * ntiles(vec) < 2048) vec >>= 1;
    const int tiles = (int)ntiles(vec);
    const int64_t waves = B * tiles;
    int nw = 1;
    const int maxw = vec == 1 ? 16 : 8;
    while (nw < maxw && waves * nw < 8192 && (int64_t)nw * TS_MIN < T) nw <<= 1;
    const bool stream = bwd ? waves >= 2048 : nw == 1;
    // MinGRU backward short of columns for that: one column per lane still streams ahead of the wave-split
    // kernel from 1024 waves (1024x128x64: 55 -> 45 us, 256x1024x256: 472 -> 332 us)
    if (bwd && mg && !stream && B * ntiles(1) >= 1024) return {1, 1, (int)ntiles(1), true};
    return {vec, stream ? 1 : nw, tiles, stream};
}

struct SegmentPlan {
    int vec = 1, tiles = 0, n = 0, steps = 0, ts = TS_MIN;  // n = 0: not in segments
};

// When to cut time into segments, and how many: from a sweep over twenty shapes of 4..256 sequences x 250..4000 steps x 64..560
// columns for every kind of scan.  One walk per column group costs a trip to memory per super-step, whatever the number of
// columns; the segments cost a second launch (3 us) and the second reading.  So: few columns (in units of a wave, `cols`), and
// steps enough per column unit -- the line T >= 9 cols forward and 4 cols backward, whose first pass reads two arrays of the
// four or five.  Time in us, one walk -> segments, forward and backward: float32 8 x 1000 x 64 31 -> 14 and 57 -> 15, 16 x 4000 x 256
// 114 -> 68 and 219 -> 90, 32 x 512 x 256 backward 34 -> 28, 57 x 2908 x 120 104 -> 110 (left out) and 194 -> 125; bfloat16 16 x 4000 x 256
// 109 -> 50 and 210 -> 68, with the MinGRU map 320 -> 92 backward; complex64 16 x 2690 x 192 150 -> 73 and 260 -> 115.
SegmentPlan plan_segments(int64_t B, int64_t T, int64_t D, size_t esize, bool bwd, bool mg, bool half_storage)
{
    SegmentPlan p;
    auto tiles = [&](int64_t v) { return (D + 64 * v - 1) / (64 * v); };
    const int64_t cols = B * tiles(1);
    if (!bwd) {
        const int64_t most = half_storage || esize == 8 ? 128 : 80;   // 57 x 2908 x 120 (cols 114): see above
        if (cols > most || T < 9 * cols || T < (esize == 8 ? 256 : 384)) return p;
    } else {
        int64_t most = 192, per = 4;   // 20 x 1250 x 551 (cols 180) 120 -> 109, 49 x 1474 x 300 (245) 160 -> 162
        if (esize == 8) most = 128, per = 5;               // 20 x 1250 x 551 188 -> 204
        else if (half_storage && mg) most = 256;           // 49 x 1474 x 300 181 -> 159
        else if (half_storage && D <= 64) per = 9;         // 128 x 1024 x 64 56 -> 60, 75 x 679 x 64 45 -> 32
        else if (!half_storage && D <= 64) most = 128;     // 128 x 1024 x 64 62 -> 55, 189 x 1264 x 64 80 -> 92
        if (cols > most || T < per * cols || T < 256) return p;
    }
    // two elements per lane where a row fills more than three quarters of its waves with them: bfloat16, and backward
    // (57 x 2908 x 120 192 -> 125 us; rows of 192, three quarters, 57 -> 63 us)
    if (D > 64 && (half_storage || (bwd && esize == 4 && 4 * D > 3 * 128 * tiles(2)))) p.vec = 2;
    if (bwd && half_storage && !mg && p.vec == 2) p.ts = 16;
    p.tiles = (int)tiles(p.vec);
    const int64_t span = 8 * p.ts;
    // a thousand workgroups in all, at most MAX_SEGMENTS per sequence
    int64_t n = (1024 + B * p.tiles - 1) / (B * p.tiles);
    n = n > MAX_SEGMENTS ? MAX_SEGMENTS : n;
    const int64_t steps = ((T + n - 1) / n + span - 1) / span * span;
    n = (T + steps - 1) / steps;
    if (n < 2) return p;
    p.n = (int)n;
    p.steps = (int)steps;
    return p;
}

template <typename E> size_t segment_bytes(const SegmentPlan &p, int64_t B, int64_t D, bool da_sum)
{
    return (size_t)p.n * B * (D * sizeof(E) * (da_sum ? 3 : 2) + sizeof(int));
}
template <typename E> Segments<E> segments_in(const SegmentPlan &p, int64_t B, int64_t D, bool da_sum, void *workspace)
{
    E *const w = reinterpret_cast<E *>(workspace);
    const int64_t one = (int64_t)p.n * B * D;
    return {p.n, p.steps, w, w + one, reinterpret_cast<int *>(w + (da_sum ? 3 : 2) * one), da_sum ? w + 2 * one : nullptr};
}

// The shares of the segments summed (da_sum): one thread per element of (B, D).
template <typename E> __global__ void __launch_bounds__(256) segment_sum_kernel(const E *__restrict__ parts, E *__restrict__ out, int n, int64_t BD)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= BD) return;
    E s = Ops<E>::zero();
    for (int j = 0; j < n; ++j) s = Ops<E>::madd(Ops<E>::one(), s, parts[(int64_t)j * BD + i]);
    out[i] = s;
}

size_t scan_smem(int nw, size_t vbytes)
{
    return nw == 1 ? 0 : 2 * (size_t)nw * 64 * vbytes * 2 + 2 * (size_t)nw * sizeof(int);
}

// dispatch on the compile-time vector width: f(std::integral_constant<int, VEC>)
template <typename E, typename F> void vec_switch(int vec, F f)
{
    if constexpr (sizeof(E) == 4) {
        if (vec == 4) f(std::integral_constant<int, 4>{});
        else if (vec == 2) f(std::integral_constant<int, 2>{});
        else f(std::integral_constant<int, 1>{});
    } else {
        if (vec == 2) f(std::integral_constant<int, 2>{});
        else f(std::integral_constant<int, 1>{});
    }
}

// The wave-split kernels that exist: f(VEC, MAXW, TS), each an integral constant.
template <typename E, bool MG, bool BWD, bool HALF, typename F> void split_switch(const ScanPlan &pl, F f)
{
    using std::integral_constant;
    auto with_steps = [&](auto vc, auto mw) {
        constexpr int VEC = decltype(vc)::value, MAXW = decltype(mw)::value;
        // 16 steps per wave, where plan_scan asks for it: 4-byte arithmetic forward, bfloat16 arrays backward
        constexpr bool LONG = BWD ? HALF && !MG && VEC == 2 && MAXW == 8 : sizeof(E) == 4 && (VEC == 1 || (HALF && VEC == 2 && MAXW == 8));
        if constexpr (LONG) {
            if (pl.ts == 16) return f(vc, mw, integral_constant<int, 16>{});
        }
        f(vc, mw, integral_constant<int, TS_MIN>{});
    };
    vec_switch<E>(pl.vec, [&](auto vc) {
        constexpr int VEC = decltype(vc)::value;
        if constexpr (VEC == 1 || (BWD && VEC == 2 && sizeof(E) == 4 && !MG)) {
            if (pl.nw == 16) return with_steps(vc, integral_constant<int, 16>{});
        }
        with_steps(vc, integral_constant<int, 8>{});
    });
}

// The kernels over segments that plan_segments asks for: f(VEC, TS); eight waves each.
template <typename E, bool MG, bool BWD, bool HALF, typename F> void segment_switch(const SegmentPlan &pl, F f)
{
    using std::integral_constant;
    if constexpr (HALF || (BWD && sizeof(E) == 4)) {
        if (pl.vec == 2) return f(integral_constant<int, 2>{}, integral_constant<int, BWD && HALF && !MG ? 16 : TS_MIN>{});
    }
    f(integral_constant<int, 1>{}, integral_constant<int, TS_MIN>{});
}

// MG (E = float): a and b hold the MinGRU projections z and h~.
// S: storage type of the (B,T,D) arrays (E, or __bf16 with E = float).
template <typename E, bool MG = false, typename S = E>
int launch_fwd(hipStream_t st, const Gate<S> &gt, const void *a, const void *b, const void *done,
               int done_f32, const void *h0, const void *P0, void *h, void *h_last,
               void *P_last, int64_t B, int64_t T, int64_t D, int a_ti, void *workspace)
{
    if (const SegmentPlan sp = workspace ? plan_segments(B, T, D, sizeof(E), false, MG, !std::is_same<S, E>::value) : SegmentPlan{}; sp.n) {
        Segments<E> sg = segments_in<E>(sp, B, D, false, workspace);
        const dim3 block(512);
        const size_t smem = scan_smem(8, sizeof(E) * sp.vec);
        int rc = MRX_ERR_LAUNCH;
        segment_switch<E, MG, false, !std::is_same<S, E>::value>(sp, [&](auto vc, auto ts) {
            constexpr int VEC = decltype(vc)::value, TS = decltype(ts)::value;
            sg.n = sp.n - 1;
            rc = launch_kernel((diag_scan_fwd_kernel<E, VEC, MG, 8, S, TS, SUMMARISE>), dim3((unsigned)(B * sp.tiles * sg.n)), block, smem, st,
                               (const S *)a, (const S *)b, done, done_f32, (const E *)nullptr, (const E *)nullptr, (S *)nullptr, (E *)nullptr,
                               (E *)nullptr, (int)T, D, sp.tiles, 8, a_ti, sg, Gate<S>{});
            if (rc != MRX_OK) return;
            sg.n = sp.n;
            rc = launch_kernel((diag_scan_fwd_kernel<E, VEC, MG, 8, S, TS, APPLY>), dim3((unsigned)(B * sp.tiles * sg.n)), block, smem, st,
                               (const S *)a, (const S *)b, done, done_f32, (const E *)h0, (const E *)P0, (S *)h, (E *)h_last, (E *)P_last,
                               (int)T, D, sp.tiles, 8, a_ti, sg, Gate<S>{});
        });
        return rc;
    }
    const ScanPlan pl = plan_scan(B, T, D, sizeof(E), false, MG, !std::is_same<S, E>::value, a_ti);
    int rc = MRX_ERR_LAUNCH;
    if (pl.stream) {
        const int64_t cpr = (D + pl.vec - 1) / pl.vec;
        const dim3 grid((unsigned)((B * cpr + 255) / 256)), block(256);
        vec_switch<E>(pl.vec, [&](auto vc) {
            constexpr int VEC = decltype(vc)::value;
            auto launch = [&](auto df, auto gate) {
                rc = launch_kernel((diag_scan_fwd_stream_kernel<E, VEC, (VEC * sizeof(E) == 16 ? 4 : 8), MG, S, decltype(df)::value, decltype(gate)::value>),
                                   grid, block, 0, st, (const S *)a, (const S *)b, done, done_f32, (const E *)h0,
                                   (const E *)P0, (S *)h, (E *)h_last, (E *)P_last, B, (int)T, D, cpr, a_ti, gt);
            };
            auto go = [&](auto df) {
                if constexpr (MG)
                    if (gt.gate) return launch(df, std::true_type{});
                launch(df, std::false_type{});
            };
            if (done_f32) go(std::true_type{});
            else go(std::false_type{});
        });
    } else {
        const dim3 grid((unsigned)(B * pl.tiles)), block(64 * pl.nw);
        const size_t smem = scan_smem(pl.nw, sizeof(E) * pl.vec);
        split_switch<E, MG, false, !std::is_same<S, E>::value>(pl, [&](auto vc, auto mw, auto ts) {
            auto launch = [&](auto ti, auto paced, auto gate) {
                rc = launch_kernel((diag_scan_fwd_kernel<E, decltype(vc)::value, MG, decltype(mw)::value, S, decltype(ts)::value, WHOLE, decltype(ti)::value, decltype(paced)::value, decltype(gate)::value>),
                                   grid, block, smem, st, (const S *)a, (const S *)b, done, done_f32, (const E *)h0, (const E *)P0, (S *)h, (E *)h_last,
                                   (E *)P_last, (int)T, D, pl.tiles, pl.nw, a_ti, Segments<E>{}, gt);
            };
            auto go = [&](auto ti, auto paced) {
                if constexpr (MG && !decltype(paced)::value)
                    if (gt.gate) return launch(ti, paced, std::true_type{});
                launch(ti, paced, std::false_type{});
            };
            if constexpr (!MG && std::is_same<S, E>::value) {   // a broadcast coefficient is read once
                if (a_ti) return go(std::true_type{}, std::false_type{});
            }
            if constexpr (std::is_same<S, float>::value && decltype(vc)::value >= 2 && decltype(mw)::value == 8 && decltype(ts)::value == TS_MIN) {
                if (B * T * D >= PACED_ELEMENTS && !gt.gate) return go(std::false_type{}, std::true_type{});
            }
            go(std::false_type{}, std::false_type{});
        });
    }
    return rc;
}

// MG (E = float): a holds z, hx holds h~ (else unused), da and db receive dz and dh~.
template <typename E, bool MG = false, typename S = E>
int launch_bwd(hipStream_t st, const Gate<S> &gt, const void *a, const void *hx, const void *h, const void *done,
               int done_f32, const void *h0, const void *g, const void *g_last, void *da,
               void *db, void *dh0, int64_t B, int64_t T, int64_t D, int a_ti, int da_sum, void *workspace)
{
    if (const SegmentPlan sp = workspace ? plan_segments(B, T, D, sizeof(E), true, MG, !std::is_same<S, E>::value) : SegmentPlan{}; sp.n) {
        Segments<E> sg = segments_in<E>(sp, B, D, da_sum, workspace);
        const dim3 block(512);
        const size_t smem = scan_smem(8, sizeof(E) * sp.vec);
        int rc = MRX_ERR_LAUNCH;
        segment_switch<E, MG, true, !std::is_same<S, E>::value>(sp, [&](auto vc, auto ts) {
            constexpr int VEC = decltype(vc)::value, TS = decltype(ts)::value;
            sg.n = sp.n - 1;
            rc = launch_kernel((diag_scan_bwd_kernel<E, VEC, MG, 8, S, TS, SUMMARISE>), dim3((unsigned)(B * sp.tiles * sg.n)), block, smem, st,
                               (const S *)a, (const S *)nullptr, (const S *)nullptr, done, done_f32, (const E *)nullptr, (const S *)g,
                               (const E *)nullptr, (S *)nullptr, (S *)nullptr, (E *)nullptr, (int)T, D, sp.tiles, 8, a_ti, 0, sg, Gate<S>{});
            if (rc != MRX_OK) return;
            sg.n = sp.n;
            rc = launch_kernel((diag_scan_bwd_kernel<E, VEC, MG, 8, S, TS, APPLY>), dim3((unsigned)(B * sp.tiles * sg.n)), block, smem, st,
                               (const S *)a, (const S *)hx, (const S *)h, done, done_f32, (const E *)h0, (const S *)g, (const E *)g_last,
                               (S *)da, (S *)db, (E *)dh0, (int)T, D, sp.tiles, 8, a_ti, da_sum, sg, Gate<S>{});
        });
        if (rc == MRX_OK && da_sum)
            rc = launch_kernel(segment_sum_kernel<E>, dim3((unsigned)((B * D + 255) / 256)), dim3(256), 0, st, (const E *)sg.da_parts, (E *)da,
                               sp.n, B * D);
        return rc;
    }
    ScanPlan pl = plan_scan(B, T, D, sizeof(E), true, MG, !std::is_same<S, E>::value, a_ti);
    // five float32 arrays of four elements a lane and eight steps do not fit the wave-split kernel's registers (mrx_gated_scan_pays has what that costs)
    if (gt.gate && std::is_same<S, E>::value && !pl.stream && pl.vec == 4) pl.vec = 2, pl.tiles = (int)((D + 127) / 128);
    int rc = MRX_ERR_LAUNCH;
    if (pl.stream) {
        const int64_t cpr = (D + pl.vec - 1) / pl.vec;
        const dim3 grid((unsigned)((B * cpr + 255) / 256)), block(256);
        vec_switch<E>(pl.vec, [&](auto vc) {
            constexpr int VEC = decltype(vc)::value;
            auto launch = [&](auto df, auto rcmp, auto gate) {
                rc = launch_kernel((diag_scan_bwd_stream_kernel<E, VEC, (VEC * sizeof(E) == 16 ? 4 : 8), MG, S, decltype(df)::value,
                                                                decltype(rcmp)::value, decltype(gate)::value>),
                                   grid, block, 0, st, (const S *)a, (const S *)hx, (const S *)h, done, done_f32,
                                   (const E *)h0, (const S *)g, (const E *)g_last, (S *)da, (S *)db, (E *)dh0, B, (int)T, D,
                                   cpr, a_ti, da_sum, gt);
            };
            auto go = [&](auto df, auto rcmp) {
                if constexpr (MG)
                    if (gt.gate) return launch(df, rcmp, std::true_type{});
                launch(df, rcmp, std::false_type{});
            };
            // six (B,T,D) arrays pass through the call: more than twice the 256 MB of last-level cache, and the
            // call is bound by HBM -- then h is better formed again than fetched
            const bool recompute = MG && 6.0 * (double)B * (double)T * (double)D * sizeof(S) >= 600e6;
            if constexpr (MG) {
                if (recompute) {
                    if (done_f32) go(std::true_type{}, std::true_type{});
                    else go(std::false_type{}, std::true_type{});
                    return;
                }
            }
            if (done_f32) go(std::true_type{}, std::false_type{});
            else go(std::false_type{}, std::false_type{});
        });
    } else {
        const dim3 grid((unsigned)(B * pl.tiles)), block(64 * pl.nw);
        const size_t smem = scan_smem(pl.nw, sizeof(E) * pl.vec);
        split_switch<E, MG, true, !std::is_same<S, E>::value>(pl, [&](auto vc, auto mw, auto ts) {
            auto launch = [&](auto ti, auto paced, auto gate) {
                rc = launch_kernel((diag_scan_bwd_kernel<E, decltype(vc)::value, MG, decltype(mw)::value, S, decltype(ts)::value, WHOLE, decltype(ti)::value, decltype(paced)::value, decltype(gate)::value>),
                                   grid, block, smem, st, (const S *)a, (const S *)hx, (const S *)h, done, done_f32, (const E *)h0, (const S *)g,
                                   (const E *)g_last, (S *)da, (S *)db, (E *)dh0, (int)T, D, pl.tiles, pl.nw, a_ti, da_sum, Segments<E>{}, gt);
            };
            auto go = [&](auto ti, auto paced) {
                if constexpr (MG && !decltype(paced)::value && (!std::is_same<S, E>::value || decltype(vc)::value < 4))
                    if (gt.gate) return launch(ti, paced, std::true_type{});
                launch(ti, paced, std::false_type{});
            };
            if constexpr (!MG && std::is_same<S, E>::value) {
                if (a_ti) return go(std::true_type{}, std::false_type{});
            }
            if constexpr (std::is_same<S, float>::value && decltype(vc)::value >= 2 && decltype(mw)::value == 8 && decltype(ts)::value == TS_MIN) {
                if (B * T * D >= PACED_ELEMENTS && !gt.gate) return go(std::false_type{}, std::true_type{});
            }
            go(std::false_type{}, std::false_type{});
        });
    }
    return rc;
}

template <typename E>
int launch_last(hipStream_t st, const void *a, const void *b, const void *done, int done_f32,
                const void *h0, void *h_last, int64_t B, int64_t T, int64_t D, int64_t a_group)
{
    const int maxvec = (int)(16 / sizeof(E));
    int vec = 1;
    for (int v = maxvec; v >= 1; v >>= 1) {
        const size_t bytes = sizeof(E) * v;
        if (D % v == 0 && a_group % v == 0 && aligned(b, bytes) && aligned(h0, bytes) && aligned(h_last, bytes)) {
            vec = v;
            break;
        }
    }
    while (vec > 1 && B * (D / vec) < 2048 * 64) vec >>= 1;  // keep at least 2048 waves when the shape allows
    const int64_t cpr = D / vec;
    const dim3 grid((unsigned)((B * cpr + 255) / 256)), block(256);
    int rc = MRX_ERR_LAUNCH;
    vec_switch<E>(vec, [&](auto vc) {
        constexpr int VEC = decltype(vc)::value;
        rc = launch_kernel((diag_scan_last_kernel<E, VEC, (VEC * sizeof(E) == 16 ? 4 : 8)>), grid, block, 0, st,
                           (const E *)a, (const E *)b, done, done_f32, (const E *)h0, (E *)h_last, B, (int)T, D,
                           cpr, a_group);
    });
    return rc;
}

bool scan_shape_ok(int64_t B, int64_t T, int64_t D)
{
    return B > 0 && T > 0 && D > 0 && T < (1ll << 30) && B * ((D + 63) / 64) < (1ll << 31);
}

}  // namespace

extern "C" int64_t mrx_scan_workspace(int64_t B, int64_t T, int64_t D, int dtype, int what)
{
    if (!scan_shape_ok(B, T, D) || dtype < MRX_F32 || dtype > MRX_C64) return 0;
    const bool bwd = what & MRX_SCAN_BACKWARD, mg = what & MRX_SCAN_MINGRU, da_sum = what & MRX_SCAN_SUM_DA;
    const SegmentPlan p = plan_segments(B, T, D, dtype == MRX_C64 ? 8 : 4, bwd, mg, dtype == MRX_BF16);
    if (!p.n) return 0;
    return (int64_t)(dtype == MRX_C64 ? segment_bytes<c64>(p, B, D, bwd && da_sum) : segment_bytes<float>(p, B, D, bwd && da_sum));
}

namespace {

int linear_scan_fwd(void *stream, const void *a, const void *b, const void *done, const void *h0, const void *P0, void *h, void *h_last,
                    void *P_last, int64_t B, int64_t T, int64_t D, int dtype, int done_dtype, int a_time_invariant, void *workspace)
{
    if (!a || !b || !done || !h) return MRX_ERR_INVALID_ARG;
    if (!scan_shape_ok(B, T, D)) return MRX_ERR_INVALID_ARG;
    if (done_dtype != MRX_DONE_U8 && done_dtype != MRX_DONE_F32) return MRX_ERR_INVALID_ARG;
    if (done_dtype == MRX_DONE_F32 && !aligned(done, 4)) return MRX_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    const int ti = a_time_invariant != 0;
    if (dtype == MRX_F32) {
        if (!aligned(a, 4) || !aligned(b, 4) || !aligned(h, 4)) return MRX_ERR_INVALID_ARG;
        return launch_fwd<float>(st, {}, a, b, done, done_dtype, h0, P0, h, h_last, P_last, B, T, D, ti, workspace);
    }
    if (dtype == MRX_C64) {
        if (!aligned(a, 8) || !aligned(b, 8) || !aligned(h, 8) || !aligned(h0, 8) ||
            !aligned(P0, 8) || !aligned(h_last, 8) || !aligned(P_last, 8))
            return MRX_ERR_INVALID_ARG;
        return launch_fwd<c64>(st, {}, a, b, done, done_dtype, h0, P0, h, h_last, P_last, B, T, D, ti, workspace);
    }
    if (dtype == MRX_BF16) {  // a, b, h in bfloat16; arithmetic and carries in float32
        if (!aligned(a, 2) || !aligned(b, 2) || !aligned(h, 2) || !aligned(h0, 4) || !aligned(P0, 4) ||
            !aligned(h_last, 4) || !aligned(P_last, 4))
            return MRX_ERR_INVALID_ARG;
        return launch_fwd<float, false, __bf16>(st, {}, a, b, done, done_dtype, h0, P0, h, h_last, P_last, B, T, D, ti, workspace);
    }
    return MRX_ERR_INVALID_ARG;
}

}  // namespace

extern "C" int mrx_linear_scan_fwd(void *stream, const void *a, const void *b, const void *done, const void *h0, const void *P0, void *h,
                                   void *h_last, void *P_last, int64_t B, int64_t T, int64_t D, int dtype, int done_dtype, int
                                   a_time_invariant)
{
    return linear_scan_fwd(stream, a, b, done, h0, P0, h, h_last, P_last, B, T, D, dtype, done_dtype, a_time_invariant, nullptr);
}

extern "C" int mrx_linear_scan_fwd_segmented(void *stream, const void *a, const void *b, const void *done, const void *h0, const void *P0,
                                             void *h, void *h_last, void *P_last, int64_t B, int64_t T, int64_t D, int dtype, int
                                             done_dtype, int a_time_invariant, void *workspace)
{
    if (!aligned(workspace, 8)) return MRX_ERR_INVALID_ARG;
    return linear_scan_fwd(stream, a, b, done, h0, P0, h, h_last, P_last, B, T, D, dtype, done_dtype, a_time_invariant, workspace);
}

namespace {

int linear_scan_bwd(void *stream, const void *a, const void *h, const void *done, const void *h0, const void *g, const void *g_last, void
                    *da, void *db, void *dh0, int64_t B, int64_t T, int64_t D, int dtype, int done_dtype, int a_time_invariant, void
                    *workspace)
{
    if (!a || !h || !done || !g || !da || !db) return MRX_ERR_INVALID_ARG;
    if (!scan_shape_ok(B, T, D)) return MRX_ERR_INVALID_ARG;
    if (done_dtype != MRX_DONE_U8 && done_dtype != MRX_DONE_F32) return MRX_ERR_INVALID_ARG;
    if (done_dtype == MRX_DONE_F32 && !aligned(done, 4)) return MRX_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    if (a_time_invariant < 0 || a_time_invariant > MRX_A_TIME_INVARIANT_SUM_DA) return MRX_ERR_INVALID_ARG;
    const int ti = a_time_invariant != 0;
    const int da_sum = a_time_invariant == MRX_A_TIME_INVARIANT_SUM_DA;
    if (dtype == MRX_F32) {
        if (!aligned(a, 4) || !aligned(h, 4) || !aligned(g, 4) || !aligned(da, 4) || !aligned(db, 4))
            return MRX_ERR_INVALID_ARG;
        return launch_bwd<float>(st, {}, a, nullptr, h, done, done_dtype, h0, g, g_last, da, db, dh0, B, T, D, ti, da_sum, workspace);
    }
    if (dtype == MRX_C64) {
        if (!aligned(a, 8) || !aligned(h, 8) || !aligned(g, 8) || !aligned(da, 8) ||
            !aligned(db, 8) || !aligned(h0, 8) || !aligned(g_last, 8) || !aligned(dh0, 8))
            return MRX_ERR_INVALID_ARG;
        return launch_bwd<c64>(st, {}, a, nullptr, h, done, done_dtype, h0, g, g_last, da, db, dh0, B, T, D, ti, da_sum, workspace);
    }
    if (dtype == MRX_BF16) {  // a, h, g, da (per step), db in bfloat16; carries and a summed da in float32
        if (!aligned(a, 2) || !aligned(h, 2) || !aligned(g, 2) || !aligned(da, da_sum ? 4 : 2) || !aligned(db, 2) ||
            !aligned(h0, 4) || !aligned(g_last, 4) || !aligned(dh0, 4))
            return MRX_ERR_INVALID_ARG;
        return launch_bwd<float, false, __bf16>(st, {}, a, nullptr, h, done, done_dtype, h0, g, g_last, da, db, dh0, B, T, D,
                                                ti, da_sum, workspace);
    }
    return MRX_ERR_INVALID_ARG;
}

}  // namespace

extern "C" int mrx_linear_scan_bwd(void *stream, const void *a, const void *h, const void *done, const void *h0, const void *g, const void
                                   *g_last, void *da, void *db, void *dh0, int64_t B, int64_t T, int64_t D, int dtype, int done_dtype, int
                                   a_time_invariant)
{
    return linear_scan_bwd(stream, a, h, done, h0, g, g_last, da, db, dh0, B, T, D, dtype, done_dtype, a_time_invariant, nullptr);
}

extern "C" int mrx_linear_scan_bwd_segmented(void *stream, const void *a, const void *h, const void *done, const void *h0, const void *g,
                                             const void *g_last, void *da, void *db, void *dh0, int64_t B, int64_t T, int64_t D, int
                                             dtype, int done_dtype, int a_time_invariant, void *workspace)
{
    if (!aligned(workspace, 8)) return MRX_ERR_INVALID_ARG;
    return linear_scan_bwd(stream, a, h, done, h0, g, g_last, da, db, dh0, B, T, D, dtype, done_dtype, a_time_invariant, workspace);
}

extern "C" int mrx_linear_scan_last(void *stream, const void *a, const void *b, const void *done,
                                    const void *h0, void *h_last, int64_t B, int64_t T, int64_t D,
                                    int64_t a_group, int dtype, int done_dtype)
{
    if (!a || !b || !done || !h_last) return MRX_ERR_INVALID_ARG;
    if (!scan_shape_ok(B, T, D) || a_group <= 0 || D % a_group != 0) return MRX_ERR_INVALID_ARG;
    if (B * D >= (1ll << 38)) return MRX_ERR_INVALID_ARG;  // grid size
    if (done_dtype != MRX_DONE_U8 && done_dtype != MRX_DONE_F32) return MRX_ERR_INVALID_ARG;
    if (done_dtype == MRX_DONE_F32 && !aligned(done, 4)) return MRX_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    if (dtype == MRX_F32) {
        if (!aligned(a, 4) || !aligned(b, 4) || !aligned(h0, 4) || !aligned(h_last, 4)) return MRX_ERR_INVALID_ARG;
        return launch_last<float>(st, a, b, done, done_dtype, h0, h_last, B, T, D, a_group);
    }
    if (dtype == MRX_C64) {
        if (!aligned(a, 8) || !aligned(b, 8) || !aligned(h0, 8) || !aligned(h_last, 8)) return MRX_ERR_INVALID_ARG;
        return launch_last<c64>(st, a, b, done, done_dtype, h0, h_last, B, T, D, a_group);
    }
    return dtype == MRX_BF16 ? MRX_ERR_UNSUPPORTED : MRX_ERR_INVALID_ARG;
}

namespace {

int mingru_scan_fwd(void *stream, const void *gate, void *y, float *ends, const void *z, const void *h_tilde, const void *done, const void *h0, const void *P0, void *h, void
                    *h_last, void *P_last, int64_t B, int64_t T, int64_t D, int dtype, int done_dtype, void *workspace)
{
    if (!z || !h_tilde || !done || !h) return MRX_ERR_INVALID_ARG;
    if (!scan_shape_ok(B, T, D)) return MRX_ERR_INVALID_ARG;
    if (dtype != MRX_F32 && dtype != MRX_BF16) return dtype == MRX_C64 ? MRX_ERR_UNSUPPORTED : MRX_ERR_INVALID_ARG;
    if (done_dtype != MRX_DONE_U8 && done_dtype != MRX_DONE_F32) return MRX_ERR_INVALID_ARG;
    if (done_dtype == MRX_DONE_F32 && !aligned(done, 4)) return MRX_ERR_INVALID_ARG;
    const size_t ea = dtype == MRX_BF16 ? 2 : 4;  // z, h~, h in `dtype`; the carries in float32
    for (const void *p : {z, h_tilde, (const void *)h, gate, (const void *)y})
        if (!aligned(p, ea)) return MRX_ERR_INVALID_ARG;
    for (const void *p : {h0, P0, (const void *)h_last, (const void *)P_last, (const void *)ends})
        if (!aligned(p, 4)) return MRX_ERR_INVALID_ARG;
    float *const last = ends ? ends + B * D : nullptr;
    if (dtype == MRX_BF16)
        return launch_fwd<float, true, __bf16>((hipStream_t)stream, {(const __bf16 *)gate, (__bf16 *)y, nullptr, ends, last}, z, h_tilde, done, done_dtype, h0, P0, h,
                                               h_last, P_last, B, T, D, 0, workspace);
    return launch_fwd<float, true>((hipStream_t)stream, {(const float *)gate, (float *)y, nullptr, ends, last}, z, h_tilde, done, done_dtype, h0, P0, h, h_last, P_last, B, T,
                                   D, 0, workspace);
}

}  // namespace

extern "C" int mrx_mingru_scan_fwd(void *stream, const void *z, const void *h_tilde, const void *done, const void *h0, const void *P0,
                                   void *h, void *h_last, void *P_last, int64_t B, int64_t T, int64_t D, int dtype, int done_dtype)
{
    return mingru_scan_fwd(stream, nullptr, nullptr, nullptr, z, h_tilde, done, h0, P0, h, h_last, P_last, B, T, D, dtype, done_dtype, nullptr);
}

extern "C" int mrx_mingru_scan_fwd_segmented(void *stream, const void *z, const void *h_tilde, const void *done, const void *h0, const
                                             void *P0, void *h, void *h_last, void *P_last, int64_t B, int64_t T, int64_t D, int dtype,
                                             int done_dtype, void *workspace)
{
    if (!aligned(workspace, 8)) return MRX_ERR_INVALID_ARG;
    return mingru_scan_fwd(stream, nullptr, nullptr, nullptr, z, h_tilde, done, h0, P0, h, h_last, P_last, B, T, D, dtype, done_dtype, workspace);
}

namespace {

int mingru_scan_bwd(void *stream, const void *gate, void *dgate, const float *ends, const void *z, const void *h_tilde, const void *h, const void *done, const void *h0, const void *g,
                    const void *g_last, void *dz, void *dh_tilde, void *dh0, int64_t B, int64_t T, int64_t D, int dtype, int done_dtype,
                    void *workspace)
{
    if (!z || !h_tilde || !h || !done || !g || !dz || !dh_tilde) return MRX_ERR_INVALID_ARG;
    if (!scan_shape_ok(B, T, D)) return MRX_ERR_INVALID_ARG;
    if (dtype != MRX_F32 && dtype != MRX_BF16) return dtype == MRX_C64 ? MRX_ERR_UNSUPPORTED : MRX_ERR_INVALID_ARG;
    if (done_dtype != MRX_DONE_U8 && done_dtype != MRX_DONE_F32) return MRX_ERR_INVALID_ARG;
    if (done_dtype == MRX_DONE_F32 && !aligned(done, 4)) return MRX_ERR_INVALID_ARG;
    const size_t ea = dtype == MRX_BF16 ? 2 : 4;  // z, h~, h, g, dz, dh~ in `dtype`; the carries in float32
    for (const void *p : {z, h_tilde, h, g, (const void *)dz, (const void *)dh_tilde, gate, (const void *)dgate})
        if (!aligned(p, ea)) return MRX_ERR_INVALID_ARG;
    for (const void *p : {h0, g_last, (const void *)dh0, (const void *)ends})
        if (!aligned(p, 4)) return MRX_ERR_INVALID_ARG;
    float *const last = ends ? const_cast<float *>(ends) + B * D : nullptr;   // (read only)
    if (dtype == MRX_BF16)
        return launch_bwd<float, true, __bf16>((hipStream_t)stream, {(const __bf16 *)gate, nullptr, (__bf16 *)dgate, nullptr, last}, z, h_tilde, h, done, done_dtype, h0, g, g_last, dz,
                                               dh_tilde, dh0, B, T, D, 0, 0, workspace);
    return launch_bwd<float, true>((hipStream_t)stream, {(const float *)gate, nullptr, (float *)dgate, nullptr, last}, z, h_tilde, h, done, done_dtype, h0, g, g_last, dz, dh_tilde,
                                   dh0, B, T, D, 0, 0, workspace);
}

}  // namespace

extern "C" int mrx_mingru_scan_bwd(void *stream, const void *z, const void *h_tilde, const void *h, const void *done, const void *h0,
                                   const void *g, const void *g_last, void *dz, void *dh_tilde, void *dh0, int64_t B, int64_t T, int64_t
                                   D, int dtype, int done_dtype)
{
    return mingru_scan_bwd(stream, nullptr, nullptr, nullptr, z, h_tilde, h, done, h0, g, g_last, dz, dh_tilde, dh0, B, T, D, dtype, done_dtype, nullptr);
}

extern "C" int mrx_mingru_scan_bwd_segmented(void *stream, const void *z, const void *h_tilde, const void *h, const void *done, const void
                                             *h0, const void *g, const void *g_last, void *dz, void *dh_tilde, void *dh0, int64_t B,
                                             int64_t T, int64_t D, int dtype, int done_dtype, void *workspace)
{
    if (!aligned(workspace, 8)) return MRX_ERR_INVALID_ARG;
    return mingru_scan_bwd(stream, nullptr, nullptr, nullptr, z, h_tilde, h, done, h0, g, g_last, dz, dh_tilde, dh0, B, T, D, dtype, done_dtype, workspace);
}

// Where the gate inside the scan takes less time than the operations that it stands for, which read and write flat arrays in whole lines whatever the rows
// are.  Behind 512 MB of other traffic, us, operations / one; shapes drawn over 3 to 120 million elements, 32 to 1024 columns: of 290 drawn once the rule stood,
// time by it over time apart is 0.88 forward and 0.91 backward in float32, 0.94 and 0.93 in bfloat16, worst 1.12, 26 of 580 above 1.03.
extern "C" int mrx_gated_scan_pays(int64_t B, int64_t T, int64_t D, int dtype, int backward)
{
    if (!scan_shape_ok(B, T, D) || (dtype != MRX_F32 && dtype != MRX_BF16)) return 0;
    const bool half = dtype == MRX_BF16;
    const ScanPlan pl = plan_scan(B, T, D, 4, backward != 0, true, half, false);
    const int64_t n = B * T * D, row = D * (half ? 2 : 4);
    if (!backward) {
        if (n < (half ? 10000000 : 12000000)) return 1;   // launches saved weigh more: bfloat16 878 x 245 x 39 50 / 48, float32 268 x 195 x 86 50 / 49
        // One more array each way of loads and stores that begin in the middle of a line.  bfloat16, wave-split, rows of no whole lines: 2010 x 675 x 34 191 / 264,
        // 1006 x 266 x 144 134 / 159, 170 x 521 x 810 235 / 279, at 10 to 15 million 0.97 to 1.11; whole lines 896 x 442 x 192 204 / 204, 1024 x 512 x 256 325 / 271.
        // Streams of two elements a lane are even (0.87 to 1.06), of one 68282 x 25 x 37 269 / 317.
        if (half) return row % 128 == 0 || (pl.stream && pl.vec > 1);
        // float32: single elements, unless a row is one wave's: 4274 x 38 x 131 145 / 173, 271 x 963 x 68 155 / 184, 25735 x 26 x 44 194 / 213; 28605 x 70 x 43 503 / 463,
        // rows of whole half lines 17302 x 23 x 144 305 / 259, two elements and more 0.59 to 1.06
        return pl.vec > 1 || row % 64 == 0 || (!pl.stream && D <= 64);
    }
    // whole rows streaming, few columns each: single elements of rows narrower than a wave, bfloat16 68282 x 25 x 37 394 / 449, float32 1416 x 449 x 49 456 / 515 (43772 x 30 x 40
    // 521 / 495), bfloat16 also four elements of rows narrower than two, 6904 x 106 x 41 281 / 340, 2514 x 125 x 124 260 / 281; whole half lines 16384 x 64 x 128 533 / 380
    if (pl.stream && row % 64 && n >= 9000000 && ((pl.vec == 1 && D < 64) || (half && pl.vec == 4 && D < 128))) return 0;
    // float32 plans of four elements run with two (launch_bwd): a second column tile that is half empty costs more than the pass, 917 x 141 x 165 200 / 250, 2843 x 220 x 158
    // 935 / 1075, 674 x 76 x 147 81 / 87; whole half lines 563 x 667 x 144 590 / 502, wider rows 3939 x 115 x 216 876 / 832
    return half || pl.stream || pl.vec < 4 || D > 208 || row % 64 == 0 || n < 6000000;
}

extern "C" int mrx_gated_scan_fwd(void *stream, const void *z, const void *h_tilde, const void *gate, const void *done, const float *log_state,
                                  const float *log_decay, void *h, void *y, float *log_state_out, float *log_decay_out, float *ends, int64_t B, int64_t T,
                                  int64_t D, int dtype, int done_dtype)
{
    if (!gate || !y) return MRX_ERR_INVALID_ARG;
    return mingru_scan_fwd(stream, gate, y, ends, z, h_tilde, done, log_state, log_decay, h, log_state_out, log_decay_out, B, T, D, dtype, done_dtype, nullptr);
}

extern "C" int mrx_gated_scan_bwd(void *stream, const void *z, const void *h_tilde, const void *gate, const void *h, const void *done,
                                  const float *ends, const void *dy, const float *g_last, void *dz, void *dh_tilde, void *dgate,
                                  float *dlog_state, int64_t B, int64_t T, int64_t D, int dtype, int done_dtype)
{
    if (!gate || !dgate || !ends) return MRX_ERR_INVALID_ARG;
    return mingru_scan_bwd(stream, gate, dgate, ends, z, h_tilde, h, done, ends, dy, g_last, dz, dh_tilde, dlog_state, B, T, D, dtype, done_dtype, nullptr);
}

namespace {

// One acting step of the MinGRU cell with its carry in the reference's log-space leaves, and the gated read-out of the
// block around it: exp of the carried state, the element map, the update, its logarithm and the product with silu(gate) are
// one pass over (B,D) arrays of a few hundred kilobytes -- eight launches as separate operations.
template <typename S, int VEC>
__global__ void __launch_bounds__(256) mingru_step_kernel(const S *__restrict__ z, const S *__restrict__ x, const S *__restrict__ gate,
                                                          const void *__restrict__ done, int done_f32, const float *log_state,
                                                          const float *log_decay, S *__restrict__ y, float *log_state_out,
                                                          float *log_decay_out, int64_t n, int64_t D)  // the carry may be updated in place
{
    const int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * VEC;
    if (at >= n) return;
    const bool reset = done_at(done, done_f32, at / D);
    const Vec<float, VEC> zv = cvtv<S, float, VEC>(ldraw<S, VEC>(z + at)), xv = cvtv<S, float, VEC>(ldraw<S, VEC>(x + at));
    Vec<float, VEC> gv = vfill<float, VEC>(0.f), ls = ldc<float, VEC>(log_state + at), ld = ldc<float, VEC>(log_decay + at), out;
    if (gate) gv = cvtv<S, float, VEC>(ldraw<S, VEC>(gate + at));
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
        float a = zv.v[i], b = xv.v[i];
        const float log_a = -(fmaxf(a, 0.f) + log1pf(expf(-fabsf(a))));   // log sigma(-z)
        MinGru::coeffs(a, b);
        const float h = reset ? b : a * expf(ls.v[i]) + b;
        ls.v[i] = logf(h);
        ld.v[i] = reset ? log_a : ld.v[i] + log_a;
        const float hs = (float)(S)h, g = gv.v[i];   // the state as the cell hands it on
        out.v[i] = gate ? hs * g / (1.f + __expf(-g)) : hs;
    }
    stc<float, VEC>(log_state_out + at, ls);
    stc<float, VEC>(log_decay_out + at, ld);
    stv<S, float, VEC>(y + at, out);
}

}  // namespace

extern "C" int mrx_mingru_step(void *stream, const void *z, const void *h_tilde, const void *gate, const void *done, const float *log_state,
                               const float *log_decay, void *y, float *log_state_out, float *log_decay_out, int64_t B, int64_t D, int dtype,
                               int done_dtype)
{
    if (!z || !h_tilde || !done || !log_state || !log_decay || !y || !log_state_out || !log_decay_out || B <= 0 || D <= 0)
        return MRX_ERR_INVALID_ARG;
    if ((dtype != MRX_F32 && dtype != MRX_BF16) || (done_dtype != MRX_DONE_U8 && done_dtype != MRX_DONE_F32)) return MRX_ERR_INVALID_ARG;
    if (B >= (1ll << 31) || D >= (1ll << 31)) return MRX_ERR_INVALID_ARG;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    bool quads = D % 4 == 0;   // rows of whole quads, every array on a 16-byte boundary
    for (const void *p : {z, h_tilde, gate, (const void *)log_state, (const void *)log_decay, (const void *)y, (const void *)log_state_out,
                          (const void *)log_decay_out})
        quads = quads && aligned(p, 16);
    const int64_t n = B * D, wgs = (n / (quads ? 4 : 1) + 255) / 256;
    if (wgs >= (1ll << 31)) return MRX_ERR_INVALID_ARG;
    auto go = [&](auto s, auto vec) {
        using S = decltype(s);
        return launch_kernel(mingru_step_kernel<S, decltype(vec)::value>, dim3((unsigned)wgs), dim3(256), 0, (hipStream_t)stream,
                             (const S *)z, (const S *)h_tilde, (const S *)gate, done, int(done_dtype == MRX_DONE_F32), log_state, log_decay,
                             (S *)y, log_state_out, log_decay_out, n, D);
    };
    using One = std::integral_constant<int, 1>;
    using Four = std::integral_constant<int, 4>;
    if (dtype == MRX_BF16) return quads ? go(__bf16(), Four{}) : go(__bf16(), One{});
    return quads ? go(float(), Four{}) : go(float(), One{});
}

extern "C" int mrx_column_sum(void *stream, const float *x, float *out, int64_t rows, int64_t columns)
{
    using namespace mrx;
    if (!x || !out || rows <= 0 || columns <= 0 || rows >= (1ll << 31) || columns >= (1ll << 31)) return MRX_ERR_INVALID_ARG;
    if (const int rc = prepare_device(); rc != MRX_OK) return rc;
    return launch_column_sum((hipStream_t)stream, x, out, nullptr, (int)rows, (int)columns);
}
