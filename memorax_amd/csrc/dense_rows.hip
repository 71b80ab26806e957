// Dense layers over many rows in bfloat16, forward and with respect to their input:
//
//     y_l = x W_l^T + b_l          up to three layers of one width that read the same rows, and one of up to eight outputs beside them
//     y   = x_res + (x W^T + b)    the layer that closes a residual branch of a float32 stream; its own result is rounded first, as by itself
//     dx  = sum_l dy_l W_l         of such a group, or of one layer whose gradient is float32 (the stream's; its rounded copy, which the
//                                  parameters' gradients read, is a by-product)
//
// With a hundred thousand rows and 64 to 256 features on either side all of them are bound by reading and writing the rows: three layers
// of 256 are 268 MB and 52 GFLOP.  A product of the array library per layer reads the shared rows again for each (and writes and
// reads the sum so far of dx), takes the residual sum and the cast of its gradient as passes of their own, and re-reads the weights for
// every tile.  Here the weights stay in registers: a workgroup of eight waves lives as long as the launch, one on a compute unit, each
// wave holds the weights of its 16 or 32 output columns for the whole contraction (three layers of 256: 192 registers a lane), and
// the rows stream through LDS past all of them, so that nothing but rows moves once the launch is under way.  The rows go from memory to
// LDS without passing through registers, in a ring of tiles with as many on their way as LDS holds; each wave counts its own
// requests and there is one barrier a tile.  Pieces of 16 bytes are exchanged within a row as they are requested (`swz`), so that the
// sixteen rows of an operand fragment lie in different banks.
// 131072 rows x 256, us: three layers forward 96 -> 60 (with one of 4 beside them 113 -> 63), dx of three 110 -> 60, closing layer and sum
// 89 -> 60, its dx with the cast 70 -> 48: 4.5 to 5.6 TB/s.
#include "chunk_common.h"
#include "row_dma.h"

namespace mrx {
namespace {

constexpr int DR_WAVES = 8, DR_THREADS = 64 * DR_WAVES, DR_WIDE = 3, DR_NARROW = 8, DR_LDS = 156 * 1024;

struct DenseRowsArgs {
    const void *x[DR_WIDE];          // forward: x[0]; input gradient: the layers' dy
    const __bf16 *w[DR_WIDE];        // forward: (n, contraction) of each layer; input gradient: w[0] (n, contraction of all), w[1] (nn, n)
    const void *b[DR_WIDE], *bn;
    void *y[DR_WIDE];
    const float *res;                // (rows, n)
    const __bf16 *wn;                // the narrow layer's weights (nn, contraction; input gradient: (nn, n))
    const void *xn;                  // input gradient: the narrow layer's dy (rows, nn)
    __bf16 *yn;                      // forward: its output
    __bf16 *copy;                    // input gradient of a float32 dy: its bfloat16 copy
    int n, nn, groups, groups_per_layer;
    int64_t rows;
    bool b_bf16;
};

// What a tile is: the fewest rows whose requests divide over the waves, and as many tiles as LDS holds, at most eight.
constexpr bool whole_ops(int bytes) { return bytes % (1024 * DR_WAVES) == 0; }
template <int SEGS, int KBS, bool XF32, int RC, bool XN> struct RowsTile {
    static constexpr int RB = 32 * KBS * (XF32 ? 4 : 2);                               // bytes of a row of one input
    static constexpr int rows_for(int tr) { return whole_ops(SEGS * tr * RB) && whole_ops(tr * RC * 4) ? tr : rows_for(2 * tr); }
    static constexpr int TR = rows_for(SEGS == 1 && RC == 0 ? 32 : 16);
    static constexpr int SEG = TR * RB, RES = TR * RC * 4;
    static constexpr int NOPS = XN ? TR * DR_NARROW * 2 / 256 : 0, NB = NOPS * 256;    // the narrow rows: a copy for each wave
    static constexpr int STAGE = SEGS * SEG + RES + DR_WAVES * NB;
    static constexpr int STAGES = DR_LDS / STAGE < 8 ? DR_LDS / STAGE : 8;
    static constexpr int XOPS = SEGS * SEG / 1024 / DR_WAVES, ROPS = RES / 1024 / DR_WAVES, OPS = XOPS + ROPS + NOPS;
    static_assert(STAGES >= 2, "a tile in use and one on its way");
};

// Where the 16-byte piece q of row r lies in a tile of SPR pieces a row: at q ^ swz(r).
template <int SPR> __device__ __forceinline__ int swz(int r) { return SPR >= 16 ? r & 15 : r / (16 / SPR) & (SPR - 1); }

// SEGS inputs of 32 KBS features; XF32: float32, rounded on the way to the product; NT: 16-column tiles per wave; RC: columns of the
// residual rows that a workgroup takes (0: none); YN / XN: a narrow layer's output / input beside the wide ones.
template <int SEGS, int KBS, bool XF32, int NT, int RC, bool YN, bool XN>
__global__ void __launch_bounds__(DR_THREADS, 1) dense_rows_kernel(DenseRowsArgs a)
{
    using Tile = RowsTile<SEGS, KBS, XF32, RC, XN>;
    constexpr int TR = Tile::TR, RB = Tile::RB, SPR = RB / 16, MT = TR / 16, STAGES = Tile::STAGES;
    constexpr int STORES = MT * (RC ? NT : 1);   // of a tile, at least
    constexpr int RSPR = RC ? RC / 4 : 16;
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 15, g = lane >> 4;
    // column groups that read the same rows follow each other on one die
    const int slot = blockIdx.x >> 3, group = slot % a.groups;
    const int workers = (int)(gridDim.x >> 3) / a.groups * 8, worker = slot / a.groups * 8 + (int)(blockIdx.x & 7);
    const int l = group / a.groups_per_layer, g0 = group % a.groups_per_layer * (128 * NT), c0 = g0 + wv * 16 * NT;
    const int64_t tiles = (a.rows + TR - 1) / TR;
    if (worker >= tiles) return;
    const uint32_t lds0 = lds_address(smem);

    // every request of a tile is made whatever exists of it: rows past the last are the last one, tiles past the last are the last one
    auto request = [&](int64_t t, int stage) {
        if (t >= tiles) t = tiles - 1;
        const int64_t r0 = t * TR;
        const int last = (int)(a.rows - 1 - r0 < TR - 1 ? a.rows - 1 - r0 : TR - 1);
        const uint32_t at = lds0 + stage * Tile::STAGE;
#pragma unroll
        for (int p = 0; p < Tile::XOPS; ++p) {
            const int op = wv * Tile::XOPS + p, s = SEGS == 1 ? 0 : op / (Tile::SEG / 1024), o = SEGS == 1 ? op : op % (Tile::SEG / 1024);
            const int r = o * 64 / SPR + lane / SPR, q = lane % SPR ^ swz<SPR>(r);
            dma16(static_cast<const char *>(a.x[s]) + r0 * RB, (uint32_t)((r < last ? r : last) * RB + q * 16), at + op * 1024);
        }
        if constexpr (RC > 0)
#pragma unroll
            for (int p = 0; p < Tile::ROPS; ++p) {
                const int o = wv * Tile::ROPS + p, r = o * 64 / RSPR + lane / RSPR, q = lane % RSPR ^ swz<RSPR>(r);
                dma16(reinterpret_cast<const char *>(a.res + r0 * a.n + g0), (uint32_t)(r < last ? r : last) * (uint32_t)a.n * 4 + q * 16,
                      at + SEGS * Tile::SEG + o * 1024);
            }
        if constexpr (XN) {
            const uint32_t end = (uint32_t)((last + 1) * a.nn * 2 - 4);
#pragma unroll
            for (int p = 0; p < Tile::NOPS; ++p) {
                const uint32_t off = (uint32_t)(p * 256 + lane * 4);
                dma4(static_cast<const char *>(a.xn) + r0 * a.nn * 2, off < end ? off : end, at + SEGS * Tile::SEG + wv * Tile::NB + p * 256);
            }
        }
    };
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s) request(worker + (int64_t)s * workers, s);

    // Row m of the operand tile j is column c0 + 4 NT (m / 4) + 4 j + m % 4, so that a lane ends up with 4 NT columns in a row.  Columns past
    // the last are the last one; their results are dropped.
    bf16x8 w[SEGS * KBS][NT], wn[YN ? KBS : 1][XN ? NT : 1];
    f32x4 bias[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int c = c0 + 4 * NT * (i >> 2) + 4 * j + (i & 3), col = c < a.n ? c : a.n - 1;
#pragma unroll
        for (int k = 0; k < SEGS * KBS; ++k)
            w[k][j] = *reinterpret_cast<const bf16x8 *>(a.w[l] + (int64_t)col * (SEGS * KBS * 32) + 32 * k + 8 * g);
        if constexpr (XN) {
            wn[0][j] = bf16x8{};
            if (g == 0)
#pragma unroll
                for (int e = 0; e < DR_NARROW; ++e)
                    if (e < a.nn) wn[0][j][e] = a.wn[(int64_t)e * a.n + col];
        }
        bias[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int bc = c0 + 4 * NT * g + 4 * j;
        if (a.b[l] && bc < a.n)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                bias[j][v] = a.b_bf16 ? (float)static_cast<const __bf16 *>(a.b[l])[bc + v] : (float)(__bf16)static_cast<const float *>(a.b[l])[bc + v];
    }
    // the narrow layer's columns are row tile by row tile the work of one more wave each, of the first group
    const bool narrow = YN && group == 0 && wv < MT;
    f32x4 bias_n = {0.f, 0.f, 0.f, 0.f};
    if constexpr (YN) {
        const int c = i < a.nn ? i : a.nn - 1;
#pragma unroll
        for (int k = 0; k < KBS; ++k) wn[k][0] = *reinterpret_cast<const bf16x8 *>(a.wn + c * (KBS * 32) + 32 * k + 8 * g);
        if (a.bn)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (4 * g + v < a.nn)
                    bias_n[v] = a.b_bf16 ? (float)static_cast<const __bf16 *>(a.bn)[4 * g + v] : (float)(__bf16)static_cast<const float *>(a.bn)[4 * g + v];
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0), here and not in the loop

    // rows 16 m + i of input s, features 32 k + 8 g .. + 7
    auto fragment = [&](const unsigned char *tile, int s, int k, int m) {
        const unsigned char *row = tile + s * Tile::SEG + (16 * m + i) * RB;
        const int sw = swz<SPR>(16 * m + i);
        if constexpr (XF32) {
            const f32x4 lo = *reinterpret_cast<const f32x4 *>(row + ((8 * k + 2 * g) ^ sw) * 16),
                        hi = *reinterpret_cast<const f32x4 *>(row + ((8 * k + 2 * g + 1) ^ sw) * 16);
            const bf16x4 l4 = TT<__bf16>::pack(lo[0], lo[1], lo[2], lo[3]), h4 = TT<__bf16>::pack(hi[0], hi[1], hi[2], hi[3]);
            return __builtin_shufflevector(l4, h4, 0, 1, 2, 3, 4, 5, 6, 7);
        } else {
            return *reinterpret_cast<const bf16x8 *>(row + ((4 * k + g) ^ sw) * 16);
        }
    };

    int stage = 0, early = c0 < a.n ? STAGES - 1 : 1 << 30;   // a wave without columns stores nothing
    for (int64_t t = worker; t < tiles; t += workers) {
        // since this tile was requested this wave has requested STAGES - 2 others and stored STAGES - 1 results
        if (early > 0) {
            wait_vm<(STAGES - 2) * Tile::OPS>();
            --early;
        } else {
            wait_vm<(STAGES - 2) * Tile::OPS + (STAGES - 1) * STORES>();
        }
        sync_lds();   // every wave has its part, and is done with the tile before, whose place the next request takes
        request(t + (int64_t)(STAGES - 1) * workers, stage == 0 ? STAGES - 1 : stage - 1);
        const unsigned char *tile = smem + stage * Tile::STAGE;
        f32x4 acc[MT][NT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[m][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < SEGS; ++s)
#pragma unroll
            for (int k = 0; k < KBS; ++k)
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    const bf16x8 f = fragment(tile, s, k, m);
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[m][j] = TT<__bf16>::mma(w[s * KBS + k][j], f, acc[m][j]);
                }
        if constexpr (XN) {
            const unsigned char *rows_n = tile + SEGS * Tile::SEG + wv * Tile::NB;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                uint32_t q[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    q[e] = g == 0 && 2 * e < a.nn ? *reinterpret_cast<const uint32_t *>(rows_n + (16 * m + i) * a.nn * 2 + 4 * e) : 0u;
                typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
                const bf16x8 f = __builtin_bit_cast(bf16x8, u32x4{q[0], q[1], q[2], q[3]});
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[m][j] = TT<__bf16>::mma(wn[0][j], f, acc[m][j]);
            }
        }
        const int64_t r0 = t * TR;
        const int col = c0 + 4 * NT * g;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int64_t r = r0 + 16 * m + i;
            if (r >= a.rows || col >= a.n) continue;
            if constexpr (RC > 0) {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const int q = (wv * 16 * NT + 4 * NT * g) / 4 + j;
                    const f32x4 x = *reinterpret_cast<const f32x4 *>(tile + SEGS * Tile::SEG + (16 * m + i) * (RC * 4) + (q ^ swz<RSPR>(16 * m + i)) * 16);
                    const f32x4 z = acc[m][j] + bias[j];
                    const bf16x4 y = TT<__bf16>::pack(z[0], z[1], z[2], z[3]);
                    *reinterpret_cast<f32x4 *>(static_cast<float *>(a.y[l]) + r * a.n + col + 4 * j) = x + f32x4{(float)y[0], (float)y[1], (float)y[2], (float)y[3]};
                }
            } else {
                bf16x4 p[NT];
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const f32x4 y = acc[m][j] + bias[j];
                    p[j] = TT<__bf16>::pack(y[0], y[1], y[2], y[3]);
                }
                __bf16 *y = static_cast<__bf16 *>(a.y[l]) + r * a.n + col;
                if constexpr (NT == 2) *reinterpret_cast<bf16x8 *>(y) = __builtin_shufflevector(p[0], p[1], 0, 1, 2, 3, 4, 5, 6, 7);
                else *reinterpret_cast<bf16x4 *>(y) = p[0];
            }
        }
        if constexpr (XF32) {
            if (a.copy && group == 0 && wv < KBS)
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    if (r0 + 16 * m + i < a.rows)
                        *reinterpret_cast<bf16x8 *>(a.copy + (r0 + 16 * m + i) * (32 * KBS) + 32 * wv + 8 * g) = fragment(tile, 0, wv, m);
        }
        if constexpr (YN) {
            if (narrow) {
                f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < KBS; ++k) y = TT<__bf16>::mma(wn[k][0], fragment(tile, 0, k, wv), y);
                y += bias_n;
                const int64_t r = r0 + 16 * wv + i;
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (r < a.rows && 4 * g + v < a.nn) a.yn[r * a.nn + 4 * g + v] = (__bf16)y[v];
            }
        }
        stage = stage == STAGES - 1 ? 0 : stage + 1;
    }
    wait_vm<0>();   // LDS goes to another workgroup once this one is gone
}

template <int SEGS, int KBS, bool XF32, int NT, int RC, bool YN, bool XN> struct Launch {
    using Tile = RowsTile<SEGS, KBS, XF32, RC, XN>;
    static constexpr auto kernel = dense_rows_kernel<SEGS, KBS, XF32, NT, RC, YN, XN>;
    static inline const KernelRegistrar registrar{reinterpret_cast<const void *>(kernel), Tile::STAGES * Tile::STAGE};
    static int go(hipStream_t st, const DenseRowsArgs &a, int cus)
    {
        (void)&registrar;
        const int64_t tiles = (a.rows + Tile::TR - 1) / Tile::TR;
        // workgroups of a column group on one die: as many as it has compute units for, no more than there are tiles
        int64_t per = cus / 8 / a.groups;
        per = per < 1 ? 1 : per;
        per = (tiles + 7) / 8 < per ? (tiles + 7) / 8 : per;
        return launch_kernel(kernel, dim3((unsigned)(8 * a.groups * per)), dim3(DR_THREADS), Tile::STAGES * Tile::STAGE, st, a);
    }
};

// 32-feature blocks of a contraction of 64, 128 or 256; 0 otherwise: `swz` exchanges the pieces of a row within a power of two
int blocks_of(int64_t k) { return k == 64 ? 2 : k == 128 ? 4 : k == 256 ? 8 : 0; }

struct Group {
    int wide = 0, narrow = -1;   // layers of n outputs, the one of nn
    int64_t n = 0, nn = 0;
    int at[DR_WIDE] = {};
    bool ok = true;
};
Group group_of(const int64_t *n, int layers)
{
    Group r;
    for (int l = 0; l < layers; ++l) {
        if (n[l] <= DR_NARROW && r.narrow < 0) {
            r.narrow = l, r.nn = n[l];
            continue;
        }
        r.ok = r.ok && r.wide < DR_WIDE && n[l] >= 64 && (r.wide == 0 || n[l] == r.n);
        if (r.ok) r.at[r.wide++] = l, r.n = n[l];
    }
    r.ok = r.ok && r.wide > 0;
    return r;
}
int columns_per_group(int64_t n) { return n <= 128 ? 128 : 256; }

// No line at few rows: a layer's launch is then its weights' way into registers (11 us for 256 x 256, the pack included, 7 to 10 as the array
// library's cast and product), but the calls cost more than that -- us, forward and backward here / as the array library's, issued by the host: three
// layers of 256 104 / 169 at 16 rows and 106 / 172 at 1024, one of 64 71 / 113 and 76 / 116; in a graph 31 / 36 and 42 / 46, 11.8 / 11.2 and
// 17.3 / 16.0, one of 256 22 / 18 and 30 / 24.

bool forward_suits(const Group &gr, int64_t K)
{
    return gr.ok && blocks_of(K) && gr.n % 8 == 0 && gr.n <= 1024 && gr.wide * ((gr.n + 255) / 256) <= 4;
}
bool residual_suits(const Group &gr, int64_t K) { return gr.ok && gr.wide == 1 && gr.narrow < 0 && blocks_of(K) && blocks_of(gr.n); }
bool input_suits(const Group &gr, int64_t K)
{
    return gr.ok && blocks_of(gr.n) && K % 8 == 0 && K >= 64 && K <= 1024 && (gr.narrow < 0 || (gr.wide == DR_WIDE && gr.nn % 2 == 0));
}

template <int KBS> int forward(hipStream_t st, const DenseRowsArgs &a, int cus)
{
    const bool narrow = a.n <= 128;
    if (a.yn) return narrow ? Launch<1, KBS, false, 1, 0, true, false>::go(st, a, cus) : Launch<1, KBS, false, 2, 0, true, false>::go(st, a, cus);
    return narrow ? Launch<1, KBS, false, 1, 0, false, false>::go(st, a, cus) : Launch<1, KBS, false, 2, 0, false, false>::go(st, a, cus);
}
template <int KBS> int closing(hipStream_t st, const DenseRowsArgs &a, int cus)
{
    return a.n == 64 ? Launch<1, KBS, false, 1, 64, false, false>::go(st, a, cus)
           : a.n == 128 ? Launch<1, KBS, false, 1, 128, false, false>::go(st, a, cus)
                        : Launch<1, KBS, false, 2, 256, false, false>::go(st, a, cus);
}
template <int KBS> int input_grad(hipStream_t st, const DenseRowsArgs &a, int segs, bool f32, int cus)
{
    const bool one = a.n <= 128;
    if (f32) return one ? Launch<1, KBS, true, 1, 0, false, false>::go(st, a, cus) : Launch<1, KBS, true, 2, 0, false, false>::go(st, a, cus);
    if (segs == 1) return one ? Launch<1, KBS, false, 1, 0, false, false>::go(st, a, cus) : Launch<1, KBS, false, 2, 0, false, false>::go(st, a, cus);
    if (segs == 2) return one ? Launch<2, KBS, false, 1, 0, false, false>::go(st, a, cus) : Launch<2, KBS, false, 2, 0, false, false>::go(st, a, cus);
    if (a.xn) return one ? Launch<3, KBS, false, 1, 0, false, true>::go(st, a, cus) : Launch<3, KBS, false, 2, 0, false, true>::go(st, a, cus);
    return one ? Launch<3, KBS, false, 1, 0, false, false>::go(st, a, cus) : Launch<3, KBS, false, 2, 0, false, false>::go(st, a, cus);
}

// ---- the weights as the products read them: bfloat16 copies, and the wide layers' transposed side by side, (K, wide n)
struct PackArgs {
    const void *w[MRX_DENSE_LAYERS];
    __bf16 *copy[MRX_DENSE_LAYERS], *transposed;
    int n[MRX_DENSE_LAYERS], first[MRX_DENSE_LAYERS + 1], at[MRX_DENSE_LAYERS];   // first 64 x 64 tile; column in `transposed`, -1: not there
    int layers, K, wide;
    bool w_bf16;
};
__global__ void __launch_bounds__(256) dense_pack_kernel(PackArgs a)
{
    __shared__ __bf16 tile[64][65];
    const int b = blockIdx.x, tid = threadIdx.x, kt = (a.K + 63) / 64;
    int l = 0;
    while (b >= a.first[l + 1]) ++l;
    const int n0 = (b - a.first[l]) / kt * 64, k0 = (b - a.first[l]) % kt * 64, N = a.n[l];
    // four columns of four rows a thread, all of them requested before the first is used; K and thus a row's quads are whole
    const int c = tid % 16 * 4;
    bf16x4 v[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int r = n0 + tid / 16 + 16 * p;
        v[p] = bf16x4{};
        if (r >= N || k0 + c >= a.K) continue;
        const int64_t at = (int64_t)r * a.K + k0 + c;
        if (a.w_bf16) {
            v[p] = *reinterpret_cast<const bf16x4 *>(static_cast<const __bf16 *>(a.w[l]) + at);
        } else {
            const f32x4 x = *reinterpret_cast<const f32x4 *>(static_cast<const float *>(a.w[l]) + at);
            v[p] = TT<__bf16>::pack(x[0], x[1], x[2], x[3]);
        }
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int r = tid / 16 + 16 * p;
        if (a.copy[l] && n0 + r < N && k0 + c < a.K) *reinterpret_cast<bf16x4 *>(a.copy[l] + (int64_t)(n0 + r) * a.K + k0 + c) = v[p];
#pragma unroll
        for (int e = 0; e < 4; ++e) tile[r][c + e] = v[p][e];
    }
    if (!a.transposed || a.at[l] < 0) return;
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 16; ++p) {
        const int k = tid / 64 + 4 * p, r = tid % 64;
        if (n0 + r < N && k0 + k < a.K) a.transposed[(int64_t)(k0 + k) * a.wide + a.at[l] + n0 + r] = tile[r][k];
    }
}

}  // namespace
}  // namespace mrx

extern "C" int mrx_dense_rows_suit(int64_t rows, int64_t K, const int64_t *n_out, int layers)
{
    using namespace mrx;
    if (!n_out || layers < 1 || layers > DR_WIDE + 1 || rows <= 0 || rows >= (1ll << 31)) return 0;
    const Group g = group_of(n_out, layers);
    return (forward_suits(g, K) ? MRX_DENSE_ROWS_FORWARD : 0) | (residual_suits(g, K) ? MRX_DENSE_ROWS_RESIDUAL : 0) |
           (input_suits(g, K) ? MRX_DENSE_ROWS_INPUT : 0);
}

extern "C" int mrx_dense_pack(void *stream, const void *const *weights, const int64_t *n_out, int layers, int64_t K, int w_dtype,
                              void *const *copies, void *transposed)
{
    using namespace mrx;
    if (!weights || !n_out || layers < 1 || layers > MRX_DENSE_LAYERS || K <= 0 || K % 4 != 0 || K > (1 << 16) || (w_dtype != MRX_F32 && w_dtype != MRX_BF16))
        return MRX_ERR_INVALID_ARG;
    PackArgs a{};
    a.layers = layers, a.K = (int)K, a.w_bf16 = w_dtype == MRX_BF16, a.transposed = static_cast<__bf16 *>(transposed);
    for (int l = 0; l < layers; ++l) {
        if (!weights[l] || n_out[l] <= 0 || n_out[l] > (1 << 16) || !aligned(weights[l], 16) || (copies && !aligned(copies[l], 8))) return MRX_ERR_INVALID_ARG;
        a.w[l] = weights[l], a.copy[l] = copies ? static_cast<__bf16 *>(copies[l]) : nullptr, a.n[l] = (int)n_out[l];
        a.first[l + 1] = a.first[l] + (int)((n_out[l] + 63) / 64 * ((K + 63) / 64));
        a.at[l] = n_out[l] <= DR_NARROW ? -1 : a.wide;
        if (a.at[l] >= 0) a.wide += a.n[l];
    }
    return launch_kernel(dense_pack_kernel, dim3((unsigned)a.first[layers]), dim3(256), 0, static_cast<hipStream_t>(stream), a);
}

extern "C" int mrx_dense_rows(void *stream, const void *x, const void *const *weights, const void *const *biases, void *const *outs,
                              const int64_t *n_out, int layers, const float *residual, int64_t rows, int64_t K, int b_dtype)
{
    using namespace mrx;
    if (!x || !weights || !biases || !outs || (b_dtype != MRX_F32 && b_dtype != MRX_BF16)) return MRX_ERR_INVALID_ARG;
    if (!(mrx_dense_rows_suit(rows, K, n_out, layers) & (residual ? MRX_DENSE_ROWS_RESIDUAL : MRX_DENSE_ROWS_FORWARD))) return MRX_ERR_UNSUPPORTED;
    const Group gr = group_of(n_out, layers);
    DenseRowsArgs a{};
    a.x[0] = x, a.res = residual, a.n = (int)gr.n, a.rows = rows, a.b_bf16 = b_dtype == MRX_BF16;
    a.groups_per_layer = (int)((gr.n + columns_per_group(gr.n) - 1) / columns_per_group(gr.n)), a.groups = a.groups_per_layer * gr.wide;
    if (!aligned(x, 16) || !aligned(residual, 16)) return MRX_ERR_INVALID_ARG;
    for (int l = 0; l < layers; ++l)
        if (!weights[l] || !outs[l] || !aligned(weights[l], 16) || !aligned(outs[l], l == gr.narrow ? 2 : 16)) return MRX_ERR_INVALID_ARG;
    for (int s = 0; s < gr.wide; ++s) a.w[s] = static_cast<const __bf16 *>(weights[gr.at[s]]), a.b[s] = biases[gr.at[s]], a.y[s] = outs[gr.at[s]];
    if (gr.narrow >= 0)
        a.nn = (int)gr.nn, a.wn = static_cast<const __bf16 *>(weights[gr.narrow]), a.bn = biases[gr.narrow], a.yn = static_cast<__bf16 *>(outs[gr.narrow]);
    int cus = 0;
    if (const int rc = prepare_device(&cus); rc != MRX_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int kbs = blocks_of(K);
    if (residual) return kbs == 2 ? closing<2>(st, a, cus) : kbs == 4 ? closing<4>(st, a, cus) : closing<8>(st, a, cus);
    return kbs == 2 ? forward<2>(st, a, cus) : kbs == 4 ? forward<4>(st, a, cus) : forward<8>(st, a, cus);
}

extern "C" int mrx_dense_rows_input_grad(void *stream, const void *const *dys, const int64_t *n_out, int layers, const void *transposed,
                                         const void *narrow_weights, void *dx, void *dy_copy, int64_t rows, int64_t K, int dy_dtype)
{
    using namespace mrx;
    if (!dys || !transposed || !dx || (dy_dtype != MRX_F32 && dy_dtype != MRX_BF16)) return MRX_ERR_INVALID_ARG;
    if (!(mrx_dense_rows_suit(rows, K, n_out, layers) & MRX_DENSE_ROWS_INPUT)) return MRX_ERR_UNSUPPORTED;
    const Group gr = group_of(n_out, layers);
    const bool f32 = dy_dtype == MRX_F32;
    if (f32 && layers != 1) return MRX_ERR_UNSUPPORTED;
    if (gr.narrow >= 0 && (!narrow_weights || !aligned(narrow_weights, 2))) return MRX_ERR_INVALID_ARG;
    if (!aligned(transposed, 16) || !aligned(dx, 16) || !aligned(dy_copy, 16)) return MRX_ERR_INVALID_ARG;
    for (int l = 0; l < layers; ++l)
        if (!dys[l] || !aligned(dys[l], l == gr.narrow ? 4 : 16)) return MRX_ERR_INVALID_ARG;
    DenseRowsArgs a{};
    for (int s = 0; s < gr.wide; ++s) a.x[s] = dys[gr.at[s]];
    a.w[0] = static_cast<const __bf16 *>(transposed), a.y[0] = dx, a.n = (int)K, a.rows = rows, a.copy = static_cast<__bf16 *>(dy_copy);
    a.groups = a.groups_per_layer = (int)((K + columns_per_group(K) - 1) / columns_per_group(K));
    if (gr.narrow >= 0) a.nn = (int)gr.nn, a.xn = dys[gr.narrow], a.wn = static_cast<const __bf16 *>(narrow_weights);
    int cus = 0;
    if (const int rc = prepare_device(&cus); rc != MRX_OK) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int kbs = blocks_of(gr.n);
    return kbs == 2 ? input_grad<2>(st, a, gr.wide, f32, cus) : kbs == 4 ? input_grad<4>(st, a, gr.wide, f32, cus) : input_grad<8>(st, a, gr.wide, f32, cus);
}
