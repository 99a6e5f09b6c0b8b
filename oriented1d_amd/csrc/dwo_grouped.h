// NHWC kernels for channel groups of one orientation (the networks give contiguous channels the same
// angle): fprop, dgrad and wgrad at strides 1 and 2, any extent (dgrad at stride 1 is fprop with reversed
// weights).
//
// A workgroup owns one 16-byte piece of a pixel (8 channels of a 16-bit type, 4 of fp32) over a tile of
// outputs.  It stages the tile's window as it lies in memory, pixel by pixel, and four lanes
// evaluate an item of four neighbouring outputs for the piece's channels, one 32-bit word (two channels
// of a 16-bit type) each, with the orientation's straight-line body: every read at an
// immediate offset, every source feeding up to four outputs.  Results leave straight from registers.
// Next to the slice kernels (dwo_nhwc_plane.h: four channels of any orientations, one fp32 plane each)
// nothing is transposed on the way in or out, a read brings two channels, and a line of memory is
// looked up by half as many workgroups; the price is a weight per lane in vector registers
// (two channels: 62), and two shifts or masks per read.
//
// What bounds them, from counters (K = 31): at stride 1 in bf16 the issue slots of the multiply-adds and those
// unpacking instructions (64 x 512 x 56 x 56 fprop 151 of 233 us; L2 lookups 42 %, LDS 25 %); at stride 2 (64 x 64 x 224 x 224) no unit
// is busy much more than half the time: fprop L2 lookups 52 %, vector instructions 38 %, x read 1.07 times; dgrad L2 lookups 56 %, dx
// written 1.46 times, as a line leaves the L2 before its pieces are there; wgrad L2 lookups 44 %, x and dy read 3.2 times at 4.7 TB/s, as the
// eight groups of a line come to it at different times.  Two workgroups per CU (80 KB of LDS,
// 128 registers) overlap staging and evaluation.
// Measured (us, fprop / wgrad, K = 31, angles of the networks): 64 x 512 x 56 x 56 bf16 233 / 264 (slice
// kernels 335 / 428), 64 x 1024 x 28 x 28 bf16 114 / 121 (129 / 190), 64 x 384 x 56 x 56 fp32 298 / 355 (326 / 551);
// stride 2, 64 x 64 x 224 x 224 bf16 298 / 357 (tile kernels 574 / 817).
#pragma once

#include "dwo_grouped_dispatch.h"
#include "dwo_static.h"
#include "dwo_window.h"

namespace dwo {

// Plan at stride S: positions in input pixels relative to the item's first output's own pixel.
constexpr Plan make_strided_plan(int o, int K, int L, int S) {
    Plan p{};
    const int eh = step_h(o) * S, ew = step_w(o) * S;
    constexpr int G = 48, GS = 2 * G + 1;
    int8_t grid[GS][GS] = {};
    for (int i = 0; i < GS; i++)
        for (int j = 0; j < GS; j++) grid[i][j] = -1;
    for (int s = 0; s < K; s++) {
        const int dh = canon_dh(o, K, s), dw = canon_dw(o, K, s);
        if (grid[dh + G][dw + G] < 0) grid[dh + G][dw + G] = (int8_t)s, p.ndistinct++;
        p.rep[s] = grid[dh + G][dw + G];
        for (int l = 0; l < L; l++) {
            p.hmin = cmin(p.hmin, dh + l * eh), p.hmax = cmax(p.hmax, dh + l * eh);
            p.wmin = cmin(p.wmin, dw + l * ew), p.wmax = cmax(p.wmax, dw + l * ew);
        }
    }
    for (int h = p.hmin; h <= p.hmax; h++)
        for (int w = p.wmin; w <= p.wmax; w++) {
            bool any = false;
            int8_t u[kMaxL] = {};
            for (int l = 0; l < kMaxL; l++) {
                u[l] = l < L ? grid[h - l * eh + G][w - l * ew + G] : (int8_t)-1;
                any = any || u[l] >= 0;
            }
            if (!any) continue;
            p.sh[p.nsrc] = (int16_t)h, p.sw[p.nsrc] = (int16_t)w;
            for (int l = 0; l < kMaxL; l++) p.user[p.nsrc][l] = u[l];
            p.nsrc++;
        }
    return p;
}

// Layout of a tile's window in LDS, in pixels of 16 bytes.  Window rows (columns) step by the stride
// where no tap leaves its row (column).
template <int O, int K, int S>
struct GrpGeo {
    static constexpr int CLS = orient_class(O), L = 4, EH = step_h(O);
    static constexpr int DH = win_extent(O, K, true), DW = win_extent(O, K, false);
    static constexpr int SR = DH == 0 ? 1 : S, SC = DW == 0 ? 1 : S;  // window rows, columns per output
    static constexpr int LR = CLS == CLS_H ? 1 : L;                   // output rows per row-block
    static constexpr int P0 = CLS == CLS_D && EH < 0 ? L - 1 : 0;
    static constexpr int PADL = CLS == CLS_D ? (L - 1) * SC : 0;  // diagonal items start left of the tile
    static constexpr int EXTRA = 2 * DW + 2 * PADL;               // columns besides the outputs' own
    static constexpr int WIDTH = (grp_tile_cols(S) - 1) * SC + 1 + EXTRA;
    // row-direction class: the four outputs of an item lie side by side, so column u is kept in sub-row
    // u % M at u / M: neighbouring items read neighbouring pixels
    static constexpr int M = L * SC, SUB = (WIDTH + M - 1) / M;
    static constexpr int RS = CLS == CLS_H ? M * SUB : WIDTH;
    static constexpr int col(int u) { return CLS == CLS_H ? (u % M) * SUB + u / M : u; }
    static constexpr Plan plan = make_strided_plan(O, K, L, S);
    static constexpr int imm(int sh, int sw) { return (sh + P0 * SR + DH) * RS + col(sw + DW); }
    static constexpr int round_rows(int th) { return (th + LR - 1) / LR * LR; }
    static constexpr int rows(int th) { return (round_rows(th) - 1) * SR + 1 + 2 * DH; }
    static constexpr int pixels(int th) { return rows(th) * RS; }
    // highest tile whose window fits
    static constexpr int max_rows() {
        int t = 64;
        while (pixels(t) > kGrpPixels) t--;
        return t;
    }
};
// Plan of dgrad at stride 2.  The dx pixels come in quads, (2 i + a, 2 j + b) for a, b in {0, 1}; tap
// (dh, dw) feeds the quad's pixel of its own parities from dy(i - floor(dh / 2), j - floor(dw / 2)), so a
// quad takes every tap once, and an item of L neighbouring quads shares its sources as outputs do.
struct QuadPlan {
    int nsrc = 0, nfma = 0;
    int16_t sh[kMaxSrc] = {}, sw[kMaxSrc] = {};
    int8_t user[kMaxSrc][2][4] = {};  // [quad][2 a + b]: first tap with that offset, or -1
    int8_t rep[64] = {};
};
constexpr int floor_half(int v) { return v >= 0 ? v / 2 : -((1 - v) / 2); }
constexpr QuadPlan make_quad_plan(int o, int K, int L) {
    QuadPlan p{};
    const int eh = step_h(o), ew = step_w(o);
    constexpr int G = 24, GS = 2 * G + 1;
    int16_t at[GS][GS] = {};
    for (int i = 0; i < GS; i++)
        for (int j = 0; j < GS; j++) at[i][j] = -1;
    for (int s = 0; s < K; s++) {
        const int dh = canon_dh(o, K, s), dw = canon_dw(o, K, s);
        int r = 0;
        while (canon_dh(o, K, r) != dh || canon_dw(o, K, r) != dw) r++;
        p.rep[s] = (int8_t)r;
        if (r != s) continue;
        for (int l = 0; l < L; l++) {
            const int h = l * eh - floor_half(dh), w = l * ew - floor_half(dw);
            int16_t &m = at[h + G][w + G];
            if (m < 0) {
                m = (int16_t)p.nsrc++;
                p.sh[m] = (int16_t)h, p.sw[m] = (int16_t)w;
                for (int q = 0; q < 2; q++)
                    for (int k = 0; k < 4; k++) p.user[m][q][k] = -1;
            }
            p.user[m][l][2 * (dh - 2 * floor_half(dh)) + dw - 2 * floor_half(dw)] = (int8_t)s;
            p.nfma++;
        }
    }
    return p;
}
// its window of dy: the interface of GrpGeo, in quads, at stride 1
template <int O, int K>
struct GrpQuadGeo {
    static constexpr int CLS = orient_class(O), L = 2, EH = step_h(O);
    static constexpr int DH = (win_extent(O, K, true) + 1) / 2, DW = (win_extent(O, K, false) + 1) / 2;
    static constexpr int SR = 1, SC = 1;
    static constexpr int LR = CLS == CLS_H ? 1 : L;
    static constexpr int P0 = CLS == CLS_D && EH < 0 ? L - 1 : 0;
    static constexpr int PADL = CLS == CLS_D ? L - 1 : 0;
    static constexpr int EXTRA = 2 * DW + 2 * PADL;
    static constexpr int WIDTH = grp_tile_cols(1) + EXTRA;
    static constexpr int M = L, SUB = (WIDTH + M - 1) / M;
    static constexpr int RS = CLS == CLS_H ? M * SUB : WIDTH;
    static constexpr int col(int u) { return CLS == CLS_H ? (u % M) * SUB + u / M : u; }
    static constexpr QuadPlan plan = make_quad_plan(O, K, L);
    static constexpr int imm(int sh, int sw) { return (sh + P0 + DH) * RS + col(sw + DW); }
    static constexpr int rows(int th) { return (th + LR - 1) / LR * LR + 2 * DH; }
    static constexpr int pixels(int th) { return rows(th) * RS; }
    static constexpr int max_rows() {
        int t = 64;
        while (pixels(t) > kGrpPixels) t--;
        return t;
    }
};

// the geometries of a kernel for all orientations
template <int K, int S>
struct ConvSet {
    static constexpr int TW = grp_tile_cols(S);
    template <int O>
    using Geo = GrpGeo<O, K, S>;
};
template <int K>
struct QuadSet {
    static constexpr int TW = grp_tile_cols(1);
    template <int O>
    using Geo = GrpQuadGeo<O, K>;
};
template <class Set, int... Os>
constexpr int grp_max_rows_impl(std::integer_sequence<int, Os...>) {
    int m = 64;
    ((m = cmin(m, Set::template Geo<Os>::max_rows())), ...);
    return m;
}
// most output rows per tile, whatever the orientation (one tile grid for all of them keeps the groups
// of a tile together)
template <class Set>
constexpr int grp_max_rows() {
    return grp_max_rows_impl<Set>(std::make_integer_sequence<int, 8>{});
}
template <class Set, int... Os>
constexpr int grp_pixels_impl(int th, std::integer_sequence<int, Os...>) {
    int m = 0;
    ((m = cmax(m, Set::template Geo<Os>::pixels(th))), ...);
    return m;
}
template <class Set>
constexpr int grp_pixels(int th) {
    return grp_pixels_impl<Set>(th, std::make_integer_sequence<int, 8>{});
}

typedef unsigned grp_u4 __attribute__((ext_vector_type(4)));

// the channels of a lane's word
template <typename T>
struct Word {
    static constexpr int N = 4 / (int)sizeof(T);
    static __device__ __forceinline__ float get(unsigned v, int e) {
        if constexpr (sizeof(T) == 4) return __uint_as_float(v);
        else if constexpr (std::is_same<T, bf16_t>::value)
            return __uint_as_float(e == 0 ? v << 16 : v & 0xffff0000u);
        else return (float)__builtin_bit_cast(_Float16, (uint16_t)(e == 0 ? v : v >> 16));
    }
    static __device__ __forceinline__ unsigned pack(const float (&a)[N]) {
        if constexpr (sizeof(T) == 4) return __float_as_uint(a[0]);
        else
            return (unsigned)__builtin_bit_cast(uint16_t, from_float<T>(a[0])) |
                   (unsigned)__builtin_bit_cast(uint16_t, from_float<T>(a[1])) << 16;
    }
};

// one tile of one image
struct GrpTile {
    int n, p, q, th, tw;  // image, corner, nominal extents
    int vh, vw;           // extents inside the image
    // NEAR: where tiles are dealt in runs (grp_run)
    template <bool NEAR>
    __device__ __forceinline__ void set(const ConvDims &d, const GrpTiles &t, int unit) {
        int row, col;
        th = t.th, tw = t.tw;
        if (NEAR && t.run > 0) {
            grp_run_tile(t, unit, n, row, col);
        } else {
            const int per = t.nth * t.ntw;
            n = unit / per;
            const int k = unit - n * per;
            row = k / t.ntw, col = k - row * t.ntw;
        }
        p = row * th, q = col * tw;
        vh = min(th, d.P - p), vw = min(tw, d.Q - q);
    }
};

// The tile's window of the group's pixel pieces into LDS; zeros outside the image.
template <class G, int S, typename T>
__device__ __forceinline__ void grp_stage(grp_u4 *lds, const T *xn, const ConvDims &d, const GrpTile &t, int c0) {
    const __amdgpu_buffer_rsrc_t rsrc =
        win_rsrc(xn, xn + (size_t)d.H * d.W * d.C - c0);
    const unsigned ww = (((t.tw + G::L - 1) / G::L * G::L) - 1) * G::SC + 1 + G::EXTRA;
    const unsigned nwin = G::rows(t.th) * ww, magic = win_magic(ww);
    const int r0 = t.p * S - G::DH, q0 = t.q * S - G::DW - G::PADL;
    const unsigned pix = (unsigned)d.C * (unsigned)sizeof(T);
    constexpr int U = 5;  // loads in flight per thread: all but the last few of a window
    for (unsigned f0 = threadIdx.x; f0 < nwin; f0 += U * kGrpThreads) {
        grp_u4 v[U];
        unsigned at[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const unsigned f = f0 + u * kGrpThreads, i = win_div(f, magic), j = f - i * ww;
            const int r = r0 + (int)i * (S / G::SR), q = q0 + (int)j * (S / G::SC);
            const bool in = f < nwin && (unsigned)r < (unsigned)d.H && (unsigned)q < (unsigned)d.W;
            at[u] = i * G::RS + G::col(j);
            v[u] = __builtin_bit_cast(grp_u4, __builtin_amdgcn_raw_buffer_load_b128(
                                                  rsrc, in ? ((unsigned)r * d.W + (unsigned)q) * pix : kWinNowhere,
                                                  0, 0));
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (f0 + u * kGrpThreads < nwin) lds[at[u]] = v[u];
    }
}

// A lane's item: LDS word of its origin, first output (row, column) in the tile.
template <class G>
struct GrpItems {
    unsigned ipr, magic, count;
    __device__ __forceinline__ explicit GrpItems(const GrpTile &t) {
        ipr = G::CLS == CLS_H ? (t.tw + G::L - 1) / G::L : (G::CLS == CLS_V ? t.tw : t.tw + G::L - 1);
        count = (G::CLS == CLS_H ? t.th : (t.th + G::L - 1) / G::L) * ipr;
        magic = win_magic(ipr);
    }
    __device__ __forceinline__ void at(unsigned item, unsigned &word, int &row, int &col) const {
        const unsigned rb = win_div(item, magic), j = item - rb * ipr;
        word = (rb * (G::LR * G::SR * G::RS) + (G::CLS == CLS_H ? j : j * G::SC)) * 4 + threadIdx.x % 4;
        row = (int)rb * G::LR + G::P0;
        col = G::CLS == CLS_H ? (int)j * G::L : (int)j - (G::CLS == CLS_D ? G::L - 1 : 0);
    }
    // output l of the item
    static __device__ __forceinline__ int row_of(int row, int l) {
        return G::CLS == CLS_H ? row : row + l * (G::CLS == CLS_V ? 1 : G::EH);
    }
    static __device__ __forceinline__ int col_of(int col, int l) { return G::CLS == CLS_V ? col : col + l; }
};

// byte offset of output (row, col) of the tile in its image's pieces, or nowhere
template <typename T>
__device__ __forceinline__ unsigned grp_offset(const GrpTile &t, const ConvDims &d, int row, int col) {
    const bool in = ((unsigned)row < (unsigned)t.vh) & ((unsigned)col < (unsigned)t.vw);
    const unsigned o = ((unsigned)(t.p + row) * d.Q + (unsigned)(t.q + col)) * d.C * (unsigned)sizeof(T);
    return in ? o + threadIdx.x % 4 * 4 : kWinNowhere;
}

// outputs of a staged window
template <int O, int S, typename T, int K>
__device__ __forceinline__ void grp_conv_items(const grp_u4 *lds, const float *lw, T *yn, const float *bias,
                                               const ConvDims &d, const GrpTile &t, int c0) {
    using G = GrpGeo<O, K, S>;
    constexpr int N = Word<T>::N, L = G::L;
    __syncthreads();
    // this lane's weights, taps at one offset added up
    const int ch = (int)(threadIdx.x % 4) * N;
    float wv[K][N], b[N];
#pragma unroll
    for (int e = 0; e < N; e++) {
        b[e] = bias != nullptr ? bias[c0 + ch + e] : 0.f;
        const float *row = lw + (ch + e) * K;
#pragma unroll
        for (int s = 0; s < K; s++) wv[s][e] = row[s];
        static_for<K>([&](auto s) {
            constexpr int r = G::plan.rep[s];
            if constexpr (r != s) wv[r][e] += wv[s][e];
        });
    }
    const __amdgpu_buffer_rsrc_t out = win_rsrc(yn, yn + (size_t)d.P * d.Q * d.C - c0);
    const unsigned *words = reinterpret_cast<const unsigned *>(lds);
    const GrpItems<G> items(t);
    for (unsigned it = threadIdx.x / 4; it < items.count; it += kGrpThreads / 4) {
        unsigned word;
        int row, col;
        items.at(it, word, row, col);
        float acc[L][N];
#pragma unroll
        for (int l = 0; l < L; l++)
#pragma unroll
            for (int e = 0; e < N; e++) acc[l][e] = b[e];
        const unsigned *base = words + word;
        static_for<G::plan.nsrc>([&](auto m) {
            constexpr int off = G::imm(G::plan.sh[m], G::plan.sw[m]) * 4;
            const unsigned v = base[off];
#pragma unroll
            for (int e = 0; e < N; e++) {
                const float x = Word<T>::get(v, e);
                static_for<L>([&](auto l) {
                    constexpr int s = G::plan.user[m][l];
                    if constexpr (s >= 0) acc[l][e] = __builtin_fmaf(x, wv[s][e], acc[l][e]);
                });
            }
        });
        pipeline_reads_and_fmas<G::plan.nsrc, N * plan_fma_count(G::plan, L) + (N - 1) * 2 * G::plan.nsrc>();
        // (the sums are due here: left alone, the compiler moves each output's multiply-adds next to its
        // store and keeps all sources alive, in scratch memory)
#pragma unroll
        for (int l = 0; l < L; l++)
#pragma unroll
            for (int e = 0; e < N; e++) asm volatile("" : "+v"(acc[l][e]));
#pragma unroll
        for (int l = 0; l < L; l++)
            __builtin_amdgcn_raw_buffer_store_b32(
                Word<T>::pack(acc[l]), out,
                grp_offset<T>(t, d, GrpItems<G>::row_of(row, l), GrpItems<G>::col_of(col, l)), 0, 0);
    }
}

template <int O, int S, typename T, int K>
__device__ __forceinline__ void grp_conv_body(grp_u4 *lds, float *lw, const T *xn, T *yn, const float *bias,
                                              const ConvDims &d, const GrpTile &t, int c0) {
    grp_stage<GrpGeo<O, K, S>, S>(lds, xn, d, t, c0);
    grp_conv_items<O, S, T, K>(lds, lw, yn, bias, d, t, c0);
}

// A group whose channels do not share a canonical orientation (the caller's claim did not hold):
// one output and channel per thread, straight from memory.
template <int S, typename T, int K>
__device__ void grp_conv_any(const T *xn, T *yn, const float *wt, const float *bias, const int8_t *dhdw,
                             const ConvDims &d, const GrpTile &t, int c0, int flip) {
    constexpr int CG = grp_channels(sizeof(T));
    for (int f = threadIdx.x; f < t.vh * t.vw * CG; f += kGrpThreads) {
        const int k = f % CG, o = f / CG, p = t.p + o / t.vw, q = t.q + o % t.vw, c = c0 + k;
        float a = bias != nullptr ? bias[c] : 0.f;
        for (int s = 0; s < K; s++) {
            const int h = p * S + dhdw[((size_t)c * K + s) * 2], w = q * S + dhdw[((size_t)c * K + s) * 2 + 1];
            if ((unsigned)h < (unsigned)d.H && (unsigned)w < (unsigned)d.W)
                a = __builtin_fmaf(to_float(xn[((size_t)h * d.W + w) * d.C + k]),
                                   wt[(size_t)c * K + (flip ? K - 1 - s : s)], a);
        }
        yn[((size_t)p * d.Q + q) * d.C + k] = from_float<T>(a);
    }
}

// orientation shared by the channels of the group, or -1
template <int CG>
__device__ __forceinline__ int grp_class(const int32_t *cls) {
    int o = cls[0];
#pragma unroll
    for (int k = 1; k < CG; k++)
        if (cls[k] != o) o = -1;
    return __builtin_amdgcn_readfirstlane(o);
}

template <int S, typename T, int K>
__global__ __launch_bounds__(kGrpThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void grouped_conv_kernel(
    const T *__restrict__ x, const float *__restrict__ wt, const float *__restrict__ bias,
    const void *__restrict__ blob, T *__restrict__ y, ConvDims d, GrpTiles tiles, int pixels, int flip) {
    extern __shared__ float lds_f[];
    grp_u4 *lds = reinterpret_cast<grp_u4 *>(lds_f);
    float *lw = lds_f + 4 * pixels;  // the group's weights
    constexpr int CG = grp_channels(sizeof(T));
    int unit, group;
    if (!grp_task(blockIdx.x, d.N * tiles.nth * tiles.ntw, d.C / CG, unit, group)) return;
    const int c0 = group * CG;
    GrpTile t;
    t.set<S == 2>(d, tiles, unit);
    const T *xn = x + (size_t)t.n * d.H * d.W * d.C + c0;
    T *yn = y + (size_t)t.n * d.P * d.Q * d.C + c0;
    if (threadIdx.x < CG * K) {  // (dgrad: in reverse tap order)
        const int s = threadIdx.x % K;
        lw[flip ? threadIdx.x - s + K - 1 - s : threadIdx.x] = wt[(size_t)c0 * K + threadIdx.x];
    }
#define DWO_CASE(O)                                                            \
    case O:                                                                    \
        grp_conv_body<O, S, T, K>(lds, lw, xn, yn, bias, d, t, c0);            \
        break;
    switch (grp_class<CG>(taps_class(blob, d.C, K) + c0)) {
        DWO_CASE(0)
        DWO_CASE(1)
        DWO_CASE(2)
        DWO_CASE(3)
        DWO_CASE(4)
        DWO_CASE(5)
        DWO_CASE(6)
        DWO_CASE(7)
        default: grp_conv_any<S, T, K>(xn, yn, wt, bias, taps_dhdw(blob), d, t, c0, flip);
    }
#undef DWO_CASE
}

// ---------------------------------------------------------------------------------------------
// fprop behind a pointwise layer of CIN inputs (the stem's dw1(pw1(x)) at inference): a workgroup
// projects the window's pixels to its group's channels while it stages them, rounded to T as the
// layer's own output would be.  The image is read once per channel group (eight times at 64 channels of a
// 16-bit type), and the C-channel tensor never exists.  Compiled for stride 2 and the three channels of an
// image: the stem.  In ConvNeXt-T inference of 128 images in bf16 489 us, with the tile kernel 986.
template <typename T>
__device__ __forceinline__ float grp_value(__amdgpu_buffer_rsrc_t r, unsigned off) {
    if constexpr (sizeof(T) == 4) return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
    else return Word<T>::get((unsigned)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0), 0);
}

template <typename T, int CIN>
struct Projection {
    static constexpr int CG = grp_channels(sizeof(T));
    float w[CG][CIN], b[CG];  // uniform: scalar registers
    __device__ __forceinline__ Projection(const float *pw_w, const float *pw_b, int c0) {
#pragma unroll
        for (int c = 0; c < CG; c++) {
            b[c] = pw_b != nullptr ? pw_b[c0 + c] : 0.f;
#pragma unroll
            for (int k = 0; k < CIN; k++) w[c][k] = pw_w[(size_t)(c0 + c) * CIN + k];
        }
    }
    __device__ __forceinline__ float channel(const float (&x)[CIN], int c) const {
        float a = b[c];
#pragma unroll
        for (int k = 0; k < CIN; k++) a = __builtin_fmaf(x[k], w[c][k], a);
        return a;
    }
};

template <class G, int S, typename T, int CIN>
__device__ __forceinline__ void grp_stage_projected(grp_u4 *lds, const T *img, const Projection<T, CIN> &pw,
                                                    const ConvDims &d, const GrpTile &t) {
    constexpr int N = Word<T>::N;
    const __amdgpu_buffer_rsrc_t rsrc = win_rsrc(img, img + (size_t)d.H * d.W * CIN);
    const unsigned ww = (((t.tw + G::L - 1) / G::L * G::L) - 1) * G::SC + 1 + G::EXTRA;
    const unsigned nwin = G::rows(t.th) * ww, magic = win_magic(ww);
    const int r0 = t.p * S - G::DH, q0 = t.q * S - G::DW - G::PADL;
    constexpr int U = 4;
    for (unsigned f0 = threadIdx.x; f0 < nwin; f0 += U * kGrpThreads) {
        float v[U][CIN];
        unsigned at[U];
        bool in[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const unsigned f = f0 + u * kGrpThreads, i = win_div(f, magic), j = f - i * ww;
            const int r = r0 + (int)i * (S / G::SR), q = q0 + (int)j * (S / G::SC);
            in[u] = f < nwin && (unsigned)r < (unsigned)d.H && (unsigned)q < (unsigned)d.W;
            at[u] = i * G::RS + G::col(j);
            const unsigned o = ((unsigned)r * d.W + (unsigned)q) * (unsigned)(CIN * sizeof(T));
#pragma unroll
            for (int k = 0; k < CIN; k++)
                v[u][k] = grp_value<T>(rsrc, in[u] ? o + k * (unsigned)sizeof(T) : kWinNowhere);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            grp_u4 px;
#pragma unroll
            for (int m = 0; m < 4; m++) {
                float a[N];
#pragma unroll
                for (int e = 0; e < N; e++) a[e] = pw.channel(v[u], m * N + e);
                px[m] = in[u] ? Word<T>::pack(a) : 0u;
            }
            if (f0 + u * kGrpThreads < nwin) lds[at[u]] = px;
        }
    }
}

template <int S, typename T, int K, int CIN>
__device__ void grp_projected_any(const T *img, T *yn, const float *wt, const float *bias, const float *pw_w,
                                  const float *pw_b, const int8_t *dhdw, const ConvDims &d, const GrpTile &t, int c0) {
    constexpr int CG = grp_channels(sizeof(T));
    for (int f = threadIdx.x; f < t.vh * t.vw * CG; f += kGrpThreads) {
        const int k = f % CG, o = f / CG, p = t.p + o / t.vw, q = t.q + o % t.vw, c = c0 + k;
        float a = bias != nullptr ? bias[c] : 0.f;
        for (int s = 0; s < K; s++) {
            const int h = p * S + dhdw[((size_t)c * K + s) * 2], w = q * S + dhdw[((size_t)c * K + s) * 2 + 1];
            if ((unsigned)h >= (unsigned)d.H || (unsigned)w >= (unsigned)d.W) continue;
            float v = pw_b != nullptr ? pw_b[c] : 0.f;
            for (int i = 0; i < CIN; i++)
                v = __builtin_fmaf(to_float(img[((size_t)h * d.W + w) * CIN + i]), pw_w[(size_t)c * CIN + i], v);
            a = __builtin_fmaf(to_float(from_float<T>(v)), wt[(size_t)c * K + s], a);
        }
        yn[((size_t)p * d.Q + q) * d.C + k] = from_float<T>(a);
    }
}

template <int S, typename T, int K, int CIN>
__global__ __launch_bounds__(kGrpThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void grouped_projected_kernel(
    const T *__restrict__ x, const float *__restrict__ pw_w, const float *__restrict__ pw_b,
    const float *__restrict__ wt, const float *__restrict__ bias, const void *__restrict__ blob, T *__restrict__ y,
    ConvDims d, GrpTiles tiles, int pixels) {
    extern __shared__ float lds_f[];
    grp_u4 *lds = reinterpret_cast<grp_u4 *>(lds_f);
    float *lw = lds_f + 4 * pixels;
    constexpr int CG = grp_channels(sizeof(T));
    int unit, group;
    if (!grp_task(blockIdx.x, d.N * tiles.nth * tiles.ntw, d.C / CG, unit, group)) return;
    const int c0 = group * CG;
    GrpTile t;
    t.set<false>(d, tiles, unit);  // (the image is small: in runs 0 to 2 % slower)
    const T *img = x + (size_t)t.n * d.H * d.W * CIN;
    T *yn = y + (size_t)t.n * d.P * d.Q * d.C + c0;
    if (threadIdx.x < CG * K) lw[threadIdx.x] = wt[(size_t)c0 * K + threadIdx.x];
    const Projection<T, CIN> pw(pw_w, pw_b, c0);
#define DWO_CASE(O)                                                              \
    case O:                                                                      \
        grp_stage_projected<GrpGeo<O, K, S>, S, T, CIN>(lds, img, pw, d, t);     \
        grp_conv_items<O, S, T, K>(lds, lw, yn, bias, d, t, c0);                 \
        break;
    switch (grp_class<CG>(taps_class(blob, d.C, K) + c0)) {
        DWO_CASE(0)
        DWO_CASE(1)
        DWO_CASE(2)
        DWO_CASE(3)
        DWO_CASE(4)
        DWO_CASE(5)
        DWO_CASE(6)
        DWO_CASE(7)
        default:
            grp_projected_any<S, T, K, CIN>(img, yn, wt, bias, pw_w, pw_b, taps_dhdw(blob), d, t, c0);
    }
#undef DWO_CASE
}

// ---------------------------------------------------------------------------------------------
// dgrad at stride 2 (QuadPlan).  `d` describes dy as both the source and the plane of quads (H = P,
// W = Q); dx is dxh x dxw.  64 x 64 x 224 x 224 bf16, K = 31: 198 us, 1.46 times dx written in 16-byte
// pieces (the residue classes one after the other from a sorted tap table, dwo_nhwc_tile.h: 544).
template <int O, typename T, int K>
__device__ __forceinline__ void grp_dgrad2_body(grp_u4 *lds, float *lw, const T *dyn, T *dxn, const ConvDims &d,
                                                const GrpTile &t, int c0, int dxh, int dxw) {
    using G = GrpQuadGeo<O, K>;
    constexpr int N = Word<T>::N, L = G::L;
    grp_stage<G, 1>(lds, dyn, d, t, c0);
    __syncthreads();
    const int ch = (int)(threadIdx.x % 4) * N;
    float wv[K][N];
#pragma unroll
    for (int e = 0; e < N; e++) {
        const float *row = lw + (ch + e) * K;
#pragma unroll
        for (int s = 0; s < K; s++) wv[s][e] = row[s];
        static_for<K>([&](auto s) {
            constexpr int r = G::plan.rep[s];
            if constexpr (r != s) wv[r][e] += wv[s][e];
        });
    }
    const __amdgpu_buffer_rsrc_t out = win_rsrc(dxn, dxn + (size_t)dxh * dxw * d.C - c0);
    const unsigned *words = reinterpret_cast<const unsigned *>(lds);
    const unsigned pix = (unsigned)d.C * (unsigned)sizeof(T);
    const GrpItems<G> items(t);
    for (unsigned it = threadIdx.x / 4; it < items.count; it += kGrpThreads / 4) {
        unsigned word;
        int row, col;
        items.at(it, word, row, col);
        float acc[L][4][N];
#pragma unroll
        for (int l = 0; l < L; l++)
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int e = 0; e < N; e++) acc[l][k][e] = 0.f;
        const unsigned *base = words + word;
        static_for<G::plan.nsrc>([&](auto m) {
            constexpr int off = G::imm(G::plan.sh[m], G::plan.sw[m]) * 4;
            const unsigned v = base[off];
#pragma unroll
            for (int e = 0; e < N; e++) {
                const float x = Word<T>::get(v, e);
                static_for<4 * L>([&](auto i) {
                    constexpr int l = i / 4, k = i % 4, s = G::plan.user[m][l][k];
                    if constexpr (s >= 0) acc[l][k][e] = __builtin_fmaf(x, wv[s][e], acc[l][k][e]);
                });
            }
        });
        pipeline_reads_and_fmas<G::plan.nsrc, N * G::plan.nfma + (N - 1) * 2 * G::plan.nsrc>();
#pragma unroll
        for (int l = 0; l < L; l++)
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int e = 0; e < N; e++) asm volatile("" : "+v"(acc[l][k][e]));  // (as in grp_conv_body)
#pragma unroll
        for (int l = 0; l < L; l++) {
            const int r = GrpItems<G>::row_of(row, l), c = GrpItems<G>::col_of(col, l);
            const int h = 2 * (t.p + r), w = 2 * (t.q + c);
            const bool in = ((unsigned)r < (unsigned)t.vh) & ((unsigned)c < (unsigned)t.vw);
            const unsigned o = ((unsigned)h * dxw + (unsigned)w) * pix + threadIdx.x % 4 * 4;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const bool ok = in & (h + k / 2 < dxh) & (w + k % 2 < dxw);
                __builtin_amdgcn_raw_buffer_store_b32(Word<T>::pack(acc[l][k]), out,
                                                      ok ? o + (k / 2 * dxw + k % 2) * pix : kWinNowhere, 0, 0);
            }
        }
    }
}

// the claim did not hold: one dx pixel and channel per thread
template <typename T, int K>
__device__ void grp_dgrad2_any(const T *dyn, T *dxn, const float *wt, const int8_t *dhdw, const ConvDims &d,
                               const GrpTile &t, int c0, int dxh, int dxw) {
    constexpr int CG = grp_channels(sizeof(T));
    for (int f = threadIdx.x; f < 4 * t.vh * t.vw * CG; f += kGrpThreads) {
        const int k = f % CG, o = f / CG, c = c0 + k;
        const int h = 2 * t.p + o / (2 * t.vw), w = 2 * t.q + o % (2 * t.vw);
        if (h >= dxh || w >= dxw) continue;
        float a = 0.f;
        for (int s = 0; s < K; s++) {
            const int ph = h - dhdw[((size_t)c * K + s) * 2], pw = w - dhdw[((size_t)c * K + s) * 2 + 1];
            if (((ph | pw) & 1) == 0 && (unsigned)(ph / 2) < (unsigned)d.H && (unsigned)(pw / 2) < (unsigned)d.W &&
                ph >= 0 && pw >= 0)
                a = __builtin_fmaf(to_float(dyn[((size_t)(ph / 2) * d.W + pw / 2) * d.C + k]),
                                   wt[(size_t)c * K + s], a);
        }
        dxn[((size_t)h * dxw + w) * d.C + k] = from_float<T>(a);
    }
}

template <typename T, int K>
__global__ __launch_bounds__(kGrpThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void grouped_dgrad2_kernel(
    const T *__restrict__ dy, const float *__restrict__ wt, const void *__restrict__ blob, T *__restrict__ dx,
    ConvDims d, GrpTiles tiles, int pixels, int dxh, int dxw) {
    extern __shared__ float lds_f[];
    grp_u4 *lds = reinterpret_cast<grp_u4 *>(lds_f);
    float *lw = lds_f + 4 * pixels;
    constexpr int CG = grp_channels(sizeof(T));
    int unit, group;
    if (!grp_task(blockIdx.x, d.N * tiles.nth * tiles.ntw, d.C / CG, unit, group)) return;
    const int c0 = group * CG;
    GrpTile t;
    t.set<true>(d, tiles, unit);
    const T *dyn = dy + (size_t)t.n * d.H * d.W * d.C + c0;
    T *dxn = dx + (size_t)t.n * dxh * dxw * d.C + c0;
    if (threadIdx.x < CG * K) lw[threadIdx.x] = wt[(size_t)c0 * K + threadIdx.x];
#define DWO_CASE(O)                                                     \
    case O:                                                             \
        grp_dgrad2_body<O, T, K>(lds, lw, dyn, dxn, d, t, c0, dxh, dxw); \
        break;
    switch (grp_class<CG>(taps_class(blob, d.C, K) + c0)) {
        DWO_CASE(0)
        DWO_CASE(1)
        DWO_CASE(2)
        DWO_CASE(3)
        DWO_CASE(4)
        DWO_CASE(5)
        DWO_CASE(6)
        DWO_CASE(7)
        default: grp_dgrad2_any<T, K>(dyn, dxn, wt, taps_dhdw(blob), d, t, c0, dxh, dxw);
    }
#undef DWO_CASE
}

// ---------------------------------------------------------------------------------------------
// wgrad: the same windows and items; a lane keeps the running sums of its channels' taps (62 for
// two channels) over all tiles of its workgroup and reads the item's dy words from memory.  Lanes
// and waves are added up at the end, in a fixed order.
template <int O, int S, bool NEAR, typename T, int K>
__device__ __forceinline__ void grp_wgrad_body(grp_u4 *lds, const T *x, const T *dy, float *part,
                                               const ConvDims &d, const GrpTiles &tiles, int c0, int g, int NG) {
    using G = GrpGeo<O, K, S>;
    constexpr int N = Word<T>::N, L = G::L, CG = grp_channels(sizeof(T));
    float acc[K][N], db[N];
#pragma unroll
    for (int e = 0; e < N; e++) {
        db[e] = 0.f;
#pragma unroll
        for (int s = 0; s < K; s++) acc[s][e] = 0.f;
    }
    const unsigned *words = reinterpret_cast<const unsigned *>(lds);
    const int units = d.N * tiles.nth * tiles.ntw;
    for (int u = g; u < units; u += NG) {
        GrpTile t;
        t.set<NEAR>(d, tiles, u);
        const T *dyn = dy + (size_t)t.n * d.P * d.Q * d.C + c0;
        const __amdgpu_buffer_rsrc_t in = win_rsrc(dyn, dyn + (size_t)d.P * d.Q * d.C - c0);
        __syncthreads();  // the previous window is consumed
        grp_stage<G, S>(lds, x + (size_t)t.n * d.H * d.W * d.C + c0, d, t, c0);
        const GrpItems<G> items(t);
        auto load_dy = [&](unsigned it, unsigned (&v)[L], unsigned &word) {
            int row, col;
            items.at(min(it, items.count - 1), word, row, col);
#pragma unroll
            for (int l = 0; l < L; l++) {
                const unsigned o =
                    grp_offset<T>(t, d, GrpItems<G>::row_of(row, l), GrpItems<G>::col_of(col, l));
                v[l] = __builtin_amdgcn_raw_buffer_load_b32(in, it < items.count ? o : kWinNowhere, 0, 0);
            }
        };
        unsigned cur[L], nxt[L], word, next_word;
        load_dy(threadIdx.x / 4, cur, word);
        __syncthreads();
        for (unsigned it = threadIdx.x / 4; it < items.count; it += kGrpThreads / 4) {
            load_dy(it + kGrpThreads / 4, nxt, next_word);  // (travels while this item is evaluated)
            float gy[L][N];
#pragma unroll
            for (int l = 0; l < L; l++)
#pragma unroll
                for (int e = 0; e < N; e++) gy[l][e] = Word<T>::get(cur[l], e), db[e] += gy[l][e];
            const unsigned *base = words + word;
            static_for<G::plan.nsrc>([&](auto m) {
                constexpr int off = G::imm(G::plan.sh[m], G::plan.sw[m]) * 4;
                const unsigned v = base[off];
#pragma unroll
                for (int e = 0; e < N; e++) {
                    const float xv = Word<T>::get(v, e);
                    static_for<L>([&](auto l) {
                        constexpr int s = G::plan.user[m][l];
                        if constexpr (s >= 0) acc[s][e] = __builtin_fmaf(xv, gy[l][e], acc[s][e]);
                    });
                }
            });
            pipeline_reads_and_fmas<G::plan.nsrc, N * plan_fma_count(G::plan, L) + (N - 1) * 2 * G::plan.nsrc>();
#pragma unroll
            for (int l = 0; l < L; l++) cur[l] = nxt[l];
            word = next_word;
        }
    }
    __syncthreads();
    // the four lanes of a row of 16 that hold the same channels (rotations inside the row: no LDS), then
    // rows and waves: red[row of the workgroup][channel][tap]
    float *red = reinterpret_cast<float *>(lds);
    const int ch = (int)(threadIdx.x % 4) * N, row16 = threadIdx.x / 16;
    auto lanes = [](float v) {
        v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x124, 0xf,
                                                                   0xf, false));  // row_ror:4
        v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xf,
                                                                   0xf, false));  // row_ror:8
        return v;
    };
#pragma unroll
    for (int e = 0; e < N; e++) {
        float *out = red + (row16 * CG + ch + e) * (K + 1);
        const float b = lanes(db[e]);
        static_for<K>([&](auto s) {
            if constexpr (G::plan.rep[s] == s) acc[s][e] = lanes(acc[s][e]);
        });
        if (threadIdx.x % 16 < 4) {
            out[K] = b;
            static_for<K>([&](auto s) { out[s] = acc[(int)G::plan.rep[s]][e]; });
        }
    }
    __syncthreads();
    if (threadIdx.x < CG * (K + 1)) {
        float total = 0.f;
#pragma unroll 8
        for (int r = 0; r < kGrpThreads / 16; r++) total += red[r * CG * (K + 1) + threadIdx.x];
        part[((size_t)c0 * (K + 1) + threadIdx.x) * NG + g] = total;
    }
}

// a group without a common canonical orientation: a thread per (channel, tap), straight from memory
template <int S, bool NEAR, typename T, int K>
__device__ void grp_wgrad_any(const T *x, const T *dy, const int8_t *dhdw, float *part, const ConvDims &d,
                              const GrpTiles &tiles, int c0, int g, int NG) {
    constexpr int CG = grp_channels(sizeof(T));
    if (threadIdx.x >= CG * (K + 1)) return;
    const int k = threadIdx.x / (K + 1), s = threadIdx.x % (K + 1), c = c0 + k;
    const int dh = s < K ? dhdw[((size_t)c * K + s) * 2] : 0, dw = s < K ? dhdw[((size_t)c * K + s) * 2 + 1] : 0;
    float total = 0.f;
    for (int u = g; u < d.N * tiles.nth * tiles.ntw; u += NG) {
        GrpTile t;
        t.set<NEAR>(d, tiles, u);
        for (int o = 0; o < t.vh * t.vw; o++) {
            const int p = t.p + o / t.vw, q = t.q + o % t.vw, h = p * S + dh, w = q * S + dw;
            const float gy = to_float(dy[(((size_t)t.n * d.P + p) * d.Q + q) * d.C + c]);
            if (s == K) total += gy;
            else if ((unsigned)h < (unsigned)d.H && (unsigned)w < (unsigned)d.W)
                total = __builtin_fmaf(gy, to_float(x[(((size_t)t.n * d.H + h) * d.W + w) * d.C + c]), total);
        }
    }
    part[((size_t)c0 * (K + 1) + threadIdx.x) * NG + g] = total;
}

template <int S, bool NEAR, typename T, int K>
__global__ __launch_bounds__(kGrpThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void grouped_wgrad_kernel(
    const T *__restrict__ x, const T *__restrict__ dy, const void *__restrict__ blob, float *__restrict__ part,
    ConvDims d, GrpTiles tiles, int NG) {
    extern __shared__ float lds_f[];
    grp_u4 *lds = reinterpret_cast<grp_u4 *>(lds_f);
    constexpr int CG = grp_channels(sizeof(T));
    int g, group;
    if (!grp_task(blockIdx.x, NG, d.C / CG, g, group)) return;
    const int c0 = group * CG;
#define DWO_CASE(O)                                                               \
    case O:                                                                       \
        grp_wgrad_body<O, S, NEAR, T, K>(lds, x, dy, part, d, tiles, c0, g, NG);  \
        break;
    switch (grp_class<CG>(taps_class(blob, d.C, K) + c0)) {
        DWO_CASE(0)
        DWO_CASE(1)
        DWO_CASE(2)
        DWO_CASE(3)
        DWO_CASE(4)
        DWO_CASE(5)
        DWO_CASE(6)
        DWO_CASE(7)
        default: grp_wgrad_any<S, NEAR, T, K>(x, dy, taps_dhdw(blob), part, d, tiles, c0, g, NG);
    }
#undef DWO_CASE
}

// Tiles of a P x Q output plane, even in size (the last is no sliver); planes x groups that would leave
// workgroup slots empty are cut into lower tiles.
template <class Set>
GrpTiles grp_tiles(int P, int Q, long planes) {
    constexpr int TH = grp_max_rows<Set>(), TW = Set::TW;
    static_assert(TH >= 4, "a window of four output rows must fit");
    GrpTiles t;
    t.nth = (P + TH - 1) / TH, t.ntw = (Q + TW - 1) / TW;
    t.th = (P + t.nth - 1) / t.nth, t.tw = (Q + t.ntw - 1) / t.ntw;
    // whole items where that does not make a tile too high or wide
    t.th = cmin((t.th + 3) & ~3, TH), t.tw = cmin((t.tw + 3) & ~3, TW);
    if (t.nth == 1) t.th = P;
    if (t.ntw == 1) t.tw = Q;
    t.nth = (P + t.th - 1) / t.th, t.ntw = (Q + t.tw - 1) / t.tw;
    while (planes * t.nth * t.ntw < kGrpSlots && t.th > kGrpLeastRows) {
        t.th = cmax((t.th / 2 + 3) & ~3, kGrpLeastRows);
        t.nth = (P + t.th - 1) / t.th;
    }
    t.run = 0;
    return t;
}

template <typename T, int K, int S>
int launch_grouped_conv_s(const void *src, const float *w, const float *bias, const void *taps, void *dst,
                          const ConvDims &d, int flip, hipStream_t st) {
    constexpr int CG = grp_channels(sizeof(T));
    static int cache[kMaxDevices];
    per_device_once(cache, [&] {
        allow_large_lds(grouped_conv_kernel<S, T, K>, (kGrpPixels * 4 + CG * K) * sizeof(float));
        return 1;
    });
    if (d.N == 0) return 0;  // set-up only
    const int ngroups = d.C / CG;
    GrpTiles t = grp_tiles<ConvSet<K, S>>(d.P, d.Q, (long)d.N * ngroups);
    if (S == 2) t.run = grp_run(t, d, sizeof(T), GRP_FPROP);
    const int pixels = grp_pixels<ConvSet<K, S>>(t.th);
    const long grid = grp_grid((long)d.N * t.nth * t.ntw, ngroups);
    if (!grp_grid_fits(grid)) return -100;
    grouped_conv_kernel<S, T, K><<<dim3((unsigned)grid), dim3(kGrpThreads), (pixels * 4 + CG * K) * sizeof(float),
                                   st>>>((const T *)src, w, bias, taps, (T *)dst, d, t, pixels, flip);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}

template <typename T, int K>
int launch_grouped_dgrad2(const void *dy, const float *w, const void *taps, void *dx, const ConvDims &d_,
                          hipStream_t st) {
    using Set = QuadSet<K>;
    constexpr int CG = grp_channels(sizeof(T));
    static int cache[kMaxDevices];
    per_device_once(cache, [&] {
        allow_large_lds(grouped_dgrad2_kernel<T, K>, (kGrpPixels * 4 + CG * K) * sizeof(float));
        return 1;
    });
    if (d_.N == 0) return 0;  // set-up only
    ConvDims d = d_;
    d.H = d.P, d.W = d.Q;
    const int ngroups = d.C / CG;
    GrpTiles t = grp_tiles<Set>(d.P, d.Q, (long)d.N * ngroups);
    t.run = grp_run(t, d_, sizeof(T), GRP_DGRAD);
    const int pixels = grp_pixels<Set>(t.th);
    const long grid = grp_grid((long)d.N * t.nth * t.ntw, ngroups);
    if (!grp_grid_fits(grid)) return -100;
    grouped_dgrad2_kernel<T, K><<<dim3((unsigned)grid), dim3(kGrpThreads), (pixels * 4 + CG * K) * sizeof(float),
                                  st>>>((const T *)dy, w, taps, (T *)dx, d, t, pixels, d_.H, d_.W);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}

template <typename T, int K>
int launch_grouped_conv(const void *src, const float *w, const float *bias, const void *taps, void *dst,
                        const ConvDims &d, int flip, hipStream_t st) {
    if (flip && d.stride == 2) return launch_grouped_dgrad2<T, K>(src, w, taps, dst, d, st);
    return d.stride == 1 ? launch_grouped_conv_s<T, K, 1>(src, w, bias, taps, dst, d, flip, st)
                         : launch_grouped_conv_s<T, K, 2>(src, w, bias, taps, dst, d, flip, st);
}

template <typename T, int K, int S>
int launch_grouped_wgrad_s(const void *x, const void *dy, const void *taps, float *part, const ConvDims &d,
                           int NG, hipStream_t st) {
    constexpr int CG = grp_channels(sizeof(T));
    constexpr int kRed = kGrpThreads / 16 * CG * (K + 1);  // floats
    static_assert(kRed <= kGrpPixels * 4, "the waves' sums fit where the window was");
    static int cache[kMaxDevices];
    per_device_once(cache, [&] {
        allow_large_lds(grouped_wgrad_kernel<S, false, T, K>, kGrpPixels * 16);
        if constexpr (S == 2) allow_large_lds(grouped_wgrad_kernel<S, true, T, K>, kGrpPixels * 16);
        return 1;
    });
    if (d.N == 0) return 0;  // set-up only
    const int ngroups = d.C / CG;
    GrpTiles t = grp_tiles<ConvSet<K, S>>(d.P, d.Q, kGrpSlots);  // (lower tiles would cost more partial sums)
    if (S == 2) t.run = grp_run(t, d, sizeof(T), GRP_WGRAD);
    const size_t lds = cmax(grp_pixels<ConvSet<K, S>>(t.th) * 4, kRed) * sizeof(float);
    const dim3 grid((unsigned)grp_grid(NG, ngroups)), block(kGrpThreads);
    // (a kernel of its own where tiles are dealt in turn: finding a tile's place in its run costs scalar registers)
    if (S == 2 && t.run > 0)
        grouped_wgrad_kernel<S, S == 2, T, K><<<grid, block, lds, st>>>((const T *)x, (const T *)dy, taps, part, d, t, NG);
    else grouped_wgrad_kernel<S, false, T, K><<<grid, block, lds, st>>>((const T *)x, (const T *)dy, taps, part, d, t, NG);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}

template <typename T, int K>
int launch_grouped_wgrad(const void *x, const void *dy, const void *taps, float *part, const ConvDims &d,
                         int *groups_out, hipStream_t st) {
    const int NG = d.N == 0 ? 8 : grp_wgrad_groups(d, sizeof(T));
    *groups_out = NG;
    return d.stride == 1 ? launch_grouped_wgrad_s<T, K, 1>(x, dy, taps, part, d, NG, st)
                         : launch_grouped_wgrad_s<T, K, 2>(x, dy, taps, part, d, NG, st);
}

template <typename T, int K>
int launch_grouped_projected(const void *x, const float *pw_w, const float *pw_b, const float *w, const float *bias,
                             const void *taps, void *y, const ConvDims &d, hipStream_t st) {
    constexpr int CG = grp_channels(sizeof(T));
    static int cache[kMaxDevices];
    per_device_once(cache, [&] {
        allow_large_lds(grouped_projected_kernel<2, T, K, kGrpProjected>, (kGrpPixels * 4 + CG * K) * sizeof(float));
        return 1;
    });
    if (d.N == 0) return 0;  // set-up only
    const int ngroups = d.C / CG;
    const GrpTiles t = grp_tiles<ConvSet<K, 2>>(d.P, d.Q, (long)d.N * ngroups);
    const int pixels = grp_pixels<ConvSet<K, 2>>(t.th);
    const long grid = grp_grid((long)d.N * t.nth * t.ntw, ngroups);
    if (!grp_grid_fits(grid)) return -100;
    grouped_projected_kernel<2, T, K, kGrpProjected>
        <<<dim3((unsigned)grid), dim3(kGrpThreads), (pixels * 4 + CG * K) * sizeof(float), st>>>(
            (const T *)x, pw_w, pw_b, w, bias, taps, (T *)y, d, t, pixels);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}

}  // namespace dwo
