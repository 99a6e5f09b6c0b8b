// LDS-staged NCHW kernels for stride 1 at any plane extent (kernel sizes of DWO_WINDOW_KS).
//
// Same straight-line bodies as the plane kernels of dwo_static.h (taps known when compiled, every
// LDS read at an immediate offset, four outputs per lane sharing their sources), with the extents as
// run-time data: only the LDS row stride is fixed when compiled (rows of up to WM columns).  A
// workgroup owns one channel and walks a run of units:
//   plane mode (planes of at most 64 x 64): a unit is PB whole planes of consecutive images.  The
//     zero halo is written once, units rewrite the interiors.  Rows share their halos (what lies
//     right of a row is what lies left of the next), and so do the planes of a unit;
//   tile mode (larger planes): a unit is one th x tw tile of a plane, staged with its halo
//     (zeros where the halo leaves the image).
// The next unit is on its way from memory into registers while one is evaluated.
//
// What bounds these kernels is the instruction rate (the multiply-adds of 8 x 96 x 128 x 128 take
// 10 us of the chip's issue slots, the tensors 10 us of HBM in bf16), so everything but the
// multiply-adds and their reads is kept off the lanes: a wave's lanes lie along the columns of the
// staged row (WM of them; 64 / WM row-blocks per wave), which leaves rows, planes and units uniform
// per wave, i.e. scalar; global accesses go through buffer descriptors, where an out-of-range offset
// stands for "not there" (loads give zeros, stores are dropped) and takes the place of branches.
// Measured (us, fprop / wgrad, eight orientations): 8 x 96 x 128 x 128 bf16 28 / 38 (the tile kernels
// of dwo_nhwc_tile.h, one LDS read per multiply-add: 43 / 134; these bodies with items dealt to the
// threads one by one, with divisions, predicates and 64-bit addresses per lane: 53 / 66); 64 x 96 x
// 60 x 60 fp32 41 / 48, where 64 x 64 with compile-time extents takes 41 / 42.  Workgroups of 512
// threads: with 256, twice the workgroups and the same LDS per wave, 64 x 192 x 31 x 31 took 41
// instead of 29 (LDS then holds 16 waves per CU instead of 24).
#pragma once

#include "dwo_static.h"
#include "dwo_window_dispatch.h"

namespace dwo {

constexpr int kWinL = 4;  // outputs per lane, every class

// Threads, staged chunks per thread (at most) and waves per SIMD (fprop, wgrad) of a variant.
template <int WM, bool TILE>
struct WinMode {
    static constexpr int NT = kWinThreads, PF = win_slots_per_thread(TILE);
    static constexpr int kWaves = 6, kWavesWgrad = TILE ? 4 : 6;
};

// LDS layout of one orientation (the interface of Geo that the plans use).
template <int CLS_, int DH_, int DW_, int P0_, int Q0_, int EH_, int WM, bool TILE>
struct WinLayout {
    static constexpr int CLS = CLS_, DH = DH_, DW = DW_, P0 = P0_, Q0 = Q0_, EH = EH_;
    static constexpr int LR = CLS == CLS_H ? 1 : kWinL;         // rows per row-block
    static constexpr int JW = CLS == CLS_H ? WM / kWinL : WM;   // lanes along a row
    static constexpr int RPW = 64 / JW;                         // row-blocks per wave
    static constexpr int PL = (Q0 + DW + 3) & ~3;               // column 0 in LDS (DH rows lie above)
    // columns from one row to the next: the halo between two rows serves both, unless both sides
    // of a row hold data (tile mode)
    static constexpr int WIDTH = WM + DW + 4 + (TILE ? PL : 0);
    // row-direction class: a row is split into four sub-rows, column u lives in sub-row u % 4 at
    // u / 4; sub-rows are sized so that the rows of a wave continue on the banks where the
    // previous one left off
    static constexpr int SUB = [] {
        int s = (WIDTH + 3) / 4 + 1;
        while ((4 * s - JW) % 32 != 0 && (4 * s) % 32 != 16) s++;
        return s;
    }();
    static constexpr int RS = CLS == CLS_H ? 4 * SUB : (WIDTH + 7) / 8 * 8;
    static constexpr int col(int u) { return CLS == CLS_H ? (u % 4) * SUB + u / 4 : u; }
    // rows from one plane to the next, and LDS words of PB planes (or one tile) of th output rows
    static constexpr int pitch(int th) { return ((th + LR - 1) / LR + RPW - 1) / RPW * RPW * LR + DH; }
    static constexpr int words(int th, int PB) { return (DH + PB * pitch(th)) * RS + PL + DW + 8; }
};
template <int O, int K, int WM, bool TILE>
using WinLayoutOf = WinLayout<orient_class(O), win_extent(O, K, true), win_extent(O, K, false),
                              orient_class(O) == CLS_D && step_h(O) < 0 ? kWinL - 1 : 0,
                              orient_class(O) == CLS_D ? kWinL - 1 : 0, step_h(O), WM, TILE>;
template <int O, int K, int WM, bool TILE>
struct WinGeo : WinLayoutOf<O, K, WM, TILE> {
    using B = WinLayoutOf<O, K, WM, TILE>;
    static constexpr int L_ = kWinL;
    static constexpr Plan plan = make_plan(O, K, kWinL, 256, 256);
    // immediate offset of source (sh, sw) from an item's base
    static constexpr int imm(int sh, int sw) {
        return (sh + B::P0 + B::DH) * B::RS + (B::CLS == CLS_H ? B::col(sw + B::PL) : sw + B::PL - B::Q0);
    }
};
// any angle: stacked items, square halo of K / 2
template <int K, int WM, bool TILE>
using WinTableGeo = WinLayout<CLS_V, K / 2, K / 2, 0, 0, 1, WM, TILE>;

template <int K, int WM, bool TILE, int... Os>
constexpr int win_words_impl(int th, int PB, std::integer_sequence<int, Os...>) {
    int m = WinTableGeo<K, WM, TILE>::words(th, PB);
    ((m = cmax(m, WinGeo<Os, K, WM, TILE>::words(th, PB))), ...);
    return m;
}
// LDS words of a unit, whatever its orientation
template <int K, int WM, bool TILE>
constexpr int win_words(int th, int PB) {
    return (win_words_impl<K, WM, TILE>(th, PB, std::make_integer_sequence<int, 8>{}) + 3) & ~3;
}

// The layout as values (constants, once inlined).
struct WinRt {
    int cls, LR, RPW, JW, DH, DW, PL, RS, SUB, P0, Q0, EH;
    template <class G>
    __device__ __forceinline__ void set() {
        cls = G::CLS, LR = G::LR, RPW = G::RPW, JW = G::JW, DH = G::DH, DW = G::DW, PL = G::PL, RS = G::RS,
        SUB = G::SUB, P0 = G::P0, Q0 = G::Q0, EH = G::EH;
    }
};

// floor(n / d) for n < 2^16, 1 <= d < 2^16 (m = 0 stands for d = 1)
__device__ __forceinline__ unsigned win_div(unsigned n, unsigned m) { return m ? __umulhi(n, m) : n; }
__device__ __forceinline__ unsigned win_magic(unsigned d) { return d > 1 ? 0xffffffffu / d + 1 : 0; }

constexpr unsigned kWinNowhere = 0x80000000u;  // an offset that no descriptor covers

// Raw descriptor from p to the end of a tensor at `end`.  p may lie before the tensor where only
// offsets inside it are used.
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t win_rsrc(const T *p, const T *end) {
    const long left = reinterpret_cast<const char *>(end) - reinterpret_cast<const char *>(p);
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(p), 0, (unsigned)min(left, 0x7fffffffL),
                                             0x00020000);
}

// Four consecutive activations through a descriptor, at any element alignment.
template <typename T>
struct Quad;
template <>
struct Quad<float> {
    typedef float f4 __attribute__((ext_vector_type(4)));
    f4 v;
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned soff) {
        v = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0));
    }
    __device__ __forceinline__ void store(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned soff) const {
        typedef unsigned u4 __attribute__((ext_vector_type(4)));
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), r, off, soff, 2);
    }
    __device__ __forceinline__ void set(const float (&a)[4]) { v = f4{a[0], a[1], a[2], a[3]}; }
    // drop the first s elements (s = 0..3), zeros behind
    __device__ __forceinline__ void drop(unsigned s) {
        if (s & 1) v = f4{v[1], v[2], v[3], 0.f};
        if (s & 2) v = f4{v[2], v[3], 0.f, 0.f};
    }
    __device__ __forceinline__ float get(int i) const { return v[i]; }
};
template <typename T>
struct Quad16 {
    unsigned long long v;
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned soff) {
        v = __builtin_bit_cast(unsigned long long, __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, 0));
    }
    __device__ __forceinline__ void store(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned soff) const {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, off, soff, 2);
    }
    __device__ __forceinline__ void set(const float (&a)[4]) {
        Vec4<T> t;
        t.set(a[0], a[1], a[2], a[3]);
        v = __builtin_bit_cast(unsigned long long, t.v);
    }
    __device__ __forceinline__ void drop(unsigned s) { v >>= 16 * s; }
    __device__ __forceinline__ float get(int i) const {
        return to_float(__builtin_bit_cast(T, (uint16_t)(v >> (16 * i))));
    }
};
template <>
struct Quad<bf16_t> : Quad16<bf16_t> {};
template <>
struct Quad<f16_t> : Quad16<f16_t> {};

// one element
__device__ __forceinline__ void win_store(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned soff, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, soff, 2);
}
template <typename T>
__device__ __forceinline__ void win_store(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned soff, T v) {
    __builtin_amdgcn_raw_buffer_store_b16(raw16(v), r, off, soff, 0);
}

// One unit of the walk: planes n .. of the channel, rows from p, columns from q (uniform).
template <bool TILE>
struct WinUnit {
    int n, p, q;
    __device__ __forceinline__ void first(const WinDims &d, int u) {
        n = u * d.PB, p = 0, q = 0;
        if (TILE) {
            const unsigned tiles = d.nth * d.ntw;
            n = (int)((unsigned)u / tiles);
            const unsigned t = u - n * tiles, a = t / (unsigned)d.ntw;
            p = (int)a * d.th, q = (int)(t - a * d.ntw) * d.tw;
        }
    }
    __device__ __forceinline__ void advance(const WinDims &d) {
        if (TILE) {
            q += d.tw;
            if (q >= d.W) q = 0, p += d.th;
            if (p >= d.H) p = 0, n++;
        } else {
            n += d.PB;
        }
    }
    __device__ __forceinline__ int planes(const WinDims &d) const { return TILE ? 1 : min(d.PB, d.N - n); }
    __device__ __forceinline__ int rows(const WinDims &d) const { return TILE ? min(d.th, d.H - p) : d.H; }
    __device__ __forceinline__ int cols(const WinDims &d) const { return TILE ? min(d.tw, d.W - q) : d.W; }
};

// Staging of a unit: the rectangle of four-column chunks that the unit's planes (plane mode) or its
// window (tile mode) consists of, dealt over the threads once; slot k of a thread is chunk
// tid + k * NT (threads beyond the last chunk repeat it).  A chunk that the right edge of the image
// cuts is loaded from column W - 4 and shifted, so that no load leaves its row.
template <typename T, int WM, bool TILE>
struct WinStager {
    static constexpr int NT = WinMode<WM, TILE>::NT, PF = WinMode<WM, TILE>::PF;
    Quad<T> pre[PF];
    unsigned off[PF];     // byte offset from the unit's corner
    unsigned lds_at[PF];  // word offset in LDS
    unsigned rc[TILE ? PF : 1];  // tile mode: row (high half) and column in the window
    unsigned nslots;
    int p_lo, q_lo;       // the rectangle's corner relative to the unit's

    __device__ __forceinline__ void setup(const WinDims &d, const WinRt &rt, unsigned pls) {
        p_lo = TILE ? -rt.DH : 0, q_lo = TILE ? -((rt.DW + 3) & ~3) : 0;
        const unsigned nr = TILE ? d.th + 2 * rt.DH : d.th;
        const unsigned nc = (unsigned)((TILE ? d.tw + rt.DW : d.tw) - q_lo + 3) / 4;
        nslots = nr * nc * (TILE ? 1 : d.PB);
        const unsigned m_nc = win_magic(nc), m_pl = win_magic(nr * nc);
#pragma unroll
        for (int k = 0; k < PF; k++) {
            const unsigned f = min(threadIdx.x + k * NT, nslots - 1);
            const unsigned pl = TILE ? 0 : win_div(f, m_pl), g = f - pl * (nr * nc);
            const unsigned i = win_div(g, m_nc), j = g - i * nc;
            const int w = (int)(4 * j);
            off[k] = (i * d.W + (TILE ? w : min(w, d.W - 4)) + pl * (unsigned)(d.C * d.H * d.W)) * (unsigned)sizeof(T);
            lds_at[k] = pl * pls + (p_lo + rt.DH + (int)i) * rt.RS +
                        (rt.cls == CLS_H ? (q_lo + rt.PL + w) / 4 : q_lo + rt.PL + w);
            if (TILE) rc[k] = i << 16 | (unsigned)w;
        }
    }
    __device__ __forceinline__ void prefetch(const T *x, const WinDims &d, int c, const WinUnit<TILE> &u) {
        const size_t plane = (size_t)d.H * d.W;
        const int p = u.p + p_lo, q = u.q + q_lo;
        const T *base = x + ((size_t)u.n * d.C + c) * plane + (long)p * d.W + q;
        const __amdgpu_buffer_rsrc_t rsrc = win_rsrc(base, x + (size_t)d.N * d.C * plane);
        // (chunks of planes beyond the last image lie beyond the descriptor)
#pragma unroll
        for (int k = 0; k < PF; k++) {
            if (k * NT >= (int)nslots) break;
            unsigned o = off[k];
            if (TILE) {
                const int r = (int)(rc[k] >> 16), w = (int)(rc[k] & 0xffff);
                const bool in = (unsigned)(p + r) < (unsigned)d.H && (unsigned)(q + w) < (unsigned)d.W;
                if (d.W % 4 != 0) o += (unsigned)min(0, d.W - 4 - q - w) * (unsigned)sizeof(T);  // uniform
                o = in ? o : kWinNowhere;
            }
            pre[k].load(rsrc, o, 0);
        }
    }
    __device__ __forceinline__ void commit(float *lds, const WinDims &d, const WinRt &rt,
                                           const WinUnit<TILE> &u) {
#pragma unroll
        for (int k = 0; k < PF; k++) {
            if (k * NT >= (int)nslots) break;
            if (d.W % 4 != 0) {  // uniform
                int w;
                if (TILE) {
                    w = (int)(rc[k] & 0xffff) + u.q + q_lo;
                } else {  // (the last chunk of a row: its offset was moved back)
                    const unsigned f = min(threadIdx.x + k * NT, nslots - 1), nc = (unsigned)(d.tw + 3) / 4;
                    w = (int)(4 * (f - win_div(f, win_magic(nc)) * nc));
                }
                pre[k].drop((unsigned)max(0, min(3, w - (d.W - 4))));
            }
            float *q = lds + lds_at[k];
            if (rt.cls == CLS_H) {  // uniform
#pragma unroll
                for (int e = 0; e < 4; e++) q[e * rt.SUB] = pre[k].get(e);
            } else {
                typedef float f4 __attribute__((ext_vector_type(4)));
                *reinterpret_cast<f4 *>(__builtin_assume_aligned(q, 16)) =
                    f4{pre[k].get(0), pre[k].get(1), pre[k].get(2), pre[k].get(3)};
            }
        }
    }
};

// A wave's items of a unit: group i of the unit (uniform) is 64 items, RPW row-blocks of JW lanes.
// Diagonal items number three more than a tile's columns; those beyond WM of all row-blocks are
// gathered in groups of their own (16 row-blocks x 4 lanes).
template <int WM, bool TILE>
struct WinGroups {
    unsigned per_plane, main_groups, m_pp, nblk, pls, plane_elems;
    __device__ __forceinline__ void setup(const WinDims &d, const WinRt &rt) {
        nblk = (unsigned)(d.th + rt.LR - 1) / (unsigned)rt.LR;
        main_groups = (nblk + rt.RPW - 1) / (unsigned)rt.RPW;
        per_plane = main_groups + (rt.cls == CLS_D && d.tw + rt.Q0 > WM ? (nblk + 15) / 16 : 0);
        m_pp = win_magic(per_plane);
        pls = (main_groups * rt.RPW * rt.LR + rt.DH) * rt.RS;
        plane_elems = (unsigned)(d.C * d.H * d.W);
    }
};
// One item: uniform plane and first row of its group, this lane's row and column from there.
struct WinItem {
    unsigned pl;
    int row0;        // uniform
    int lrow, col;   // output 0 of the lane lies at (row0 + lrow, col)
    const float *base;
};
template <int WM, bool TILE>
__device__ __forceinline__ WinItem win_item(const WinGroups<WM, TILE> &g, const WinRt &rt, const float *lds,
                                            unsigned i) {
    WinItem it;
    it.pl = TILE ? 0 : win_div(i, g.m_pp);
    unsigned b = i - it.pl * g.per_plane;
    const unsigned lane = threadIdx.x & 63;
    unsigned lrb = rt.RPW == 1 ? 0 : lane / (unsigned)rt.JW, j = rt.RPW == 1 ? lane : lane % (unsigned)rt.JW;
    b *= rt.RPW;
    bool spare = false;
    if (rt.cls == CLS_D && b >= g.main_groups * rt.RPW) {
        b = (b / (unsigned)rt.RPW - g.main_groups) * 16;
        lrb = lane / 4, j = WM + lane % 4;
        spare = lrb > g.nblk - 1 - b;  // (more lanes than row-blocks: no such rows, some LDS address)
        lrb = spare ? 0 : lrb;
    }
    it.row0 = (int)(b * rt.LR);
    it.lrow = spare ? 0x10000 : (int)(lrb * rt.LR) + rt.P0;
    it.col = rt.cls == CLS_H ? (int)(4 * j) : (int)j - rt.Q0;
    it.base = lds + (it.pl * g.pls + b * (unsigned)(rt.LR * rt.RS)) + (lrb * (unsigned)(rt.LR * rt.RS) + j);
    return it;
}

// The results of an item of a unit of `rows` x `cols` outputs whose corner the descriptor starts
// at.  32-bit results of the stacked and diagonal classes go out one per lane and row (consecutive
// lanes, consecutive columns); 16-bit ones are exchanged between neighbouring lanes first, so that
// a lane stores two adjacent columns of every second row as one word (2-byte stores run far below
// the rate of wider ones).  The row-direction class stores four columns.
template <typename T>
__device__ __forceinline__ void win_emit(__amdgpu_buffer_rsrc_t rsrc, const WinRt &rt, const WinItem &it,
                                         unsigned W, int rows, int cols, unsigned plane_elems,
                                         const float (&acc)[kWinL]) {
    constexpr unsigned ES = sizeof(T);
    const unsigned soff = (it.pl * plane_elems + (unsigned)it.row0 * W) * ES;  // uniform
    const int left = rows - it.row0;  // rows of the unit from row0 on (uniform)
    if (rt.cls == CLS_H) {
        Quad<T> v;
        v.set(acc);
        const unsigned off = ((unsigned)it.lrow * W + (unsigned)it.col) * ES;
        const bool row = it.lrow < left;
        v.store(rsrc, row && it.col + 4 <= cols ? off : kWinNowhere, soff);
        if (cols % 4 != 0) {  // uniform
            const bool part = row && it.col + 4 > cols;
#pragma unroll
            for (int l = 0; l < 3; l++)
                if (part && it.col + l < cols) win_store(rsrc, off + l * ES, soff, from_float<T>(acc[l]));
        }
        return;
    }
    const bool diag = rt.cls == CLS_D;
    const int ew = diag ? 1 : 0;
    // (stacked class: all rows of the group are there)
    const bool whole = !diag && left >= rt.RPW * kWinL;
    if constexpr (ES == 4) {
        const unsigned off = ((unsigned)it.lrow * W + (unsigned)it.col) * ES;
        if (whole) {  // uniform
            const unsigned o = it.col < cols ? off : kWinNowhere;
#pragma unroll
            for (int l = 0; l < kWinL; l++) win_store(rsrc, o, soff + l * W * ES, acc[l]);
        } else {
#pragma unroll
            for (int l = 0; l < kWinL; l++) {
                const bool in = it.lrow + l * rt.EH < left && (unsigned)(it.col + l * ew) < (unsigned)cols;
                win_store(rsrc, in ? off + (unsigned)(l * rt.EH * (int)W + l * ew) * ES : kWinNowhere, soff, acc[l]);
            }
        }
    } else {
        // lanes 2i and 2i+1 hold neighbouring columns: the even one stores row l, the odd one row l+1
        const int odd = threadIdx.x & 1;
        const unsigned off = (unsigned)((it.lrow + (odd ? rt.EH : 0)) * (int)W + it.col + (odd ? ew - 1 : 0)) * ES;
#pragma unroll
        for (int l = 0; l < kWinL; l += 2) {
            const float send = odd ? acc[l] : acc[l + 1], keep = odd ? acc[l + 1] : acc[l];
            const float got = __builtin_bit_cast(
                float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, send), 0xB1, 0xf, 0xf, true));
            Vec4<T> pk;
            pk.set(odd ? got : keep, odd ? keep : got, 0.f, 0.f);
            const unsigned word = (unsigned)__builtin_bit_cast(unsigned long long, pk.v);
            const int q = it.col + l * ew + (odd ? ew - 1 : 0);
            const bool row = whole || it.lrow + l * rt.EH + (odd ? rt.EH : 0) < left;
            const bool both = row && q + 1 < cols && (!diag || q >= 0);
            if (!diag) {
                __builtin_amdgcn_raw_buffer_store_b32(word, rsrc, both ? off : kWinNowhere, soff + l * W * ES, 2);
                if (cols % 2 != 0) {  // uniform
                    if (row && q == cols - 1)
                        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)word, rsrc, off, soff + l * W * ES, 0);
                }
            } else {
                const unsigned o = off + (unsigned)(l * rt.EH * (int)W + l) * ES;
                __builtin_amdgcn_raw_buffer_store_b32(word, rsrc, both ? o : kWinNowhere, soff, 2);
                const bool lo = row && q == cols - 1, hi = row && q == -1;
                if (lo || hi)
                    __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(hi ? word >> 16 : word), rsrc,
                                                          hi ? o + 2u : o, soff, 0);
            }
        }
    }
}

// Taps of one channel for the table-driven body, one per lane (LDS offset and weight bits), fetched
// with lane reads.
template <int K, int WM, bool TILE>
struct WinTableTaps {
    using G = WinTableGeo<K, WM, TILE>;
    int off, wbits;
    __device__ __forceinline__ void load(const int8_t *__restrict__ dhdw, const float *__restrict__ wt,
                                         int c, int flip) {
        const int s = min((int)(threadIdx.x & 63), K - 1);
        const int dh = dhdw[((size_t)c * K + s) * 2], dw = dhdw[((size_t)c * K + s) * 2 + 1];
        off = (flip ? -1 : 1) * (dh * G::RS + dw) + G::DH * G::RS + G::PL;
        wbits = wt != nullptr ? __builtin_bit_cast(int, wt[(size_t)c * K + s]) : 0;
    }
    // (opaque to the optimiser, once per item: the lane reads stay with the item instead of being
    // hoisted into 2 K scalar registers for the whole walk)
    __device__ __forceinline__ void touch() { asm volatile("" : "+v"(off), "+v"(wbits)); }
    __device__ __forceinline__ int offset(int s) const { return __builtin_amdgcn_readlane(off, s); }
    __device__ __forceinline__ float weight(int s) const {
        return __builtin_bit_cast(float, __builtin_amdgcn_readlane(wbits, s));
    }
    // body(s, v): v[k] = source of tap s for the item's output k; the reads of tap s + 2 are issued
    // before tap s is used
    template <class F>
    __device__ __forceinline__ void sweep(const float *base, F &&body) const {
        float v[3][kWinL];
        auto read = [&](int s) {
            const float *q = base + offset(s);
#pragma unroll
            for (int k = 0; k < kWinL; k++) v[s % 3][k] = q[k * G::RS];
        };
        read(0);
        if (K > 1) read(1);
#pragma unroll
        for (int s = 0; s < K; s++) {
            if (s + 2 < K) read(s + 2);
            body(s, v[s % 3]);
        }
    }
};

// f(orientation) with the orientation as a compile-time constant, or table() for any other angle
template <class F, class G>
__device__ __forceinline__ void win_switch(int o, F &&f, G &&table) {
    switch (o) {
        case 0: f(std::integral_constant<int, 0>{}); break;
        case 1: f(std::integral_constant<int, 1>{}); break;
        case 2: f(std::integral_constant<int, 2>{}); break;
        case 3: f(std::integral_constant<int, 3>{}); break;
        case 4: f(std::integral_constant<int, 4>{}); break;
        case 5: f(std::integral_constant<int, 5>{}); break;
        case 6: f(std::integral_constant<int, 6>{}); break;
        case 7: f(std::integral_constant<int, 7>{}); break;
        default: table();
    }
}

// The walk over units [u0, u1).  start(unit) runs under the first loads' latency, eval(unit, next,
// more) between the commit of a unit and that of the next, with the next one's loads in flight.
template <typename T, int WM, bool TILE, class Start, class Eval>
__device__ __forceinline__ void win_walk(const T *__restrict__ x, float *lds, unsigned words, const WinDims &d,
                                         const WinRt &rt, unsigned pls, int c, int u0, int u1,
                                         Start &&start, Eval &&eval) {
    WinStager<T, WM, TILE> sg;
    sg.setup(d, rt, pls);
    WinUnit<TILE> cur;
    cur.first(d, u0);
    sg.prefetch(x, d, c, cur);
    start(cur);
    lds_zero<WinMode<WM, TILE>::NT>(lds, words);
    for (int u = u0; u < u1; u++) {
        set_progress_priority(u - u0, u1 - u0);
        __syncthreads();
        wait_vmem_done();
        sg.commit(lds, d, rt, cur);
        __syncthreads();
        const WinUnit<TILE> now = cur;
        if (u + 1 < u1) {
            cur.advance(d);
            sg.prefetch(x, d, c, cur);
        }
        eval(now, cur, u + 1 < u1);
    }
}

// units of group g of `groups`
__device__ __forceinline__ void win_range(unsigned units, unsigned groups, unsigned g, int &u0, int &u1) {
    const unsigned per = (units + groups - 1) / groups;
    u0 = (int)min(units, g * per);
    u1 = (int)min(units, g * per + per);
}

// Outputs of channel c over the units [u0, u1): body(base, acc) adds up one item from its place in LDS.
template <typename T, class G, int WM, bool TILE, class Start, class Body>
__device__ __forceinline__ void win_conv(const T *__restrict__ src, T *__restrict__ dst, float *lds,
                                         unsigned words, const WinDims &d, int c, int u0, int u1, float bv,
                                         Start &&start, Body &&body) {
    WinRt rt;
    rt.set<G>();
    WinGroups<WM, TILE> grp;
    grp.setup(d, rt);
    const size_t plane = (size_t)d.H * d.W;
    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    win_walk<T, WM, TILE>(
        src, lds, words, d, rt, grp.pls, c, u0, u1, [&](const WinUnit<TILE> &) { start(); },
        [&](const WinUnit<TILE> &now, const WinUnit<TILE> &, bool) {
            const T *out = dst + ((size_t)now.n * d.C + c) * plane + (size_t)now.p * d.W + now.q;
            const __amdgpu_buffer_rsrc_t rsrc = win_rsrc(out, dst + (size_t)d.N * d.C * plane);
            const unsigned total = now.planes(d) * grp.per_plane;
            const int rows = now.rows(d), cols = now.cols(d);
            for (unsigned i = wave; i < total; i += WinMode<WM, TILE>::NT / 64) {
                const WinItem it = win_item(grp, rt, lds, i);
                float acc[kWinL];
#pragma unroll
                for (int l = 0; l < kWinL; l++) acc[l] = bv;
                body(it.base, acc);
                // (opaque: results first used behind a branch of the stores would be computed
                // there, with all of the item's sources kept in registers until then)
#pragma unroll
                for (int l = 0; l < kWinL; l++) asm volatile("" : "+v"(acc[l]));
                win_emit<T>(rsrc, rt, it, (unsigned)d.W, rows, cols, grp.plane_elems, acc);
            }
        });
}

// fprop, and dgrad with flip = 1 (the weights in reverse tap order)
template <typename T, int K, int WM, bool TILE>
__global__ __launch_bounds__((WinMode<WM, TILE>::NT)) __attribute__((amdgpu_waves_per_eu(WinMode<WM, TILE>::kWaves, 8))) void window_kernel(
    const T *__restrict__ src, const float *__restrict__ wt, const float *__restrict__ bias,
    const void *__restrict__ blob, T *__restrict__ dst, WinDims d, unsigned words, int groups, int flip) {
    extern __shared__ __align__(16) float lds[];
    int c, group, u0, u1;
    plane_task(blob, d.C, K, groups, c, group);
    win_range(d.units, groups, group, u0, u1);
    const float bv = bias != nullptr ? bias[c] : 0.f;
    win_switch(
        taps_class(blob, d.C, K)[c],
        [&](auto O) {
            using G = WinGeo<O, K, WM, TILE>;
            ChannelTaps<G, OP_FPROP, T, K, false> taps;
            win_conv<T, G, WM, TILE>(
                src, dst, lds, words, d, c, u0, u1, bv, [&] { taps.load(wt, bias, c, flip); },
                [&](const float *base, float (&acc)[kWinL]) {
                    static_for<G::plan.nsrc>([&](auto m) {
                        constexpr int off = G::imm(G::plan.sh[m], G::plan.sw[m]);
                        const float v = base[off];
                        static_for<kWinL>([&](auto l) {
                            constexpr int t = G::plan.user[m][l];
                            if constexpr (t >= 0) acc[l] = __builtin_fmaf(v, taps.wv[t], acc[l]);
                        });
                    });
                    pipeline_reads_and_fmas<G::plan.nsrc, plan_fma_count(G::plan, kWinL)>();
                });
        },
        [&] {
            WinTableTaps<K, WM, TILE> table;
            win_conv<T, WinTableGeo<K, WM, TILE>, WM, TILE>(
                src, dst, lds, words, d, c, u0, u1, bv, [&] { table.load(taps_dhdw(blob), wt, c, flip); },
                [&](const float *base, float (&acc)[kWinL]) {
                    table.touch();
                    table.sweep(base, [&](int s, const float (&v)[kWinL]) {
                        const float ws = table.weight(s);
#pragma unroll
                        for (int k = 0; k < kWinL; k++) acc[k] = __builtin_fmaf(v[k], ws, acc[k]);
                    });
                });
        });
}

// dy of one item, straight from memory to the registers of the lane that uses it: four columns at
// once in the row-direction class, one element per row otherwise; zeros where the output does not
// exist.
template <typename T>
struct WinDy {
    unsigned raw[kWinL];  // a Quad, or one element each
    unsigned cut;
    __device__ __forceinline__ unsigned one(__amdgpu_buffer_rsrc_t rsrc, unsigned off, unsigned soff) const {
        if constexpr (sizeof(T) == 4) return __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, soff, 0);
        else return (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rsrc, off, soff, 0);
    }
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rsrc, const WinRt &rt, const WinItem &it,
                                         unsigned W, int rows, int cols, unsigned plane_elems) {
        constexpr unsigned ES = sizeof(T);
        const unsigned soff = (it.pl * plane_elems + (unsigned)it.row0 * W) * ES;
        const int left = rows - it.row0;
        if (rt.cls == CLS_H) {
            // (a quad that the unit's last column cuts is loaded from four columns before its end
            // and shifted: units are at least four columns wide)
            cut = (unsigned)max(0, it.col - (cols - 4));
            const unsigned off = ((unsigned)it.lrow * W + (unsigned)it.col - cut) * ES;
            Quad<T> q;
            q.load(rsrc, it.lrow < left && it.col < cols ? off : kWinNowhere, soff);
            __builtin_memcpy(raw, &q.v, sizeof(q.v));
            return;
        }
        const bool diag = rt.cls == CLS_D;
        const int ew = diag ? 1 : 0;
        const unsigned off = ((unsigned)it.lrow * W + (unsigned)it.col) * ES;
        if (!diag && left >= rt.RPW * kWinL) {  // uniform: all rows of the group are there
            const unsigned o = it.col < cols ? off : kWinNowhere;
#pragma unroll
            for (int l = 0; l < kWinL; l++) raw[l] = one(rsrc, o, soff + l * W * ES);
        } else {
#pragma unroll
            for (int l = 0; l < kWinL; l++) {
                const bool in = it.lrow + l * rt.EH < left && (unsigned)(it.col + l * ew) < (unsigned)cols;
                raw[l] = one(rsrc, in ? off + (unsigned)(l * rt.EH * (int)W + l * ew) * ES : kWinNowhere, soff);
            }
        }
    }
    __device__ __forceinline__ void get(const WinRt &rt, float (&o)[kWinL], bool ragged) {
        if (rt.cls == CLS_H) {
            Quad<T> q;
            __builtin_memcpy(&q.v, raw, sizeof(q.v));
            if (ragged) q.drop(min(cut, 3u));
#pragma unroll
            for (int l = 0; l < kWinL; l++) o[l] = q.get(l);
        } else {
#pragma unroll
            for (int l = 0; l < kWinL; l++) {
                if constexpr (sizeof(T) == 4) o[l] = __builtin_bit_cast(float, raw[l]);
                else o[l] = to_float(__builtin_bit_cast(T, (uint16_t)raw[l]));
            }
        }
    }
};

// Sums of channel c over the units [u0, u1): add(base, dy, acc) runs for every item.  The dy of a
// wave's next item is loaded while it works on one.
template <typename T, class G, int K, int WM, bool TILE, class Add, class SlotOf>
__device__ __forceinline__ void win_wgrad(const T *__restrict__ x, const T *__restrict__ dy,
                                          const WgradOut &out, float *lds, unsigned words, const WinDims &d,
                                          int c, int u0, int u1, int group, Add &&add, SlotOf slot_of) {
    constexpr int NT = WinMode<WM, TILE>::NT;
    WinRt rt;
    rt.set<G>();
    WinGroups<WM, TILE> grp;
    grp.setup(d, rt);
    const size_t plane = (size_t)d.H * d.W;
    const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    WinDy<T> g;
    float acc[K + 1];  // acc[s] for representative taps s, acc[K] = sum of dy (bias gradient)
#pragma unroll
    for (int s = 0; s <= K; s++) acc[s] = 0.f;
    // (Item i of the unit.  A wave without one loads the last again and drops it: behind that lie planes that
    // need not be there, and the descriptor's bound covers the per-lane part of an address only, not soff.  The
    // loads sent nowhere instead, as rows that do not exist, took 19 x 829 x 35 x 35 in bf16 from 74 to 84 us.)
    auto fetch = [&](const WinUnit<TILE> &u, unsigned i) {
        const T *at = dy + ((size_t)u.n * d.C + c) * plane + (size_t)u.p * d.W + u.q;
        const __amdgpu_buffer_rsrc_t rsrc = win_rsrc(at, dy + (size_t)d.N * d.C * plane);
        const WinItem it = win_item(grp, rt, lds, min(i, u.planes(d) * grp.per_plane - 1));
        g.load(rsrc, rt, it, (unsigned)d.W, u.rows(d), u.cols(d), grp.plane_elems);
    };
    win_walk<T, WM, TILE>(
        x, lds, words, d, rt, grp.pls, c, u0, u1, [&](const WinUnit<TILE> &u) { fetch(u, wave); },
        [&](const WinUnit<TILE> &now, const WinUnit<TILE> &next, bool more) {
            const unsigned total = now.planes(d) * grp.per_plane;
            const bool ragged = now.cols(d) % 4 != 0;
            for (unsigned i = wave; i < total; i += NT / 64) {
                float gy[kWinL];
                g.get(rt, gy, ragged);
                const bool last = i + NT / 64 >= total;
                if (!last || more) fetch(last ? next : now, last ? wave : i + NT / 64);
                add(win_item(grp, rt, lds, i).base, gy, acc);
#pragma unroll
                for (int l = 0; l < kWinL; l++) acc[K] += gy[l];
            }
            // (a wave without items in this unit still takes the next unit's first dy)
            if (wave >= total && more) fetch(next, wave);
        });
    wgrad_epilogue<K, NT>(acc, lds, out, c, group, slot_of);
}

template <typename T, int K, int WM, bool TILE>
__global__ __launch_bounds__((WinMode<WM, TILE>::NT)) __attribute__((amdgpu_waves_per_eu(WinMode<WM, TILE>::kWavesWgrad, 8))) void window_wgrad_kernel(
    const T *__restrict__ x, const T *__restrict__ dy, const void *__restrict__ blob, WgradOut out, WinDims d,
    unsigned words, int cus) {
    extern __shared__ __align__(16) float lds[];
    int c, group, u0, u1;
    if (!wgrad_task(blob, d.C, K, out.NG, cus, c, group)) return;
    win_range(d.units, out.NG, group, u0, u1);
    win_switch(
        taps_class(blob, d.C, K)[c],
        [&](auto O) {
            using G = WinGeo<O, K, WM, TILE>;
            win_wgrad<T, G, K, WM, TILE>(
                x, dy, out, lds, words, d, c, u0, u1, group,
                [&](const float *base, const float (&gy)[kWinL], float (&acc)[K + 1]) {
                    static_for<G::plan.nsrc>([&](auto m) {
                        constexpr int off = G::imm(G::plan.sh[m], G::plan.sw[m]);
                        const float v = base[off];
                        static_for<kWinL>([&](auto l) {
                            constexpr int t = G::plan.user[m][l];
                            if constexpr (t >= 0) acc[t] = __builtin_fmaf(v, gy[l], acc[t]);
                        });
                    });
                    pipeline_reads_and_fmas<G::plan.nsrc, plan_fma_count(G::plan, kWinL)>();
                },
                [](int s) { return (int)G::plan.rep[s]; });
        },
        [&] {
            WinTableTaps<K, WM, TILE> table;
            table.load(taps_dhdw(blob), nullptr, c, 0);
            win_wgrad<T, WinTableGeo<K, WM, TILE>, K, WM, TILE>(
                x, dy, out, lds, words, d, c, u0, u1, group,
                [&](const float *base, const float (&gy)[kWinL], float (&acc)[K + 1]) {
                    table.touch();
                    table.sweep(base, [&](int s, const float (&v)[kWinL]) {
#pragma unroll
                        for (int k = 0; k < kWinL; k++) acc[s] = __builtin_fmaf(v[k], gy[k], acc[s]);
                    });
                },
                [](int s) { return s; });
        });
}

// ---------------------------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------------------------
// Workgroups resident at once: the register bound comes from the occupancy query (cached, with
// little LDS), the LDS bound from the launch's own size.
template <class Kern>
int win_slots(Kern kern, int threads, int *cache, size_t lds, int &cus) {
    const int packed = per_device_once(cache, [&] {
        allow_large_lds(kern, 160 * 1024);
        return resident_slots(kern, threads, 1024);
    });
    cus = packed >> 16;
    const int by_regs = (packed & 0xffff) / cus, by_lds = (int)(160 * 1024 / lds);
    return cus * (by_lds < 1 ? 1 : (by_regs < by_lds ? by_regs : by_lds));
}
template <typename T, int K, int WM, bool TILE>
int launch_window_conv_v(const void *src, const float *w, const float *bias, const void *taps, void *dst,
                         const WinDims &d, int flip, hipStream_t st) {
    const unsigned words = win_words<K, WM, TILE>(d.th, d.PB);
    const size_t lds = (size_t)words * sizeof(float);
    static int cache[kMaxDevices];
    int cus = 0;
    const int slots = win_slots(window_kernel<T, K, WM, TILE>, WinMode<WM, TILE>::NT, cache, lds, cus);
    if (d.N == 0) return 0;  // set-up only
    const int groups = win_groups(d, slots, cus, d.units);
    window_kernel<T, K, WM, TILE><<<dim3(d.C * groups), dim3(WinMode<WM, TILE>::NT), lds, st>>>(
        (const T *)src, w, bias, taps, (T *)dst, d, words, groups, flip);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}
template <typename T, int K>
int launch_window_conv(const void *src, const float *w, const float *bias, const void *taps, void *dst,
                       const WinDims &d, int flip, hipStream_t st) {
#define DWO_GO(WM, TILE) launch_window_conv_v<T, K, WM, TILE>(src, w, bias, taps, dst, d, flip, st)
    if (d.N == 0) return DWO_GO(16, false) | DWO_GO(32, false) | DWO_GO(64, false) | DWO_GO(64, true);
    if (d.tiled()) return DWO_GO(64, true);
    return d.tw <= 16 ? DWO_GO(16, false) : (d.tw <= 32 ? DWO_GO(32, false) : DWO_GO(64, false));
#undef DWO_GO
}

template <typename T, int K, int WM, bool TILE>
int launch_window_wgrad_v(const void *x, const void *dy, const void *taps, float *part, float *dw, float *db,
                          unsigned *tickets, const WinDims &d, int *groups_out, hipStream_t st) {
    constexpr int NT = WinMode<WM, TILE>::NT;
    const unsigned words = cmax(win_words<K, WM, TILE>(d.th, d.PB), NT);  // (the epilogue's rows: NT words)
    const size_t lds = (size_t)words * sizeof(float);
    static int cache[kMaxDevices];
    int cus = 0;
    const int slots = win_slots(window_wgrad_kernel<T, K, WM, TILE>, NT, cache, lds, cus);
    if (d.N == 0) return 0;
    const int groups = win_groups(d, slots, cus, win_wgrad_groups(d.C, K));
    *groups_out = groups;
    window_wgrad_kernel<T, K, WM, TILE><<<dim3(plane_grid(d.C, groups, cus)), dim3(NT), lds, st>>>(
        (const T *)x, (const T *)dy, taps, WgradOut{part, dw, db, groups, tickets}, d, words, cus);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}
template <typename T, int K>
int launch_window_wgrad(const void *x, const void *dy, const void *taps, float *part, float *dw, float *db,
                        unsigned *tickets, const WinDims &d, int *groups_out, hipStream_t st) {
#define DWO_GO(WM, TILE) \
    launch_window_wgrad_v<T, K, WM, TILE>(x, dy, taps, part, dw, db, tickets, d, groups_out, st)
    if (d.N == 0) return DWO_GO(16, false) | DWO_GO(32, false) | DWO_GO(64, false) | DWO_GO(64, true);
    if (d.tiled()) return DWO_GO(64, true);
    return d.tw <= 16 ? DWO_GO(16, false) : (d.tw <= 32 ? DWO_GO(32, false) : DWO_GO(64, false));
#undef DWO_GO
}

}  // namespace dwo
