// Host side of the window kernels (dwo_window.h): which shapes they take, how a launch is cut into
// units, and the launchers defined in dwo_inst_window.hip, one translation unit per (element type,
// kernel size).
#pragma once

#include <hip/hip_runtime.h>

#include "dwo_common.h"
#include "dwo_plan.h"

// kernel sizes with window kernels: those of the networks and of their cropped backbones, and the
// 7 of the reference's own layer benchmark
#define DWO_WINDOW_KS(X) X(7) X(13) X(15) X(27) X(31)

namespace dwo {

struct WinDims {
    int N, C, H, W;
    int th, tw;    // rows and columns of a unit's planes or tile
    int nth, ntw;  // tiles per plane (1 x 1: plane mode)
    int PB;        // planes per unit (1 in tile mode)
    int units;     // units per channel
    __host__ __device__ bool tiled() const { return nth * ntw > 1; }
};

constexpr int kWinMaxTile = 64;
constexpr int kWinMaxPlanes = 8;
constexpr int kMaxWinGroups = 64;  // image groups per channel in wgrad (partial sums per tap), at most
// and no more than dwo_wgrad_static has room for (C x (K + 1) sums each).  The bound starts at C = 1024
// (K = 31), where a chip's slots make at most two groups per channel: no launch is cut differently for it.
inline int win_wgrad_groups(int C, int K) {
    const long fit = (long)(DWO_STATIC_SCRATCH_BYTES / sizeof(float)) / ((long)C * (K + 1));
    return fit < 1 ? 1 : (fit < kMaxWinGroups ? (int)fit : kMaxWinGroups);
}
// Threads per workgroup, and staged four-column chunks per thread at most (plane and tile mode).
constexpr int kWinThreads = 512;
constexpr int win_slots_per_thread(bool tile) { return tile ? 5 : 2; }

inline bool win_has_k(int K) {
#define DWO_MATCH(K_) if (K == K_) return true;
    DWO_WINDOW_KS(DWO_MATCH)
#undef DWO_MATCH
    return false;
}

// Cuts a launch into units; false when the window kernels do not take the shape (rows shorter than
// a four-column chunk, units beyond 32-bit byte offsets: a tile's window begins up to `pad` rows above the
// image, and its offsets count from there).
inline bool win_dims(int N, int C, int H, int W, int K, size_t esize, WinDims &d) {
    if (!win_has_k(K) || W < 4 || (double)H * W * esize >= 2147483648.0 || H > 32767) return false;
    // (a launch holds fewer than 2^32 threads: a workgroup per channel at least, on a padded grid)
    if (((long)C + 4096) * kWinThreads >= 1L << 32) return false;
    d.N = N, d.C = C, d.H = H, d.W = W;
    const int pad = K / 2;
    // a wave takes 64 lanes of row-blocks: rounds of the workgroup's waves over those of `planes`
    // planes of th x tw
    auto rounds = [](int planes, int th, int tw) {
        const int wm = tw <= 16 ? 16 : (tw <= 32 ? 32 : 64), rpw = 64 / wm, waves = kWinThreads / 64;
        return (planes * (((th + 3) / 4 + rpw - 1) / rpw) + waves - 1) / waves;
    };
    if (H <= kWinMaxTile && W <= kWinMaxTile) {
        d.th = H, d.tw = W, d.nth = d.ntw = 1, d.PB = 1;
        const int wm = W <= 16 ? 16 : (W <= 32 ? 32 : 64);
        // planes per unit: the count that keeps the waves busiest, a unit costing about one round on
        // top of its own (barriers, staging), within 53 KB of LDS (three workgroups per CU)
        const int chunks = H * ((W + 3) / 4);
        double best = 1e30;
        for (int pb = 1; pb <= kWinMaxPlanes && pb <= N; pb++) {
            if (chunks * pb > win_slots_per_thread(false) * kWinThreads) break;
            if (pb > 1 && (double)(pad + pb * (H + pad + 8)) * (wm + pad + 8) * 4 > 54000.0) break;
            if (pb > 1 && (double)pb * C * H * W * esize >= 2147483648.0) break;
            const double cost = (double)((N + pb - 1) / pb) * (1.0 + rounds(pb, H, W));
            if (cost < best) best = cost, d.PB = pb;
        }
        d.units = (N + d.PB - 1) / d.PB;
        return true;
    }
    // Thin planes.  A tile's waves stand for 32 rows of 64 columns, so of a plane of few rows or columns most
    // of the issue slots are spent on nothing, where the tile kernels fit their windows to the plane.  Those
    // take them from about the batch on at which they fill the chip (four channels of up to 32 rows per
    // workgroup); below it the window kernels' shorter chains win.  fprop us, tile / window kernels, K = 31:
    // 32 x 384 x 4 x 256 bf16 87 / 177, 64 x 200 x 7 x 256 fp32 160 / 224, 32 x 200 x 400 x 6 fp32 (any angle)
    // 263 / 459; 2 x 384 x 8 x 400 fp32 73 / 26; K = 7 in narrow planes: 64 x 96 x 190 x 5 bf16 96 / 54.
    const long planes = (long)N * C;
    if (H <= 4 ? planes >= 768 : (H <= 8 && planes >= 1536)) return false;
    if (W <= 8 && K > 7 && planes >= 6144) return false;
    const int window_rows = (H < kWinMaxTile + pad ? H : kWinMaxTile + pad) + pad;
    if ((double)window_rows * W * esize >= 2147483648.0) return false;
    // tiles of at most 64 x 64: the split with the least estimated work, per tile the rounds over
    // its row-blocks, the staging of its window and a fixed charge
    double best = 1e30;
    const int h0 = (H + kWinMaxTile - 1) / kWinMaxTile, w0 = (W + kWinMaxTile - 1) / kWinMaxTile;
    for (int a = h0; a <= h0 + 2; a++)
        for (int b = w0; b <= w0 + 2; b++) {
            const int th = ((H + a - 1) / a + 3) & ~3, tw = ((W + b - 1) / b + 3) & ~3;
            if (th > kWinMaxTile || tw > kWinMaxTile) continue;
            const int nth = (H + th - 1) / th, ntw = (W + tw - 1) / tw;
            if (W - (ntw - 1) * tw < 4 || nth * ntw == 1) continue;  // (a tile narrower than a chunk)
            const double chunks = (th + pad) * (tw + pad) / 4.0 / kWinThreads;
            const double cost = nth * ntw * (rounds(1, th, 64) + chunks * 0.3 + 0.7);
            if (cost < best) best = cost, d.th = th, d.tw = tw, d.nth = nth, d.ntw = ntw;
        }
    if (best == 1e30) return false;
    d.PB = 1;
    d.units = N * d.nth * d.ntw;
    return true;
}

// Workgroups per channel, at most `most`: as many as the chip holds at once (`slots` over all channels), or two
// rounds of them where one would leave a quarter idle (plane_groups).  With few channels these are many short
// workgroups; more than kMaxWinGroups of them only where that gives the busiest CU no more units than
// kMaxWinGroups do (8 channels of 64 x 128 x 128, any angle: nine units 26.1 us, eight 24.8; 3 channels: three
// 12.7, four 18.7).
inline int win_groups(const WinDims &d, int slots, int cus, int most) {
    // workgroups of equal length: the launch ends with its slowest
    auto even = [&d](int g) {
        const int per = (d.units + g - 1) / g;
        return (d.units + per - 1) / per;
    };
    auto busiest = [&d, cus](int g) { return ((long)d.C * g + cus - 1) / cus * ((d.units + g - 1) / g); };
    int g = slots / d.C;
    if (g < 1) g = 1;
    if ((long)d.C * g * 4 < (long)slots * 3) g = (2 * slots + d.C - 1) / d.C;
    if (g > d.units) g = d.units;
    if (g > most) g = most;
    g = even(g);
    if (g > kMaxWinGroups && busiest(g) > busiest(even(kMaxWinGroups))) g = even(kMaxWinGroups);
    return g;
}
template <typename T, int K>
int launch_window_conv(const void *src, const float *w, const float *bias, const void *taps, void *dst,
                       const WinDims &d, int flip, hipStream_t st);
template <typename T, int K>
int launch_window_wgrad(const void *x, const void *dy, const void *taps, float *part, float *dw, float *db,
                        unsigned *tickets, const WinDims &d, int *groups_out, hipStream_t st);

#define DWO_DECLARE(T, K)                                                                              \
    extern template int launch_window_conv<T, K>(const void *, const float *, const float *,          \
                                                 const void *, void *, const WinDims &, int,          \
                                                 hipStream_t);                                        \
    extern template int launch_window_wgrad<T, K>(const void *, const void *, const void *, float *,  \
                                                  float *, float *, unsigned *, const WinDims &,      \
                                                  int *, hipStream_t);
#define DWO_DECLARE_ALL(K) DWO_DECLARE(float, K) DWO_DECLARE(bf16_t, K) DWO_DECLARE(f16_t, K)
DWO_WINDOW_KS(DWO_DECLARE_ALL)
#undef DWO_DECLARE_ALL
#undef DWO_DECLARE

}  // namespace dwo
