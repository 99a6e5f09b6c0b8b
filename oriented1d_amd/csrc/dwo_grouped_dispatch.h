// Which calls the grouped kernels of dwo_grouped.h cover, how an image is cut into tiles, and the
// launchers compiled per (element type, kernel size).
#pragma once

#include "dwo_common.h"
#include "dwo_plan.h"

// X(K): the kernel sizes of the networks and of the reference's layer benchmark
#define DWO_GROUPED_KS(X) X(7) X(13) X(15) X(27) X(31)

namespace dwo {

constexpr int kGrpThreads = 512;
constexpr int kGrpPixels = 4960;  // staged pixels of 16 bytes: two workgroups per CU
constexpr int kGrpSlots = 512;     // workgroups resident on the chip
constexpr int kGrpLeastRows = 8;  // of a tile that is cut to fill the chip
// channels of one 16-byte pixel piece: they share an orientation
constexpr int grp_channels(size_t esize) { return 16 / (int)esize; }
// inputs of the pointwise layer that the projecting kernel is compiled for: the channels of an image
constexpr int kGrpProjected = 3;
// widest tile, in outputs
constexpr int grp_tile_cols(int S) { return S == 1 ? 64 : 32; }

// Workgroup -> (unit, channel group) of a launch's units x ngroups tasks.  The groups of a unit share its lines, so
// they get ids of one XCD (consecutive ids go to the eight XCDs in turn) at about the same time: unit u runs on
// XCD u % 8.  The tasks of the units beyond the last eight are dealt to all XCDs in runs of equal length instead:
// two images of 1024 x 28 x 28 fp32 ran on two of the eight (fprop 27 us; now 9.2, on the slice kernels 9.4).
// False for the ids that fill up the last run.
constexpr long grp_grid(long units, int ngroups) { return 8 * (units / 8 * ngroups + (units % 8 * ngroups + 7) / 8); }
// A launch holds fewer than 2^32 threads; what needs more goes to the kernels that would take it otherwise (the slice
// kernels walk any number of planes of 56 x 56 and 28 x 28 with the chip's slots).
constexpr bool grp_grid_fits(long grid) { return grid * kGrpThreads < 1L << 32; }
__host__ __device__ inline bool grp_task(unsigned block, int units, int ngroups, int &unit, int &group) {
    const unsigned xcd = block % 8, k = block / 8, full = (unsigned)(units / 8 * ngroups);
    if (k < full) {
        unit = (int)(k / (unsigned)ngroups * 8 + xcd);
        group = (int)(k % (unsigned)ngroups);
        return true;
    }
    const unsigned t = xcd * (unsigned)((units % 8 * ngroups + 7) / 8) + (k - full);
    unit = units / 8 * 8 + (int)(t / (unsigned)ngroups);
    group = (int)(t % (unsigned)ngroups);
    return unit < units;
}

struct GrpTiles {
    int th, tw, nth, ntw;  // tile extents and counts
    int run;               // tiles of an XCD where they are dealt in runs, else 0
};

// Tiles in runs (stride 2, where a window is up to four times its tile's share of the image): neighbouring tiles on one XCD at about
// the same time, so that they find each other's lines in its L2.  grp_task deals units to the XCDs in turn; in runs XCD x
// gets the x-th eighth of them, in bands of two tile columns (a tile shares more with the rows below than with the columns
// beside; without bands 64 x 64 x 224 x 224 wgrad in bf16 381 instead of 367).
__host__ __device__ inline void grp_run_tile(const GrpTiles &t, int unit, int &n, int &row, int &col) {
    const int per = t.nth * t.ntw;
    if (unit < 8 * t.run) unit = unit % 8 * t.run + unit / 8;
    n = unit / per;
    const int k = unit - n * per, b = k / (2 * t.nth), j = k - b * (2 * t.nth), two = 2 * b + 1 < t.ntw ? 1 : 0;
    row = j >> two, col = 2 * b + (j & two);
}
// Where that pays (us, in turn / in runs; NHWC, C = 64 unless noted, images N x H x W).  In general: images cut into tiles; tile columns
// no multiple of eight, with which an XCD has whole columns as it is; many more tasks than run at once (3 x 200 x 300, K = 31, 840 of
// them, wgrad fp32 47.5 / 50.0, bf16 40.9 / 43.0; 8 x 256 x 256, 2048, 119.6 / 112.0 and 74.7 / 63.9).
//   fprop, wgrad: always while x and y fit the 256 MB of cache behind the L2s (K = 31 64 x 112 x 112 fp32 150 / 127, 211 / 171, K = 15 fp32 12 x
//     256 x 256 100 / 87, 127 / 106, K = 7 bf16 32 x 224 x 224 94 / 83, 119 / 109).  Beyond it eight places at a time spread what is read, and
//     the halos have to weigh more:
//     fprop with K = 27 and 31 (bf16 64 x 224 x 224 312 / 300, fp32 611 / 595, 128 x 112 x 112 with 128 channels 621 / 572; K = 15 bf16 34 x 320 x 288
//     228 / 239, K = 7 293 / 323);
//     wgrad with these, in 16 bits from K = 13 on, of at most 384 bytes per pixel (bf16 64 x 224 x 224 440 / 357, K = 15 287 / 257, 12 x 448 x 448 198 /
//     204, K = 7 227 / 261; fp32 1002 / 966, K = 15 34 x 320 x 288 543 / 592; bf16 80 x 112 x 112 with 192 channels 464 / 426, 64 with 256 403 / 430; fp32 32 x
//     224 x 224 with 96 824 / 841, with 128 775 / 886).
//   dgrad: whole bands, 16 bits or K = 27 and 31, 64 channels at most beyond that cache (K = 31 bf16 64 x 224 x 224, two tile columns, 240 /
//     203, K = 15 265 / 242, K = 7 264 / 251; fp32 K = 31 506 / 490, K = 15 506 / 506; three columns, bf16 34 x 320 x 288, 270 / 290; one column, 128 x 112 x
//     112, 81 / 86; 24 x 224 x 224 with 192 channels 262 / 291).
// Behind a projection the image is small and nothing is gained.
enum GrpPass { GRP_FPROP, GRP_DGRAD, GRP_WGRAD };
inline int grp_run(const GrpTiles &t, const ConvDims &d, size_t esize, GrpPass pass) {
    const long units = (long)d.N * t.nth * t.ntw;
    if (d.stride != 2 || t.nth * t.ntw == 1 || t.ntw % 8 == 0 || units * (d.C / grp_channels(esize)) < 4 * kGrpSlots) return 0;
    const bool wide = d.K >= 27, cached = ((double)d.H * d.W + (double)d.P * d.Q) * d.C * d.N * esize <= 1 << 28;
    bool pays = wide || cached;
    if (pass == GRP_WGRAD) pays = cached || ((wide || (esize == 2 && d.K >= 13)) && d.C * esize <= 384);
    if (pass == GRP_DGRAD) pays = t.ntw % 2 == 0 && (wide || esize == 2) && (cached || d.C <= 64);
    return pays ? (int)(units / 8) : 0;
}

// Partial sums per (channel, tap): about two rounds of the chip's slots at most, and no more than there are tiles of
// 16 x 32 outputs; a multiple of eight (unit u runs on XCD u % 8) where there are as many tiles.  A workgroup's sums
// over lanes and waves cost as much as a few hundred outputs, so it gets 256 of them, or four tiles where tiles are
// that small (surplus groups would add zeros, at that cost).  K = 31, us, with a group per tile / like this:
// 107 x 16 x 5 x 64 fp32 38 / 28, 64 x 64 x 17 x 17 bf16 stride 2 44 / 33, 53 x 32 x 4 x 84 fp32 33 / 25.
inline int grp_wgrad_groups(const ConvDims &d, size_t esize) {
    const long units = (long)d.N * ((d.P + 15) / 16) * ((d.Q + 31) / 32), ngroups = d.C / grp_channels(esize);
    long most = (long)d.N * d.P * d.Q / 256;
    if (most < (units + 3) / 4) most = (units + 3) / 4;
    long G = 1024 / ngroups;
    if (G > most) G = most;
    G = ((G < 1 ? 1 : G) + 7) / 8 * 8;
    return (int)(G < units ? G : units);
}

template <typename T, int K>
int launch_grouped_conv(const void *src, const float *w, const float *bias, const void *taps, void *dst,
                        const ConvDims &d, int flip, hipStream_t st);
template <typename T, int K>
int launch_grouped_wgrad(const void *x, const void *dy, const void *taps, float *part, const ConvDims &d,
                         int *groups_out, hipStream_t st);
// fprop at stride 2 behind a pointwise layer of kGrpProjected inputs
template <typename T, int K>
int launch_grouped_projected(const void *x, const float *pw_w, const float *pw_b, const float *w, const float *bias,
                             const void *taps, void *y, const ConvDims &d, hipStream_t st);

#define DWO_DECLARE(T, K)                                                                                \
    extern template int launch_grouped_conv<T, K>(const void *, const float *, const float *,           \
                                                  const void *, void *, const ConvDims &, int,          \
                                                  hipStream_t);                                         \
    extern template int launch_grouped_wgrad<T, K>(const void *, const void *, const void *, float *,   \
                                                   const ConvDims &, int *, hipStream_t);              \
    extern template int launch_grouped_projected<T, K>(const void *, const float *, const float *,      \
                                                       const float *, const float *, const void *,      \
                                                       void *, const ConvDims &, hipStream_t);
#define DWO_DECLARE_ALL(K) DWO_DECLARE(float, K) DWO_DECLARE(bf16_t, K) DWO_DECLARE(f16_t, K)
DWO_GROUPED_KS(DWO_DECLARE_ALL)
#undef DWO_DECLARE_ALL
#undef DWO_DECLARE

}  // namespace dwo
