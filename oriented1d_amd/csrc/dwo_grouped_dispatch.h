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
    int run;               // tiles of an XCD where they are dealt in runs (GrpTile::set), else 0
};

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
