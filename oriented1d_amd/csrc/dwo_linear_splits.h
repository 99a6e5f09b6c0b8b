// How the rows that a pointwise layer's parameter gradients sum over are split (linear_wgrad_kernel, dwo_linear.h).
#pragma once

#include <cstddef>

namespace dwo {

constexpr int kLinTile = 128, kLinRows = 64;  // outputs of a tile each way, rows of a step
constexpr long kLinFew = 4, kLinAlone = 224;  // tiles
constexpr long kLinAloneWide = 54, kLinAloneTall = 128;  // steps

// Splits of the rows, each with 256 rows where they are dealt evenly; a multiple of eight where there are as many (whole splits
// per XCD).  Two workgroups per CU (512), but
//   one where the outputs are at most four tiles and the rows enough for more: memory binds, and the partial sums, 64 KB per workgroup
//   both ways, are what can be saved (us with the sums, behind a pass over other memory, 512 / 256: 401408 x 512 x 128 146 / 135,
//   200704 x 96 x 384 54.5 / 49.6, 100352 x 256 x 256 35.8 / 30.6, 24576 x 512 x 128 19.2 / 17.8, 50176 x 192 x 96 16.2 / 15.8; where
//   both are as many splits the halves only cost, 16384 x 512 x 128 14.9 / 16.2, 1000 x 96 x 64 11.0 / 12.0; eight tiles, back to
//   back, 50176 x 256 x 512, 29.1 / 31.1);
//   no split where the tiles alone give each CU its workgroup: the reduction, 11 to 12 us, is saved, and the second workgroup per CU is
//   given up, which overlaps the other's chain.  With many rows that weighs more where the workgroups of an XCD share their lines: K a
//   multiple of eight tiles, so that it has the same columns of x in both splits, the more so with fewer tiles along N (us, two
//   splits / none, K wide: 1000 x 1024 x 4096 27.5 / 18.9, 3136 rows 42.2 / 41.4, 3600 45.9 / 46.8, 6272 64 / 75, 16384 179 / 184,
//   16384 x 1792 x 2048 142 / 179; N tall: 3136 x 4096 x 1024 50.0 / 42.2, 8192 rows 100.4 / 99.9, 16384 182 / 189, 16384 x 3584 x 1024
//   170 / 184; other widths: 6272 x 1024 x 3712 88 / 76, 50176 rows 674 / 579, 50176 x 5120 x 768 653 / 608).
// Where there are half as many splits the sums of each are kept in halves (HALVES), and their error stays.
// A split holds whole steps of 64 rows, rounded up, so the last few may hold no rows: their sums are zeros.
struct LinearSplits {
    int splits, per;  // of `per` steps
    bool halves;
    LinearSplits(size_t rows, int N, int K) {
        const long tn = (N + kLinTile - 1) / kLinTile, tk = (K + kLinTile - 1) / kLinTile, tiles = tn * tk;
        const long steps = (long)((rows + kLinRows - 1) / kLinRows);
        auto deal = [&](long most) {
            long n = most < steps / 4 ? most : steps / 4;
            if (n >= 8) n = n / 8 * 8;
            return (int)(n < 1 ? 1 : n);
        };
        const bool alone = tiles > 256 || (tiles >= kLinAlone && (tk % 8 != 0 || steps <= (tn > tk ? kLinAloneTall : kLinAloneWide)));
        splits = alone ? 1 : deal(512 / tiles);
        const bool few = tiles <= kLinFew && deal(256 / tiles) < splits;
        if (few) splits = deal(256 / tiles);
        per = (int)((steps + splits - 1) / splits);
        halves = few || (alone && steps >= 8);
    }
};
// (one split writes the gradients themselves)
inline size_t linear_wgrad_scratch(size_t rows, int N, int K) {
    const int splits = LinearSplits(rows, N, K).splits;
    return splits == 1 ? 16 : (size_t)splits * ((size_t)N * K + N) * sizeof(float);
}

}  // namespace dwo
