// How the rows that a pointwise layer's parameter gradients sum over are split (linear_wgrad_kernel, dwo_linear.h).
#pragma once

#include <cstddef>

namespace dwo {

constexpr int kLinTile = 128, kLinRows = 64;  // outputs of a tile each way, rows of a step
constexpr long kLinFew = 4, kLinAlone = 224;  // tiles

// Splits of the rows, each with 256 rows where they are dealt evenly; a multiple of eight where there are as many (whole splits
// per XCD).  Two workgroups per CU (512), but
//   one where the outputs are at most four tiles and the rows enough for more: memory binds, and the partial sums, 64 KB per workgroup
//   both ways, are what can be saved (us with the sums, behind a pass over other memory, 512 / 256: 401408 x 512 x 128 146 / 135,
//   200704 x 96 x 384 54.5 / 49.6, 100352 x 256 x 256 35.8 / 30.6, 24576 x 512 x 128 19.2 / 17.8, 50176 x 192 x 96 16.2 / 15.8; where
//   both are as many splits the halves only cost, 16384 x 512 x 128 14.9 / 16.2, 1000 x 96 x 64 11.0 / 12.0; eight tiles, back to
//   back, 50176 x 256 x 512, 29.1 / 31.1);
//   no split where the tiles alone give each CU its workgroup (3136 x 4096 x 1024 53 / 44).
// Where there are half as many splits the sums of each are kept in halves (HALVES), and their error stays.
// A split holds whole steps of 64 rows, rounded up, so the last few may hold no rows: their sums are zeros.
struct LinearSplits {
    int splits, per;  // of `per` steps
    bool halves;
    LinearSplits(size_t rows, int N, int K) {
        const long tiles = (long)((N + kLinTile - 1) / kLinTile) * ((K + kLinTile - 1) / kLinTile);
        const long steps = (long)((rows + kLinRows - 1) / kLinRows);
        auto deal = [&](long most) {
            long n = most < steps / 4 ? most : steps / 4;
            if (n >= 8) n = n / 8 * 8;
            return (int)(n < 1 ? 1 : n);
        };
        const bool alone = tiles >= kLinAlone;
        splits = alone ? 1 : deal(512 / tiles);
        const bool few = tiles <= kLinFew && deal(256 / tiles) < splits;
        if (few) splits = deal(256 / tiles);
        per = (int)((steps + splits - 1) / splits);
        halves = few || (alone && steps >= 8);
    }
};
inline size_t linear_wgrad_scratch(size_t rows, int N, int K) {
    return (size_t)LinearSplits(rows, N, K).splits * ((size_t)N * K + N) * sizeof(float);
}

}  // namespace dwo
