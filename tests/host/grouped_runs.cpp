// Host-side check of the grouped kernels' tiles in runs (dwo_grouped_dispatch.h).  Without arguments: every unit of a launch has a tile
// of its own, and an XCD's units are neighbours in bands of two tile columns; one line per violation, exit status 0 when there is
// none.  With N C H W K: the tiles of the stride-2 kernels for that layer, as lines "pass bytes run rows columns".
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "dwo_grouped.h"

using namespace dwo;

template <int K>
static void print_tiles(ConvDims d) {
    for (int es : {2, 4}) {
        const int ngroups = d.C / grp_channels(es);
        const GrpTiles conv = grp_tiles<ConvSet<K, 2>>(d.P, d.Q, (long)d.N * ngroups);
        const GrpTiles quad = grp_tiles<QuadSet<K>>(d.P, d.Q, (long)d.N * ngroups);
        const GrpTiles sums = grp_tiles<ConvSet<K, 2>>(d.P, d.Q, kGrpSlots);
        printf("fprop %d %d %d %d\n", es, grp_run(conv, d, es, GRP_FPROP), conv.nth, conv.ntw);
        printf("dgrad %d %d %d %d\n", es, grp_run(quad, d, es, GRP_DGRAD), quad.nth, quad.ntw);
        printf("wgrad %d %d %d %d\n", es, grp_run(sums, d, es, GRP_WGRAD), sums.nth, sums.ntw);
    }
}

int main(int argc, char **argv) {
    if (argc == 6) {
        ConvDims d{};
        d.N = atoi(argv[1]), d.C = atoi(argv[2]), d.H = atoi(argv[3]), d.W = atoi(argv[4]), d.K = atoi(argv[5]);
        d.stride = 2, d.P = (d.H + 1) / 2, d.Q = (d.W + 1) / 2;
        switch (d.K) {
#define DWO_CASE(K) case K: print_tiles<K>(d); return 0;
            DWO_GROUPED_KS(DWO_CASE)
#undef DWO_CASE
        }
        return 1;
    }
    int failures = 0;
    for (int N : {1, 2, 3, 7, 8, 13})
        for (int nth = 1; nth < 10; nth++)
            for (int ntw = 1; ntw < 12; ntw++) {
                GrpTiles t{};
                const int units = N * nth * ntw;
                t.nth = nth, t.ntw = ntw, t.run = units / 8;
                std::vector<int> seen(units, 0);
                int before = -1;
                for (int x = 0; x < 8; x++)
                    for (int i = 0; i < t.run; i++) {
                        int n, row, col;
                        grp_run_tile(t, 8 * i + x, n, row, col);
                        // (the places in order: image, band, row, column)
                        const int wide = col / 2 * 2 + 1 < ntw ? 2 : 1, place = n * nth * ntw + col / 2 * 2 * nth + row * wide + col % 2;
                        if (place != before + 1) printf("%d x %d x %d: unit %d\n", N, nth, ntw, 8 * i + x), failures++;
                        before = place;
                    }
                for (int u = 0; u < units; u++) {
                    int n, row, col;
                    grp_run_tile(t, u, n, row, col);
                    if (n < 0 || n >= N || row < 0 || row >= nth || col < 0 || col >= ntw || seen[(n * nth + row) * ntw + col]++)
                        printf("%d x %d x %d: unit %d at %d, %d, %d\n", N, nth, ntw, u, n, row, col), failures++;
                }
            }
    return failures != 0;
}
