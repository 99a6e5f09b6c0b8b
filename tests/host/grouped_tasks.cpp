// Host-side check of the grouped kernels' task map (dwo_grouped_dispatch.h): every (unit, channel group) once, the
// eight XCDs within one task of each other.  Prints one line per violation; exit status 0 when there is none.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "dwo_grouped_dispatch.h"

using namespace dwo;

int main() {
    int failures = 0;
    for (int units : {1, 2, 3, 7, 8, 9, 64, 257})
        for (int ngroups : {1, 2, 3, 8, 12, 24, 100, 512}) {
            std::vector<int> seen((size_t)units * ngroups, 0), per_xcd(8, 0);
            const unsigned grid = (unsigned)grp_grid(units, ngroups);
            for (unsigned b = 0; b < grid; b++) {
                int unit = 0, group = 0;
                if (!grp_task(b, units, ngroups, unit, group)) continue;
                if (unit < 0 || unit >= units || group < 0 || group >= ngroups) {
                    printf("block %u of %u: unit %d, group %d\n", b, grid, unit, group), failures++;
                    continue;
                }
                seen[(size_t)unit * ngroups + group]++, per_xcd[b % 8]++;
            }
            const bool once = std::all_of(seen.begin(), seen.end(), [](int n) { return n == 1; });
            const int most = *std::max_element(per_xcd.begin(), per_xcd.end());
            // (the last runs are short)
            if (!once || most != (units * ngroups + 7) / 8)
                printf("%d units, %d groups: %s, %d tasks on one XCD\n", units, ngroups, once ? "once" : "not once", most), failures++;
        }
    // launches of fewer than 2^32 threads
    for (long units : {1L, 7L, 8L, 9L, 100L, 16384L, 131071L, 131072L, 131073L, 1L << 27})
        for (int ngroups : {1, 8, 64, 512, 1 << 20, (1 << 20) + 1}) {
            const long grid = grp_grid(units, ngroups);
            const bool fits = grid * 512 <= 0xffffffffL;
            if (grid < units * ngroups || grp_grid_fits(grid) != fits)
                printf("%ld units, %d groups: %ld workgroups\n", units, ngroups, grid), failures++;
        }
    // wgrad's groups: each has a tile, and all of them fit a launch
    for (int N : {1, 3, 64, 300})
        for (int C : {16, 64, 272, 2048, 65536})
            for (int P : {1, 2, 5, 17, 40, 112})
                for (int Q : {1, 9, 33, 128})
                    for (int es : {2, 4}) {
                        ConvDims d{};
                        d.N = N, d.C = C, d.P = P, d.Q = Q;
                        const long units = (long)N * ((P + 15) / 16) * ((Q + 31) / 32);
                        const int G = grp_wgrad_groups(d, es), ngroups = C / grp_channels(es);
                        if (G < 1 || G > units || (G > 8 && (long)G * ngroups > 1024 + 8L * ngroups) ||
                            !grp_grid_fits(grp_grid(G, ngroups)))
                            printf("%d groups of %d x %d x %d x %d\n", G, N, C, P, Q), failures++;
                    }
    return failures != 0;
}
