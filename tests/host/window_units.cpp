// Host-side checks of how the window kernels' launches are cut (dwo_window_dispatch.h), over the shapes that
// they accept.  Prints one line per violation; exit status 0 when there is none.
#include <cstdio>
#include <cstring>

#include "dwo_window_dispatch.h"

using namespace dwo;

static int failures = 0;
#define EXPECT(cond, ...)                          \
    do {                                           \
        if (!(cond)) {                             \
            if (failures++ < 20) printf(__VA_ARGS__); \
        }                                          \
    } while (0)

// Byte offsets of a tile's window count from its corner, which may lie a halo above the image: those of the
// rows and columns inside the image must stay below the descriptor's 2^31 - 1 bytes.
static void check_offsets(int H, int W, int K, int es) {
    WinDims d;
    if (!win_dims(1, 8, H, W, K, es, d) || !d.tiled()) return;
    for (int halo = 0; halo <= K / 2; halo++)
        for (int a = 0; a < d.nth; a += d.nth > 3 && a == 1 ? d.nth - 2 : 1) {
            const long corner = (long)a * d.th - halo, q_lo = (K / 2 + 3) & ~3;
            for (long i = 0; i < d.th + 2 * halo; i++) {
                if (corner + i < 0 || corner + i >= H) continue;
                const long cols = cmin(W, d.tw + 2 * (int)q_lo + 4);
                const long end = (i * W + cols) * es;
                EXPECT(end <= 0x7fffffffL, "offset %ld: %d x %d, K %d, %d bytes, halo %d, tile row %d\n", end, H, W, K,
                       es, halo, a);
            }
        }
}

int main() {
    for (int K : {7, 13, 15, 27, 31})
        for (int es : {2, 4})
            for (int H : {1, 2, 4, 5, 16, 17, 48, 63, 64, 65, 100, 128, 200})
                for (int rows = 1; rows <= 130; rows++)
                    for (int extra : {-8, -1, 0, 1, 3, 8}) {
                        const double W = 2147483648.0 / es / rows + extra;
                        if (W * H * es < 2147483648.0) check_offsets(H, (int)W, K, es);
                    }
    for (int K : {7, 31}) {
        WinDims d;
        EXPECT(win_dims(1, 8, 64, 4000000, K, 4, d) && d.tiled(), "4 million columns are refused\n");
        EXPECT(win_dims(1, 8, 1, 20000000, K, 4, d) && d.tiled(), "a row of 20 million columns is refused\n");
    }
    // a workgroup per channel, in launches of fewer than 2^32 threads
    for (long C : {1L << 20, 8000000L, 8384511L, 8388607L, 8388608L, 20000000L}) {
        WinDims d;
        if (!win_dims(1, (int)C, 4, 4, 31, 2, d)) continue;
        const long groups = win_groups(d, 1024, 256, d.units);
        EXPECT((C * groups + 255) / 256 * 256 * kWinThreads < 1L << 32, "%ld channels in %ld groups\n", C, groups);
    }
    // thin planes of more than 64 rows or columns: small batches are taken, large ones left to the tile kernels
    for (int large : {0, 1}) {
        WinDims d;
        EXPECT(win_dims(large ? 32 : 2, 200, 4, 400, 31, 2, d) == !large, "4 x 400, batch %d\n", large);
        EXPECT(win_dims(large ? 64 : 2, 200, 8, 256, 31, 4, d) == !large, "8 x 256, batch %d\n", large);
        EXPECT(win_dims(large ? 32 : 2, 200, 400, 6, 31, 4, d) == !large, "400 x 6, batch %d\n", large);
        EXPECT(win_dims(large ? 64 : 2, 200, 400, 6, 7, 4, d) && win_dims(large ? 64 : 2, 200, 9, 400, 31, 2, d) &&
                   win_dims(large ? 64 : 2, 200, 4, 64, 31, 4, d),
               "a plane that is not thin, batch %d\n", large);
    }
    // few channels: the workgroups fill the chip's slots where there are units for them, in wgrad within
    // its partial sums
    for (int C : {1, 2, 3, 5, 8, 11, 12, 64, 96})
        for (int slots : {512, 768, 1024}) {
            WinDims d;
            const int N = 4096 / C;
            EXPECT(win_dims(N, C, 128, 128, 31, 4, d), "128 x 128 is refused\n");
            const int groups = win_groups(d, slots, 256, d.units);
            const int sums = win_groups(d, slots, 256, win_wgrad_groups(C, 31));
            EXPECT((C * groups >= 512 || C * groups * 4 >= slots * 3) && groups <= d.units,
                   "%d groups of %d channels in %d slots\n", groups, C, slots);
            EXPECT(sums >= 1 && sums <= kMaxWinGroups, "%d groups of sums\n", sums);
        }
    printf("%d violations\n", failures);
    return failures != 0;
}
