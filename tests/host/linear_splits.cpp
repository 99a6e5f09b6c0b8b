// Host-side check of how the rows of the pointwise weight gradients are split (dwo_linear_splits.h): all rows are covered, launches
// stay in range, no chain of fp32 sums is longer than with two workgroups per CU (but for one step where a half is an odd number of
// them, and 5 % for three tiles, whose 168 splits become 80: 401408 x 384 x 96 is 3.18e-7 from 64 bits, with 168 3.15e-7), and sums are
// kept in halves only where there are fewer splits than that.  Prints one line per violation; exit status 0 when there is none.
#include <algorithm>
#include <cstdio>

#include "dwo_linear_splits.h"

using namespace dwo;

static int failures = 0;
#define EXPECT(cond, what)                                                                             \
    do {                                                                                               \
        if (!(cond) && failures++ < 20) printf("%s: %zu rows, %d x %d, %d splits\n", what, rows, N, K, s.splits); \
    } while (0)

int main() {
    const size_t few[] = {1, 63, 64, 65, 255, 256, 257, 448, 449, 512, 513, 960, 1000, 1024, 1025, 3136, 3456, 3457, 6272, 8192, 8193,
                          12544, 16384, 16385, 16640, 21760, 22016, 32768, 33024, 50176, 65536, 66000, 131072, 200704, 401408,
                          802816, (size_t)1 << 31};
    for (size_t rows : few)
        for (int N : {8, 64, 96, 128, 136, 192, 256, 384, 512, 768, 1024, 1536, 1792, 2048, 3072, 3584, 4096, 65536})
            for (int K : {8, 64, 96, 128, 192, 256, 384, 512, 1024, 1792, 2048, 3712, 4096, 65536}) {
                const LinearSplits s(rows, N, K);
                const long tiles = (long)((N + 127) / 128) * ((K + 127) / 128), steps = (long)((rows + 63) / 64);
                long two = std::min(512 / tiles, steps / 4);  // two workgroups per CU
                if (two >= 8) two = two / 8 * 8;
                two = std::max(two, 1L);
                EXPECT(s.splits >= 1 && (long)s.splits * s.per >= steps, "rows are left out");
                EXPECT((long)s.splits * tiles * 256 < 1L << 32, "a launch of too many threads");
                EXPECT(s.splits < 8 || s.splits % 8 == 0, "splits that no XCD takes whole");
                const long chain = s.halves ? std::max((s.per + 1) / 4 * 2, s.per - (s.per + 1) / 4 * 2) : s.per;
                const long before = (steps + two - 1) / two;
                EXPECT(chain <= before + 1 + (tiles == 3 ? before / 20 : 0), "a longer chain of sums");
                EXPECT(tiles > 256 || (K + 127) / 128 % 8 != 0 || s.splits > 1 || steps <= 128, "many rows in one workgroup per tile");
                EXPECT(!s.halves || s.splits < two || tiles > 256, "halves without fewer splits");
            }
    return failures != 0;
}
