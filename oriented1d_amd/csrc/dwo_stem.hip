// The stem's projecting convolution on the matrix cores.
#include "dwo_stem.h"

namespace dwo {

// -100 where the shape is not covered (another path takes it)
int launch_stem(const bf16_t *x, const float *pw_w, const float *pw_b, const float *w, const float *bias, const void *taps,
                bf16_t *y, const ConvDims &d, hipStream_t st) {
    if (d.C % kStemC != 0 && d.N != 0) return -100;
    if (d.K > 32 || d.stride != 2) return -100;
    StemTiles t = stem_tiles(d.N, d.P, d.Q, d.K / 2);
    const long tiles = (long)d.N * t.nth * t.ntw;
    const size_t lds = (size_t)t.rows * t.hc * 16;
    if (tiles >= 1L << 31 || d.C / kStemC > 65535 || lds > kStemWindow) return -100;
    // two workgroups per CU keep their weights for all their tiles
    t.tiles = (int)tiles;
    const dim3 grid((unsigned)(tiles < 512 ? tiles : 512), d.C / kStemC), block(kStemThreads);
    auto launch = [&](auto kernel, int *cache) {
        per_device_once(cache, [&] {
            allow_large_lds(kernel, kStemWindow);
            return 1;
        });
        if (d.N == 0) return 0;  // set-up only
        kernel<<<grid, block, lds, st>>>(x, pw_w, pw_b, w, bias, taps_dhdw(taps), y, d, t);
        const hipError_t e = hipGetLastError();
        return e == hipSuccess ? 0 : (int)e;
    };
    static int cache[3][kMaxDevices];
    if (d.K <= 8) return launch(stem_kernel<1>, cache[0]);
    if (d.K <= 16) return launch(stem_kernel<2>, cache[1]);
    return launch(stem_kernel<4>, cache[2]);
}

}  // namespace dwo
