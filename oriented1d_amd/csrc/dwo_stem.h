// The stem's first two layers at inference in bf16 (3 -> C pointwise, oriented convolution of stride 2, models/convnext.py:177-178)
// as matrix products over the image:
//   y[c][p] = b[c] + sum over taps s, inputs i < 4 of (w[c][s] * pw[c][i]) * x4[i][p + tap s]
// with x4 the three inputs and an indicator of the image (times the pointwise bias).  Eight neighbouring channels share an orientation,
// hence the pixels that a tap reads: 16 pixels x 8 channels are 31 x 4 products deep, four matrix instructions.  The other eight rows of
// these hold the low halves of the weights: fp32 weights as two bf16 (error 2^-17), where the separate layers
// round the 3 -> C result to bf16 (2^-9).
//
// A workgroup stages its window of x4 once for all channels (8 bytes per pixel, even and odd columns apart: 16 output
// pixels read 128 neighbouring bytes); a wave takes 16 channels x 16 pixels at a time and keeps its weights for all tiles.  Busiest are
// the vector instructions (54 % of the time at 128 x 224 x 224 and K = 31 by counters: staging, each input six times, and
// addresses), then LDS with eight bytes per lane and tap (36 %, bank conflicts included) and the matrix cores (18 %).  Against tap
// by tap with the projection repeated for each group (us, K = 31 unless noted): 128 x 224 x 224 520 / 114, 4 x 512 x 512
// 92 / 33, 64 x 224 x 224 at K = 15 170 / 57.  Error against 64 bits 1.64e-3 to 1.70e-3 over seven shapes with K = 7 to 31, which is the result's own
// rounding (tap by tap 1.75e-3 to 2.34e-3).  bf16 only: in fp16 the low halves of weights below 1/4 leave the normal range.
#pragma once

#include "dwo_linear.h"

namespace dwo {

constexpr int kStemThreads = 512, kStemWaves = kStemThreads / 64, kStemCin = 3;
constexpr int kStemParts = 4, kStemC = 16 * kStemParts;  // channels per workgroup, 16 of them in every fourth wave
constexpr int kStemWindow = 76 * 1024;                   // bytes of LDS for the window: two workgroups per CU

struct StemTiles {
    int th, tw16, nth, ntw;  // rows, columns / 16, tiles
    int rows, hc;            // window: rows, columns of one parity
    int tiles;               // in all
    unsigned magic;          // division by 2 hc
};
inline StemTiles stem_tiles(int N, int P, int Q, int R) {
    StemTiles t;
    const int sets = (Q + 15) / 16;
    t.ntw = (sets + 3) / 4, t.tw16 = (sets + t.ntw - 1) / t.ntw;
    t.hc = 16 * t.tw16 + R;
    const int most = (kStemWindow / (16 * t.hc) + 1 - 2 * R) / 2;
    t.nth = (P + most - 1) / most;
    // small batches: lower tiles, though the window's halo is staged again, until every CU has one
    while ((long)N * t.nth * t.ntw < 256 && (P + t.nth - 1) / t.nth > 2) t.nth *= 2;
    t.th = (P + t.nth - 1) / t.nth, t.nth = (P + t.th - 1) / t.th;
    t.rows = 2 * t.th - 1 + 2 * R;
    t.magic = (unsigned)(((1ULL << 32) + 2 * t.hc - 1) / (2 * t.hc));
    return t;
}

// NT: K <= 8 NT
template <int NT>
__global__ __launch_bounds__(kStemThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void stem_kernel(const bf16_t *__restrict__ x, const float *__restrict__ pw_w,
                                                            const float *__restrict__ pw_b, const float *__restrict__ wt,
                                                            const float *__restrict__ bias,
                                                            const int8_t *__restrict__ dhdw, bf16_t *__restrict__ y,
                                                            ConvDims d, StemTiles t) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_stem[];
    mma_u2 *win = reinterpret_cast<mma_u2 *>(lds_stem);  // [row][parity][hc]
    const int K = d.K, R = K / 2, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int g = lane >> 4, j = lane & 15;
    const int cw = blockIdx.y * kStemC, c0 = cw + wave % kStemParts * 16, rs = 2 * t.hc;
    // taps: the eight channels of a group agree, no tap leaves the window; weights: their products are finite
    bool beyond = false;
    for (int f = threadIdx.x; f < kStemC * K; f += kStemThreads) {
        const int c = cw + f / K, s = f % K;
        const int8_t *a = dhdw + ((size_t)c * K + s) * 2, *b = dhdw + ((size_t)(c & ~7) * K + s) * 2;
        beyond |= a[0] != b[0] || a[1] != b[1] || a[0] > R || a[0] < -R || a[1] > R || a[1] < -R;
        const float w = wt[(size_t)c * K + s];
        float most = pw_b != nullptr ? __builtin_fabsf(w * pw_b[c]) : 0.f;
        for (int i = 0; i < kStemCin; i++) most += __builtin_fabsf(w * pw_w[(size_t)c * kStemCin + i]);
        beyond |= !(most < 1e38f);
    }
    // weights: row j % 8 is the channel, rows 8 .. the low halves (what is left of a value above its upper 16 bits,
    // rounded: 2^-17); this lane's taps are 8 k + 2 g and the next
    mma_s8 fw[2][NT];
    unsigned off[2][NT];  // places of the two taps in the window, 16 bits each
    float cb[4];
#pragma unroll
    for (int a = 0; a < 2; a++) {
        const int c = c0 + 8 * a + j % 8;
        float pw[4];
#pragma unroll
        for (int i = 0; i < kStemCin; i++) pw[i] = pw_w[(size_t)c * kStemCin + i];
        pw[3] = pw_b != nullptr ? pw_b[c] : 0.f;
#pragma unroll
        for (int k = 0; k < NT; k++) {
            off[a][k] = 0;
            mma_u4 words;
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int s = 8 * k + 2 * g + e, ss = s < K ? s : 0;
                const float w = wt[(size_t)c * K + ss] * (s < K ? 1.f : 0.f);
                float part[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float v = w * pw[i], hi = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, v) & 0xffff0000u);
                    part[i] = j < 8 ? hi : v - hi;
                }
                words[2 * e] = lin_pack<bf16_t>(part[0], part[1]), words[2 * e + 1] = lin_pack<bf16_t>(part[2], part[3]);
                const int8_t *tap = dhdw + ((size_t)(c0 + 8 * a) * K + ss) * 2;
                const int col = tap[1] + R;
                off[a][k] |= (unsigned)((tap[0] + R) * rs + (col & 1) * t.hc + (col >> 1) + j) << (16 * e);
            }
            fw[a][k] = __builtin_bit_cast(mma_s8, words);
            __builtin_amdgcn_sched_barrier(0);  // (else all loads are in registers at once)
        }
    }
    // after the halves have met a lane has channels 4 g .. 4 g + 3 of 16
#pragma unroll
    for (int r = 0; r < 4; r++) cb[r] = bias != nullptr ? bias[c0 + 4 * g + r] : 0.f;
    for (int tile = blockIdx.x; tile < t.tiles; tile += gridDim.x) {
        const int per = t.nth * t.ntw, n = tile / per, k0 = tile - n * per;
        const int p0 = k0 / t.ntw * t.th, q0 = k0 % t.ntw * t.tw16 * 16;
        const int vh = min(t.th, d.P - p0), vw = min(t.tw16 * 16, d.Q - q0);
        const bf16_t *img = x + (size_t)n * d.H * d.W * kStemCin;
        // the window: rows 2 p0 - R .., columns 2 q0 - R ..
        bool odd = beyond;  // something that the products below do not cover
        const int total = t.rows * rs;
        __syncthreads();  // the window's last readers are done
        constexpr int U = 4;
        for (int f0 = threadIdx.x; f0 < total; f0 += U * kStemThreads) {
            uint16_t v[U][kStemCin];
            bool in[U];
            int at[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int f = f0 + u * kStemThreads, r = (int)__umulhi((unsigned)f, t.magic), q = f - r * rs;
                const int h = 2 * p0 - R + r, w = 2 * q0 - R + q;
                at[u] = r * rs + (q & 1) * t.hc + (q >> 1);
                in[u] = f < total && (unsigned)h < (unsigned)d.H && (unsigned)w < (unsigned)d.W;
                const size_t o = in[u] ? ((size_t)h * d.W + w) * kStemCin : 0;
#pragma unroll
                for (int i = 0; i < kStemCin; i++) v[u][i] = __builtin_bit_cast(uint16_t, img[o + i]);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
#pragma unroll
                for (int i = 0; i < kStemCin; i++) odd |= in[u] && (v[u][i] & 0x7f80) == 0x7f80;  // infinities and NaN
                const mma_u2 px = mma_u2{(unsigned)v[u][0] | (unsigned)v[u][1] << 16, (unsigned)v[u][2] | 0x3f800000u};
                if (f0 + u * kStemThreads < total) win[at[u]] = in[u] ? px : mma_u2{0u, 0u};
            }
        }
        if (__syncthreads_or(odd)) {  // tap by tap, the pointwise result rounded as by itself
            for (int f = threadIdx.x; f < vh * vw * kStemC; f += kStemThreads) {
                const int c = cw + f % kStemC, o = f / kStemC, p = p0 + o / vw, q = q0 + o % vw;
                float a = bias != nullptr ? bias[c] : 0.f;
                for (int s = 0; s < K; s++) {
                    const int h = 2 * p + dhdw[((size_t)c * K + s) * 2], w = 2 * q + dhdw[((size_t)c * K + s) * 2 + 1];
                    if ((unsigned)h >= (unsigned)d.H || (unsigned)w >= (unsigned)d.W) continue;
                    float v = pw_b != nullptr ? pw_b[c] : 0.f;
                    for (int i = 0; i < kStemCin; i++)
                        v = __builtin_fmaf(to_float(img[((size_t)h * d.W + w) * kStemCin + i]), pw_w[(size_t)c * kStemCin + i], v);
                    a = __builtin_fmaf(to_float(from_float<bf16_t>(v)), wt[(size_t)c * K + s], a);
                }
                y[(((size_t)n * d.P + p) * d.Q + q) * d.C + c] = from_float<bf16_t>(a);
            }
            continue;
        }
        const int sets = vh * t.tw16;
        for (int set = wave / kStemParts; set < sets; set += kStemWaves / kStemParts) {
            const int row = set / t.tw16, col = (set - row * t.tw16) * 16;
            if (col >= vw) continue;  // (uniform)
            const mma_u2 *base = win + 2 * row * rs + col;
            mma_f4 acc[2];
#pragma unroll
            for (int a = 0; a < 2; a++) {
                acc[a] = mma_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < NT; k++) {
                    const mma_u2 lo = base[off[a][k] & 0xffff], hi = base[off[a][k] >> 16];
                    acc[a] = Mma<bf16_t>::run(fw[a][k], __builtin_bit_cast(mma_s8, mma_u4{lo[0], lo[1], hi[0], hi[1]}), acc[a]);
                }
            }
            // lanes 0 .. 31 take the first group, 32 .. 63 the second: high plus low halves
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                // (scalars: a bit cast of a vector's element reads the vector's first)
                const float first = acc[0][r], second = acc[1][r];
                const auto s = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, first),
                                                                __builtin_bit_cast(unsigned, second), false, false);
                const unsigned hi = s[0], lo = s[1];
                v[r] = __builtin_bit_cast(float, hi) + __builtin_bit_cast(float, lo) + cb[r];
            }
            if (col + j < vw)
                *reinterpret_cast<mma_u2 *>(y + (((size_t)n * d.P + p0 + row) * d.Q + q0 + col + j) * d.C + c0 + 4 * g) =
                    mma_u2{lin_pack<bf16_t>(v[0], v[1]), lin_pack<bf16_t>(v[2], v[3])};
        }
    }
}

}  // namespace dwo
