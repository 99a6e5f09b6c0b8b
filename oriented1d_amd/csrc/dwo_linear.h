// Parameter gradients of a pointwise layer (the blocks' two linear layers, models/convnext.py:296-298,306-318)
// over 16-bit activations: dw[n][k] = sum over rows m of dy[m][n] * x[m][k], db[n] = sum of dy[m][n], on the
// matrix cores with fp32 accumulation.
//
// The sum runs over the pixels of a batch (3 136 to 802 816 rows) for outputs of 64 x 96 to 4096 x 1024, so
// most shapes have far fewer output tiles than the chip has CUs: the rows are split over workgroups, each
// writes fp32 partial sums and a second kernel adds them in a fixed order.  Both operands have the
// summed index as their slow one: tiles of 64 rows go to LDS as they lie in memory (rows padded by
// 32 bytes, so that the eight rows a half-wave reads lie on different banks) and come out
// transposed (ds_read_b64_tr_b16).  The order of the rows inside a product is the same for both
// operands, hence free: a read takes rows 4 g .. 4 g + 3 for its lane group g.  The bias gradient is a product with
// ones, in the workgroups of the first column of tiles.
#pragma once

#include "dwo_common.h"

namespace dwo {

typedef float mma_f4 __attribute__((ext_vector_type(4)));
typedef short mma_s4 __attribute__((ext_vector_type(4)));
typedef short mma_s8 __attribute__((ext_vector_type(8)));
typedef unsigned mma_u4 __attribute__((ext_vector_type(4)));

// D[4 g + r][j] += A[4 g + r][..] * B[..][j] for lane 16 g + j, over 32 products; a lane's eight values of
// A are row j, those of B column j
template <typename T>
struct Mma;
template <>
struct Mma<bf16_t> {
    static constexpr short kOne = 0x3f80;
    static __device__ __forceinline__ mma_f4 run(mma_s8 a, mma_s8 b, mma_f4 c) {
        typedef __bf16 v8 __attribute__((ext_vector_type(8)));
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0,
                                                       0);
    }
};
template <>
struct Mma<f16_t> {
    static constexpr short kOne = 0x3c00;
    static __device__ __forceinline__ mma_f4 run(mma_s8 a, mma_s8 b, mma_f4 c) {
        typedef _Float16 v8 __attribute__((ext_vector_type(8)));
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0,
                                                      0);
    }
};

constexpr int kLinThreads = 256, kLinTile = 128, kLinRows = 64;
constexpr int kLinPitch = kLinTile + 16;  // elements per LDS row
constexpr unsigned kLinNowhere = 0x80000000u;

// eight values of a column in rows [r, r + 4) and [r + 16, r + 20), r = 4 * (lane / 16)
__device__ __forceinline__ mma_s8 lin_column(const uint16_t *tile, int row, int col) {
    const int lane = threadIdx.x & 63, g = lane >> 4, i = lane & 15;
    const uint16_t *p = tile + (row + 4 * g + (i >> 2)) * kLinPitch + col + (i & 3) * 4;
    typedef __attribute__((address_space(3))) mma_s4 lds_s4;
    const mma_s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)p);
    const mma_s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(p + 16 * kLinPitch));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// rows [m, m + 64) of one operand's column tile, 16 bytes per load; zeros beyond its last row or column
struct LinSource {
    mma_u4 v[4];
    unsigned off[4];
    const char *at;
    long left;  // bytes from `at` to the end
    __device__ __forceinline__ void init(const void *p, long rows, long m0, int cols, int c0) {
        const unsigned pitch = (unsigned)cols * 2;
        at = reinterpret_cast<const char *>(p) + m0 * pitch;
        left = max(rows - m0, 0L) * (long)pitch;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int f = threadIdx.x + u * kLinThreads, c = c0 + f % 16 * 8;
            off[u] = c < cols ? (unsigned)(f / 16) * pitch + (unsigned)c * 2 : kLinNowhere;
        }
    }
    __device__ __forceinline__ void load(int cols) {
        const __amdgpu_buffer_rsrc_t r =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(at), 0, (unsigned)min(left, 0x7fffffffL), 0x00020000);
#pragma unroll
        for (int u = 0; u < 4; u++)
            v[u] = __builtin_bit_cast(mma_u4, __builtin_amdgcn_raw_buffer_load_b128(r, off[u], 0, 0));
        at += (long)kLinRows * cols * 2, left -= (long)kLinRows * cols * 2;
    }
    __device__ __forceinline__ void store(uint16_t *tile) const {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int f = threadIdx.x + u * kLinThreads;
            *reinterpret_cast<mma_u4 *>(tile + f / 16 * kLinPitch + f % 16 * 8) = v[u];
        }
    }
};

// part [split][N * K + N]
template <typename T>
__global__ __launch_bounds__(kLinThreads, 2) void linear_wgrad_kernel(const T *__restrict__ dy,
                                                                      const T *__restrict__ x,
                                                                      float *__restrict__ part, long rows, int N,
                                                                      int K, int splits, int steps, int with_bias) {
    __shared__ __attribute__((aligned(16))) uint16_t lds[2][kLinRows * kLinPitch];
    const int tk = (K + kLinTile - 1) / kLinTile, tiles = (N + kLinTile - 1) / kLinTile * tk;
    // the tiles of a split read the same rows: one XCD (workgroup ids modulo eight) takes whole splits
    int split, tile;
    if (splits % 8 == 0) {
        const int k = blockIdx.x / 8;
        split = k / tiles * 8 + blockIdx.x % 8, tile = k % tiles;
    } else {
        split = blockIdx.x / tiles, tile = blockIdx.x % tiles;
    }
    const int n0 = tile / tk * kLinTile, k0 = tile % tk * kLinTile;
    const long m0 = (long)split * steps * kLinRows;
    const long last = min(rows, m0 + (long)steps * kLinRows);
    const int wave = threadIdx.x >> 6, wn = wave / 2 * 64, wk = wave % 2 * 64;
    const bool bias = with_bias != 0 && k0 == 0 && wk == 0;
    mma_f4 acc[4][4], accb[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        accb[i] = mma_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = mma_f4{0.f, 0.f, 0.f, 0.f};
    }
    mma_s8 ones;
#pragma unroll
    for (int i = 0; i < 8; i++) ones[i] = Mma<T>::kOne;
    LinSource a, b;
    a.init(dy, rows, m0, N, n0);
    b.init(x, rows, m0, K, k0);
    a.load(N), b.load(K);
    for (long m = m0; m < last; m += kLinRows) {
        __syncthreads();
        a.store(lds[0]), b.store(lds[1]);
        __syncthreads();
        if (m + kLinRows < last) a.load(N), b.load(K);
#pragma unroll
        for (int r = 0; r < kLinRows; r += 32) {
            mma_s8 fa[4], fb[4];
#pragma unroll
            for (int i = 0; i < 4; i++) fa[i] = lin_column(lds[0], r, wn + 16 * i);
#pragma unroll
            for (int j = 0; j < 4; j++) fb[j] = lin_column(lds[1], r, wk + 16 * j);
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = Mma<T>::run(fa[i], fb[j], acc[i][j]);
            if (bias)
#pragma unroll
                for (int i = 0; i < 4; i++) accb[i] = Mma<T>::run(fa[i], ones, accb[i]);
        }
    }
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    float *out = part + (size_t)split * ((size_t)N * K + N);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int n = n0 + wn + 16 * i + 4 * g + r;
            if (n >= N) continue;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int k = k0 + wk + 16 * j + c;
                if (k < K) out[(size_t)n * K + k] = acc[i][j][r];
            }
            if (bias && c == 0) out[(size_t)N * K + n] = accb[i][r];
        }
}

// Sums over the splits, fixed order: eight threads share four outputs, each takes every eighth split.
template <typename TO>
__global__ __launch_bounds__(kLinThreads) void linear_reduce_kernel(const float *__restrict__ part,
                                                                    TO *__restrict__ dw, TO *__restrict__ db, int N,
                                                                    int K, int splits) {
    __shared__ mma_f4 red[kLinThreads];
    const size_t total = (size_t)N * K + N, first = (size_t)N * K;
    const size_t i = ((size_t)blockIdx.x * 32 + threadIdx.x % 32) * 4;
    mma_f4 s = mma_f4{0.f, 0.f, 0.f, 0.f};
    if (i < total)
        for (int p = threadIdx.x / 32; p < splits; p += 8)
            s += *reinterpret_cast<const mma_f4 *>(part + (size_t)p * total + i);
    red[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x >= 32 || i >= total || (i >= first && db == nullptr)) return;
#pragma unroll
    for (int p = 1; p < 8; p++) s += red[threadIdx.x + 32 * p];
    TO *out = i < first ? dw + i : db + (i - first);
#pragma unroll
    for (int e = 0; e < 4; e++) out[e] = from_float<TO>(s[e]);
}

// Splits of the rows: two workgroups per CU (512), each with at least 256 rows; a multiple of eight
// where there are as many (whole splits per XCD).
inline int linear_splits(size_t rows, int N, int K) {
    const long tiles = (long)((N + kLinTile - 1) / kLinTile) * ((K + kLinTile - 1) / kLinTile);
    const long steps = (long)((rows + kLinRows - 1) / kLinRows);
    long s = 512 / tiles;
    if (s > steps / 4) s = steps / 4;
    if (s >= 8) s = s / 8 * 8;
    return (int)(s < 1 ? 1 : s);
}
inline size_t linear_wgrad_scratch(size_t rows, int N, int K) {
    return (size_t)linear_splits(rows, N, K) * ((size_t)N * K + N) * sizeof(float);
}

template <typename T>
int launch_linear_wgrad(const void *dy, const void *x, float *part, size_t rows, int N, int K, int splits,
                        int with_bias, hipStream_t st) {
    const long steps = (long)((rows + kLinRows - 1) / kLinRows);
    const int per = (int)((steps + splits - 1) / splits);
    const unsigned tiles = (unsigned)((N + kLinTile - 1) / kLinTile) * ((K + kLinTile - 1) / kLinTile);
    linear_wgrad_kernel<T><<<dim3(tiles * (unsigned)splits), dim3(kLinThreads), 0, st>>>(
        (const T *)dy, (const T *)x, part, (long)rows, N, K, splits, per, with_bias);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}
template <typename TO>
int launch_linear_reduce(const float *part, void *dw, void *db, int N, int K, int splits, hipStream_t st) {
    const size_t vecs = ((size_t)N * K + N) / 4;
    linear_reduce_kernel<TO><<<dim3((unsigned)((vecs + 31) / 32)), dim3(kLinThreads), 0, st>>>(part, (TO *)dw,
                                                                                              (TO *)db, N, K, splits);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}

}  // namespace dwo
