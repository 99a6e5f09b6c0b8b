// Parameter gradients of a pointwise layer with few inputs (the stem's first layer,
// models/convnext.py:143,177): dw[c][k] = sum over pixels of dy[p][c] * x[p][k], db[c] = sum of dy[p][c],
// for k < CIN <= 4.
//
// What bounds it is reading dy once (64 x 224 x 224 pixels of 64 channels in bf16: 411 MB).  As a
// matrix product it is C x CIN with millions of terms per element, a single tile for a library GEMM:
// 5060 us at that size, against 91 us here (4.5 TB/s, bf16).  A thread holds one 16-byte piece of a pixel's channels
// and walks pixels, so a wave reads whole lines; sums stay in fp32 registers, workgroups write partial
// sums and a second kernel adds them in a fixed order.
#pragma once

#include "dwo_common.h"

namespace dwo {

constexpr int kPwThreads = 256, kPwBlocks = 1024, kPwMaxCin = 4;

// sixteen bytes of activations as floats
template <typename T>
struct Piece {
    static constexpr int N = 16 / (int)sizeof(T);
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    u4 v;
    __device__ __forceinline__ void load(const T *p) { v = *reinterpret_cast<const u4 *>(p); }
    __device__ __forceinline__ float get(int i) const {
        if constexpr (sizeof(T) == 4) return __uint_as_float(v[i]);
        else return to_float(__builtin_bit_cast(T, (uint16_t)(v[i / 2] >> (16 * (i % 2)))));
    }
};

template <typename T, int CIN>
__global__ __launch_bounds__(kPwThreads) void pointwise_wgrad_kernel(const T *__restrict__ dy,
                                                                     const T *__restrict__ x,
                                                                     float *__restrict__ part, long rows,
                                                                     int C) {
    constexpr int N = Piece<T>::N, A = N * (CIN + 1), U = 4;
    __shared__ float red[kPwThreads * (A + 1)];
    const int lpp = C / N, ppb = kPwThreads / lpp;  // threads per pixel, pixels per workgroup
    const int slot = threadIdx.x / lpp, piece = threadIdx.x - slot * lpp;
    float acc[A];
#pragma unroll
    for (int i = 0; i < A; i++) acc[i] = 0.f;
    if (slot < ppb) {
        const long step = (long)gridDim.x * ppb;
        for (long p = (long)blockIdx.x * ppb + slot; p < rows; p += U * step) {
            Piece<T> g[U];
            T xv[U][CIN];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const long r = min(p + u * step, rows - 1);  // (repeats are dropped below)
                g[u].load(dy + r * C + piece * N);
#pragma unroll
                for (int k = 0; k < CIN; k++) xv[u][k] = x[r * CIN + k];
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (p + u * step >= rows) break;
#pragma unroll
                for (int i = 0; i < N; i++) {
                    const float v = g[u].get(i);
                    acc[i * (CIN + 1) + CIN] += v;
#pragma unroll
                    for (int k = 0; k < CIN; k++)
                        acc[i * (CIN + 1) + k] = __builtin_fmaf(v, to_float(xv[u][k]), acc[i * (CIN + 1) + k]);
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < A; i++) red[threadIdx.x * (A + 1) + i] = acc[i];
    __syncthreads();
    // cell (piece, i) is channel piece * N + i / (CIN + 1), term i % (CIN + 1)
    for (int cell = threadIdx.x; cell < lpp * A; cell += kPwThreads) {
        const int pc = cell / A, i = cell - pc * A;
        float t = 0.f;
        for (int s = 0; s < ppb; s++) t += red[(s * lpp + pc) * (A + 1) + i];
        part[(size_t)cell * gridDim.x + blockIdx.x] = t;
    }
}

// one wave per cell
__global__ void pointwise_reduce_kernel(const float *__restrict__ part, float *__restrict__ dw,
                                        float *__restrict__ db, int CIN, int blocks) {
    const int cell = blockIdx.x;
    float t = 0.f;
    for (int b = threadIdx.x; b < blocks; b += 64) t += part[(size_t)cell * blocks + b];
    t = wave_sum(t);
    if (threadIdx.x != 0) return;
    const int c = cell / (CIN + 1), k = cell - c * (CIN + 1);
    if (k < CIN) dw[(size_t)c * CIN + k] = t;
    else if (db != nullptr) db[c] = t;
}

// C a multiple of a 16-byte piece, at most kPwThreads pieces; dy 16-byte aligned
template <typename T, int CIN>
int launch_pointwise_wgrad(const void *dy, const void *x, float *dw, float *db, float *part, size_t rows, int C,
                           hipStream_t st) {
    const int ppb = kPwThreads / (C / Piece<T>::N);
    const size_t want = (rows + 4 * ppb - 1) / (4 * ppb);
    const int blocks = (int)(want < (size_t)kPwBlocks ? want : (size_t)kPwBlocks);
    pointwise_wgrad_kernel<T, CIN><<<dim3(blocks), dim3(kPwThreads), 0, st>>>((const T *)dy, (const T *)x, part,
                                                                              (long)rows, C);
    pointwise_reduce_kernel<<<dim3(C * (CIN + 1)), dim3(64), 0, st>>>(part, dw, db, CIN, blocks);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}

}  // namespace dwo
