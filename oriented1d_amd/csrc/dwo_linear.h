// Parameter gradients of a pointwise layer (the blocks' two linear layers, models/convnext.py:296-298,306-318)
// over 16-bit activations: dw[n][k] = sum over rows m of dy[m][n] * x[m][k], db[n] = sum of dy[m][n], on the
// matrix cores with fp32 accumulation.
//
// The sum runs over the pixels of a batch (3 136 to 802 816 rows) for outputs of 64 x 96 to 4096 x 1024, so
// most shapes have far fewer output tiles than the chip has CUs: the rows are split over workgroups, each
// writes fp32 partial sums and a second kernel adds them in a fixed order.  Both operands have the
// summed index as their slow one: stages of 32 rows go to LDS as they lie in memory (the 32-byte units of a row permuted by the row,
// so that the eight rows a half-wave reads lie on different banks) and come out
// transposed (ds_read_b64_tr_b16).  The order of the rows inside a product is the same for both
// operands, hence free: a read takes rows 4 g .. 4 g + 3 for its lane group g.  The bias gradient is a product with
// ones, in the workgroups of the first column of tiles.
//
// What binds it is the chain of a step, not a unit: by counters matrix cores 25 %, vector instructions 12 %, LDS 12 %, no conflicts, waves
// waiting 29 % of their cycles (12544 x 512 x 2048, 64 MB read; at 131072 x 384 x 96 129 MB in 31 us, 4.6 TB/s).  So the loads go straight to
// LDS, three stages ahead, with one barrier per stage, and where the partial sums weigh more there are fewer of them
// (LinearSplits).  us with the reduction, staging through registers with two barriers per 64 rows / so: 12544 x 512 x 2048 46.3 / 39.6,
// 3136 x 4096 x 1024 56 / 42.5, 8192 x 384 x 1536 30.4 / 25.0, 131072 x 384 x 96 37.7 / 33.9, 200704 x 512 x 128 62 / 56; slower where few splits
// or a K of one and a half tiles let workgroups that share lines drift apart, with many rows (75264 x 3072 x 768 581 / 602, 100352 x 768 x 192 73 / 79:
// 12544 x 3072 x 768 reads 582 MB, its inputs six times).  Tried: three stages and three workgroups per CU (its partial sums cost more
// than it gives, 200704 x 512 x 128 78).  Larger tiles would read less per product, but fewer tiles mean more splits.
#pragma once

#include "dwo_common.h"
#include "dwo_linear_splits.h"

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

constexpr int kLinThreads = 256;
constexpr int kLinStage = 32;  // rows that travel together
constexpr unsigned kLinNowhere = 0x80000000u;

// Place of a fragment in a stage: columns [16 unit, 16 unit + 16) of rows 4 g + i / 4 and 16 rows on, as the transposing read
// takes them (lane 16 g + i; rows of 256 bytes, their 32-byte units permuted by the row)
__device__ __forceinline__ int lin_column_at(int unit) {
    const int lane = threadIdx.x & 63, i = lane & 15, row = 4 * (lane >> 4) + (i >> 2);
    return row * kLinTile + (unit ^ (row & 7)) * 16 + (i & 3) * 4;
}
// eight values of a column in rows [r, r + 4) and [r + 16, r + 20), r = 4 * (lane / 16)
__device__ __forceinline__ mma_s8 lin_column(const uint16_t *stage, int at) {
    typedef __attribute__((address_space(3))) mma_s4 lds_s4;
    const mma_s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(stage + at));
    const mma_s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(stage + at + 16 * kLinTile));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// 32 rows of one operand's column tile straight to LDS, 16 bytes per lane and load; zeros beyond its last row or column
struct LinSource {
    unsigned off[2];
    const char *at;
    long left;  // bytes from `at` to the end
    __device__ __forceinline__ void init(const void *p, long rows, long m0, int cols, int c0) {
        const unsigned pitch = (unsigned)cols * 2;
        at = reinterpret_cast<const char *>(p) + m0 * pitch;
        left = max(rows - m0, 0L) * (long)pitch;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int f = threadIdx.x + u * kLinThreads, row = f / 16, q = f % 16;
            const int c = c0 + ((q >> 1 ^ (row & 7)) * 2 + (q & 1)) * 8;
            off[u] = c < cols ? (unsigned)row * pitch + (unsigned)c * 2 : kLinNowhere;
        }
    }
    __device__ __forceinline__ void load(uint16_t *stage, int cols) {
        typedef __attribute__((address_space(3))) void lds_void;
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<char *>(at), 0, (unsigned)max(0L, min(left, 0x7fffffffL)), 0x00020000);
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
        for (int u = 0; u < 2; u++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)(stage + (u * kLinThreads + wave * 64) * 8), 16, off[u], 0,
                                                     0, 0);
#endif
        at += (long)kLinStage * cols * 2, left -= (long)kLinStage * cols * 2;
    }
};

// dw [split][stride] and db [split][stride]: partial sums, or with one split the gradients themselves (db may be null).
// HALVES: the sums of the first half of a split's rows wait in registers of their own, so that no chain is longer than where
// twice as many splits share the rows, but for 64 rows where these are an odd number of steps (error against 64 bits at 200704 x
// 512 x 128 with 256 workgroups 3.5e-7, like this 2.5e-7, with 512 2.5e-7; 512 / 960 rows x 4096 x 1024 1.25e-7 / 1.78e-7 in
// one chain, 9.0e-8 / 1.24e-7 like this and with two splits).
template <typename T, typename TO, bool HALVES>
__global__ __launch_bounds__(kLinThreads, 2) void linear_wgrad_kernel(const T *__restrict__ dy,
                                                                      const T *__restrict__ x, TO *__restrict__ dw,
                                                                      TO *__restrict__ db, size_t stride, long rows,
                                                                      int N, int K, int splits, int steps) {
    __shared__ __attribute__((aligned(16))) uint16_t sa0[kLinStage * kLinTile];
    __shared__ __attribute__((aligned(16))) uint16_t sb0[kLinStage * kLinTile];
    __shared__ __attribute__((aligned(16))) uint16_t sa1[kLinStage * kLinTile];
    __shared__ __attribute__((aligned(16))) uint16_t sb1[kLinStage * kLinTile];
    __shared__ __attribute__((aligned(16))) uint16_t sa2[kLinStage * kLinTile];
    __shared__ __attribute__((aligned(16))) uint16_t sb2[kLinStage * kLinTile];
    __shared__ __attribute__((aligned(16))) uint16_t sa3[kLinStage * kLinTile];
    __shared__ __attribute__((aligned(16))) uint16_t sb3[kLinStage * kLinTile];
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
    const bool bias = db != nullptr && k0 == 0 && wk == 0;
    mma_f4 acc[4][4], accb[4];
    int ca[4], cb[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        accb[i] = mma_f4{0.f, 0.f, 0.f, 0.f};
        ca[i] = lin_column_at(wn / 16 + i), cb[i] = lin_column_at(wk / 16 + i);
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = mma_f4{0.f, 0.f, 0.f, 0.f};
    }
    mma_s8 ones;
#pragma unroll
    for (int i = 0; i < 8; i++) ones[i] = Mma<T>::kOne;
    LinSource a, b;
    a.init(dy, min(rows, max(last, m0)), m0, N, n0);
    b.init(x, min(rows, max(last, m0)), m0, K, k0);
    // a stage is multiplied while the next three travel (loads beyond the split's last row read nowhere)
    auto stage = [&](uint16_t *sa, uint16_t *sb, uint16_t *na, uint16_t *nb) {
        // vmcnt(8) lgkmcnt(0): this wave's part of the stage is there, and what it read of the one before ..
        __builtin_amdgcn_s_waitcnt(0x0078);
        asm volatile("s_barrier" ::: "memory");  // .. and the other waves'; nobody reads the one before any more
        a.load(na, N), b.load(nb, K);
        __builtin_amdgcn_sched_barrier(0);
        mma_s8 fa[4], fb[4];
#pragma unroll
        for (int i = 0; i < 4; i++) fa[i] = lin_column(sa, ca[i]);
#pragma unroll
        for (int j = 0; j < 4; j++) fb[j] = lin_column(sb, cb[j]);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[i][j] = Mma<T>::run(fa[i], fb[j], acc[i][j]);
        if (bias)
#pragma unroll
            for (int i = 0; i < 4; i++) accb[i] = Mma<T>::run(fa[i], ones, accb[i]);
    };
    a.load(sa0, N), b.load(sb0, K);
    a.load(sa1, N), b.load(sb1, K);
    a.load(sa2, N), b.load(sb2, K);
    const int pairs = (int)((max(last - m0, 0L) + 2 * kLinStage - 1) / (2 * kLinStage));
    auto run = [&](int n) {
        for (int p = 0; p < n; p++) {
            stage(sa0, sb0, sa3, sb3), stage(sa1, sb1, sa0, sb0);
            stage(sa2, sb2, sa1, sb1), stage(sa3, sb3, sa2, sb2);
        }
    };
    mma_f4 half[4][4], halfb[4];
    if constexpr (HALVES) {
        run((pairs + 1) / 4);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            halfb[i] = accb[i], accb[i] = mma_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 4; j++) half[i][j] = acc[i][j], acc[i][j] = mma_f4{0.f, 0.f, 0.f, 0.f};
        }
        run(pairs / 2 - (pairs + 1) / 4);
    } else {
        run(pairs / 2);
    }
    if (pairs % 2 != 0) stage(sa0, sb0, sa3, sb3), stage(sa1, sb1, sa0, sb0);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // (nothing may arrive in LDS behind the workgroup's end)
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    TO *out = dw + (size_t)split * stride;
    if constexpr (HALVES)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            accb[i] += halfb[i];
#pragma unroll
            for (int j = 0; j < 4; j++) acc[i][j] += half[i][j];
        }
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int n = n0 + wn + 16 * i + 4 * g + r;
            if (n >= N) continue;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int k = k0 + wk + 16 * j + c;
                if (k < K) out[(size_t)n * K + k] = from_float<TO>(acc[i][j][r]);
            }
            if (bias && c == 0) db[(size_t)split * stride + n] = from_float<TO>(accb[i][r]);
        }
}

// Sums over the splits, fixed order: SHARE threads share four outputs, each takes every SHARE-th split.
template <typename TO, int SHARE>
__global__ __launch_bounds__(kLinThreads) void linear_reduce_kernel(const float *__restrict__ part,
                                                                    TO *__restrict__ dw, TO *__restrict__ db, int N,
                                                                    int K, int splits) {
    constexpr int VECS = kLinThreads / SHARE;
    __shared__ mma_f4 red[SHARE > 1 ? kLinThreads : 1];
    const size_t total = (size_t)N * K + N, first = (size_t)N * K;
    const size_t i = ((size_t)blockIdx.x * VECS + threadIdx.x % VECS) * 4;
    mma_f4 s = mma_f4{0.f, 0.f, 0.f, 0.f};
    if (i < total)
#pragma unroll 4
        for (int p = threadIdx.x / VECS; p < splits; p += SHARE)
            s += *reinterpret_cast<const mma_f4 *>(part + (size_t)p * total + i);
    if constexpr (SHARE > 1) {
        red[threadIdx.x] = s;
        __syncthreads();
    }
    if (threadIdx.x >= VECS || i >= total || (i >= first && db == nullptr)) return;
#pragma unroll
    for (int p = 1; p < SHARE; p++) s += red[threadIdx.x + VECS * p];
    TO *out = i < first ? dw + i : db + (i - first);
#pragma unroll
    for (int e = 0; e < 4; e++) out[e] = from_float<TO>(s[e]);
}

template <typename T, typename TO>
int launch_linear_products(const void *dy, const void *x, TO *dw, TO *db, size_t stride, size_t rows, int N, int K,
                           const LinearSplits &s, hipStream_t st) {
    const unsigned tiles = (unsigned)((N + kLinTile - 1) / kLinTile) * ((K + kLinTile - 1) / kLinTile);
    const dim3 grid(tiles * (unsigned)s.splits), block(kLinThreads);
    if (s.halves)
        linear_wgrad_kernel<T, TO, true><<<grid, block, 0, st>>>((const T *)dy, (const T *)x, dw, db, stride, (long)rows, N, K,
                                                                 s.splits, s.per);
    else
        linear_wgrad_kernel<T, TO, false><<<grid, block, 0, st>>>((const T *)dy, (const T *)x, dw, db, stride, (long)rows, N,
                                                                  K, s.splits, s.per);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}
template <typename T, typename TO>
int launch_linear_wgrad(const void *dy, const void *x, void *dw, void *db, float *part, size_t rows, int N, int K,
                        hipStream_t st) {
    const LinearSplits s(rows, N, K);
    const int splits = s.splits;
    if (splits == 1) return launch_linear_products<T, TO>(dy, x, (TO *)dw, (TO *)db, 0, rows, N, K, s, st);
    const size_t outputs = (size_t)N * K, stride = outputs + N;
    const int e = launch_linear_products<T, float>(dy, x, part, db != nullptr ? part + outputs : nullptr, stride, rows, N, K,
                                                   s, st);
    if (e != 0) return e;
    const size_t vecs = stride / 4;
    const int share = splits < 8 ? 1 : 8, per = kLinThreads / share;
    const dim3 grid((unsigned)((vecs + per - 1) / per)), block(kLinThreads);
    if (share == 1) linear_reduce_kernel<TO, 1><<<grid, block, 0, st>>>(part, (TO *)dw, (TO *)db, N, K, splits);
    else linear_reduce_kernel<TO, 8><<<grid, block, 0, st>>>(part, (TO *)dw, (TO *)db, N, K, splits);
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? 0 : (int)err;
}

// ------------------------------------------------------------------------------------------------- inference
// y[m][n] = b[n] + sum_k x[m][k] * w[n][k] with what follows it in a block at inference (models/convnext.py:306-318):
//   rows     exact GELU on the way out, [M][N]: the first layer
//   planes   res + scale[n] * y as [image][N][HW]: the second layer, layer scale, permute and residual
// so that neither the 4 C-channel tensor before GELU nor the product of the second layer goes through memory by itself.
//
// A product D = P * Q^T puts four neighbouring rows of P into a lane's registers: P is the operand whose index is the
// fast one in the output (channels for rows, pixels for planes), and its rows are dealt to the fragments of a wave
// so that a lane ends up with twice eight neighbours, and four lanes with 64 bytes of output per store (8-byte
// stores left the L2 with four times as many writes: 401408 x 384 x 96 208 us, now 172).  Where planes are no multiple of four pixels
// lanes run along the pixels instead (single values, 32 bytes per store).

template <typename T>
struct LinearArgs {
    const T *x, *w, *bias, *scale, *res;
    T *out;
    long M;
    int N, K, HW, gelu;
};

// GELU of a sum that nothing has rounded: |u| (1/2 - q) + u / 2 with q = Phi(-|u|) = 2^p(|u|), p the polynomial of degree eight for
// log2 Phi(-t) on [0, 5] whose largest error, weighted with Phi(-t) + 1e-5, is least (from there on it falls, to -infinity).  The
// logarithm is so smooth that no quotient is needed, and v_rcp_f32 takes four issue slots: 15 a value instead of 20
// with erf from Abramowitz and Stegun 7.1.26 and further from 64 bits (in fp32, q off by 2.6e-7 at most, here 5.4e-8, GELU over N(0,1)
// by 5.5e-8 and 2.2e-8 rms, mean relative error on [-4, -3] 2.1e-4 and 8e-5).  us, bf16, with that / this: both layers of a block
// 401408 x 96 120 / 113, 100352 x 192 108.5 / 105; the first one 401408 x 384 x 96 173 / 167, 25088 x 1536 x 384 60 / 57.
// gelu_rounded, whose tail is exact to the result's rounding, has no place here: a separate layer's rounding of u, which the
// tail magnifies by u^2, is gone, and was worth five to nine times the difference.  Infinities and NaN give what u * (1 + erf) gives.
__device__ __forceinline__ float lin_gelu(float u) {
    const float t = __builtin_fabsf(u);
    float p = __builtin_fmaf(t, -2.09645073e-06f, 3.15079535e-05f);
    p = __builtin_fmaf(t, p, -0.000153187882f);
    p = __builtin_fmaf(t, p, -0.000206634976f);
    p = __builtin_fmaf(t, p, 0.00714238625f);
    p = __builtin_fmaf(t, p, -0.0525433468f);
    p = __builtin_fmaf(t, p, -0.459194624f);
    p = __builtin_fmaf(t, p, -1.15110672f);
    p = __builtin_fmaf(t, p, -0.999999963f);
    return __builtin_fmaf(t, 0.5f - __builtin_amdgcn_exp2f(p), 0.5f * u);
}

typedef unsigned mma_u2 __attribute__((ext_vector_type(2)));
template <typename T>
__device__ __forceinline__ unsigned lin_pack(float a, float b) {
    return (unsigned)__builtin_bit_cast(uint16_t, from_float<T>(a)) |
           (unsigned)__builtin_bit_cast(uint16_t, from_float<T>(b)) << 16;
}
template <typename T>
__device__ __forceinline__ float lin_value(unsigned v, int e) {
    return to_float(__builtin_bit_cast(T, (uint16_t)(v >> (16 * e))));
}

// Q neighbouring channels n .. n + Q - 1 of row m (Q 4 or 8, n a multiple of it; N is a multiple of eight)
template <int Q, typename T>
__device__ __forceinline__ void lin_emit_rows(const LinearArgs<T> &a, long m, int n, float (&v)[Q], const float (&b)[Q]) {
    if (m >= a.M || n >= a.N) return;
#pragma unroll
    for (int r = 0; r < Q; r++) v[r] += b[r];
    if (a.gelu) {
#pragma unroll
        for (int r = 0; r < Q; r++) v[r] = lin_gelu(v[r]);
    }
    T *at = a.out + m * a.N + n;
    if constexpr (Q == 8)
        *reinterpret_cast<mma_u4 *>(at) = mma_u4{lin_pack<T>(v[0], v[1]), lin_pack<T>(v[2], v[3]),
                                                 lin_pack<T>(v[4], v[5]), lin_pack<T>(v[6], v[7])};
    else *reinterpret_cast<mma_u2 *>(at) = mma_u2{lin_pack<T>(v[0], v[1]), lin_pack<T>(v[2], v[3])};
}
template <int Q, typename T>
__device__ __forceinline__ void lin_bias(const LinearArgs<T> &a, int n, float (&b)[Q]) {
#pragma unroll
    for (int r = 0; r < Q; r++) b[r] = a.bias != nullptr && n < a.N ? to_float(a.bias[n + r]) : 0.f;
}
// bias and scale of channel n
template <typename T>
__device__ __forceinline__ void lin_affine(const LinearArgs<T> &a, int n, float &b, float &s) {
    b = a.bias != nullptr && n < a.N ? to_float(a.bias[n]) : 0.f;
    s = a.scale != nullptr && n < a.N ? to_float(a.scale[n]) : 1.f;
}
// place of pixel m in channel 0 of its image
template <typename T>
__device__ __forceinline__ size_t lin_pixel(const LinearArgs<T> &a, long m) {
    const long img = (unsigned)m / (unsigned)a.HW;
    return (size_t)img * a.N * a.HW + (m - img * a.HW);
}
template <typename T>
__device__ __forceinline__ void lin_emit_pixel(const LinearArgs<T> &a, size_t at, float v, float b, float s) {
    a.out[at] = from_float<T>(__builtin_fmaf(v + b, s, a.res != nullptr ? to_float(a.res[at]) : 0.f));
}
// four neighbouring pixels m .. m + 3 of channel n (m a multiple of four)
template <typename T>
__device__ __forceinline__ void lin_emit_pixels4(const LinearArgs<T> &a, long m, int n, mma_f4 v, float b, float s) {
    if (m >= a.M || n >= a.N) return;
    if (a.HW % 4 == 0) {  // the four lie in one image, M is a multiple of four
        const size_t at = lin_pixel(a, m) + (size_t)n * a.HW;
        mma_u2 r = mma_u2{0u, 0u};
        if (a.res != nullptr) r = *reinterpret_cast<const mma_u2 *>(a.res + at);
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = __builtin_fmaf(v[e] + b, s, a.res != nullptr ? lin_value<T>(r[e / 2], e % 2) : 0.f);
        *reinterpret_cast<mma_u2 *>(a.out + at) = mma_u2{lin_pack<T>(o[0], o[1]), lin_pack<T>(o[2], o[3])};
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (m + e < a.M) lin_emit_pixel(a, lin_pixel(a, m + e) + (size_t)n * a.HW, v[e], b, s);
}
// eight neighbouring pixels m .. m + 7 of channel n (m a multiple of eight)
template <typename T>
__device__ __forceinline__ void lin_emit_pixels8(const LinearArgs<T> &a, long m, int n, mma_f4 v, mma_f4 w, float b, float s) {
    if (a.HW % 8 != 0) {
        lin_emit_pixels4(a, m, n, v, b, s);
        lin_emit_pixels4(a, m + 4, n, w, b, s);
        return;
    }
    if (m >= a.M || n >= a.N) return;
    const size_t at = lin_pixel(a, m) + (size_t)n * a.HW;
    mma_u4 r = mma_u4{0u, 0u, 0u, 0u};
    if (a.res != nullptr) r = *reinterpret_cast<const mma_u4 *>(a.res + at);
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; e++)
        o[e] = __builtin_fmaf((e < 4 ? v[e] : w[e - 4]) + b, s, a.res != nullptr ? lin_value<T>(r[e / 2], e % 2) : 0.f);
    *reinterpret_cast<mma_u4 *>(a.out + at) = mma_u4{lin_pack<T>(o[0], o[1]), lin_pack<T>(o[2], o[3]),
                                                     lin_pack<T>(o[4], o[5]), lin_pack<T>(o[6], o[7])};
}

// Tiles of 64 columns lie in LDS as rows of 128 bytes whose 16-byte pieces are permuted by the row, so that eight lanes of
// a fragment read meet on all banks.
constexpr int kLinK = 64;

// R rows x BK columns of a row-major operand from memory straight to LDS, zeros beyond its last row or column: a lane
// brings sixteen bytes per load, a wave 1 KB (the permutation is in the addresses it reads).
// DEAL: slot 32 h + 16 i + 4 g + r holds row 32 h + 8 g + 4 i + r.
template <int R, int BK, bool DEAL>
struct LinAsync {
    static constexpr int PIECES = BK / 8, U = R * PIECES / kLinThreads;  // pieces per row, loads
    unsigned off[U];
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ void init(const void *p, long rows, long r0, int K) {
        r = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(reinterpret_cast<const char *>(p) + r0 * K * 2), 0,
                                              (unsigned)min(max(rows - r0, 0L) * K * 2, 0x7fffffffL), 0x00020000);
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int f = (int)threadIdx.x + u * kLinThreads, s = f / PIECES;
            const int row = DEAL ? (s & ~31) + (s >> 2 & 3) * 8 + (s >> 4 & 1) * 4 + (s & 3) : s;
            off[u] = (unsigned)row * (unsigned)K * 2 + piece() * 16;
        }
    }
    // (the piece a lane reads is the same one in all its rows: they are a multiple of PIECES apart)
    static __device__ __forceinline__ int piece() {
        return (threadIdx.x % PIECES) ^ (threadIdx.x / PIECES % PIECES);
    }
    __device__ __forceinline__ void load(uint16_t *lds, int k0, int K) const {
        typedef __attribute__((address_space(3))) void lds_void;
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        // beyond the last column a lane reads nowhere, which writes zeros
        const unsigned kill = piece() * 8 < K - k0 ? 0u : kLinNowhere;
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
        for (int u = 0; u < U; u++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)(lds + (wave + 4 * u) * 512), 16, off[u] | kill,
                                                     k0 * 2, 0, 0);
#endif
    }
};
// 16 rows x 32 columns for a product, columns 32 kk .. of the tile
template <int BK>
__device__ __forceinline__ mma_s8 lin_fragment(const uint16_t *lds, int slot0, int kk) {
    const int lane = threadIdx.x & 63, s = slot0 + (lane & 15);
    return *reinterpret_cast<const mma_s8 *>(lds + s * BK + ((kk * 4 + (lane >> 4)) ^ (s & (BK / 8 - 1))) * 8);
}

// Outputs of a wave's fragments: P rows p0 + 32 h + 8 g + 4 i + r of fragments (2 h + i, j) against Q row q0 + 16 j + c.
enum { LIN_ROWS, LIN_PLANES, LIN_PIXELS };  // rows, planes, planes with lanes along the pixels (P rows not dealt)
template <int OUT, typename T, int H, int QF>
__device__ __forceinline__ void lin_emit(const LinearArgs<T> &a, long p0, long q0, const mma_f4 (&acc)[2 * H][QF]) {
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    if constexpr (OUT == LIN_PLANES) {
#pragma unroll
        for (int j = 0; j < QF; j++) {
            const int n = (int)q0 + 16 * j + c;
            float b, s;
            lin_affine(a, n, b, s);
#pragma unroll
            for (int h = 0; h < H; h++) lin_emit_pixels8(a, p0 + 32 * h + 8 * g, n, acc[2 * h][j], acc[2 * h + 1][j], b, s);
        }
    } else if constexpr (OUT == LIN_PIXELS) {
        size_t at[QF];
#pragma unroll
        for (int j = 0; j < QF; j++) at[j] = lin_pixel(a, q0 + 16 * j + c);
#pragma unroll
        for (int i = 0; i < 2 * H; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int n = (int)p0 + 16 * i + 4 * g + r;
                float b, s;
                lin_affine(a, n, b, s);
#pragma unroll
                for (int j = 0; j < QF; j++)
                    if (n < a.N && q0 + 16 * j + c < a.M) lin_emit_pixel(a, at[j] + (size_t)n * a.HW, acc[i][j][r], b, s);
            }
    } else {
#pragma unroll
        for (int h = 0; h < H; h++) {
            const int n = (int)p0 + 32 * h + 8 * g;
            float b[8];
            lin_bias(a, n, b);
#pragma unroll
            for (int j = 0; j < QF; j++) {
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = acc[2 * h + e / 4][j][e % 4];
                lin_emit_rows(a, q0 + 16 * j + c, n, v, b);
            }
        }
    }
}

// Large tiles: 128 rows of P, 32 * QF of Q, four waves of 64 x 16 QF products, two buffers: the next 64 columns travel
// to LDS while these are multiplied, one barrier per step, two workgroups per CU.  bf16, us: 25088 x 1536 x 384 with GELU 57 (MFMA
// 12, the GELU's vector instructions 30; library product and GELU kernel 92), 401408 x 384 x 96 167 (290); planes
// 25088 x 384 x 1536 58 (library and scale kernel 57), 401408 x 96 x 384 109 (193).  Tried: staging through registers
// (the same; -20 % where few workgroups run), three buffers with one workgroup per CU (+30 %), stages of 32 columns, three ahead (half
// lines; 6272 x 3072 x 768 52 / 63, planes 6272 x 768 x 3072 60 / 69).
template <typename T, int QF>
__device__ __forceinline__ void lin_products(const uint16_t *lp, const uint16_t *lq, int wp, int wq, mma_f4 (&acc)[4][QF]) {
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
        mma_s8 fp[4], fq[QF];
#pragma unroll
        for (int i = 0; i < 4; i++) fp[i] = lin_fragment<kLinK>(lp, wp + 16 * i, kk);
#pragma unroll
        for (int j = 0; j < QF; j++) fq[j] = lin_fragment<kLinK>(lq, wq + 16 * j, kk);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < QF; j++) acc[i][j] = Mma<T>::run(fp[i], fq[j], acc[i][j]);
    }
    // the second half's fragments are read between the products of the first
    __builtin_amdgcn_sched_group_barrier(0x100, 4 + QF, 0);
#pragma unroll
    for (int i = 0; i < 4 + QF; i++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 8 * QF - 2 * (4 + QF), 0);
}
template <typename T, int OUT, int QF>
__global__ __launch_bounds__(kLinThreads, 2) void linear_kernel(LinearArgs<T> a, int mtiles, int ntiles) {
    constexpr bool PLANES = OUT == LIN_PLANES;  // P is x
    constexpr int RP = 128, RQ = 32 * QF;
    __shared__ __attribute__((aligned(16))) uint16_t lp0[RP * kLinK];
    __shared__ __attribute__((aligned(16))) uint16_t lq0[RQ * kLinK];
    __shared__ __attribute__((aligned(16))) uint16_t lp1[RP * kLinK];
    __shared__ __attribute__((aligned(16))) uint16_t lq1[RQ * kLinK];
    const int k = blockIdx.x / 8, mt = k / ntiles * 8 + blockIdx.x % 8, nt = k % ntiles;
    if (mt >= mtiles) return;
    const long m0 = (long)mt * (PLANES ? RP : RQ);
    const int n0 = nt * (PLANES ? RQ : RP);
    LinAsync<RP, kLinK, OUT != LIN_PIXELS> tp;
    LinAsync<RQ, kLinK, false> tq;
    if (PLANES) tp.init(a.x, a.M, m0, a.K), tq.init(a.w, a.N, n0, a.K);
    else tp.init(a.w, a.N, n0, a.K), tq.init(a.x, a.M, m0, a.K);
    const int wave = threadIdx.x >> 6, wp = wave / 2 * 64, wq = wave % 2 * 16 * QF;
    mma_f4 acc[4][QF];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < QF; j++) acc[i][j] = mma_f4{0.f, 0.f, 0.f, 0.f};
    tp.load(lp0, 0, a.K), tq.load(lq0, 0, a.K);
    for (int k0 = 0; k0 < a.K; k0 += 2 * kLinK) {
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's pieces are there ..
        __syncthreads();                     // .. and the other waves'; nobody reads the other buffer any more
        if (k0 + kLinK < a.K) tp.load(lp1, k0 + kLinK, a.K), tq.load(lq1, k0 + kLinK, a.K);
        lin_products<T, QF>(lp0, lq0, wp, wq, acc);
        if (k0 + kLinK >= a.K) break;
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
        if (k0 + 2 * kLinK < a.K) tp.load(lp0, k0 + 2 * kLinK, a.K), tq.load(lq0, k0 + 2 * kLinK, a.K);
        lin_products<T, QF>(lp1, lq1, wp, wq, acc);
    }
    lin_emit<OUT, T, 2, QF>(a, (PLANES ? m0 : n0) + wp, (PLANES ? n0 : m0) + wq, acc);
}

// Fewer tiles than CUs, but not few (launch_few_tiles): 64 x 64, and the four waves share the columns, a quarter of every 128 each
// (a chain half as long per column, four times as many workgroups); their sums meet in LDS.  us, large tiles / these: 784 x
// 1536 x 384 9.7 / 6.8, 3136 x 384 x 96 7.6 / 6.2; 3136 x 1536 x 384 (300 large tiles) 13.3 / 17.2.
template <typename T, int OUT>
__global__ __launch_bounds__(kLinThreads, 2) void linear_split_kernel(LinearArgs<T> a, int mtiles) {
    constexpr bool PLANES = OUT == LIN_PLANES;
    constexpr int BK = 128, R = 64;
    __shared__ __attribute__((aligned(16))) uint16_t lp0[R * BK];
    __shared__ __attribute__((aligned(16))) uint16_t lq0[R * BK];
    __shared__ __attribute__((aligned(16))) uint16_t lp1[R * BK];
    __shared__ __attribute__((aligned(16))) uint16_t lq1[R * BK];
    const long m0 = (long)(blockIdx.x % mtiles) * R;
    const int n0 = blockIdx.x / mtiles * R;
    LinAsync<R, BK, OUT != LIN_PIXELS> tp;
    LinAsync<R, BK, false> tq;
    if (PLANES) tp.init(a.x, a.M, m0, a.K), tq.init(a.w, a.N, n0, a.K);
    else tp.init(a.w, a.N, n0, a.K), tq.init(a.x, a.M, m0, a.K);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    mma_f4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 16; i++) acc[i / 4][i % 4] = mma_f4{0.f, 0.f, 0.f, 0.f};
    auto products = [&](const uint16_t *lp, const uint16_t *lq) {
        mma_s8 fp[4], fq[4];
#pragma unroll
        for (int i = 0; i < 4; i++) fp[i] = lin_fragment<BK>(lp, 16 * i, wave), fq[i] = lin_fragment<BK>(lq, 16 * i, wave);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[i][j] = Mma<T>::run(fp[i], fq[j], acc[i][j]);
    };
    tp.load(lp0, 0, a.K), tq.load(lq0, 0, a.K);
    for (int k0 = 0; k0 < a.K; k0 += 2 * BK) {
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
        if (k0 + BK < a.K) tp.load(lp1, k0 + BK, a.K), tq.load(lq1, k0 + BK, a.K);
        products(lp0, lq0);
        if (k0 + BK >= a.K) break;
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
        if (k0 + 2 * BK < a.K) tp.load(lp0, k0 + 2 * BK, a.K), tq.load(lq0, k0 + 2 * BK, a.K);
        products(lp1, lq1);
    }
    // four arrays of 16 KB: fragments (i, ..) of all waves in array i; wave 2 h + x ends up with fragments (2 h + .., 2 x + ..)
    __syncthreads();
    auto give = [&](uint16_t *to, int i) {
#pragma unroll
        for (int j = 0; j < 4; j++) reinterpret_cast<mma_f4 *>(to)[(j * 4 + wave) * 64 + lane] = acc[i][j];
    };
    give(lp0, 0), give(lq0, 1), give(lp1, 2), give(lq1, 3);
    __syncthreads();
    const int h = wave / 2, x = wave % 2;
    mma_f4 sum[2][2];
    auto take = [&](const uint16_t *from, int i) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const mma_f4 *r = reinterpret_cast<const mma_f4 *>(from) + (2 * x + j) * 256 + lane;
            sum[i][j] = (r[0] + r[64]) + (r[128] + r[192]);
        }
    };
    if (h == 0) take(lp0, 0), take(lq0, 1);
    else take(lp1, 0), take(lq1, 1);
    lin_emit<OUT, T, 1, 2>(a, (PLANES ? m0 : n0) + 32 * h, (PLANES ? n0 : m0) + 32 * x, sum);
}

// Fewer tiles still (launch_few_tiles): 32 rows of P and 16 * QF of Q.  No two waves read the same value (every fourth 64 columns are
// a wave's), so each has its own four stages of LDS, three of them on their way, and no barrier until the sums meet: with the
// kernel above two stages and few workgroups left the loads of a long row one after the other.  Through LDS and not straight to
// registers, because a fragment's neighbouring lanes lie in different rows (196 x 384 x 1536 7.2, 49 x 768 x 3072 12.8).
// Waiting for memory bounds it (half of the waves' cycles by counters, no unit above 6 %).  bf16, us, 64 x 64 tiles / these, behind a
// pass over other memory, as in a network, whose weights come from beyond the L2: 49 x 3072 x 768 7.1 / 4.7, planes 196 x 384 x 1536 12.6 / 5.0, 784 x
// 192 x 768 7.8 / 4.8, 98 x 1024 x 4096 27.9 / 9.7, 49 x 768 x 3072 21.5 / 8.1, rows 196 x 384 x 96 4.3 / 4.3 (an empty launch 3).
template <typename T, int OUT, int QF>
__global__ __launch_bounds__(kLinThreads, 1) void linear_wave_kernel(LinearArgs<T> a, int xtiles, int tiles) {
    constexpr bool PLANES = OUT == LIN_PLANES;
    constexpr int RP = 32, RQ = 16 * QF, BK = 64, WAVES = kLinThreads / 64, LP = RP / 8, LQ = RQ / 8;  // (a load is eight rows)
    constexpr int SIZE = WAVES * (RP + RQ) * BK;
    __shared__ __attribute__((aligned(16))) uint16_t s0[SIZE];
    __shared__ __attribute__((aligned(16))) uint16_t s1[SIZE];
    __shared__ __attribute__((aligned(16))) uint16_t s2[SIZE];
    __shared__ __attribute__((aligned(16))) uint16_t s3[SIZE];
    // an XCD (workgroup ids modulo eight) takes a run of tiles, those of x against the same weights next to each other
    const int tile = blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8;
    if (tile >= tiles) return;
    const long m0 = (long)(tile % xtiles) * (PLANES ? RP : RQ);
    const int n0 = tile / xtiles * (PLANES ? RQ : RP);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const long pitch = (long)a.K * 2;
    auto operand = [&](const T *p, long rows, long r0) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(reinterpret_cast<const char *>(p) + r0 * pitch), 0,
                                                 (unsigned)min((rows - r0) * pitch, 0x7fffffffL), 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rp = PLANES ? operand(a.x, a.M, m0) : operand(a.w, a.N, n0);
    const __amdgpu_buffer_rsrc_t rq = PLANES ? operand(a.w, a.N, n0) : operand(a.x, a.M, m0);
    const int piece = (lane % 8) ^ (lane / 8);
    unsigned op[LP], oq[LQ];  // (rows beyond the last lie beyond the operand's end: zeros)
#pragma unroll
    for (int u = 0; u < LP; u++) {
        const int s = 8 * u + lane / 8;
        const int row = OUT == LIN_PIXELS ? s : (s >> 2 & 3) * 8 + (s >> 4 & 1) * 4 + (s & 3);
        op[u] = (unsigned)row * (unsigned)pitch + piece * 16;
    }
#pragma unroll
    for (int u = 0; u < LQ; u++) oq[u] = (unsigned)(8 * u + lane / 8) * (unsigned)pitch + piece * 16;
    int k0 = wave * BK;  // of the next load
    auto load = [&](uint16_t *stage) {
        typedef __attribute__((address_space(3))) void lds_void;
        const unsigned kill = piece * 8 < a.K - k0 ? 0u : kLinNowhere;
        uint16_t *at = stage + wave * (RP + RQ) * BK;
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
        for (int u = 0; u < LP; u++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rp, (lds_void *)(at + u * 8 * BK), 16, op[u] | kill, k0 * 2, 0, 0);
#pragma unroll
        for (int u = 0; u < LQ; u++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rq, (lds_void *)(at + (RP + u * 8) * BK), 16, oq[u] | kill, k0 * 2, 0, 0);
#endif
        k0 += WAVES * BK;
    };
    mma_f4 acc[2][QF];
#pragma unroll
    for (int i = 0; i < 2 * QF; i++) acc[i / QF][i % QF] = mma_f4{0.f, 0.f, 0.f, 0.f};
    auto step = [&](const uint16_t *stage, uint16_t *next) {
        // all but the next two stages' loads have arrived, and the reads of the one before, which `next` was
        constexpr int N = 2 * (LP + LQ);
        __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | N >> 4 << 14);  // vmcnt(N) lgkmcnt(0)
        asm volatile("" ::: "memory");
        load(next);
        __builtin_amdgcn_sched_barrier(0);
        const uint16_t *at = stage + wave * (RP + RQ) * BK;
        mma_s8 fp[2][2], fq[2][QF];
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
#pragma unroll
            for (int i = 0; i < 2; i++) fp[kk][i] = lin_fragment<BK>(at, 16 * i, kk);
#pragma unroll
            for (int j = 0; j < QF; j++) fq[kk][j] = lin_fragment<BK>(at + RP * BK, 16 * j, kk);
        }
#pragma unroll
        for (int kk = 0; kk < 2; kk++)
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < QF; j++) acc[i][j] = Mma<T>::run(fp[kk][i], fq[kk][j], acc[i][j]);
    };
    load(s0), load(s1), load(s2);
    int left = (a.K + WAVES * BK - 1) / (WAVES * BK);
    for (; left > 2; left -= 4) {
        step(s0, s3), step(s1, s0), step(s2, s1);
        if (left == 3) { left = 0; break; }
        step(s3, s2);
    }
    if (left > 0) step(s0, s3);
    if (left > 1) step(s1, s0);
    __builtin_amdgcn_s_waitcnt(0x0070);  // (nothing may arrive behind the sums)
    {
        mma_f4 *mine = reinterpret_cast<mma_f4 *>(s0 + wave * (RP + RQ) * BK) + lane;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < QF; j++) mine[(2 * j + i) * 64] = acc[i][j];
    }
    __syncthreads();
    if (wave >= QF) return;
    mma_f4 sum[2][1];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        mma_f4 v[WAVES];
#pragma unroll
        for (int w = 0; w < WAVES; w++)
            v[w] = reinterpret_cast<const mma_f4 *>(s0 + w * (RP + RQ) * BK)[(2 * wave + i) * 64 + lane];
        sum[i][0] = (v[0] + v[1]) + (v[2] + v[3]);
    }
    lin_emit<OUT, T, 1, 1>(a, PLANES ? m0 : n0, (PLANES ? n0 : m0) + 16 * wave, sum);
}

// Workgroups of linear_wave_kernel, one per CU: the narrow tiles where they fit the chip at once, the others up to twice its CUs.
// The second round pays where rows are long, as long as what it reads has to come from beyond the L2 (us, bf16, behind a pass over
// other memory, 64 x 64 tiles / these: planes 300 tiles 784 x 384 x 1536 12.5 / 10.5, 484 x 320 x 1280 10.8 / 9.3, 784 x 512 x 2048 15.2 /
// 11.6, 512 tiles 1024 x 512 x 2048 13.9 / 13.3, 512 x 1024 x 4096 24.3 / 17.5, 1024 x 320 x 1280 10.9 / 10.5); rows of 1024 gain nothing (1176 x
// 256 x 1024 9.8 / 9.5, 1536 rows 8.7 / 9.1, 2048 rows 8.9 / 9.8, odd planes 15.0 / 15.9) and lose back to back (1176 x 256 x 1024 7.7 / 8.0, odd
// planes 9.9 / 11.4), shorter ones lose (rows, 189 x 1536 x 384 5.7 / 7.1).  The third round does not pay (1056 x 512 x 2048 14.7 / 18.2).
constexpr long kLinCus = 256;
constexpr int kLinLongRow = 1280;
template <typename T, int OUT, int QF>
bool launch_wave_tiles(const LinearArgs<T> &a, long most, hipStream_t st) {
    constexpr int X = OUT == LIN_PLANES ? 32 : 16 * QF, W = OUT == LIN_PLANES ? 16 * QF : 32;
    const long xtiles = (a.M + X - 1) / X, tiles = xtiles * ((a.N + W - 1) / W);
    if (tiles > most) return false;
    linear_wave_kernel<T, OUT, QF><<<dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(kLinThreads), 0, st>>>(a, (int)xtiles, (int)tiles);
    return true;
}
template <typename T, int OUT>
int launch_few_tiles(const LinearArgs<T> &a, hipStream_t st) {
    if (!launch_wave_tiles<T, OUT, 1>(a, kLinCus, st) &&
        !launch_wave_tiles<T, OUT, 2>(a, a.K < kLinLongRow ? kLinCus : 2 * kLinCus, st)) {
        const int mt = (int)((a.M + 63) / 64);
        linear_split_kernel<T, OUT><<<dim3((unsigned)((long)mt * ((a.N + 63) / 64))), dim3(kLinThreads), 0, st>>>(a, mt);
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}

constexpr long kLinLargeTiles = 160;
template <typename T, bool PLANES>
int launch_linear(const LinearArgs<T> &a, hipStream_t st) {
    // channels per large tile: 96 where that leaves no partial tile and 128 does (planes only)
    const bool three = PLANES && a.HW % 4 == 0 && a.N % 128 != 0 && a.N % 96 == 0;
    const int nt = three ? 96 : 128;
    const long mtiles = (a.M + 127) / 128;
    const int ntiles = (a.N + nt - 1) / nt;
    if (mtiles * ntiles >= kLinLargeTiles) {  // (both kernels take the same time at 150 to 170 tiles)
        const dim3 grid((unsigned)((mtiles + 7) / 8 * 8 * ntiles)), block(kLinThreads);
        if constexpr (!PLANES) linear_kernel<T, LIN_ROWS, 4><<<grid, block, 0, st>>>(a, (int)mtiles, ntiles);
        else if (a.HW % 4 != 0) linear_kernel<T, LIN_PIXELS, 4><<<grid, block, 0, st>>>(a, (int)mtiles, ntiles);
        else if (three) linear_kernel<T, LIN_PLANES, 3><<<grid, block, 0, st>>>(a, (int)mtiles, ntiles);
        else linear_kernel<T, LIN_PLANES, 4><<<grid, block, 0, st>>>(a, (int)mtiles, ntiles);
    } else {
        constexpr int OUT = PLANES ? LIN_PLANES : LIN_ROWS;
        if constexpr (PLANES)
            if (a.HW % 4 != 0) return launch_few_tiles<T, LIN_PIXELS>(a, st);
        return launch_few_tiles<T, OUT>(a, st);
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}

// ------------------------------------------------------------------------------------------------- norm behind a layer
// out[image][n][p] = LayerNorm over n of (b[n] + sum_k w[n][k] z[image][p][k]) with z = GELU(LayerNorm over k of x), rounded as a layer
// of its own would: the stem's last layers with the planes that follow (models/convnext.py:184-190), K = 64 and N = 16 NB <= 128.
// A wave holds the weights as fragments and takes 32 pixels at a time with all their channels, so that a LayerNorm is a sum
// over its registers and a few lanes.  GELU's vector instructions bound it, 68 % of the time by counters: 401408 x 64 -> 96 in bf16 56
// us (without the first norm 38, which is reading x and writing the planes; as a norm pass, the library's product, a norm pass and a
// transposition 200), one image 9.6 behind other work (back to back 8, 20), waiting for its one tile per wave.
constexpr int kNormK = 64, kNormGroups = 1024;
struct NormArgs {
    const float *gamma, *beta, *gamma_in, *beta_in;
    float eps, eps_in;
};
template <typename T, int NB>
__global__ __launch_bounds__(kLinThreads, 2) void linear_norm_kernel(LinearArgs<T> a, NormArgs na, long tiles) {
    __shared__ __attribute__((aligned(16))) float affine[2 * kNormK];  // of the norm before
    if (threadIdx.x < 2 * kNormK)
        affine[threadIdx.x] = threadIdx.x < kNormK ? na.gamma_in[threadIdx.x] : na.beta_in[threadIdx.x - kNormK];
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    mma_s8 fw[2][NB];
    float bias[NB], gm[NB], bt[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const int n = 16 * j + c;
#pragma unroll
        for (int k = 0; k < 2; k++) fw[k][j] = *reinterpret_cast<const mma_s8 *>(a.w + n * kNormK + k * 32 + g * 8);
        bias[j] = a.bias != nullptr ? to_float(a.bias[n]) : 0.f, gm[j] = na.gamma[n], bt[j] = na.beta[n];
    }
    auto lanes = [](float v) {  // over the sixteen lanes of a row
        auto add = [](float v, auto ctrl) {
            return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value,
                                                                             0xf, 0xf, true));
        };
        v = add(v, std::integral_constant<int, 0xB1>{});      // quad_perm [1,0,3,2]
        v = add(v, std::integral_constant<int, 0x4E>{});      // quad_perm [2,3,0,1]
        v = add(v, std::integral_constant<int, 0x141>{});     // row_half_mirror
        return add(v, std::integral_constant<int, 0x140>{});  // row_mirror
    };
    mma_s8 fx[2][2], next[2][2];
    auto fetch = [&](mma_s8 (&f)[2][2], long tile) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const long m = min(tile * 32 + 8 * (c >> 2) + 4 * i + (c & 3), a.M - 1);  // (pixels beyond the last are not written)
#pragma unroll
            for (int k = 0; k < 2; k++) f[k][i] = *reinterpret_cast<const mma_s8 *>(a.x + m * kNormK + k * 32 + g * 8);
        }
    };
    const long step = (long)gridDim.x * (kLinThreads / 64);
    long tile = (long)blockIdx.x * (kLinThreads / 64) + wave;
    if (tile >= tiles) return;
    fetch(next, tile);
    for (; tile < tiles; tile += step) {
#pragma unroll
        for (int k = 0; k < 2; k++) fx[k][0] = next[k][0], fx[k][1] = next[k][1];
        if (tile + step < tiles) fetch(next, tile + step);
#pragma unroll
        for (int i = 0; i < 2; i++) {  // a lane has 16 of its pixel's channels, the lanes 16, 32 and 48 on the others
            float u[2][8], s = 0.f, q = 0.f;
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int e = 0; e < 8; e++)
                    u[k][e] = to_float(__builtin_bit_cast(T, (uint16_t)fx[k][i][e])), s += u[k][e];
            s += __shfl_xor(s, 16, 64), s += __shfl_xor(s, 32, 64);
            s *= 1.f / kNormK;
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int e = 0; e < 8; e++) u[k][e] -= s, q = __builtin_fmaf(u[k][e], u[k][e], q);
            q += __shfl_xor(q, 16, 64), q += __shfl_xor(q, 32, 64);
            q = rsqrtf(q * (1.f / kNormK) + na.eps_in);
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const float *p = affine + 32 * k + 8 * g;
                mma_u4 o;
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const mma_f4 gi = *reinterpret_cast<const mma_f4 *>(p + 4 * h);
                    const mma_f4 bi = *reinterpret_cast<const mma_f4 *>(p + kNormK + 4 * h);
                    float w[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) w[e] = gelu_rounded(__builtin_fmaf(u[k][4 * h + e] * q, gi[e], bi[e]));
                    o[2 * h] = lin_pack<T>(w[0], w[1]), o[2 * h + 1] = lin_pack<T>(w[2], w[3]);
                }
                fx[k][i] = __builtin_bit_cast(mma_s8, o);
            }
        }
        mma_f4 v[2][NB];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            mma_f4 s = mma_f4{0.f, 0.f, 0.f, 0.f}, q = s;
#pragma unroll
            for (int j = 0; j < NB; j++) {
                v[i][j] = mma_f4{bias[j], bias[j], bias[j], bias[j]};
#pragma unroll
                for (int k = 0; k < 2; k++) v[i][j] = Mma<T>::run(fx[k][i], fw[k][j], v[i][j]);
#pragma unroll
                for (int r = 0; r < 4; r++) s[r] += v[i][j][r];
            }
#pragma unroll
            for (int r = 0; r < 4; r++) s[r] = lanes(s[r]) * (1.f / (16 * NB));
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) v[i][j][r] -= s[r], q[r] = __builtin_fmaf(v[i][j][r], v[i][j][r], q[r]);
#pragma unroll
            for (int r = 0; r < 4; r++) q[r] = rsqrtf(lanes(q[r]) / (float)(16 * NB) + na.eps);
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) v[i][j][r] = __builtin_fmaf(v[i][j][r] * q[r], gm[j], bt[j]);
        }
#pragma unroll
        for (int j = 0; j < NB; j++) lin_emit_pixels8(a, tile * 32 + 8 * g, 16 * j + c, v[0][j], v[1][j], 0.f, 1.f);
    }
}

template <typename T>
int launch_linear_norm(const LinearArgs<T> &a, const NormArgs &na, hipStream_t st) {
    const long tiles = (a.M + 31) / 32, want = (tiles + 3) / 4;
    const dim3 grid((unsigned)(want < kNormGroups ? want : kNormGroups)), block(kLinThreads);
    if (a.N == 96) linear_norm_kernel<T, 6><<<grid, block, 0, st>>>(a, na, tiles);
    else linear_norm_kernel<T, 8><<<grid, block, 0, st>>>(a, na, tiles);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}

// ------------------------------------------------------------------------------------------------- few inputs
// y[m][n] = b[n] + sum_k x[m][k] * w[n][k] for K <= 4 (the stem's first layer, models/convnext.py:143,177) and N a multiple of
// 64.  Writing y bounds it (64 x 224 x 224 pixels of 64 channels in bf16: 411 MB; back to back 147 us, as a library product 330;
// in a training pass 118).
// One matrix instruction per 16 pixels x 16 channels, 28 of its 32 columns zero: the same sums, bit for
// bit, as a library product's.
constexpr int kFewThreads = 256;
template <typename T, int K>
__global__ __launch_bounds__(kFewThreads) void few_inputs_kernel(const T *__restrict__ x, const T *__restrict__ w,
                                                                 const T *__restrict__ b, T *__restrict__ y, long M,
                                                                 int N) {
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    const int n0 = blockIdx.y * 64;
    // fragment 2 h + i: channels 32 h + 8 g' + 4 i + r for its rows 4 g' + r
    mma_s8 fw[4];
#pragma unroll
    for (int f = 0; f < 4; f++) {
        fw[f] = mma_s8{0, 0, 0, 0, 0, 0, 0, 0};
        const int n = n0 + 32 * (f / 2) + 8 * (c / 4) + 4 * (f % 2) + c % 4;
        if (g == 0)
#pragma unroll
            for (int k = 0; k < K; k++) fw[f][k] = __builtin_bit_cast(short, w[(size_t)n * K + k]);
    }
    float bias[4][4];
#pragma unroll
    for (int f = 0; f < 4; f++)
#pragma unroll
        for (int r = 0; r < 4; r++)
            bias[f][r] = b != nullptr ? to_float(b[n0 + 32 * (f / 2) + 8 * g + 4 * (f % 2) + r]) : 0.f;
    constexpr int U = 4;  // groups of 16 pixels per step
    const long step = (long)gridDim.x * (kFewThreads / 64) * 16 * U;
    for (long m0 = ((long)blockIdx.x * (kFewThreads / 64) + (threadIdx.x >> 6)) * 16 * U; m0 < M; m0 += step) {
        mma_s8 fx[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            fx[u] = mma_s8{0, 0, 0, 0, 0, 0, 0, 0};
            const long m = m0 + 16 * u + c;
            if (g == 0 && m < M)
#pragma unroll
                for (int k = 0; k < K; k++) fx[u][k] = __builtin_bit_cast(short, x[m * K + k]);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const long m = m0 + 16 * u + c;
            mma_f4 v[4];
#pragma unroll
            for (int f = 0; f < 4; f++) {
                v[f] = Mma<T>::run(fw[f], fx[u], mma_f4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                for (int r = 0; r < 4; r++) v[f][r] += bias[f][r];
            }
            if (m < M)
#pragma unroll
                for (int h = 0; h < 2; h++)
                    *reinterpret_cast<mma_u4 *>(y + m * N + n0 + 32 * h + 8 * g) =
                        mma_u4{lin_pack<T>(v[2 * h][0], v[2 * h][1]), lin_pack<T>(v[2 * h][2], v[2 * h][3]),
                               lin_pack<T>(v[2 * h + 1][0], v[2 * h + 1][1]), lin_pack<T>(v[2 * h + 1][2], v[2 * h + 1][3])};
        }
    }
}

template <typename T>
int launch_few_inputs(const void *x, const void *w, const void *b, void *y, long M, int N, int K, hipStream_t st) {
    const long want = (M + 255) / 256, most = 8192 / (N / 64) > 0 ? 8192 / (N / 64) : 1;
    const dim3 grid((unsigned)(want < most ? want : most), N / 64), block(kFewThreads);
#define DWO_FEW(K_) \
    case K_: few_inputs_kernel<T, K_><<<grid, block, 0, st>>>((const T *)x, (const T *)w, (const T *)b, (T *)y, M, N); break;
    switch (K) { DWO_FEW(1) DWO_FEW(2) DWO_FEW(3) DWO_FEW(4) }
#undef DWO_FEW
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}

}  // namespace dwo
