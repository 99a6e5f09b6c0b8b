// What a ConvNeXt-1D block and the stem do around the operator and the pointwise layers when they are
// trained (models/convnext.py:176-190,306-318), forward and backward, each as one pass over its tensors:
//
//   ln_tile     y [N,C,HW] -> LayerNorm over C -> [N,HW,C]        permute + LayerNorm of a block
//   ln_rows     rows of C  -> LayerNorm -> (GELU)                 the stem's
//   ln_patch    y [N,C,H,W] -> LayerNorm over C -> 2 x 2 patches  in front of a downsampling layer
//   tail        res + scale[c] * y, y [N,HW,C] -> [N,C,HW]        layer scale + permute + residual
//
// Memory bounds them (ln_tile 5.4 TB/s with the VALU busy for 85 %, tail 6.5, backward 5.7) but for ln_rows with GELU, where it
// is the vector instructions (87 % of the time forward, 94 % backward with an fp32 gradient), and small tensors.  PyTorch's
// compositions move each tensor three to six times (permuted copies, conversions, separate parameter gradients).  Input and output
// have types of their own, so the conversions of autocast happen on the way out (fp32 stream, 16-bit pointwise layers).
// Channels are handled in pieces of eight, rows by groups of 8 to 64 lanes, and parameter gradients are kept in registers
// over all the tiles of a workgroup, written as partial sums and added in a fixed order by a second kernel.  Statistics and
// sums are fp32.
#pragma once

#include "dwo_common.h"

namespace dwo {

constexpr int kBlkThreads = 256, kBlkMaxC = 1024, kBlkGroups = 1024;

typedef unsigned blk_u4 __attribute__((ext_vector_type(4)));
typedef unsigned blk_u2 __attribute__((ext_vector_type(2)));
typedef float blk_f4 __attribute__((ext_vector_type(4)));
typedef float blk_f2 __attribute__((ext_vector_type(2)));

// eight neighbouring values as floats
template <typename T>
__device__ __forceinline__ void load8(const T *p, float (&v)[8]) {
    if constexpr (sizeof(T) == 4) {
        const blk_f4 a = reinterpret_cast<const blk_f4 *>(p)[0], b = reinterpret_cast<const blk_f4 *>(p)[1];
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = a[i], v[4 + i] = b[i];
    } else {
        const blk_u4 a = *reinterpret_cast<const blk_u4 *>(p);
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = to_float(__builtin_bit_cast(T, (uint16_t)(a[i / 2] >> (16 * (i % 2)))));
    }
}
template <typename T>
__device__ __forceinline__ unsigned pack2(float a, float b) {
    return (unsigned)__builtin_bit_cast(uint16_t, from_float<T>(a)) |
           (unsigned)__builtin_bit_cast(uint16_t, from_float<T>(b)) << 16;
}
template <typename T>
__device__ __forceinline__ void store8(T *p, const float (&v)[8]) {
    if constexpr (sizeof(T) == 4) {
        reinterpret_cast<blk_f4 *>(p)[0] = blk_f4{v[0], v[1], v[2], v[3]};
        reinterpret_cast<blk_f4 *>(p)[1] = blk_f4{v[4], v[5], v[6], v[7]};
    } else {
        *reinterpret_cast<blk_u4 *>(p) =
            blk_u4{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]), pack2<T>(v[4], v[5]), pack2<T>(v[6], v[7])};
    }
}
// VEC = 4 or 1 neighbouring values
template <typename T, int VEC>
__device__ __forceinline__ void load_run(const T *p, float (&v)[VEC]) {
    if constexpr (VEC == 1) v[0] = to_float(*p);
    else if constexpr (sizeof(T) == 4) {
        const blk_f4 a = *reinterpret_cast<const blk_f4 *>(p);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = a[i];
    } else {
        const blk_u2 a = *reinterpret_cast<const blk_u2 *>(p);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = to_float(__builtin_bit_cast(T, (uint16_t)(a[i / 2] >> (16 * (i % 2)))));
    }
}
template <typename T, int VEC>
__device__ __forceinline__ void store_run(T *p, const float (&v)[VEC]) {
    if constexpr (VEC == 1) *p = from_float<T>(v[0]);
    else if constexpr (sizeof(T) == 4) *reinterpret_cast<blk_f4 *>(p) = blk_f4{v[0], v[1], v[2], v[3]};
    else *reinterpret_cast<blk_u2 *>(p) = blk_u2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
}

// Total over the aligned group of LPR lanes, in every lane.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int LPR>
__device__ __forceinline__ float group_total(float v) {
    v = dpp_add<0xB1>(v);   // quad_perm [1,0,3,2]
    v = dpp_add<0x4E>(v);   // quad_perm [2,3,0,1]
    v = dpp_add<0x141>(v);  // row_half_mirror: the other four of eight
    if constexpr (LPR >= 16) v = dpp_add<0x140>(v);  // row_mirror: the other eight of sixteen
    if constexpr (LPR >= 32) v += __shfl_xor(v, 16, 64);
    if constexpr (LPR >= 64) v += __shfl_xor(v, 32, 64);
    return v;
}

// flags of the row kernels
enum { ROWS_GELU = 1, ROWS_ROUNDED = 2 };  // GELU; what it takes (and its gradient) rounded to the output's type
template <typename T>
__device__ __forceinline__ float rounded(float v) { return to_float(from_float<T>(v)); }

__device__ __forceinline__ float blk_gelu(float u) { return 0.5f * u * (1.f + erff(u * 0.70710678118654752f)); }
__device__ __forceinline__ float blk_gelu_slope(float u) {
    return 0.5f * (1.f + erff(u * 0.70710678118654752f)) + u * 0.39894228040143268f * expf(-0.5f * u * u);
}

// Channels of a lane: pieces lane % LPR + k * LPR for k < NV.
template <int LPR, int NV>
struct Lanes {
    int l, slot;                          // place in the group, row within a step of the workgroup
    __device__ __forceinline__ Lanes() : l(threadIdx.x % LPR), slot(threadIdx.x / LPR) {}
    static constexpr int ROWS = kBlkThreads / LPR;  // rows per step of the workgroup
    __device__ __forceinline__ int chan(int k) const { return 8 * (l + k * LPR); }
};

// Sums of a workgroup's lanes of equal channels: [2][C] partial sums per workgroup.
template <int LPR, int NV>
__device__ __forceinline__ void write_param_partials(float (&dg)[NV][8], float (&db)[NV][8], int C, float *red,
                                                     float *part) {
    constexpr int ROWS = Lanes<LPR, NV>::ROWS;
#pragma unroll
    for (int k = 0; k < NV; k++)
#pragma unroll
        for (int which = 0; which < 2; which++) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 8; i++) red[i * kBlkThreads + threadIdx.x] = which == 0 ? dg[k][i] : db[k][i];
            __syncthreads();
            // value i of lane l, summed over the rows
            for (int f = threadIdx.x; f < 8 * LPR; f += kBlkThreads) {
                const int l = f / 8, i = f % 8, c = 8 * (l + k * LPR) + i;
                float s = 0.f;
#pragma unroll
                for (int r = 0; r < ROWS; r++) s += red[i * kBlkThreads + r * LPR + l];
                if (c < C) part[(size_t)blockIdx.x * 2 * C + which * C + c] = s;
            }
        }
}

// part [groups][L] -> out0 [split], out1 [L - split], fixed order.  Few columns and up to a thousand groups: latency binds,
// so 32 threads share a column, each with eight loads in flight (eight threads, one load at a
// time: 23 us for 1024 groups of 1024 columns, now 8).
constexpr int kColThreads = 1024;
template <typename TO>
__global__ __launch_bounds__(kColThreads) void column_sums_kernel(const float *__restrict__ part, TO *out0, TO *out1,
                                                                  int L, int split, int groups) {
    __shared__ float red[kColThreads];
    const int c = blockIdx.x * 32 + threadIdx.x % 32;
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (c < L)
        for (int g = threadIdx.x / 32; g < groups; g += 256) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = g + 32 * u < groups ? part[(size_t)(g + 32 * u) * L + c] : 0.f;
#pragma unroll
            for (int u = 0; u < 8; u++) s[u] += v[u];
        }
    red[threadIdx.x] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    __syncthreads();
    if (threadIdx.x >= 32 || c >= L) return;
    float t = red[threadIdx.x];
#pragma unroll
    for (int k = 1; k < 32; k++) t += red[threadIdx.x + 32 * k];
    TO *out = c < split ? out0 : out1;
    if (out != nullptr) out[c < split ? c : c - split] = from_float<TO>(t);
}

// ------------------------------------------------------------------------------------------------- rows
template <typename TI, typename TO, int LPR, int NV>
__global__ __launch_bounds__(kBlkThreads) void ln_rows_kernel(const TI *__restrict__ x, const float *__restrict__ gamma,
                                                              const float *__restrict__ beta, TO *__restrict__ out,
                                                              float2 *__restrict__ stats, long rows, int C, float eps,
                                                              int gelu) {
    const Lanes<LPR, NV> ln;
    float gm[NV][8], bt[NV][8];
#pragma unroll
    for (int k = 0; k < NV; k++)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int c = ln.chan(k) + i;
            gm[k][i] = c < C ? gamma[c] : 0.f, bt[k][i] = c < C ? beta[c] : 0.f;
        }
    const long step = (long)gridDim.x * ln.ROWS;
    for (long r0 = (long)blockIdx.x * ln.ROWS; r0 < rows; r0 += step) {
        const long r = r0 + ln.slot;
        const bool row = r < rows;
        float v[NV][8], s = 0.f;
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const bool ok = row && ln.chan(k) < C;
            if (ok) load8(x + r * C + ln.chan(k), v[k]);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                if (!ok) v[k][i] = 0.f;
                s += v[k][i];
            }
        }
        const float mean = group_total<LPR>(s) / (float)C;
        float q = 0.f;
#pragma unroll
        for (int k = 0; k < NV; k++)
            if (ln.chan(k) < C)
#pragma unroll
                for (int i = 0; i < 8; i++) v[k][i] -= mean, q = __builtin_fmaf(v[k][i], v[k][i], q);
        const float rstd = rsqrtf(group_total<LPR>(q) / (float)C + eps);
        if (!row) continue;
#pragma unroll
        for (int k = 0; k < NV; k++)
            if (ln.chan(k) < C) {
                float o[8];
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    o[i] = __builtin_fmaf(v[k][i] * rstd, gm[k][i], bt[k][i]);
                    if (gelu & ROWS_ROUNDED) o[i] = rounded<TO>(o[i]);
                    if (gelu & ROWS_GELU) o[i] = sizeof(TO) == 2 ? gelu_rounded(o[i]) : blk_gelu(o[i]);
                }
                store8(out + r * C + ln.chan(k), o);
            }
        if (stats != nullptr && ln.l == 0) stats[r] = make_float2(mean, rstd);
    }
}

template <typename TI, typename TO, int LPR, int NV>
__global__ __launch_bounds__(kBlkThreads) void ln_rows_backward_kernel(
    const TO *__restrict__ dout, const TI *__restrict__ x, const float2 *__restrict__ stats,
    const float *__restrict__ gamma, const float *__restrict__ beta, TI *__restrict__ dx, float *__restrict__ part,
    long rows, int C, int gelu) {
    __shared__ float red[8 * kBlkThreads];
    const Lanes<LPR, NV> ln;
    float gm[NV][8], bt[NV][8], dg[NV][8], db[NV][8];
#pragma unroll
    for (int k = 0; k < NV; k++)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int c = ln.chan(k) + i;
            gm[k][i] = c < C ? gamma[c] : 0.f, bt[k][i] = c < C ? beta[c] : 0.f;
            dg[k][i] = db[k][i] = 0.f;
        }
    const long step = (long)gridDim.x * ln.ROWS;
    for (long r0 = (long)blockIdx.x * ln.ROWS; r0 < rows; r0 += step) {
        const long r = r0 + ln.slot;
        const bool row = r < rows;
        const float2 st = row ? stats[r] : make_float2(0.f, 0.f);
        float h[NV][8], g[NV][8], s1 = 0.f, s2 = 0.f;
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const bool ok = row && ln.chan(k) < C;
            if (ok) load8(x + r * C + ln.chan(k), h[k]), load8(dout + r * C + ln.chan(k), g[k]);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                if (!ok) h[k][i] = st.x, g[k][i] = 0.f;
                h[k][i] = (h[k][i] - st.x) * st.y;
                if ((gelu & ROWS_GELU) && ok) {
                    float u = __builtin_fmaf(h[k][i], gm[k][i], bt[k][i]);
                    if (gelu & ROWS_ROUNDED) u = rounded<TO>(u);
                    // (a gradient that stays in 32 bits takes erff's slope)
                    g[k][i] *= sizeof(TO) == 2 && (gelu & ROWS_ROUNDED) ? gelu_slope_rounded(u) : blk_gelu_slope(u);
                    if (gelu & ROWS_ROUNDED) g[k][i] = rounded<TO>(g[k][i]);
                }
                dg[k][i] = __builtin_fmaf(g[k][i], h[k][i], dg[k][i]);
                db[k][i] += g[k][i];
                g[k][i] *= gm[k][i];
                s1 += g[k][i];
                s2 = __builtin_fmaf(g[k][i], h[k][i], s2);
            }
        }
        s1 = group_total<LPR>(s1) / (float)C;
        s2 = group_total<LPR>(s2) / (float)C;
#pragma unroll
        for (int k = 0; k < NV; k++)
            if (row && ln.chan(k) < C) {
                float o[8];
#pragma unroll
                for (int i = 0; i < 8; i++) o[i] = st.y * (g[k][i] - s1 - h[k][i] * s2);
                store8(dx + r * C + ln.chan(k), o);
            }
    }
    write_param_partials<LPR, NV>(dg, db, C, red, part);
}

// ------------------------------------------------------------------------------------------------- quads
// LayerNorm over the channels of planes.  A lane holds eight channels of four pixels: eight runs of the planes on one
// side, four runs of eight channels (16 bytes and more) on the other, so the transposition is the order of the registers
// and LDS only carries the sums over channels from wave to wave.  A wave covers 64 channels x 32 pixels: 64-byte pieces and longer
// both ways.  Neighbouring tiles stay on one XCD (they share the lines at their edges).
//
// The four pixels are neighbours (their index m runs over the images' pixels), or a 2 x 2 patch of a
// downsampling layer (m = 4 * patch + pixel; out is [patch][C][2][2], the operand of that 2 x 2 convolution of stride 2
// as a product with its weights as they lie, models/convnext.py:548-553).
//
// Memory bounds it from a few thousand pixels on, latency below.  Through LDS tiles of [C][pixels], value by value (before) / so,
// us: forward bf16 128 x 96 x 56 x 56 57 / 28 (5.6 TB/s), 128 x 384 x 14 x 14 25 / 12, 128 x 768 x 7 x 7 36 / 13, fp32 to bf16
// 64 x 512 x 14 x 14 24 / 9.5; patches of 128 x 96 x 56 x 56 72 / 37.  Backward with the parameter sums, fp32 stream: 64 x 512 x
// 14 x 14 42 / 22, 64 x 128 x 56 x 56 64 / 49; above 512 channels the 1024 threads have 128 registers each, which spills: 64
// x 1024 x 7 x 7 40 / 43.
enum { QUAD_RUN, QUAD_SINGLE, QUAD_PATCH, QUAD_PATCH_SINGLE };  // four pixels by one load, by four; patches by two, by four

struct BlkQuads {
    int C, HW, H, W;
    int wc, pt;        // waves across the channels, tiles of 32 pixels per workgroup
    int per;           // workgroup tiles per XCD
    unsigned M;        // pixels (in patches)
};

// places of the four pixels m .. m + 3 in channel `chan` of their image (a tensor has fewer than 2^31 values)
template <int MODE>
struct QuadAt {
    static constexpr int RUNS = MODE == QUAD_RUN ? 1 : MODE == QUAD_PATCH ? 2 : 4;
    unsigned at[RUNS];
    __device__ __forceinline__ QuadAt(const BlkQuads &t, unsigned m, int chan) {
        if constexpr (MODE == QUAD_RUN || MODE == QUAD_SINGLE) {
#pragma unroll
            for (int e = 0; e < RUNS; e++) {
                const unsigned img = (m + e) / (unsigned)t.HW;
                at[e] = (img * t.C + chan) * t.HW + (m + e - img * t.HW);
            }
        } else {
            const unsigned w2 = (unsigned)t.W / 2, h2 = (unsigned)t.H / 2, k = m / 4;
            const unsigned row = k / w2, img = row / h2;
            const unsigned o = (img * t.C + chan) * t.HW + (row - img * h2) * 2 * t.W + (k - row * w2) * 2;
            if constexpr (MODE == QUAD_PATCH) at[0] = o, at[1] = o + t.W;
            else at[0] = o, at[1] = o + 1, at[2] = o + t.W, at[3] = o + t.W + 1;
        }
    }
    // the addresses made from these are made again where they are used next, instead of being kept in registers
    __device__ __forceinline__ void forget() {
#pragma unroll
        for (int e = 0; e < RUNS; e++) asm volatile("" : "+v"(at[e]));
    }
};
// two neighbouring values
template <typename T>
__device__ __forceinline__ void store_pair(T *p, float a, float b) {
    if constexpr (sizeof(T) == 4) *reinterpret_cast<blk_f2 *>(p) = blk_f2{a, b};
    else *reinterpret_cast<unsigned *>(p) = pack2<T>(a, b);
}
// N neighbouring values as they lie in memory
template <typename T, int N>
struct RawRun {
    static constexpr int WORDS = N * (int)sizeof(T) / 4;
    typedef unsigned vec __attribute__((ext_vector_type(WORDS < 4 ? WORDS : 4)));
    unsigned w[WORDS];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int k = 0; k < WORDS; k++) w[k] = 0u;
    }
    // L of them, from value `at` on
    template <int L>
    __device__ __forceinline__ void load(const T *p, int at) {
        constexpr int n = L * (int)sizeof(T) / 4;
        if constexpr (n == 0) w[at / 2] |= (unsigned)__builtin_bit_cast(uint16_t, *p) << (16 * (at % 2));
        else if constexpr (n == 1) w[at * (int)sizeof(T) / 4] = *reinterpret_cast<const unsigned *>(p);
        else if constexpr (n == 2) {
            const blk_u2 v = *reinterpret_cast<const blk_u2 *>(p);
            w[at * (int)sizeof(T) / 4] = v[0], w[at * (int)sizeof(T) / 4 + 1] = v[1];
        } else {
#pragma unroll
            for (int k = 0; k < n / 4; k++) {
                const blk_u4 v = reinterpret_cast<const blk_u4 *>(p)[k];
#pragma unroll
                for (int j = 0; j < 4; j++) w[4 * k + j] = v[j];
            }
        }
    }
    __device__ __forceinline__ float get(int i) const {
        if constexpr (sizeof(T) == 4) return __builtin_bit_cast(float, w[i]);
        else return to_float(__builtin_bit_cast(T, (uint16_t)(w[i / 2] >> (16 * (i % 2)))));
    }
    // what was made of these values is made again, instead of being kept in registers beside them
    __device__ __forceinline__ void forget() {
#pragma unroll
        for (int k = 0; k < WORDS; k++) asm volatile("" : "+v"(w[k]));
    }
};
// eight channels (planes HW apart) of four pixels, of which `live` exist (all or none but for QUAD_SINGLE)
template <int MODE, typename T>
struct QuadPlanes {
    RawRun<T, 4> run[8];
    __device__ __forceinline__ void load(const T *x, const QuadAt<MODE> &q, int HW, int live) {
#pragma unroll
        for (int i = 0; i < 8; i++) run[i].clear();
        if (live == 0) return;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const T *xi = x + (size_t)i * HW;  // (uniform)
            if constexpr (MODE == QUAD_RUN) {
                run[i].template load<4>(xi + q.at[0], 0);
            } else if constexpr (MODE == QUAD_PATCH) {
                run[i].template load<2>(xi + q.at[0], 0), run[i].template load<2>(xi + q.at[1], 2);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (MODE == QUAD_PATCH_SINGLE || e < live) run[i].template load<1>(xi + q.at[e], e);
            }
        }
    }
    __device__ __forceinline__ float get(int i, int e) const { return run[i].get(e); }
    __device__ __forceinline__ void forget() {
#pragma unroll
        for (int i = 0; i < 8; i++) run[i].forget();
    }
};
// the same values as rows: [m][C], or [patch][C][4]
template <int MODE, typename T>
struct QuadRows {
    static constexpr bool PATCHES = MODE == QUAD_PATCH || MODE == QUAD_PATCH_SINGLE;
    RawRun<T, 8> piece[4];  // a pixel's eight channels; two channels' four pixels
    __device__ __forceinline__ void load(const T *rows, unsigned m, int chan, int C, int live) {
#pragma unroll
        for (int k = 0; k < 4; k++) piece[k].clear();
        if (live == 0) return;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (MODE != QUAD_SINGLE || k < live)
                piece[k].template load<8>(PATCHES ? rows + ((size_t)(m / 4) * C + chan + 2 * k) * 4
                                                  : rows + (size_t)(m + k) * C + chan, 0);
        }
    }
    __device__ __forceinline__ float get(int i, int e) const {
        return PATCHES ? piece[i / 2].get(i % 2 * 4 + e) : piece[e].get(i);
    }
    __device__ __forceinline__ void forget() {
#pragma unroll
        for (int k = 0; k < 4; k++) piece[k].forget();
    }
};
template <int MODE, typename T>
__device__ __forceinline__ void quad_store(T *x, const QuadAt<MODE> &q, int HW, int live, const float (&v)[8][4]) {
    if (live == 0) return;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        T *xi = x + (size_t)i * HW;
        if constexpr (MODE == QUAD_RUN) {
            store_run<T, 4>(xi + q.at[0], v[i]);
        } else if constexpr (MODE == QUAD_PATCH) {
            store_pair(xi + q.at[0], v[i][0], v[i][1]), store_pair(xi + q.at[1], v[i][2], v[i][3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (MODE == QUAD_PATCH_SINGLE || e < live) xi[q.at[e]] = from_float<T>(v[i][e]);
        }
    }
}
template <int MODE, typename T>
__device__ __forceinline__ void quad_store_rows(T *rows, unsigned m, int chan, int C, int live, const float (&v)[8][4]) {
    if (live == 0) return;
    if constexpr (MODE == QUAD_RUN || MODE == QUAD_SINGLE) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float o[8];
#pragma unroll
            for (int i = 0; i < 8; i++) o[i] = v[i][e];
            if (MODE == QUAD_RUN || e < live) store8(rows + (size_t)(m + e) * C + chan, o);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
            float o[8];
#pragma unroll
            for (int e = 0; e < 8; e++) o[e] = v[i + e / 4][e % 4];
            store8(rows + (size_t)(m / 4) * C * 4 + (chan + i) * 4, o);
        }
    }
}

// Lane: pixels 4 * (lane % 8) .. of the wave's 32, channels 8 * (lane / 8) .. of its 64
struct QuadLane {
    int wave, wch, wp, pq, chan, step;  // step: pixels per workgroup tile
    __device__ __forceinline__ QuadLane(const BlkQuads &t)
        : wave(threadIdx.x >> 6), wch(wave % t.wc), wp(wave / t.wc), pq(threadIdx.x % 8),
          chan(wch * 64 + (int)(threadIdx.x >> 3 & 7) * 8), step(32 * t.pt) {}
    // pixel of tile `tile`
    __device__ __forceinline__ unsigned pixel(int tile) const { return (unsigned)tile * step + wp * 32 + pq * 4; }
    // pixels that exist, 0 beyond the channels
    __device__ __forceinline__ int live(const BlkQuads &t, unsigned m) const {
        return chan < t.C && m < t.M ? (int)min(4u, t.M - m) : 0;
    }
    // this wave's sums over its channels go to red, [wave][32]
    __device__ __forceinline__ void give(float *red, float (&s)[4]) const {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            s[e] = dpp_add<0x128>(s[e]);  // row_ror:8
            s[e] += __shfl_xor(s[e], 16, 64);
            s[e] += __shfl_xor(s[e], 32, 64);
        }
        if ((threadIdx.x & 63) < 8) *reinterpret_cast<blk_f4 *>(red + wave * 32 + pq * 4) = blk_f4{s[0], s[1], s[2], s[3]};
    }
    __device__ __forceinline__ void take(const float *red, const BlkQuads &t, float (&s)[4]) const {
        blk_f4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
        for (int w = 0; w < t.wc; w++) v += *reinterpret_cast<const blk_f4 *>(red + (wp * t.wc + w) * 32 + pq * 4);
#pragma unroll
        for (int e = 0; e < 4; e++) s[e] = v[e];
    }
};

template <typename TI, typename TO, int MODE, int THREADS>
__global__ __launch_bounds__(THREADS) void ln_quad_kernel(const TI *__restrict__ x, const float *__restrict__ gamma,
                                                          const float *__restrict__ beta, TO *__restrict__ out,
                                                          float2 *__restrict__ stats, BlkQuads t, float eps) {
    __shared__ __attribute__((aligned(16))) float red[2][THREADS / 64 * 32];
    const QuadLane ln(t);
    const int tile = blockIdx.x % 8 * t.per + blockIdx.x / 8;
    const unsigned m = ln.pixel(tile);
    if (m - ln.pq * 4 - ln.wp * 32 >= t.M) return;  // (the whole workgroup)
    const int live = ln.live(t, m);
    float v[8][4], mean[4], rstd[4];
    QuadPlanes<MODE, TI> in;
    in.load(x, QuadAt<MODE>(t, m, ln.chan), t.HW, live);
    float gm[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, bt[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (ln.chan < t.C)
#pragma unroll
        for (int i = 0; i < 8; i++) gm[i] = gamma[ln.chan + i], bt[i] = beta[ln.chan + i];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        mean[e] = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) v[i][e] = in.get(i, e), mean[e] += v[i][e];
    }
    ln.give(red[0], mean);
    __syncthreads();
    ln.take(red[0], t, mean);
#pragma unroll
    for (int e = 0; e < 4; e++) {
        mean[e] /= (float)t.C;
        rstd[e] = 0.f;
        if (e < live)
#pragma unroll
            for (int i = 0; i < 8; i++) v[i][e] -= mean[e], rstd[e] = __builtin_fmaf(v[i][e], v[i][e], rstd[e]);
    }
    ln.give(red[1], rstd);
    __syncthreads();
    ln.take(red[1], t, rstd);
#pragma unroll
    for (int e = 0; e < 4; e++) {
        rstd[e] = rsqrtf(rstd[e] / (float)t.C + eps);
#pragma unroll
        for (int i = 0; i < 8; i++) v[i][e] = __builtin_fmaf(v[i][e] * rstd[e], gm[i], bt[i]);
        if (stats != nullptr && ln.chan == 0 && e < live) stats[m + e] = make_float2(mean[e], rstd[e]);
    }
    quad_store_rows<MODE>(out, m, ln.chan, t.C, live, v);
}

// part: [workgroups][2][C].  The tensors' own values stay in registers over the barrier, not the floats made of them.
template <typename TI, typename TO, int MODE, int THREADS>
__global__ __launch_bounds__(THREADS) void ln_quad_backward_kernel(
    const TO *__restrict__ dout, const TI *__restrict__ x, const float2 *__restrict__ stats,
    const float *__restrict__ gamma, TI *__restrict__ dx, float *__restrict__ part, BlkQuads t) {
    __shared__ __attribute__((aligned(16))) float red[2][2][THREADS / 64 * 32];
    const QuadLane ln(t);
    float gm[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, dg[8], db[8];
    if (ln.chan < t.C)
#pragma unroll
        for (int i = 0; i < 8; i++) gm[i] = gamma[ln.chan + i];
#pragma unroll
    for (int i = 0; i < 8; i++) dg[i] = db[i] = 0.f;
    int turn = 0;
    // (the sums of a turn are read before the barrier of the next one, and written again after it)
    for (int k = blockIdx.x / 8; k < t.per; k += gridDim.x / 8, turn ^= 1) {
        const unsigned m = ln.pixel(blockIdx.x % 8 * t.per + k);
        if (m - ln.pq * 4 - ln.wp * 32 >= t.M) break;  // (the whole workgroup)
        const int live = ln.live(t, m);
        QuadAt<MODE> at(t, m, ln.chan);
        QuadPlanes<MODE, TI> xs;
        QuadRows<MODE, TO> gs;
        xs.load(x, at, t.HW, live), gs.load(dout, m, ln.chan, t.C, live);
        float s1[4], s2[4];
        float2 st[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            st[e] = e < live ? stats[m + e] : make_float2(0.f, 0.f), s1[e] = s2[e] = 0.f;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float g = gs.get(i, e), h = (xs.get(i, e) - st[e].x) * st[e].y, v = g * gm[i];
                dg[i] = __builtin_fmaf(g, h, dg[i]);
                db[i] += g;
                s1[e] += v;
                s2[e] = __builtin_fmaf(v, h, s2[e]);
            }
            __builtin_amdgcn_sched_barrier(0);  // (a pixel's floats are gone before the next one's are made)
        }
        ln.give(red[turn][0], s1), ln.give(red[turn][1], s2);
        __syncthreads();
        at.forget(), xs.forget(), gs.forget();
        ln.take(red[turn][0], t, s1), ln.take(red[turn][1], t, s2);
        float o[8][4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            s1[e] /= (float)t.C, s2[e] /= (float)t.C;
#pragma unroll
            for (int i = 0; i < 8; i++)
                o[i][e] = st[e].y * (gs.get(i, e) * gm[i] - s1[e] - (xs.get(i, e) - st[e].x) * st[e].y * s2[e]);
            __builtin_amdgcn_sched_barrier(0);
        }
        quad_store<MODE>(dx, at, t.HW, live, o);
    }
    // the waves of equal channels meet in LDS
#pragma unroll
    for (int i = 0; i < 8; i++) dg[i] = group_total<8>(dg[i]), db[i] = group_total<8>(db[i]);
    __shared__ __attribute__((aligned(16))) float sums[4][2][64];
    if (t.pt > 1) {
        const int l = ln.chan - ln.wch * 64;
        if (ln.pq == 0) store8(&sums[ln.wave][0][l], dg), store8(&sums[ln.wave][1][l], db);
        __syncthreads();
        if (ln.wp == 0 && ln.pq == 0)
            for (int p = 1; p < t.pt; p++) {
                float a[8], b[8];
                load8(&sums[p * t.wc + ln.wch][0][l], a), load8(&sums[p * t.wc + ln.wch][1][l], b);
#pragma unroll
                for (int i = 0; i < 8; i++) dg[i] += a[i], db[i] += b[i];
            }
    }
    if (ln.wp == 0 && ln.pq == 0 && ln.chan < t.C) {
        float *to = part + (size_t)blockIdx.x * 2 * t.C + ln.chan;
        store8(to, dg), store8(to + t.C, db);
    }
}

// ------------------------------------------------------------------------------------------------- tail
// 64 pixels x 64 channels through LDS; thread = (piece of eight channels, pixel), piece threadIdx % 8
constexpr int kTailP = 64, kTailC = 64, kTailPitch = kTailP + 1;

struct TailTiles {
    int C, HW, per, ctiles, units;  // pixel tiles per image, channel tiles, (image, pixel tile) pairs
};

// (TS: the type of res; without res out is y in planes; round: scale * y is rounded to y's type, as a product by itself is)
template <typename TY, typename TS, typename TR, int VEC>
__global__ __launch_bounds__(kBlkThreads) void tail_kernel(const TY *__restrict__ y, const float *__restrict__ scale,
                                                           const TS *__restrict__ res, TR *__restrict__ out,
                                                           TailTiles t, int round) {
    __shared__ float tile[kTailC * kTailPitch];
    const int u = blockIdx.x / t.ctiles, c0 = blockIdx.x % t.ctiles * kTailC;
    const int n = u / t.per, p0 = u % t.per * kTailP, np = min(kTailP, t.HW - p0), nc = min(kTailC, t.C - c0);
    const size_t base = ((size_t)n * t.C + c0) * t.HW + p0;
    constexpr int PER = kTailP / VEC, R = kTailC * PER / kBlkThreads;  // residual runs per thread
    float rs[R][VEC];
    const int c = threadIdx.x % 8 * 8;
    float v[2][8];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int p = threadIdx.x / 8 + 32 * k;
        if (c < nc && p < np) load8(y + ((size_t)n * t.HW + p0 + p) * t.C + c0 + c, v[k]);
    }
#pragma unroll
    for (int k = 0; k < R; k++) {
        const int f = threadIdx.x + k * kBlkThreads, cc = f / PER, p = f % PER * VEC;
#pragma unroll
        for (int e = 0; e < VEC; e++) rs[k][e] = 0.f;
        if (res != nullptr && cc < nc && p < np) load_run<TS, VEC>(res + base + (size_t)cc * t.HW + p, rs[k]);
    }
    float sc[8];
#pragma unroll
    for (int i = 0; i < 8; i++) sc[i] = scale != nullptr && c < nc ? scale[c0 + c + i] : 1.f;
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int p = threadIdx.x / 8 + 32 * k;
        if (c < nc && p < np)
#pragma unroll
            for (int i = 0; i < 8; i++)
                tile[(c + i) * kTailPitch + p] = round ? rounded<TY>(v[k][i] * sc[i]) : v[k][i] * sc[i];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < R; k++) {
        const int f = threadIdx.x + k * kBlkThreads, cc = f / PER, p = f % PER * VEC;
        if (cc < nc && p < np) {
#pragma unroll
            for (int e = 0; e < VEC; e++) rs[k][e] += tile[cc * kTailPitch + p + e];
            store_run<TR, VEC>(out + base + (size_t)cc * t.HW + p, rs[k]);
        }
    }
}

// dy [N,HW,C] = scale * dout, part [groups][C] = sums of dout * y; a workgroup keeps its channel tile (y may be null: no
// sums)
template <typename TY, typename TR, int VEC>
__global__ __launch_bounds__(kBlkThreads) void tail_backward_kernel(const TR *__restrict__ dout,
                                                                    const TY *__restrict__ y,
                                                                    const float *__restrict__ scale,
                                                                    TY *__restrict__ dy, float *__restrict__ part,
                                                                    TailTiles t) {
    __shared__ float tile[kTailC * kTailPitch];
    const int c0 = blockIdx.x % t.ctiles * kTailC, nc = min(kTailC, t.C - c0);
    const int group = blockIdx.x / t.ctiles, groups = gridDim.x / t.ctiles;
    const int c = threadIdx.x % 8 * 8;
    float sc[8], ds[8];
#pragma unroll
    for (int i = 0; i < 8; i++) sc[i] = scale != nullptr && c < nc ? scale[c0 + c + i] : 1.f, ds[i] = 0.f;
    constexpr int PER = kTailP / VEC, R = kTailC * PER / kBlkThreads;
    for (int u = group; u < t.units; u += groups) {
        const int n = u / t.per, p0 = u % t.per * kTailP, np = min(kTailP, t.HW - p0);
        const size_t base = ((size_t)n * t.C + c0) * t.HW + p0;
        float v[R][VEC], yv[2][8];
#pragma unroll
        for (int k = 0; k < R; k++) {
            const int f = threadIdx.x + k * kBlkThreads, cc = f / PER, p = f % PER * VEC;
            if (cc < nc && p < np) load_run<TR, VEC>(dout + base + (size_t)cc * t.HW + p, v[k]);
        }
        const size_t row = ((size_t)n * t.HW + p0) * t.C + c0 + c;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int p = threadIdx.x / 8 + 32 * k;
            if (y != nullptr && c < nc && p < np) load8(y + row + (size_t)p * t.C, yv[k]);
            else
#pragma unroll
                for (int i = 0; i < 8; i++) yv[k][i] = 0.f;
        }
        __syncthreads();  // the tile's last readers are done
#pragma unroll
        for (int k = 0; k < R; k++) {
            const int f = threadIdx.x + k * kBlkThreads, cc = f / PER, p = f % PER * VEC;
            if (cc < nc && p < np)
#pragma unroll
                for (int e = 0; e < VEC; e++) tile[cc * kTailPitch + p + e] = v[k][e];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int p = threadIdx.x / 8 + 32 * k;
            if (c < nc && p < np) {
                float o[8];
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float g = tile[(c + i) * kTailPitch + p];
                    ds[i] = __builtin_fmaf(g, yv[k][i], ds[i]);
                    o[i] = g * sc[i];
                }
                store8(dy + row + (size_t)p * t.C, o);
            }
        }
    }
    if (y == nullptr) return;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; i++) tile[i * kBlkThreads + threadIdx.x] = ds[i];
    __syncthreads();
    if (threadIdx.x < nc) {  // channel threadIdx: value threadIdx % 8 of piece threadIdx / 8
        float s = 0.f;
#pragma unroll
        for (int r = 0; r < kBlkThreads / 8; r++) s += tile[threadIdx.x % 8 * kBlkThreads + r * 8 + threadIdx.x / 8];
        part[(size_t)group * t.C + c0 + threadIdx.x] = s;
    }
}

}  // namespace dwo
