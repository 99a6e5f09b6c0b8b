// What a ConvNeXt-1D block and the stem do around the operator and the pointwise layers when they are
// trained (models/convnext.py:176-190,306-318), forward and backward, each as one pass over its tensors:
//
//   ln_tile     y [N,C,HW] -> LayerNorm over C -> [N,HW,C]        permute + LayerNorm of a block
//   ln_rows     rows of C  -> LayerNorm -> (GELU)                 the stem's
//   ln_patch    y [N,C,H,W] -> LayerNorm over C -> 2 x 2 patches  in front of a downsampling layer
//   tail        res + scale[c] * y, y [N,HW,C] -> [N,C,HW]        layer scale + permute + residual
//
// All of them are bound by memory: PyTorch's compositions move each tensor three to six times (permuted
// copies, conversions, separate parameter gradients) at 0.4 to 2 TB/s.  Input and output have types of their
// own, so the conversions of autocast happen on the way out (fp32 stream, 16-bit pointwise layers).  Channels
// are handled in pieces of eight by groups of 8 to 64 lanes, sums over channels stay inside a group, and
// parameter gradients are kept in registers over all the tiles of a workgroup, written as
// partial sums and added in a fixed order by a second kernel.  Statistics and sums are fp32.
#pragma once

#include "dwo_common.h"

namespace dwo {

constexpr int kBlkThreads = 256, kBlkMaxC = 1024, kBlkGroups = 1024;

typedef unsigned blk_u4 __attribute__((ext_vector_type(4)));
typedef unsigned blk_u2 __attribute__((ext_vector_type(2)));
typedef float blk_f4 __attribute__((ext_vector_type(4)));

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

// Channels of a lane: pieces lane % LPR + k * LPR for k < NV, of which `live` exist.
template <int LPR, int NV>
struct Lanes {
    static constexpr int PER = 64 / LPR;  // rows of channels per wave and step
    int l, slot;                          // place in the group, row within a step of the workgroup
    __device__ __forceinline__ Lanes() : l(threadIdx.x % LPR), slot(threadIdx.x / LPR) {}
    static constexpr int ROWS = kBlkThreads / LPR;  // rows per step of the workgroup
    __device__ __forceinline__ int chan(int k) const { return 8 * (l + k * LPR); }
};

// Sums of a workgroup's lanes of equal channels: [2][C] partial sums per workgroup.
template <int LPR, int NV>
__device__ __forceinline__ void write_param_partials(float (&dg)[NV][8], float (&db)[NV][8], int C, float *red,
                                                     float *part) {
    const Lanes<LPR, NV> ln;
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
// so 32 threads share a column, each with four loads in flight (eight threads one load at a time: 23 us for 1024 groups of 1024 columns, now 8).
constexpr int kColThreads = 1024;
template <typename TO>
__global__ __launch_bounds__(kColThreads) void column_sums_kernel(const float *__restrict__ part, TO *out0, TO *out1,
                                                                  int L, int split, int groups) {
    __shared__ float red[kColThreads];
    const int c = blockIdx.x * 32 + threadIdx.x % 32;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    if (c < L)
        for (int g = threadIdx.x / 32; g < groups; g += 128)
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (g + 32 * u < groups) s[u] += part[(size_t)(g + 32 * u) * L + c];
    red[threadIdx.x] = (s[0] + s[1]) + (s[2] + s[3]);
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
                    g[k][i] *= sizeof(TI) == 2 ? gelu_slope_rounded(u) : blk_gelu_slope(u);
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

// ------------------------------------------------------------------------------------------------- tiles
// P pixels x C channels of an image in LDS as [C][P + 1] values of the tensor's type: four workgroups per CU, but 16
// pixels (whole 64-byte pieces of fp32 rows) while they fit the 64 KB that need no attribute
// Fewer pixels where the tiles would not fill the chip (a single image: the chain of one tile is what counts).
inline int blk_tile_pixels(int C, int esize, long pixels) {
    int p = 64;
    while (p > 16 && (long)C * (p + 1) * esize > 36 * 1024) p >>= 1;
    while (p > 8 && pixels / p < 256) p >>= 1;
    return (long)C * (p + 1) * esize > 64 * 1024 ? 8 : p;
}
inline size_t blk_tile_bytes(int C, int P, int esize) { return ((size_t)C * (P + 1) * esize + 15) / 16 * 16; }

struct BlkTiles {
    int C, HW, P, log2P, per, tiles;  // tiles per image, in all
    int H, W, W2;                     // patches: image extents, patches per row
};

template <typename T, int VEC>
__device__ __forceinline__ void tile_in(const T *xn, T *tile, const BlkTiles &t, int np) {
    const int sh = t.log2P - (VEC == 4 ? 2 : 0), total = t.C << sh;
    constexpr int U = 8;  // loads in flight
    for (int f0 = threadIdx.x; f0 < total; f0 += U * kBlkThreads) {
        float v[U][VEC];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int f = f0 + u * kBlkThreads, c = f >> sh, p = (f - (c << sh)) * VEC;
            if (f < total && p < np) load_run<T, VEC>(xn + (size_t)c * t.HW + p, v[u]);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int f = f0 + u * kBlkThreads, c = f >> sh, p = (f - (c << sh)) * VEC;
            if (f < total && p < np)
#pragma unroll
                for (int e = 0; e < VEC; e++) tile[c * (t.P + 1) + p + e] = from_float<T>(v[u][e]);
        }
    }
}
template <typename T, int VEC>
__device__ __forceinline__ void tile_out(T *xn, const T *tile, const BlkTiles &t, int np) {
    const int sh = t.log2P - (VEC == 4 ? 2 : 0), total = t.C << sh;
    for (int f = threadIdx.x; f < total; f += kBlkThreads) {
        const int c = f >> sh, p = (f - (c << sh)) * VEC;
        if (p >= np) continue;
        float v[VEC];
#pragma unroll
        for (int e = 0; e < VEC; e++) v[e] = to_float(tile[c * (t.P + 1) + p + e]);
        store_run<T, VEC>(xn + (size_t)c * t.HW + p, v);
    }
}

template <typename TI, typename TO, int LPR, int NV, int VEC>
__global__ __launch_bounds__(kBlkThreads) void ln_tile_kernel(const TI *__restrict__ x, const float *__restrict__ gamma,
                                                              const float *__restrict__ beta, TO *__restrict__ out,
                                                              float2 *__restrict__ stats, BlkTiles t, float eps) {
    extern __shared__ float lds_block[];
    TI *tile = reinterpret_cast<TI *>(lds_block);
    const Lanes<LPR, NV> ln;
    const int n = blockIdx.x / t.per, p0 = blockIdx.x % t.per * t.P, np = min(t.P, t.HW - p0);
    tile_in<TI, VEC>(x + (size_t)n * t.C * t.HW + p0, tile, t, np);
    float gm[NV][8], bt[NV][8];
#pragma unroll
    for (int k = 0; k < NV; k++)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int c = ln.chan(k) + i;
            gm[k][i] = c < t.C ? gamma[c] : 0.f, bt[k][i] = c < t.C ? beta[c] : 0.f;
        }
    __syncthreads();
    const long row0 = (long)n * t.HW + p0;
    for (int q0 = 0; q0 < np; q0 += ln.ROWS) {
        const int p = q0 + ln.slot;
        const bool row = p < np;
        float v[NV][8], s = 0.f;
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const bool ok = row && ln.chan(k) < t.C;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                v[k][i] = ok ? to_float(tile[(ln.chan(k) + i) * (t.P + 1) + p]) : 0.f;
                s += v[k][i];
            }
        }
        const float mean = group_total<LPR>(s) / (float)t.C;
        float q = 0.f;
#pragma unroll
        for (int k = 0; k < NV; k++)
            if (ln.chan(k) < t.C)
#pragma unroll
                for (int i = 0; i < 8; i++) v[k][i] -= mean, q = __builtin_fmaf(v[k][i], v[k][i], q);
        const float rstd = rsqrtf(group_total<LPR>(q) / (float)t.C + eps);
        if (!row) continue;
#pragma unroll
        for (int k = 0; k < NV; k++)
            if (ln.chan(k) < t.C) {
                float o[8];
#pragma unroll
                for (int i = 0; i < 8; i++) o[i] = __builtin_fmaf(v[k][i] * rstd, gm[k][i], bt[k][i]);
                store8(out + (row0 + p) * t.C + ln.chan(k), o);
            }
        if (stats != nullptr && ln.l == 0) stats[row0 + p] = make_float2(mean, rstd);
    }
}

template <typename TI, typename TO, int LPR, int NV, int VEC>
__global__ __launch_bounds__(kBlkThreads) void ln_tile_backward_kernel(
    const TO *__restrict__ dout, const TI *__restrict__ x, const float2 *__restrict__ stats,
    const float *__restrict__ gamma, TI *__restrict__ dx, float *__restrict__ part, BlkTiles t) {
    extern __shared__ float lds_block[];
    TI *tile = reinterpret_cast<TI *>(lds_block);
    const Lanes<LPR, NV> ln;
    float gm[NV][8], dg[NV][8], db[NV][8];
#pragma unroll
    for (int k = 0; k < NV; k++)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int c = ln.chan(k) + i;
            gm[k][i] = c < t.C ? gamma[c] : 0.f;
            dg[k][i] = db[k][i] = 0.f;
        }
    for (int u = blockIdx.x; u < t.tiles; u += gridDim.x) {
        const int n = u / t.per, p0 = u % t.per * t.P, np = min(t.P, t.HW - p0);
        const size_t base = (size_t)n * t.C * t.HW + p0;
        const long row0 = (long)n * t.HW + p0;
        __syncthreads();
        tile_in<TI, VEC>(x + base, tile, t, np);
        __syncthreads();
        for (int q0 = 0; q0 < np; q0 += ln.ROWS) {
            const int p = q0 + ln.slot;
            const bool row = p < np;
            const float2 st = row ? stats[row0 + p] : make_float2(0.f, 0.f);
            float h[NV][8], g[NV][8], s1 = 0.f, s2 = 0.f;
#pragma unroll
            for (int k = 0; k < NV; k++) {
                const bool ok = row && ln.chan(k) < t.C;
                if (ok) load8(dout + (row0 + p) * t.C + ln.chan(k), g[k]);
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    h[k][i] = ok ? (to_float(tile[(ln.chan(k) + i) * (t.P + 1) + p]) - st.x) * st.y : 0.f;
                    if (!ok) g[k][i] = 0.f;
                    dg[k][i] = __builtin_fmaf(g[k][i], h[k][i], dg[k][i]);
                    db[k][i] += g[k][i];
                    g[k][i] *= gm[k][i];
                    s1 += g[k][i];
                    s2 = __builtin_fmaf(g[k][i], h[k][i], s2);
                }
            }
            s1 = group_total<LPR>(s1) / (float)t.C;
            s2 = group_total<LPR>(s2) / (float)t.C;
#pragma unroll
            for (int k = 0; k < NV; k++)
                if (row && ln.chan(k) < t.C)
#pragma unroll
                    for (int i = 0; i < 8; i++)
                        tile[(ln.chan(k) + i) * (t.P + 1) + p] =
                            from_float<TI>(st.y * (g[k][i] - s1 - h[k][i] * s2));
        }
        __syncthreads();
        tile_out<TI, VEC>(dx + base, tile, t, np);
    }
    write_param_partials<LPR, NV>(dg, db, t.C, lds_block, part);
}

// ------------------------------------------------------------------------------------------------- patches
// x [N,C,H,W] -> LayerNorm over C -> patches [N,H/2,W/2][C][2][2], the operand of the downsampling 2 x 2 convolution of stride
// 2 as a product with its weights as they lie (models/convnext.py:548-553).  A tile is a run of
// P / 4 patches of one row; a lane holds eight channels of the four pixels of a patch, 32 neighbouring values of the output.
struct PatchTile {
    int n, h, p0, np;  // image, row of patches, first patch, patches
    __device__ __forceinline__ PatchTile(const BlkTiles &t, int u) {
        const int P = t.P / 4, h2 = t.H / 2, row = u / t.per;
        n = row / h2, h = row - n * h2;
        p0 = u % t.per * P, np = min(P, t.W2 - p0);
    }
};
template <typename T, int VEC, bool IN>
__device__ __forceinline__ void patch_move(T *x, T *tile, const BlkTiles &t, const PatchTile &at) {
    const int sh = t.log2P - (VEC == 4 ? 2 : 0), half = t.P / 2 / VEC, total = t.C << sh;
    T *xn = x + (size_t)at.n * t.C * t.HW + (size_t)2 * at.h * t.W + 2 * at.p0;
    constexpr int U = IN ? 8 : 1;
    for (int f0 = threadIdx.x; f0 < total; f0 += U * kBlkThreads) {
        float v[U][VEC];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int f = f0 + u * kBlkThreads, c = f >> sh, k = f - (c << sh), r = k >= half, q = (k - r * half) * VEC;
            if (f >= total || q >= 2 * at.np) continue;
            T *m = xn + (size_t)c * t.HW + r * t.W + q;
            const T *l = tile + c * (t.P + 1) + r * (t.P / 2) + q;
            if constexpr (IN) load_run<T, VEC>(m, v[u]);
            else {
#pragma unroll
                for (int e = 0; e < VEC; e++) v[u][e] = to_float(l[e]);
                store_run<T, VEC>(m, v[u]);
            }
        }
        if constexpr (IN) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int f = f0 + u * kBlkThreads, c = f >> sh, k = f - (c << sh), r = k >= half, q = (k - r * half) * VEC;
                if (f >= total || q >= 2 * at.np) continue;
#pragma unroll
                for (int e = 0; e < VEC; e++) tile[c * (t.P + 1) + r * (t.P / 2) + q + e] = from_float<T>(v[u][e]);
            }
        }
    }
}

template <typename TI, typename TO, int LPR, int NV, int VEC>
__global__ __launch_bounds__(kBlkThreads) void ln_patch_kernel(const TI *__restrict__ x, const float *__restrict__ gamma,
                                                               const float *__restrict__ beta, TO *__restrict__ out,
                                                               float2 *__restrict__ stats, BlkTiles t, float eps) {
    extern __shared__ float lds_block[];
    TI *tile = reinterpret_cast<TI *>(lds_block);
    const Lanes<LPR, NV> ln;
    const PatchTile at(t, blockIdx.x);
    patch_move<TI, VEC, true>(const_cast<TI *>(x), tile, t, at);
    float gm[NV][8], bt[NV][8];
#pragma unroll
    for (int k = 0; k < NV; k++)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int c = ln.chan(k) + i;
            gm[k][i] = c < t.C ? gamma[c] : 0.f, bt[k][i] = c < t.C ? beta[c] : 0.f;
        }
    __syncthreads();
    const size_t first = ((size_t)at.n * (t.H / 2) + at.h) * t.W2 + at.p0;
    for (int q0 = 0; q0 < at.np; q0 += ln.ROWS) {
        const int p = q0 + ln.slot;
        const bool row = p < at.np;
        float v[NV][8][4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const TI *px = tile + q / 2 * (t.P / 2) + 2 * p + q % 2;
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < NV; k++)
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    v[k][i][q] = row && ln.chan(k) < t.C ? to_float(px[(ln.chan(k) + i) * (t.P + 1)]) : 0.f;
                    s += v[k][i][q];
                }
            const float mean = group_total<LPR>(s) / (float)t.C;
            float d = 0.f;
#pragma unroll
            for (int k = 0; k < NV; k++)
                if (ln.chan(k) < t.C)
#pragma unroll
                    for (int i = 0; i < 8; i++) v[k][i][q] -= mean, d = __builtin_fmaf(v[k][i][q], v[k][i][q], d);
            const float rstd = rsqrtf(group_total<LPR>(d) / (float)t.C + eps);
#pragma unroll
            for (int k = 0; k < NV; k++)
#pragma unroll
                for (int i = 0; i < 8; i++) v[k][i][q] = __builtin_fmaf(v[k][i][q] * rstd, gm[k][i], bt[k][i]);
            if (stats != nullptr && row && ln.l == 0) stats[(first + p) * 4 + q] = make_float2(mean, rstd);
        }
        if (!row) continue;
#pragma unroll
        for (int k = 0; k < NV; k++)
            if (ln.chan(k) < t.C)
#pragma unroll
                for (int i = 0; i < 8; i += 2) {
                    float o[8];
#pragma unroll
                    for (int e = 0; e < 8; e++) o[e] = v[k][i + e / 4][e % 4];
                    store8(out + ((first + p) * t.C + ln.chan(k) + i) * 4, o);
                }
    }
}

template <typename TI, typename TO, int LPR, int NV, int VEC>
__global__ __launch_bounds__(kBlkThreads) void ln_patch_backward_kernel(
    const TO *__restrict__ dout, const TI *__restrict__ x, const float2 *__restrict__ stats,
    const float *__restrict__ gamma, TI *__restrict__ dx, float *__restrict__ part, BlkTiles t) {
    extern __shared__ float lds_block[];
    TI *tile = reinterpret_cast<TI *>(lds_block);
    const Lanes<LPR, NV> ln;
    float gm[NV][8], dg[NV][8], db[NV][8];
#pragma unroll
    for (int k = 0; k < NV; k++)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int c = ln.chan(k) + i;
            gm[k][i] = c < t.C ? gamma[c] : 0.f;
            dg[k][i] = db[k][i] = 0.f;
        }
    for (int u = blockIdx.x; u < t.tiles; u += gridDim.x) {
        const PatchTile at(t, u);
        __syncthreads();
        patch_move<TI, VEC, true>(const_cast<TI *>(x), tile, t, at);
        __syncthreads();
        const size_t first = ((size_t)at.n * (t.H / 2) + at.h) * t.W2 + at.p0;
        for (int q0 = 0; q0 < at.np; q0 += ln.ROWS) {
            const int p = q0 + ln.slot;
            const bool row = p < at.np;
            float g[NV][8][4];
#pragma unroll
            for (int k = 0; k < NV; k++)
#pragma unroll
                for (int i = 0; i < 8; i += 2) {
                    float o[8];
                    if (row && ln.chan(k) < t.C) load8(dout + ((first + p) * t.C + ln.chan(k) + i) * 4, o);
#pragma unroll
                    for (int e = 0; e < 8; e++) g[k][i + e / 4][e % 4] = row && ln.chan(k) < t.C ? o[e] : 0.f;
                }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                TI *px = tile + q / 2 * (t.P / 2) + 2 * p + q % 2;
                const float2 st = row ? stats[(first + p) * 4 + q] : make_float2(0.f, 0.f);
                float h[NV][8], s1 = 0.f, s2 = 0.f;
#pragma unroll
                for (int k = 0; k < NV; k++)
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        const bool ok = row && ln.chan(k) < t.C;
                        h[k][i] = ok ? (to_float(px[(ln.chan(k) + i) * (t.P + 1)]) - st.x) * st.y : 0.f;
                        dg[k][i] = __builtin_fmaf(g[k][i][q], h[k][i], dg[k][i]);
                        db[k][i] += g[k][i][q];
                        g[k][i][q] *= gm[k][i];
                        s1 += g[k][i][q];
                        s2 = __builtin_fmaf(g[k][i][q], h[k][i], s2);
                    }
                s1 = group_total<LPR>(s1) / (float)t.C;
                s2 = group_total<LPR>(s2) / (float)t.C;
#pragma unroll
                for (int k = 0; k < NV; k++)
                    if (row && ln.chan(k) < t.C)
#pragma unroll
                        for (int i = 0; i < 8; i++)
                            px[(ln.chan(k) + i) * (t.P + 1)] = from_float<TI>(st.y * (g[k][i][q] - s1 - h[k][i] * s2));
            }
        }
        __syncthreads();
        patch_move<TI, VEC, false>(dx, tile, t, at);
    }
    write_param_partials<LPR, NV>(dg, db, t.C, lds_block, part);
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
