// Both pointwise layers of a block at inference as one kernel (models/convnext.py:306-318), 16-bit types:
//   out[n][c][p] = res[n][c][p] + scale[c] * (b2[c] + sum_j w2[c][j] * gelu(b1[j] + sum_k w1[j][k] * x[n][p][k]))
// for x [N,HW,C] (normalised), 4 C hidden channels, planes out: the hidden tensor, four times the size of the others, never exists.
//
// A wave owns 16 PF pixels: their C inputs as fragments in registers, their C sums in registers.  It walks the hidden
// channels in steps of 32: H^T = W1 X^T leaves a lane with eight hidden channels of one pixel, after GELU
// and rounding that is, as it stands, the operand of Y^T += W2 H^T (the rows of W1 are dealt to LDS slots so that they
// are eight neighbours): nothing passes through LDS or between lanes.  The weights of a step travel to LDS
// while the previous ones are used and are shared by the waves; 16 PF is what leaves two waves per SIMD, so that one's
// GELU runs under the other's matrix instructions.
//
// What bounds it, by counters: at C = 96 the vector instructions, mostly of GELU (16 issue slots per hidden value), 66 % of the time
// (matrix cores 19 %, LDS 27 %); the share falls to 40 % at 192 and 29 % at 384, where the LDS reads of the weights, which
// eight waves of 16 pixels share, lead with 39 % and no unit is busy for half the time.  us, bf16, two product kernels / this
// one: 401408 x 96 269 / 113, 100352 x 192 159 / 105, 25088 x 384 119 / 100; slower from C = 512 (spills) and where its
// workgroups of 128 pixels are few (its chain is 4 C / 32 steps of 1.5 to 1.9 us: 12544 x 384 60 / 90).  Tried: at 384 four waves
// of 32 pixels, half the LDS reads (one wave per SIMD overlaps nothing, 98 / 205); GELU of a step under the first products of the
// next one, same sums (48 registers more: at 96 two waves per SIMD instead of three, 113 / 134, from 192 on spills, twice the time).
#pragma once

#include "dwo_linear.h"

namespace dwo {

template <typename T>
struct MlpArgs {
    const T *x, *w1, *b1, *w2, *b2, *scale, *res;
    T *out;
    long M;
    int HW, vec;  // pixels per plane; values per access of a plane: 8, 4 or 1
};

template <int C>
struct Mlp {
    static constexpr int PF = C <= 192 ? 2 : 1, WAVES = C <= 192 ? 4 : 8;
    static constexpr int THREADS = 64 * WAVES, PIXELS = 16 * PF * WAVES, HIDDEN = 4 * C;
    static constexpr int LOADS = (C / 16 + WAVES - 1) / WAVES;  // of 1 KB per wave, operand and step
    // rows of C values in LDS: the 16-byte pieces of a row are permuted so that the sixteen rows of a fragment meet on all banks
    static constexpr int RB = C * 2 / 4 % 64;  // banks from row to row
    static __device__ __forceinline__ int swizzle(int s) {
        if constexpr (RB == 0) return s & 15;
        else if constexpr (RB == 32) return s >> 1 & 7;
        else return s >> 2 & 3;
    }
    static_assert(C % 32 == 0 && (RB == 0 || RB == 32 || RB == 48 || RB == 16), "a permutation for this row length");
    static_assert(C / 8 % (RB == 0 ? 16 : RB == 32 ? 8 : 4) == 0, "it stays inside the row");
};

template <typename T, int C>
__global__ __launch_bounds__(Mlp<C>::THREADS, 2) void mlp_kernel(MlpArgs<T> a) {
    using G = Mlp<C>;
    constexpr int PF = G::PF, KS = C / 32, NB = C / 16, LOADS = G::LOADS;
    // two buffers of the weights of 32 hidden channels; afterwards the waves' output pixels
    __shared__ __attribute__((aligned(16))) uint16_t w1a[32 * C];
    __shared__ __attribute__((aligned(16))) uint16_t w2a[32 * C];
    __shared__ __attribute__((aligned(16))) uint16_t w1b[32 * C];
    __shared__ __attribute__((aligned(16))) uint16_t w2b[32 * C];
    __shared__ __attribute__((aligned(16))) uint16_t bias1[G::HIDDEN];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    const long m0 = (long)blockIdx.x * G::PIXELS + wave * 16 * PF;
    // this lane's pieces of the weights
    const __amdgpu_buffer_rsrc_t r1 =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(a.w1), 0, G::HIDDEN * C * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t r2 =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(a.w2), 0, G::HIDDEN * C * 2, 0x00020000);
    unsigned o1[LOADS], o2[LOADS];
#pragma unroll
    for (int u = 0; u < LOADS; u++) {
        const int f = (wave + u * G::WAVES) * 64 + lane;
        const int s = f / (C / 8), p = (f % (C / 8)) ^ G::swizzle(s);
        const int row = (s >> 2 & 3) * 8 + (s >> 4 & 1) * 4 + (s & 3);  // slot 16 i + 4 g + r: hidden channel 8 g + 4 i + r
        o1[u] = (unsigned)(row * C * 2 + p * 16);
        const int n = f / 4, q = (f % 4) ^ (n >> 2 & 3);
        o2[u] = (unsigned)(n * G::HIDDEN * 2 + q * 16);
    }
    auto load = [&](uint16_t *l1, uint16_t *l2, int h0) {
        typedef __attribute__((address_space(3))) void lds_void;
#pragma unroll
        for (int u = 0; u < LOADS; u++) {
            const int k = wave + u * G::WAVES;
            if (k >= C / 16) break;  // (uniform)
#ifdef __HIP_DEVICE_COMPILE__
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r1, (lds_void *)(l1 + k * 512), 16, o1[u], h0 * C * 2, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r2, (lds_void *)(l2 + k * 512), 16, o2[u], h0 * 2, 0, 0);
#endif
        }
    };
    load(w1a, w2a, 0);
    for (int f = threadIdx.x; f < G::HIDDEN / 8; f += G::THREADS)
        reinterpret_cast<mma_u4 *>(bias1)[f] = reinterpret_cast<const mma_u4 *>(a.b1)[f];
    // the pixels' inputs, zeros beyond the last
    mma_s8 fx[KS][PF];
    {
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<T *>(a.x + m0 * C), 0, (unsigned)min(max(a.M - m0, 0L) * C * 2, 0x7fffffffL), 0x00020000);
#pragma unroll
        for (int p = 0; p < PF; p++)
#pragma unroll
            for (int k = 0; k < KS; k++)
                fx[k][p] = __builtin_bit_cast(mma_s8, __builtin_amdgcn_raw_buffer_load_b128(
                                                          rx, (16 * p + c) * C * 2 + k * 64 + g * 16, 0, 0));
    }
    mma_f4 y[NB][PF];
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
        for (int p = 0; p < PF; p++) y[n][p] = mma_f4{0.f, 0.f, 0.f, 0.f};
    auto first = [&](const uint16_t *l1, int k, int i) {
        const int s = 16 * i + c;
        return *reinterpret_cast<const mma_s8 *>(l1 + s * C + ((k * 4 + g) ^ G::swizzle(s)) * 8);
    };
    auto second = [&](const uint16_t *l2, int n) {
        const int s = 16 * n + c;
        return *reinterpret_cast<const mma_s8 *>(l2 + s * 32 + (g ^ (s >> 2 & 3)) * 8);
    };
    // fragments in flight ahead of the products that use them
    constexpr int D1 = 6 < 2 * KS ? 6 : 2 * KS, D2 = 6 < NB ? 6 : NB;
    auto step = [&](const uint16_t *l1, const uint16_t *l2, int h0) {
        mma_f4 h[2][PF];
        const mma_u4 b = *reinterpret_cast<const mma_u4 *>(bias1 + h0 + 8 * g);
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int p = 0; p < PF; p++)
#pragma unroll
                for (int r = 0; r < 4; r++) h[i][p][r] = lin_value<T>(b[2 * i + r / 2], r % 2);
        mma_s8 f1[2 * KS];
#pragma unroll
        for (int k = 0; k < 2 * KS; k++) f1[k] = first(l1, k / 2, k % 2);
#pragma unroll
        for (int k = 0; k < 2 * KS; k++)
#pragma unroll
            for (int p = 0; p < PF; p++) h[k % 2][p] = Mma<T>::run(f1[k], fx[k / 2][p], h[k % 2][p]);
        __builtin_amdgcn_sched_group_barrier(0x100, 1 + D1, 0);
#pragma unroll
        for (int k = 0; k < 2 * KS - D1; k++) {
            __builtin_amdgcn_sched_group_barrier(0x008, PF, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, D1 * PF, 0);
        __builtin_amdgcn_sched_barrier(0);
        mma_s8 f2[NB];
#pragma unroll
        for (int n = 0; n < D2; n++) f2[n] = second(l2, n);
        __builtin_amdgcn_sched_barrier(0);
        mma_s8 hb[PF];
#pragma unroll
        for (int p = 0; p < PF; p++) {
            mma_u4 v;
#pragma unroll
            for (int e = 0; e < 4; e++)
                v[e] = lin_pack<T>(lin_gelu(h[e / 2][p][2 * e % 4]), lin_gelu(h[e / 2][p][2 * e % 4 + 1]));
            hb[p] = __builtin_bit_cast(mma_s8, v);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = D2; n < NB; n++) f2[n] = second(l2, n);
#pragma unroll
        for (int n = 0; n < NB; n++)
#pragma unroll
            for (int p = 0; p < PF; p++) y[n][p] = Mma<T>::run(f2[n], hb[p], y[n][p]);
#pragma unroll
        for (int n = 0; n < NB - D2; n++) {
            __builtin_amdgcn_sched_group_barrier(0x008, PF, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, D2 * PF, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int h0 = 0; h0 < G::HIDDEN; h0 += 64) {
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's pieces are there ..
        __syncthreads();                     // .. and the other waves'; nobody reads the other buffer any more
        load(w1b, w2b, h0 + 32);
        step(w1a, w2a, h0);
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
        if (h0 + 64 < G::HIDDEN) load(w1a, w2a, h0 + 64);
        step(w1b, w2b, h0 + 32);
    }
    __syncthreads();
    // the wave's pixels as [C][16 PF] values in LDS: residual in, sums on top, out as runs of pixels
    constexpr int RUN = 16 * PF, PER = G::WAVES / 4;
    const int quarter = wave / PER;
    uint16_t *mine = (quarter == 0 ? w1a : quarter == 1 ? w2a : quarter == 2 ? w1b : w2b) + wave % PER * C * RUN;
    auto planes = [&](auto vec, auto in) {
        constexpr int V = decltype(vec)::value, CH = RUN / V;
        for (int f = lane; f < C * CH; f += 64) {
            const int n = f / CH, q = f % CH * V;
            const long m = m0 + q;
            if (m >= a.M) continue;
            const long img = (unsigned)m / (unsigned)a.HW;
            const size_t at = ((size_t)img * C + n) * a.HW + (m - img * a.HW);
            uint16_t *l = mine + n * RUN + q;
            if constexpr (decltype(in)::value) {
                if constexpr (V == 8) *reinterpret_cast<mma_u4 *>(l) = *reinterpret_cast<const mma_u4 *>(a.res + at);
                else if constexpr (V == 4) *reinterpret_cast<mma_u2 *>(l) = *reinterpret_cast<const mma_u2 *>(a.res + at);
                else *l = __builtin_bit_cast(uint16_t, a.res[at]);
            } else {
                if constexpr (V == 8) *reinterpret_cast<mma_u4 *>(a.out + at) = *reinterpret_cast<const mma_u4 *>(l);
                else if constexpr (V == 4) *reinterpret_cast<mma_u2 *>(a.out + at) = *reinterpret_cast<const mma_u2 *>(l);
                else a.out[at] = __builtin_bit_cast(T, *l);
            }
        }
    };
    auto move = [&](auto in) {
        if (a.vec == 8) planes(std::integral_constant<int, 8>{}, in);
        else if (a.vec == 4) planes(std::integral_constant<int, 4>{}, in);
        else planes(std::integral_constant<int, 1>{}, in);
    };
    move(std::true_type{});
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int ch = 16 * n + 4 * g + r;
            const float b = to_float(a.b2[ch]), s = a.scale != nullptr ? to_float(a.scale[ch]) : 1.f;
#pragma unroll
            for (int p = 0; p < PF; p++) {
                uint16_t *l = mine + ch * RUN + 16 * p + c;
                *l = __builtin_bit_cast(
                    uint16_t, from_float<T>(__builtin_fmaf(y[n][p][r] + b, s, to_float(__builtin_bit_cast(T, *l)))));
            }
        }
    __syncthreads();
    move(std::false_type{});
}

template <typename T, int C>
int launch_mlp(const MlpArgs<T> &a, hipStream_t st) {
    using G = Mlp<C>;
    mlp_kernel<T, C><<<dim3((unsigned)((a.M + G::PIXELS - 1) / G::PIXELS)), dim3(G::THREADS), 0, st>>>(a);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}

}  // namespace dwo
