// C entry points of the block's and the stem's training passes.
#include "dwo_block.h"

using namespace dwo;

namespace {

int status() {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? DWO_OK : (int)e;
}

bool channels_ok(int C) { return C >= 8 && C % 8 == 0 && C <= kBlkMaxC; }
bool aligned16(const void *p) { return (uintptr_t)p % 16 == 0; }

// f(LPR, NV) for C channels: the fewest lanes that hold them in one piece of eight each, two above 512
template <class F>
int by_channels(int C, F &&f) {
    using std::integral_constant;
    if (C <= 64) return f(integral_constant<int, 8>{}, integral_constant<int, 1>{});
    if (C <= 128) return f(integral_constant<int, 16>{}, integral_constant<int, 1>{});
    if (C <= 256) return f(integral_constant<int, 32>{}, integral_constant<int, 1>{});
    if (C <= 512) return f(integral_constant<int, 64>{}, integral_constant<int, 1>{});
    return f(integral_constant<int, 64>{}, integral_constant<int, 2>{});
}
template <typename T>
struct Type {
    typedef T type;
};
// f(TI, TO): equal types, or fp32 on one side
template <class F>
int by_types(int in, int out, F &&f) {
    if (in == DWO_F32 && out == DWO_F32) return f(Type<float>{}, Type<float>{});
    if (in == DWO_F32 && out == DWO_BF16) return f(Type<float>{}, Type<bf16_t>{});
    if (in == DWO_F32 && out == DWO_F16) return f(Type<float>{}, Type<f16_t>{});
    if (in == DWO_BF16 && out == DWO_BF16) return f(Type<bf16_t>{}, Type<bf16_t>{});
    if (in == DWO_BF16 && out == DWO_F32) return f(Type<bf16_t>{}, Type<float>{});
    if (in == DWO_F16 && out == DWO_F16) return f(Type<f16_t>{}, Type<f16_t>{});
    if (in == DWO_F16 && out == DWO_F32) return f(Type<f16_t>{}, Type<float>{});
    return DWO_ERR_BAD_DTYPE;
}

int column_sums(const float *part, void *out0, void *out1, int L, int split, int groups, int dtype, hipStream_t st) {
    const dim3 grid((L + 31) / 32), block(kColThreads);
    switch (dtype) {
        case DWO_F32:
            column_sums_kernel<float><<<grid, block, 0, st>>>(part, (float *)out0, (float *)out1, L, split, groups);
            break;
        case DWO_BF16:
            column_sums_kernel<bf16_t><<<grid, block, 0, st>>>(part, (bf16_t *)out0, (bf16_t *)out1, L, split, groups);
            break;
        case DWO_F16:
            column_sums_kernel<f16_t><<<grid, block, 0, st>>>(part, (f16_t *)out0, (f16_t *)out1, L, split, groups);
            break;
        default: return DWO_ERR_BAD_DTYPE;
    }
    return status();
}

bool tile_ok(int N, int C, int H, int W) {
    return N >= 1 && H >= 1 && W >= 1 && channels_ok(C) && (double)N * C * H * W < 2147483648.0;
}
// m runs over `pixels` pixels (in patches: four per patch)
BlkQuads quads_of(int C, int H, int W, long pixels) {
    BlkQuads t{};
    t.C = C, t.HW = H * W, t.H = H, t.W = W, t.M = (unsigned)pixels;
    t.wc = (C + 63) / 64;
    t.pt = t.wc >= 3 ? 1 : 4 / t.wc;  // four waves where that many fit
    t.per = (int)(((pixels + 32 * t.pt - 1) / (32 * t.pt) + 7) / 8);
    return t;
}
// f(MODE, THREADS)
template <class F>
int by_quads(const BlkQuads &t, bool patches, F &&f) {
    using std::integral_constant;
    auto threads = [&](auto mode) {
        if (t.C <= 256) return f(mode, integral_constant<int, 256>{});
        if (t.C <= 512) return f(mode, integral_constant<int, 512>{});
        return f(mode, integral_constant<int, 1024>{});
    };
    if (patches)
        return t.W % 2 == 0 ? threads(integral_constant<int, QUAD_PATCH>{}) : threads(integral_constant<int, QUAD_PATCH_SINGLE>{});
    return t.HW % 4 == 0 ? threads(integral_constant<int, QUAD_RUN>{}) : threads(integral_constant<int, QUAD_SINGLE>{});
}
int ln_quads(const void *x, const float *gamma, const float *beta, void *out, float *stats, const BlkQuads &t, bool patches,
             float eps, int in_dtype, int out_dtype, hipStream_t st) {
    return by_types(in_dtype, out_dtype, [&](auto ti, auto to) {
        using TI = typename decltype(ti)::type;
        using TO = typename decltype(to)::type;
        return by_quads(t, patches, [&](auto mode, auto threads) {
            ln_quad_kernel<TI, TO, decltype(mode)::value, decltype(threads)::value>
                <<<dim3((unsigned)t.per * 8), dim3(64 * t.wc * t.pt), 0, st>>>((const TI *)x, gamma, beta, (TO *)out,
                                                                               (float2 *)stats, t, eps);
            return status();
        });
    });
}
int ln_quads_backward(const void *dout, const void *x, const float *stats, const float *gamma, void *dx, void *dgamma,
                      void *dbeta, float *part, const BlkQuads &t, bool patches, int in_dtype, int out_dtype, int grad_dtype,
                      hipStream_t st) {
    const int grid = 8 * (t.per < kBlkGroups / 8 ? t.per : kBlkGroups / 8);
    const int e = by_types(in_dtype, out_dtype, [&](auto ti, auto to) {
        using TI = typename decltype(ti)::type;
        using TO = typename decltype(to)::type;
        return by_quads(t, patches, [&](auto mode, auto threads) {
            ln_quad_backward_kernel<TI, TO, decltype(mode)::value, decltype(threads)::value>
                <<<dim3(grid), dim3(64 * t.wc * t.pt), 0, st>>>((const TO *)dout, (const TI *)x, (const float2 *)stats, gamma,
                                                                (TI *)dx, part, t);
            return status();
        });
    });
    if (e != DWO_OK) return e;
    return column_sums(part, dgamma, dbeta, 2 * t.C, t.C, grid, grad_dtype, st);
}
TailTiles tail_of(int N, int C, int HW) {
    TailTiles t;
    t.C = C, t.HW = HW, t.per = (HW + kTailP - 1) / kTailP;
    t.ctiles = (C + kTailC - 1) / kTailC, t.units = N * t.per;
    return t;
}
// workgroups that keep parameter sums: four per CU at most
int groups_of(long tasks) { return (int)(tasks < kBlkGroups ? tasks : kBlkGroups); }

}  // namespace

extern "C" {

size_t dwo_block_scratch_bytes(int C) { return (size_t)kBlkGroups * 2 * (C > 0 ? C : 0) * sizeof(float); }

int dwo_ln_rows(const void *x, const float *gamma, const float *beta, void *out, float *stats, size_t rows, int C,
                float eps, int gelu, int in_dtype, int out_dtype, void *stream) {
    if (!x || !gamma || !beta || !out) return DWO_ERR_NULL_POINTER;
    if (rows < 1 || rows > (size_t)1 << 31 || !channels_ok(C) || !aligned16(x) || !aligned16(out)) return DWO_ERR_BAD_SHAPE;
    (void)hipGetLastError();
    return by_types(in_dtype, out_dtype, [&](auto ti, auto to) {
        using TI = typename decltype(ti)::type;
        using TO = typename decltype(to)::type;
        return by_channels(C, [&](auto lpr, auto nv) {
            constexpr int LPR = decltype(lpr)::value, NV = decltype(nv)::value;
            const long steps = ((long)rows + kBlkThreads / LPR - 1) / (kBlkThreads / LPR);
            ln_rows_kernel<TI, TO, LPR, NV><<<dim3((unsigned)(steps < 4096 ? steps : 4096)), dim3(kBlkThreads), 0,
                                              (hipStream_t)stream>>>((const TI *)x, gamma, beta, (TO *)out,
                                                                     (float2 *)stats, (long)rows, C, eps, gelu);
            return status();
        });
    });
}

int dwo_ln_rows_backward(const void *dout, const void *x, const float *stats, const float *gamma, const float *beta,
                         void *dx, void *dgamma, void *dbeta, void *scratch, size_t scratch_bytes, size_t rows, int C,
                         int gelu, int in_dtype, int out_dtype, int grad_dtype, void *stream) {
    if (!dout || !x || !stats || !gamma || !beta || !dx || !scratch) return DWO_ERR_NULL_POINTER;
    if (rows < 1 || rows > (size_t)1 << 31 || !channels_ok(C) || !aligned16(x) || !aligned16(dout) || !aligned16(dx))
        return DWO_ERR_BAD_SHAPE;
    if (scratch_bytes < dwo_block_scratch_bytes(C)) return DWO_ERR_SCRATCH_TOO_SMALL;
    (void)hipGetLastError();
    hipStream_t st = (hipStream_t)stream;
    int groups = 0;
    const int e = by_types(in_dtype, out_dtype, [&](auto ti, auto to) {
        using TI = typename decltype(ti)::type;
        using TO = typename decltype(to)::type;
        return by_channels(C, [&](auto lpr, auto nv) {
            constexpr int LPR = decltype(lpr)::value, NV = decltype(nv)::value;
            groups = groups_of(((long)rows + kBlkThreads / LPR - 1) / (kBlkThreads / LPR));
            ln_rows_backward_kernel<TI, TO, LPR, NV><<<dim3(groups), dim3(kBlkThreads), 0, st>>>(
                (const TO *)dout, (const TI *)x, (const float2 *)stats, gamma, beta, (TI *)dx, (float *)scratch,
                (long)rows, C, gelu);
            return status();
        });
    });
    if (e != DWO_OK) return e;
    return column_sums((const float *)scratch, dgamma, dbeta, 2 * C, C, groups, grad_dtype, st);
}

int dwo_ln_tile(const void *x, const float *gamma, const float *beta, void *out, float *stats, int N, int C, int H,
                int W, float eps, int in_dtype, int out_dtype, void *stream) {
    if (!x || !gamma || !beta || !out) return DWO_ERR_NULL_POINTER;
    if (!tile_ok(N, C, H, W) || !aligned16(x) || !aligned16(out)) return DWO_ERR_BAD_SHAPE;
    (void)hipGetLastError();
    return ln_quads(x, gamma, beta, out, stats, quads_of(C, H, W, (long)N * H * W), false, eps, in_dtype, out_dtype,
                    (hipStream_t)stream);
}

int dwo_ln_tile_backward(const void *dout, const void *x, const float *stats, const float *gamma, void *dx,
                         void *dgamma, void *dbeta, void *scratch, size_t scratch_bytes, int N, int C, int H, int W,
                         int in_dtype, int out_dtype, int grad_dtype, void *stream) {
    if (!dout || !x || !stats || !gamma || !dx || !scratch) return DWO_ERR_NULL_POINTER;
    if (!tile_ok(N, C, H, W) || !aligned16(x) || !aligned16(dout) || !aligned16(dx)) return DWO_ERR_BAD_SHAPE;
    if (scratch_bytes < dwo_block_scratch_bytes(C)) return DWO_ERR_SCRATCH_TOO_SMALL;
    (void)hipGetLastError();
    return ln_quads_backward(dout, x, stats, gamma, dx, dgamma, dbeta, (float *)scratch,
                             quads_of(C, H, W, (long)N * H * W), false, in_dtype, out_dtype, grad_dtype,
                             (hipStream_t)stream);
}

int dwo_ln_patch(const void *x, const float *gamma, const float *beta, void *out, float *stats, int N, int C, int H,
                 int W, float eps, int in_dtype, int out_dtype, void *stream) {
    if (!x || !gamma || !beta || !out) return DWO_ERR_NULL_POINTER;
    if (!tile_ok(N, C, H, W) || H < 2 || W < 2 || !aligned16(x) || !aligned16(out)) return DWO_ERR_BAD_SHAPE;
    (void)hipGetLastError();
    return ln_quads(x, gamma, beta, out, stats, quads_of(C, H, W, (long)N * (H / 2) * (W / 2) * 4), true, eps, in_dtype,
                    out_dtype, (hipStream_t)stream);
}

int dwo_ln_patch_backward(const void *dout, const void *x, const float *stats, const float *gamma, void *dx,
                          void *dgamma, void *dbeta, void *scratch, size_t scratch_bytes, int N, int C, int H, int W,
                          int in_dtype, int out_dtype, int grad_dtype, void *stream) {
    if (!dout || !x || !stats || !gamma || !dx || !scratch) return DWO_ERR_NULL_POINTER;
    if (!tile_ok(N, C, H, W) || H < 2 || W < 2 || !aligned16(x) || !aligned16(dout) || !aligned16(dx))
        return DWO_ERR_BAD_SHAPE;
    if (scratch_bytes < dwo_block_scratch_bytes(C)) return DWO_ERR_SCRATCH_TOO_SMALL;
    (void)hipGetLastError();
    return ln_quads_backward(dout, x, stats, gamma, dx, dgamma, dbeta, (float *)scratch,
                             quads_of(C, H, W, (long)N * (H / 2) * (W / 2) * 4), true, in_dtype, out_dtype, grad_dtype,
                             (hipStream_t)stream);
}

int dwo_block_tail(const void *y, const float *scale, const void *res, void *out, int N, int C, int H, int W,
                   int rounded, int y_dtype, int res_dtype, int dtype, void *stream) {
    if (!y || !out) return DWO_ERR_NULL_POINTER;
    if (N < 1 || H < 1 || W < 1 || C < 8 || C % 8 != 0 || (double)N * C * H * W >= 2147483648.0 || !aligned16(y) ||
        !aligned16(res) || !aligned16(out))
        return DWO_ERR_BAD_SHAPE;
    (void)hipGetLastError();
    const TailTiles t = tail_of(N, C, H * W);
    const dim3 grid((unsigned)t.units * t.ctiles), block(kBlkThreads);
    // out is y's type or fp32, res has out's type or y's
    return by_types(dtype, y_dtype, [&](auto tr, auto ty) {
        using TR = typename decltype(tr)::type;
        using TY = typename decltype(ty)::type;
        auto launch = [&](auto ts) {
            using TS = typename decltype(ts)::type;
            if (t.HW % 4 == 0)
                tail_kernel<TY, TS, TR, 4><<<grid, block, 0, (hipStream_t)stream>>>((const TY *)y, scale, (const TS *)res,
                                                                                    (TR *)out, t, rounded);
            else
                tail_kernel<TY, TS, TR, 1><<<grid, block, 0, (hipStream_t)stream>>>((const TY *)y, scale, (const TS *)res,
                                                                                    (TR *)out, t, rounded);
            return status();
        };
        if (res == nullptr || res_dtype == dtype) return launch(Type<TR>{});
        if (res_dtype == y_dtype) return launch(Type<TY>{});
        return (int)DWO_ERR_BAD_DTYPE;
    });
}

int dwo_block_tail_backward(const void *dout, const void *y, const float *scale, void *dy, void *dscale, void *scratch,
                            size_t scratch_bytes, int N, int C, int H, int W, int y_dtype, int dtype, int grad_dtype,
                            void *stream) {
    if (!dout || !dy || (y && !scratch)) return DWO_ERR_NULL_POINTER;
    if (N < 1 || H < 1 || W < 1 || C < 8 || C % 8 != 0 || (double)N * C * H * W >= 2147483648.0 || !aligned16(y) ||
        !aligned16(dout) || !aligned16(dy))
        return DWO_ERR_BAD_SHAPE;
    if (y && scratch_bytes < dwo_block_scratch_bytes(C)) return DWO_ERR_SCRATCH_TOO_SMALL;
    (void)hipGetLastError();
    hipStream_t st = (hipStream_t)stream;
    const TailTiles t = tail_of(N, C, H * W);
    // without sums a workgroup per tile, else workgroups that keep them over several tiles
    long g = y ? 2048 / t.ctiles : t.units;
    if (g < 1) g = 1;
    if (g > t.units) g = t.units;
    const int groups = y ? groups_of(g) : (int)g;
    const int e = by_types(dtype, y_dtype, [&](auto tr, auto ty) {
        using TR = typename decltype(tr)::type;
        using TY = typename decltype(ty)::type;
        const dim3 grid((unsigned)groups * t.ctiles), block(kBlkThreads);
        if (t.HW % 4 == 0)
            tail_backward_kernel<TY, TR, 4><<<grid, block, 0, st>>>((const TR *)dout, (const TY *)y, scale, (TY *)dy,
                                                                    (float *)scratch, t);
        else
            tail_backward_kernel<TY, TR, 1><<<grid, block, 0, st>>>((const TR *)dout, (const TY *)y, scale, (TY *)dy,
                                                                    (float *)scratch, t);
        return status();
    });
    if (e != DWO_OK || !y) return e;
    return column_sums((const float *)scratch, dscale, nullptr, C, C, groups, grad_dtype, st);
}

}  // extern "C"
