// C entry points of the pointwise layers' parameter gradients.
#include "dwo_linear.h"

using namespace dwo;

extern "C" {

size_t dwo_linear_wgrad_scratch_bytes(size_t rows, int N, int K) {
    if (rows < 1 || rows > (size_t)1 << 31 || N < 8 || K < 8 || N % 8 != 0 || K % 8 != 0 || N > 65536 || K > 65536)
        return 0;
    return linear_wgrad_scratch(rows, N, K);
}

int dwo_linear_wgrad(const void *dy, const void *x, void *dw, void *db, void *scratch, size_t scratch_bytes,
                     size_t rows, int N, int K, int dtype, int grad_dtype, void *stream) {
    if (!dy || !x || !dw || !scratch) return DWO_ERR_NULL_POINTER;
    const size_t need = dwo_linear_wgrad_scratch_bytes(rows, N, K);
    if (need == 0 || ((uintptr_t)dy | (uintptr_t)x | (uintptr_t)scratch) % 16 != 0) return DWO_ERR_BAD_SHAPE;
    if (scratch_bytes < need) return DWO_ERR_SCRATCH_TOO_SMALL;
    hipStream_t st = (hipStream_t)stream;
    (void)hipGetLastError();  // (an earlier call's error is not this call's status)
    float *part = (float *)scratch;
#define DWO_TYPES(T)                                                                                    \
    switch (grad_dtype) {                                                                               \
        case DWO_F32: return launch_linear_wgrad<T, float>(dy, x, dw, db, part, rows, N, K, st);        \
        case DWO_BF16: return launch_linear_wgrad<T, bf16_t>(dy, x, dw, db, part, rows, N, K, st);      \
        case DWO_F16: return launch_linear_wgrad<T, f16_t>(dy, x, dw, db, part, rows, N, K, st);        \
        default: return DWO_ERR_BAD_DTYPE;                                                              \
    }
    switch (dtype) {
        case DWO_BF16: DWO_TYPES(bf16_t)
        case DWO_F16: DWO_TYPES(f16_t)
        default: return DWO_ERR_BAD_DTYPE;
    }
#undef DWO_TYPES
}

// y = x w^T + b over 16-bit activations; x, w and out 16-byte aligned, N and K multiples of eight, offsets inside 31 bits
static bool linear_ok(size_t rows, int N, int K, const void *x, const void *w, const void *out) {
    return rows >= 1 && rows < (size_t)1 << 31 && N >= 8 && K >= 8 && N % 8 == 0 && K % 8 == 0 && N <= 65536 &&
           K <= 65536 && ((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) % 16 == 0;
}

int dwo_linear_rows(const void *x, const void *w, const void *bias, void *out, size_t rows, int N, int K, int gelu,
                    int dtype, void *stream) {
    if (!x || !w || !out) return DWO_ERR_NULL_POINTER;
    if (!linear_ok(rows, N, K, x, w, out)) return DWO_ERR_BAD_SHAPE;
    (void)hipGetLastError();
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
        case DWO_BF16:
            return launch_linear<bf16_t, false>({(const bf16_t *)x, (const bf16_t *)w, (const bf16_t *)bias, nullptr,
                                                 nullptr, (bf16_t *)out, (long)rows, N, K, 1, gelu}, st);
        case DWO_F16:
            return launch_linear<f16_t, false>({(const f16_t *)x, (const f16_t *)w, (const f16_t *)bias, nullptr,
                                                nullptr, (f16_t *)out, (long)rows, N, K, 1, gelu}, st);
        default: return DWO_ERR_BAD_DTYPE;
    }
}

int dwo_linear_planes(const void *x, const void *w, const void *bias, const void *scale, const void *res, void *out,
                      int images, int HW, int N, int K, int dtype, void *stream) {
    if (!x || !w || !out) return DWO_ERR_NULL_POINTER;
    if (images < 1 || HW < 1 || (double)images * HW >= 2147483648.0 ||
        !linear_ok((size_t)images * HW, N, K, x, w, out) || (uintptr_t)res % 16 != 0)
        return DWO_ERR_BAD_SHAPE;
    (void)hipGetLastError();
    hipStream_t st = (hipStream_t)stream;
    const long M = (long)images * HW;
    switch (dtype) {
        case DWO_BF16:
            return launch_linear<bf16_t, true>({(const bf16_t *)x, (const bf16_t *)w, (const bf16_t *)bias,
                                                (const bf16_t *)scale, (const bf16_t *)res, (bf16_t *)out, M, N, K, HW,
                                                0}, st);
        case DWO_F16:
            return launch_linear<f16_t, true>({(const f16_t *)x, (const f16_t *)w, (const f16_t *)bias,
                                               (const f16_t *)scale, (const f16_t *)res, (f16_t *)out, M, N, K, HW, 0},
                                              st);
        default: return DWO_ERR_BAD_DTYPE;
    }
}

int dwo_linear_norm_planes(const void *x, const float *gamma_in, const float *beta_in, float eps_in, const void *w,
                           const void *bias, const float *gamma, const float *beta, float eps, void *out, int images, int HW,
                           int N, int K, int dtype, void *stream) {
    if (!x || !gamma_in || !beta_in || !w || !gamma || !beta || !out) return DWO_ERR_NULL_POINTER;
    if (images < 1 || HW < 1 || (double)images * HW >= 2147483648.0 || K != kNormK || (N != 96 && N != 128) ||
        ((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) % 16 != 0)
        return DWO_ERR_BAD_SHAPE;
    (void)hipGetLastError();
    hipStream_t st = (hipStream_t)stream;
    const long M = (long)images * HW;
    const NormArgs na{gamma, beta, gamma_in, beta_in, eps, eps_in};
    switch (dtype) {
        case DWO_BF16:
            return launch_linear_norm<bf16_t>({(const bf16_t *)x, (const bf16_t *)w, (const bf16_t *)bias, nullptr, nullptr,
                                               (bf16_t *)out, M, N, K, HW, 0}, na, st);
        case DWO_F16:
            return launch_linear_norm<f16_t>({(const f16_t *)x, (const f16_t *)w, (const f16_t *)bias, nullptr, nullptr,
                                              (f16_t *)out, M, N, K, HW, 0}, na, st);
        default: return DWO_ERR_BAD_DTYPE;
    }
}

int dwo_pointwise_forward(const void *x, const void *w, const void *b, void *y, size_t rows, int Cin, int C, int dtype,
                          void *stream) {
    if (!x || !w || !y) return DWO_ERR_NULL_POINTER;
    if (rows < 1 || rows > (size_t)1 << 40 || Cin < 1 || Cin > 4 || C < 64 || C % 64 != 0 || C > 65536 ||
        (uintptr_t)y % 16 != 0)
        return DWO_ERR_BAD_SHAPE;
    (void)hipGetLastError();
    switch (dtype) {
        case DWO_BF16: return launch_few_inputs<bf16_t>(x, w, b, y, (long)rows, C, Cin, (hipStream_t)stream);
        case DWO_F16: return launch_few_inputs<f16_t>(x, w, b, y, (long)rows, C, Cin, (hipStream_t)stream);
        default: return DWO_ERR_BAD_DTYPE;
    }
}

}  // extern "C"
