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
    const int splits = linear_splits(rows, N, K);
    float *part = (float *)scratch;
    int e;
    switch (dtype) {
        case DWO_BF16: e = launch_linear_wgrad<bf16_t>(dy, x, part, rows, N, K, splits, db != nullptr, st); break;
        case DWO_F16: e = launch_linear_wgrad<f16_t>(dy, x, part, rows, N, K, splits, db != nullptr, st); break;
        default: return DWO_ERR_BAD_DTYPE;
    }
    if (e != 0) return e;
    switch (grad_dtype) {
        case DWO_F32: return launch_linear_reduce<float>(part, dw, db, N, K, splits, st);
        case DWO_BF16: return launch_linear_reduce<bf16_t>(part, dw, db, N, K, splits, st);
        case DWO_F16: return launch_linear_reduce<f16_t>(part, dw, db, N, K, splits, st);
        default: return DWO_ERR_BAD_DTYPE;
    }
}

}  // extern "C"
