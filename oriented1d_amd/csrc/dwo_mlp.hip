// C entry point of a block's two pointwise layers as one kernel.
#include "dwo_mlp.h"

using namespace dwo;

namespace {
template <typename T>
int mlp(const void *x, const void *w1, const void *b1, const void *w2, const void *b2, const void *scale, const void *res,
        void *out, long M, int HW, int C, hipStream_t st) {
    const MlpArgs<T> a{(const T *)x, (const T *)w1, (const T *)b1, (const T *)w2, (const T *)b2, (const T *)scale,
                       (const T *)res, (T *)out, M, HW, HW % 8 == 0 ? 8 : HW % 4 == 0 ? 4 : 1};
    switch (C) {
        case 96: return launch_mlp<T, 96>(a, st);
        case 128: return launch_mlp<T, 128>(a, st);
        case 192: return launch_mlp<T, 192>(a, st);
        case 384: return launch_mlp<T, 384>(a, st);
        default: return DWO_ERR_BAD_SHAPE;
    }
}
}  // namespace

extern "C" {

int dwo_block_mlp(const void *x, const void *w1, const void *b1, const void *w2, const void *b2, const void *scale,
                  const void *res, void *out, int images, int HW, int C, int dtype, void *stream) {
    if (!x || !w1 || !b1 || !w2 || !b2 || !res || !out) return DWO_ERR_NULL_POINTER;
    if (images < 1 || HW < 1 || (double)images * HW >= 2147483648.0 ||
        ((uintptr_t)x | (uintptr_t)w1 | (uintptr_t)b1 | (uintptr_t)w2 | (uintptr_t)res | (uintptr_t)out) % 16 != 0)
        return DWO_ERR_BAD_SHAPE;
    (void)hipGetLastError();
    const long M = (long)images * HW;
    switch (dtype) {
        case DWO_BF16: return mlp<bf16_t>(x, w1, b1, w2, b2, scale, res, out, M, HW, C, (hipStream_t)stream);
        case DWO_F16: return mlp<f16_t>(x, w1, b1, w2, b2, scale, res, out, M, HW, C, (hipStream_t)stream);
        default: return DWO_ERR_BAD_DTYPE;
    }
}

}  // extern "C"
