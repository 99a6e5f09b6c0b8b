// One translation unit per (element type, kernel size) of the window kernels: compile with
//   -DDWO_INST_T=<float|bf16_t|f16_t> -DDWO_INST_K=<K>
#include "dwo_window.h"

namespace dwo {
template int launch_window_conv<DWO_INST_T, DWO_INST_K>(const void *, const float *, const float *,
                                                        const void *, void *, const WinDims &, int,
                                                        hipStream_t);
template int launch_window_wgrad<DWO_INST_T, DWO_INST_K>(const void *, const void *, const void *, float *,
                                                         float *, float *, unsigned *, const WinDims &,
                                                         int *, hipStream_t);
}  // namespace dwo
