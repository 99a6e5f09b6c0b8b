// One translation unit per (element type, kernel size) of the grouped NHWC kernels: compile with
//   -DDWO_INST_T=<float|bf16_t|f16_t> -DDWO_INST_K=<K>
#include "dwo_grouped.h"

namespace dwo {
template int launch_grouped_conv<DWO_INST_T, DWO_INST_K>(const void *, const float *, const float *,
                                                         const void *, void *, const ConvDims &, int,
                                                         hipStream_t);
template int launch_grouped_wgrad<DWO_INST_T, DWO_INST_K>(const void *, const void *, const void *, float *,
                                                          const ConvDims &, int *, hipStream_t);
template int launch_grouped_projected<DWO_INST_T, DWO_INST_K>(const void *, const float *, const float *,
                                                              const float *, const float *, const void *, void *,
                                                              const ConvDims &, hipStream_t);
}  // namespace dwo
