// FP64 (complex128) instantiation of the fused sweeps.
#define WH_S double
#define WH_T double
#define WH_SUFFIX f64
#include "wh_sweeps_inst.inc"

namespace wh {
// narrow: one-wave blocks of radix 8 (kGpNarrow) instead of kGpWide
hipError_t launch_gpshift(bool narrow, const SweepArgs& a, int nwork, hipStream_t s) {
  if (narrow)
    hipLaunchKernelGGL((gpshift_kernel<kGpNarrow.R, kGpNarrow.block>), dim3(nwork), dim3(kGpNarrow.block), 0, s, a);
  else
    hipLaunchKernelGGL((gpshift_kernel<kGpWide.R, kGpWide.block>), dim3(nwork), dim3(kGpWide.block), 0, s, a);
  return hipGetLastError();
}
}  // namespace wh
