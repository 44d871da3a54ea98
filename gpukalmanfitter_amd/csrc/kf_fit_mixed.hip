// kf_fit_mixed.hip -- the fit kernels of the FP32-mixed mode.
#include "kf_fit_kernels.hpp"

extern "C" hipError_t kfd_launch_fit_mixed(const kfd::FitArgs *args, hipStream_t stream,
                                           hipEvent_t between, const KfdLaunch *launch) {
  return kfd::launchFit<float>(args, stream, between, launch);
}
