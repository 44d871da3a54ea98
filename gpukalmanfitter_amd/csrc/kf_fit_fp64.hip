// kf_fit_fp64.hip -- the fit kernels of the FP64 mode.
#include "kf_fit_kernels.hpp"

extern "C" hipError_t kfd_launch_fit_fp64(const kfd::FitArgs *args, hipStream_t stream,
                                          hipEvent_t between, const KfdLaunch *launch) {
  return kfd::launchFit<double>(args, stream, between, launch);
}
