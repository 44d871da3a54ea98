// kf_kernels.hip -- the kernels around the fit (track-state export, length
// sort, counters) and the launcher of a slice of a batch.
#include <hip/hip_runtime.h>

#include "kf_kernels.hpp"

namespace kfd {

// Copies the public track-state records into kf_results.track_states
// ([state][KF_TS_STRIDE][n]).  A block moves half of the fields of one state
// slot of one 64-track chunk, each wave kExportFields of them with every load
// issued before the first store, so a launch has chunks x states x 8 waves
// whatever the batch: with one thread per track walking its states field by
// field (the records of 4,099 tracks of 8-40 states are 17 blocks then) the
// copy was a serial chain of loads, 1.85 ms of a 3.1 ms fit.
constexpr int kExportFields = KF_TS_STRIDE / 8;
static_assert(KF_TS_STRIDE % 8 == 0, "eight waves per record");
__global__ void __launch_bounds__(256) kf_export_states(FitArgs args, double *out) {
  const uint32_t lane = threadIdx.x & 63u;
  const int64_t local = (int64_t)blockIdx.x * 64 + lane;
  if (local >= args.count) return;
  const int64_t pos = args.first + local;
  const int64_t i = args.order ? (int64_t)args.order[pos] : pos;
  const int nm = (args.out_nmeas[i] < args.max_states) ? args.out_nmeas[i] : args.max_states;
  const double *base =
      args.tsf + (size_t)blockIdx.x * (size_t)args.max_states * KF_TS_STRIDE * 64u;
  const int f0 = (int)(blockIdx.z * 4 + (threadIdx.x >> 6)) * kExportFields;
  for (int k = (int)blockIdx.y; k < nm; k += (int)gridDim.y) {
    double v[kExportFields];
#pragma unroll
    for (int f = 0; f < kExportFields; ++f)
      v[f] = base[((uint32_t)k * KF_TS_STRIDE + (uint32_t)(f0 + f)) * 64u + lane];
#pragma unroll
    for (int f = 0; f < kExportFields; ++f)
      out[((size_t)k * KF_TS_STRIDE + (size_t)(f0 + f)) * (size_t)args.n + i] = v[f];
  }
}

// ------------------------------------------------------- length sort ----
// Counting sort of the tracks by decreasing sequence length (lengths >= 255
// share the top bin): tracks of one wave then take similar numbers of steps,
// and a persistent grid starts on the longest.  Per-block LDS histograms keep
// the global atomics to one per block and bin; a thread takes kSortTracks tracks,
// so that the blocks' atomics on the few bins in use do not queue up.
constexpr int kLenBins = 256;
constexpr int kSortTracks = 4;
constexpr int kSortBlock = 256 * kSortTracks;

KFD_INLINE int lengthBin(const FitArgs &a, int64_t i) {
  int l = a.seq_count[i];
  return l < 0 ? 0 : (l >= kLenBins ? kLenBins - 1 : l);
}

// zeroes the histogram and bin offsets
__global__ void __launch_bounds__(256) kf_sort_reset(uint32_t *scratch) {
  scratch[threadIdx.x] = 0u;
  scratch[kLenBins + threadIdx.x] = 0u;
}

// zeroes the redo counters of the fused fit
__global__ void __launch_bounds__(64) kf_redo_reset(uint32_t *redo) {
  if (threadIdx.x < 3) redo[threadIdx.x] = 0u;
}

// zeroes the work-queue counters (forward, backward)
__global__ void __launch_bounds__(64) kf_queue_reset(uint32_t *queue) {
  if (threadIdx.x < 2) queue[threadIdx.x] = 0u;
}

__global__ void __launch_bounds__(256) kf_len_hist(FitArgs a, uint32_t *hist) {
  __shared__ uint32_t h[kLenBins];
  h[threadIdx.x] = 0u;
  __syncthreads();
  const int64_t i0 = (int64_t)blockIdx.x * kSortBlock + threadIdx.x;
#pragma unroll
  for (int q = 0; q < kSortTracks; ++q)
    if (i0 + 256 * q < a.n) atomicAdd(&h[lengthBin(a, i0 + 256 * q)], 1u);
  __syncthreads();
  if (h[threadIdx.x]) atomicAdd(&hist[threadIdx.x], h[threadIdx.x]);
}

// off[len] = number of tracks longer than len (one block of 256)
__global__ void __launch_bounds__(256) kf_len_scan(uint32_t *hist, uint32_t *off) {
  __shared__ uint32_t s[kLenBins];
  const int t = threadIdx.x;
  s[t] = hist[kLenBins - 1 - t];
  __syncthreads();
  for (int w = 1; w < kLenBins; w <<= 1) {
    const uint32_t v = (t >= w) ? s[t - w] : 0u;
    __syncthreads();
    s[t] += v;
    __syncthreads();
  }
  off[kLenBins - 1 - t] = s[t] - hist[kLenBins - 1 - t];
}

__global__ void __launch_bounds__(256) kf_len_scatter(FitArgs a, uint32_t *off, int32_t *order) {
  __shared__ uint32_t cnt[kLenBins], base[kLenBins];
  cnt[threadIdx.x] = 0u;
  __syncthreads();
  const int64_t i0 = (int64_t)blockIdx.x * kSortBlock + threadIdx.x;
  int bin[kSortTracks];
  uint32_t local[kSortTracks];
#pragma unroll
  for (int q = 0; q < kSortTracks; ++q) {
    const int64_t i = i0 + 256 * q;
    bin[q] = (i < a.n) ? lengthBin(a, i) : 0;
    local[q] = (i < a.n) ? atomicAdd(&cnt[bin[q]], 1u) : 0u;
  }
  __syncthreads();
  if (cnt[threadIdx.x]) base[threadIdx.x] = atomicAdd(&off[threadIdx.x], cnt[threadIdx.x]);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kSortTracks; ++q)
    if (i0 + 256 * q < a.n) order[base[bin[q]] + local[q]] = (int32_t)(i0 + 256 * q);
}

}  // namespace kfd

extern "C" hipError_t kfd_launch_fit(const kfd::FitArgs *args, int precision, hipStream_t stream,
                                     double *track_states_out, hipEvent_t between,
                                     const KfdLaunch *launch) {
  if (args->count <= 0) return hipSuccess;
  // the fused kernel takes one position per lane whatever the schedule
  if (launch && launch->persistent_blocks > 0 && args->tsf)
    hipLaunchKernelGGL(kfd::kf_queue_reset, dim3(1), dim3(64), 0, stream, args->queue);
  const hipError_t e = (precision == KF_PRECISION_FP64)
                           ? kfd_launch_fit_fp64(args, stream, between, launch)
                           : kfd_launch_fit_mixed(args, stream, between, launch);
  if (e != hipSuccess) return e;
  if (track_states_out) {
    const unsigned chunks = (unsigned)((args->count + 63) / 64);
    const unsigned slots = (unsigned)(args->max_states < 32768 ? args->max_states : 32768);
    hipLaunchKernelGGL(kfd::kf_export_states, dim3(chunks, slots, 2), dim3(256), 0, stream, *args,
                       track_states_out);
  }
  return hipGetLastError();
}

extern "C" hipError_t kfd_launch_redo_reset(uint32_t *redo, hipStream_t stream) {
  hipLaunchKernelGGL(kfd::kf_redo_reset, dim3(1), dim3(64), 0, stream, redo);
  return hipGetLastError();
}

extern "C" hipError_t kfd_launch_sort(const kfd::FitArgs *args, const KfdLaunch *launch,
                                      hipStream_t stream) {
  if (args->n <= 0) return hipSuccess;
  const unsigned sb = (unsigned)((args->n + kfd::kSortBlock - 1) / kfd::kSortBlock);
  uint32_t *hist = launch->sort_scratch, *off = launch->sort_scratch + kfd::kLenBins;
  hipLaunchKernelGGL(kfd::kf_sort_reset, dim3(1), dim3(256), 0, stream, launch->sort_scratch);
  hipLaunchKernelGGL(kfd::kf_len_hist, dim3(sb), dim3(256), 0, stream, *args, hist);
  hipLaunchKernelGGL(kfd::kf_len_scan, dim3(1), dim3(256), 0, stream, hist, off);
  hipLaunchKernelGGL(kfd::kf_len_scatter, dim3(sb), dim3(256), 0, stream, *args, off,
                     launch->order);
  return hipGetLastError();
}
