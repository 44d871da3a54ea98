// kf_fit_kernels.hpp -- the batched Kalman-fit kernels for gfx950 and the
// launcher of one precision, instantiated by kf_fit_fp64.hip and
// kf_fit_mixed.hip.  The per-track program is TrackFit (kf_trackfit.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include "kf_trackfit.hpp"

namespace kfd {

// Bases of the state stores of the 64-track chunk this wave works on.
// Blocks are multiples of 64 work-items, so a wave covers exactly one chunk.
template <typename S>
struct ChunkBases {
  double *d;
  S *s;
  double *f;
  double *c;
  KFD_INLINE ChunkBases(const FitArgs &a, int64_t i) {
    const size_t chunk = __builtin_amdgcn_readfirstlane((uint32_t)(i >> 6));
    const size_t per = (size_t)a.max_states * 64u;
    d = a.tsd ? a.tsd + chunk * per * KF_SD_N : nullptr;
    s = a.tss ? (S *)a.tss + chunk * per * KF_SS_N : nullptr;
    f = a.tsf ? a.tsf + chunk * per * KF_TS_STRIDE : nullptr;
    c = a.tsc ? a.tsc + chunk * per * KF_CK_N : nullptr;
  }
};

// Fits the track at position pos (pass FWD of the two kernels); `rank` is
// the lane's index in the track's group of L lanes.
template <typename S, bool FWD, int L, bool PS, int FK, int KEEP>
KFD_INLINE void fitPosition(const FitArgs &a, int64_t local, uint32_t rank,
                            const DevPlane *planes) {
  const ChunkBases<S> cb(a, local);
  if (local >= a.count) return;
  const int64_t pos = a.first + local;
  const int64_t i = a.order ? (int64_t)a.order[pos] : pos;
  TrackFit<S, FWD, L, PS, false, FK, KEEP> tf(a, i, cb.d, cb.s, cb.f, cb.c,
                                              (uint32_t)(local & 63), local);
  tf.setRank(rank);
  tf.pls = planes;
  if constexpr (FWD)
    tf.runForward();
  else
    tf.runBackward();
}

// One thread per position, or (persistent) resident waves that take
// chunks_per_grab 64-position chunks at a time from a work-queue counter
// until every chunk is taken; the grab is one vector atomic by lane 0.
//
// LDS = true: the block first copies the plane table (at most KF_LDS_PLANES
// planes) to LDS and reads planes there.
// PERS = false: one thread per position; true: the persistent work queue
// (a separate instantiation, so the one-shot kernel does not carry the
// queue loop's registers).
// L: lanes per track (one-shot grid only): L consecutive lanes fit one
// position, a wave covers 64 / L positions of one 64-position store chunk.
// PS: store slots by plane position (kf_schedule.store_by_plane; one lane
// per track).
// FK, KEEP: the field kind and what is kept of the states.  The build is the
// one for the batch's field, so the step loop carries no code of the other
// kind, with kKeepRecords where track states are asked for (where not:
// kf_fused_kernel); plane tables read from global memory run on (kFieldAny,
// kKeepRecords).  The chi2 adjoint's forward
// pass is the kKeepCheckpoints build: without the smoother's store and with
// the checkpoint's constant half left out it writes 248 B per state instead
// of 1,000.
template <typename S, bool FWD, bool LDS, bool PERS, int L, bool PS, int FK, int KEEP>
__global__ void __launch_bounds__(KF_BLOCK) kf_fit_kernel(FitArgs args) {
  static_assert(L == 1 || !PERS, "lane groups run on the one-shot grid");
  static_assert(L == 1 || !PS, "store slots by plane with one lane per track");
  const DevPlane *planes = args.planes;
  if constexpr (LDS) {
    __shared__ DevPlane lds_planes[KF_LDS_PLANES];
    const double *src = (const double *)args.planes;
    double *dst = (double *)lds_planes;
    const int words = args.n_planes * (int)(sizeof(DevPlane) / sizeof(double));
    for (int w = threadIdx.x; w < words; w += KF_BLOCK) dst[w] = src[w];
    __syncthreads();
    planes = lds_planes;
  }
  const uint32_t lane = threadIdx.x & 63u;
  if constexpr (!PERS) {
    const int64_t t = (int64_t)blockIdx.x * KF_BLOCK + threadIdx.x;
    fitPosition<S, FWD, L, PS, FK, KEEP>(args, t / L, (uint32_t)(t % L), planes);
  } else {
    const uint32_t nchunks = (uint32_t)((args.count + 63) >> 6);
    const uint32_t grab = (uint32_t)args.chunks_per_grab;
    uint32_t *q = args.queue + (FWD ? 0 : 1);
    for (;;) {
      uint32_t c0 = 0;
      if (lane == 0) c0 = atomicAdd(q, grab);
      c0 = (uint32_t)__shfl((int)c0, 0, 64);
      if (c0 >= nchunks) break;
      const uint32_t c1 = (c0 + grab < nchunks) ? c0 + grab : nchunks;
      for (uint32_t c = c0; c < c1; ++c)
        fitPosition<S, FWD, 1, PS, FK, KEEP>(args, (int64_t)c * 64 + lane, 0u, planes);
    }
  }
}

// The whole fit in one kernel, for fits that ask for neither track states
// nor checkpoints: forward filter with the fixed-point smoother, then back to
// the perigee (TrackFit::runFused).  Per-track state in registers (one wave
// per SIMD), the smoother's sums in LDS (46 KB per block in FP64, 64 KB in the
// mixed mode), the plane table in dynamic LDS (PLDS) or global memory.  FK: the
// field kind, so the step loop carries no code of the other one (either kind where
// the plane table is in global memory).  L as in kf_fit_kernel.
//
// Bound by instruction issue: a wave of ten planes issues 24,600 vector
// instructions in FP64 (1,048,576 tracks: 1.30 ms) and 40,600 in the mixed
// mode (1.73 ms), a third of them the RTS gain and its sums (TrackFit::fxRtsStep; the
// FP64 sums round differently from the recursion over float covariances, 1e-7
// in the time variance).  Mixed, against the forward and backward kernels that
// passed 304 B per state through memory: 1,048,576 tracks 2.03 -> 1.73 ms,
// 500,003 ragged ones 2.81 -> 2.30 ms, 100,003 with material 1.93 -> 1.70 ms.
//
// Tracks for the RTS program (redoTrack), in three ways:
//  - a track near the phi wrap (nearWrap) is left out by its lane and fitted by
//    the waves at the front of the grid, rts_waves of them, which go through a
//    share of the positions each and take the tracks they pick 64 at a time;
//  - a track that the fixed-point smoother leaves, for its start covariance before
//    the pass (TrackFit::fxDefinite) or in the end (fxSafe; 1 in 2,000 of the
//    material workload spread over azimuth), is fitted by its own wave while the others go on, over a store slot of its own
//    (redoSlotPerTrack) or a chunk that the wave takes from a pool;
//  - when the pool is used up it goes to the list of the redo kernel.
// Fitted after the fused pass alone, a single handed-back track cost a small
// batch the RTS program's latency on top.  10,007 tracks of ten planes facing
// phi = pi: 318 us so, 127 beside the others, 159 in the forward and backward kernels
// (FP64; 361, 138 and 153 mixed); 1,048,576 of them 2,410, 1,791 and 2,881 us;
// facing +x 96 us and 1,300 us either way.  Waiting for the redo kernel with all of
// them cost the material workload 0.9 ms a call.
//
// redoTrack is a call so that its code and registers stay out of the fit's and
// that a track's bits do not depend on which of the three it takes; it reads the
// kernel's arguments where the kernel finds them, and the plane table in LDS
// where the kernel has it there.
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(3))) const DevPlane LdsPlane;
#else
typedef const DevPlane LdsPlane;
#endif
template <typename S, bool PLDS, int FK>
static __device__ __attribute__((noinline)) void redoTrack(const FitArgs *args, int64_t i,
                                                           int64_t slot, LdsPlane *table) {
  const FitArgs &a = *uniformArgs(args);
  const uint32_t lane = (uint32_t)(slot & 63);
  const size_t per = (size_t)(slot >> 6) * (size_t)a.max_states * 64u;
  double *d = a.tsd + per * KF_SD_N;
  S *s = (S *)a.tss + per * KF_SS_N;
  const DevPlane *planes = PLDS ? (const DevPlane *)table : a.planes;
  {
    TrackFit<S, true, 1, false, false, FK, kKeepStates> tf(a, i, d, s, nullptr, nullptr, lane,
                                                           slot);
    tf.pls = planes;
    tf.redoSlots();
    tf.runForward();
  }
  {
    TrackFit<S, false, 1, false, false, FK, kKeepStates> tf(a, i, d, s, nullptr, nullptr, lane,
                                                            slot);
    tf.pls = planes;
    tf.redoSlots();
    tf.runBackward();
  }
}

// The plane table to dynamic LDS.
KFD_INLINE const DevPlane *tableToLds(const FitArgs &args, double *lds_table) {
  const double *src = (const double *)args.planes;
  const int words = args.n_planes * (int)(sizeof(DevPlane) / sizeof(double));
  for (int w = threadIdx.x; w < words; w += (int)blockDim.x) lds_table[w] = src[w];
  __syncthreads();
  return (const DevPlane *)lds_table;
}

// One of the waves for tracks near the wrap: its share of the positions, every
// rts_waves-th 64 of them (sorted by length or by angle, each then has as much to
// do), the picked ones collected, at most 63 + 64, until a wave is full.  Its
// store slots are those of its lanes, so that a few tracks lie together; where the
// chunk is also that of the positions' own wave (redoSlotPerTrack) that one takes
// slots from the other end for the tracks it leaves, or, with several waves to a
// chunk (L > 1), both take those of the positions.
template <typename S, bool PLDS, int L, int FK>
KFD_INLINE void fitNearWrap(const FitArgs &args, int64_t wave, uint32_t *list, LdsPlane *table) {
  const FitArgs *ka = (const FitArgs *)__builtin_amdgcn_kernarg_segment_ptr();
  if (wave >= args.rts_waves) return;
  const int lane = (int)(threadIdx.x & 63u);
  int n = 0;
  for (int64_t at = wave * 64; at < args.count || n > 0;) {
    while (n < 64 && at < args.count) {
      const int64_t local = at + lane;
      bool pick = false;
      if (local < args.count) {
        const int64_t pos = args.first + local;
        const int64_t i = args.order ? (int64_t)args.order[pos] : pos;
        pick = nearWrap(ka, i);
      }
      const uint64_t m = __ballot(pick);
      if (pick) list[n + __popcll(m & ((1ull << lane) - 1ull))] = (uint32_t)local;
      n += __popcll(m);
      at += args.rts_waves * (int64_t)64;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int take = (n < 64) ? n : 64;
    const uint32_t local = (lane < take) ? list[lane] : 0u;
    const uint32_t rest = (lane + 64 < n) ? list[lane + 64] : 0u;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane + 64 < n) list[lane] = rest;
    n -= take;
    if (lane < take) {
      const int64_t pos = args.first + (int64_t)local;
      redoTrack<S, PLDS, FK>(ka, args.order ? (int64_t)args.order[pos] : pos,
                             (L > 1 && redoSlotPerTrack(args)) ? (int64_t)local
                                                               : wave * 64 + lane,
                             table);
    }
  }
}

template <typename S, bool PLDS, int L, int FK>
__global__ void __launch_bounds__(KF_FUSED_BLOCK) kf_fused_kernel(FitArgs args) {
  using Fit = TrackFit<S, true, L, false, false, FK, kKeepFirst>;
  __shared__ typename Fit::FxPair sums[Fit::kFxN * KF_FUSED_BLOCK];
  __shared__ uint32_t picked[KF_FUSED_BLOCK / 64][128];
  extern __shared__ double lds_table[];
  static_assert(sizeof sums + sizeof picked +
                        sizeof(DevPlane) * (sizeof(S) == sizeof(double) ? KF_FUSED_LDS_PLANES_FP64
                                                                        : KF_FUSED_LDS_PLANES_MIXED) <=
                    160 * 1024 / 2,
                "two blocks per compute unit");
  const DevPlane *planes = args.planes;
  if constexpr (PLDS) planes = tableToLds(args, lds_table);
  LdsPlane *table = PLDS ? (LdsPlane *)planes : nullptr;
  const FitArgs *ka = (const FitArgs *)__builtin_amdgcn_kernarg_segment_ptr();
  const uint32_t rtsBlocks = (uint32_t)rtsBlocksOf(args);
  if (blockIdx.x < rtsBlocks) {
    const int w = (int)(threadIdx.x >> 6), per = rtsPerBlock(args);
    if (w < per) fitNearWrap<S, PLDS, L, FK>(args, (int64_t)blockIdx.x * per + w, picked[w], table);
    return;
  }
  const int64_t t = (int64_t)(blockIdx.x - rtsBlocks) * KF_FUSED_BLOCK + threadIdx.x;
  const int64_t local = t / L;
  if (local >= args.count) return;
  const int64_t pos = args.first + local;
  const int64_t i = args.order ? (int64_t)args.order[pos] : pos;
  bool redo;
  {
    Fit tf(args, i, nullptr, nullptr, nullptr, nullptr, threadIdx.x & 63u, local);
    tf.setRank((uint32_t)(t % L));
    tf.pls = planes;
    tf.fx = sums + threadIdx.x;
    if (rtsBlocks > 0) tf.picker = ka;
    tf.leaveEarly = true;
    redo = !tf.runFused() && tf.lead;
  }
  const uint64_t redoMask = __ballot(redo);
  if (redoMask == 0) return;
  const int lane = (int)(threadIdx.x & 63u);
  int64_t slot = local;
  if (redoSlotPerTrack(args)) {
    if constexpr (L == 1) slot = local - lane + 63 - __popcll(redoMask & ((1ull << lane) - 1ull));
  } else {
    const int first = __ffsll((unsigned long long)redoMask) - 1;
    uint32_t chunk = 0;
    if (lane == first) chunk = atomicAdd(args.redo, 1u);
    chunk = (uint32_t)__shfl((int)chunk, first, 64);
    slot = ((int64_t)args.rts_waves + chunk) * 64 + lane;
    if (slot >= args.redo_lanes) {
      if (redo) args.redo[KF_REDO_LIST + atomicAdd(args.redo + 1, 1u)] = (uint32_t)local;
      return;
    }
  }
  if (redo) redoTrack<S, PLDS, FK>(ka, i, slot, table);
}

// The tracks that found no store chunk in the fused kernel, 64 at a time per
// wave, over all the chunks.  Usually the list is empty and the kernel ends at
// once.  The last block zeroes the counters for the next fit (every wave has read
// the count when its block takes its ticket).
template <typename S, bool PLDS, int FK>
__global__ void __launch_bounds__(KF_FUSED_BLOCK) kf_redo_kernel(FitArgs args) {
  extern __shared__ double lds_table[];
  const uint32_t n = __hip_atomic_load(args.redo + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const DevPlane *planes = args.planes;
  if constexpr (PLDS)
    if (n > 0) planes = tableToLds(args, lds_table);
  const int64_t slot = (int64_t)blockIdx.x * KF_FUSED_BLOCK + threadIdx.x;
  if (slot < args.redo_lanes)
    for (int64_t e = slot; e < (int64_t)n; e += args.redo_lanes) {
      const int64_t pos = args.first + (int64_t)args.redo[KF_REDO_LIST + e];
      redoTrack<S, PLDS, FK>((const FitArgs *)__builtin_amdgcn_kernarg_segment_ptr(),
                             args.order ? (int64_t)args.order[pos] : pos, slot,
                             PLDS ? (LdsPlane *)planes : nullptr);
    }
  __syncthreads();
  if (threadIdx.x == 0 && atomicAdd(args.redo + 2, 1u) == gridDim.x - 1) {
    args.redo[0] = 0u;
    args.redo[1] = 0u;
    args.redo[2] = 0u;
  }
}

// The launches of one precision.
template <typename S>
hipError_t launchFit(const FitArgs *args, hipStream_t stream, hipEvent_t between,
                     const KfdLaunch *launch) {
  const bool pers = launch && launch->persistent_blocks > 0;
  const int lpt = (launch && !pers && launch->lanes_per_track > 1) ? launch->lanes_per_track : 1;
  if (lpt != 1 && lpt != 2 && lpt != 4) return hipErrorInvalidValue;
  const bool ps = launch && launch->store_by_plane != 0;
  if (ps && lpt != 1) return hipErrorInvalidValue;
  const int64_t blocks =
      pers ? launch->persistent_blocks : (args->count * lpt + KF_BLOCK - 1) / KF_BLOCK;
  const dim3 grid((unsigned)blocks), block(KF_BLOCK);
  const bool rec = args->tsf != nullptr;
  if constexpr (sizeof(S) == sizeof(double)) {
    if (args->tsc) {
      const unsigned nb = (unsigned)((args->count + KF_BLOCK - 1) / KF_BLOCK);
#define KFD_CHECKPOINTS(LDS_, FK_)                                                             \
  hipLaunchKernelGGL((kf_fit_kernel<S, true, LDS_, false, 1, false, FK_, kKeepCheckpoints>), \
                     dim3(nb), block, 0, stream, *args)
      if (args->n_planes > KF_LDS_PLANES)
        KFD_CHECKPOINTS(false, kFieldAny);
      else if (args->field.grid)
        KFD_CHECKPOINTS(true, kFieldGrid);
      else
        KFD_CHECKPOINTS(true, kFieldConst);
#undef KFD_CHECKPOINTS
      if (between) {
        const hipError_t e = hipEventRecord(between, stream);
        if (e != hipSuccess) return e;
      }
      return hipGetLastError();
    }
  }
  if (rec) {
    const bool lds = args->n_planes <= KF_LDS_PLANES;
#define KFD_LAUNCH2(FWD_, LDS_, PERS_, L_, PS_, FK_, KEEP_)                                     \
  hipLaunchKernelGGL((kf_fit_kernel<S, FWD_, LDS_, PERS_, L_, PS_, FK_, KEEP_>), grid, block, 0, \
                     stream, *args)
#define KFD_LAUNCH1(FWD_, LDS_, FK_, KEEP_)                   \
  do {                                                        \
    if (pers && ps)                                           \
      KFD_LAUNCH2(FWD_, LDS_, true, 1, true, FK_, KEEP_);     \
    else if (pers)                                            \
      KFD_LAUNCH2(FWD_, LDS_, true, 1, false, FK_, KEEP_);    \
    else if (lpt == 1 && ps)                                  \
      KFD_LAUNCH2(FWD_, LDS_, false, 1, true, FK_, KEEP_);    \
    else if (lpt == 1)                                        \
      KFD_LAUNCH2(FWD_, LDS_, false, 1, false, FK_, KEEP_);   \
    else if (lpt == 2)                                        \
      KFD_LAUNCH2(FWD_, LDS_, false, 2, false, FK_, KEEP_);   \
    else                                                      \
      KFD_LAUNCH2(FWD_, LDS_, false, 4, false, FK_, KEEP_);   \
  } while (0)
#define KFD_LAUNCH(FWD_)                                      \
  do {                                                        \
    if (lds && args->field.grid)                              \
      KFD_LAUNCH1(FWD_, true, kFieldGrid, kKeepRecords);      \
    else if (lds)                                             \
      KFD_LAUNCH1(FWD_, true, kFieldConst, kKeepRecords);     \
    else                                                      \
      KFD_LAUNCH1(FWD_, false, kFieldAny, kKeepRecords);      \
  } while (0)
    KFD_LAUNCH(true);
    if (between) {
      const hipError_t e = hipEventRecord(between, stream);
      if (e != hipSuccess) return e;
    }
    // without smoothing the forward kernel finishes every track
    if (args->smoothing) KFD_LAUNCH(false);
#undef KFD_LAUNCH
#undef KFD_LAUNCH1
#undef KFD_LAUNCH2
    return hipGetLastError();
  }
  const bool plds = args->n_planes <= (sizeof(S) == sizeof(double) ? KF_FUSED_LDS_PLANES_FP64
                                                                   : KF_FUSED_LDS_PLANES_MIXED);
  const dim3 fgrid((unsigned)((args->count * lpt + KF_FUSED_BLOCK - 1) / KF_FUSED_BLOCK +
                              rtsBlocksOf(*args)));
  const unsigned table = plds ? (unsigned)(args->n_planes * sizeof(DevPlane)) : 0u;
#define KFD_FUSED2(PLDS_, L_, FK_)                                                             \
  hipLaunchKernelGGL((kf_fused_kernel<S, PLDS_, L_, FK_>), fgrid, dim3(KF_FUSED_BLOCK), table, \
                     stream, *args)
#define KFD_FUSED1(PLDS_, FK_)     \
  do {                             \
    if (lpt == 1)                  \
      KFD_FUSED2(PLDS_, 1, FK_);   \
    else if (lpt == 2)             \
      KFD_FUSED2(PLDS_, 2, FK_);   \
    else                           \
      KFD_FUSED2(PLDS_, 4, FK_);   \
  } while (0)
  if (!plds)
    KFD_FUSED1(false, kFieldAny);
  else if (args->field.grid)
    KFD_FUSED1(true, kFieldGrid);
  else
    KFD_FUSED1(true, kFieldConst);
#undef KFD_FUSED1
#undef KFD_FUSED2
  if (between) {
    const hipError_t e = hipEventRecord(between, stream);
    if (e != hipSuccess) return e;
  }
  if (args->smoothing && !redoSlotPerTrack(*args)) {
    const dim3 rgrid((unsigned)((args->redo_lanes + KF_FUSED_BLOCK - 1) / KF_FUSED_BLOCK));
#define KFD_REDO(PLDS_, FK_)                                                                  \
  hipLaunchKernelGGL((kf_redo_kernel<S, PLDS_, FK_>), rgrid, dim3(KF_FUSED_BLOCK), table, stream, \
                     *args)
    if (!plds)
      KFD_REDO(false, kFieldAny);
    else if (args->field.grid)
      KFD_REDO(true, kFieldGrid);
    else
      KFD_REDO(true, kFieldConst);
#undef KFD_REDO
  }
  return hipGetLastError();
}

}  // namespace kfd
