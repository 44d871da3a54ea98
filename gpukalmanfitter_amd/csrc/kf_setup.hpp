// kf_setup.hpp -- host-side preparation of the kernel arguments: the
// device plane record and the physics constants.  Shared by the C ABI
// (kf_api.hip) and the CPU build of the per-track code used by the tests.
#pragma once

#include <cfloat>
#include <cmath>
#include <cstring>
#include <vector>

#include "kf_kernels.hpp"

namespace kfd {

// Whether a fit sorts its tracks by length: as the schedule says, or (KF_SORT_AUTO)
// where a fused fit gains from it.  A wave takes as long as its longest track, so
// where the tracks fill fewer than 4/5 of the states they may have (the caller's
// max_states; a batch whose longest track is not stated is left alone) and the
// waves exceed one per SIMD, lengths sorted into waves shorten the launch by more
// than the sort and the scattered reads cost: filled to 0.55-0.60, 66,000 tracks
// 745 -> 450 us (FP64, 5-30 planes) and 1,334 -> 831 us (mixed, 8-40 planes with
// material), 500,003 tracks 2,719 -> 2,036 us; with equal lengths, where holes or a
// loose max_states make them look unequal, 100,000 tracks go from 191 to 205 us (four
// launches; a schedule with sort_by_length = 0 spares them).
// Up to one wave per SIMD the longest track decides, sorted or not.
inline bool sortsByLength(const kf_schedule &sc, bool fused, int64_t n_tracks, int64_t n_hits,
                          int32_t max_states, int n_cu) {
  if (sc.sort_by_length != KF_SORT_AUTO) return sc.sort_by_length != 0;
  return fused && max_states > 0 && n_tracks * sc.lanes_per_track > (int64_t)256 * n_cu &&
         (double)n_hits < 0.8 * (double)n_tracks * (double)max_states;
}

// The schedules that an autotuner times: those that differ in what a fit launches.
// Every fit: sorted and not, 1, 2 and 4 lanes per track.  One with track states
// also has its store slots by plane and its work queue, which the fused kernel of
// the others has not.
inline std::vector<kf_schedule> scheduleCandidates(bool track_states) {
  std::vector<kf_schedule> cand;
  for (int sort = 0; sort <= 1; ++sort)
    for (int byPlane = 0; byPlane <= (track_states ? 1 : 0); ++byPlane) {
      kf_schedule c{};
      c.sort_by_length = sort;
      c.waves_per_cu = 4;
      c.chunks_per_grab = 1;
      c.graph = 1;
      c.store_by_plane = byPlane;
      for (int l : {1, 2, 4}) {  // lane groups: slots by measurement
        c.lanes_per_track = l;
        if (l == 1 || !byPlane) cand.push_back(c);
      }
      if (!track_states) continue;
      c.lanes_per_track = 1;
      c.persistent = 1;
      for (int w : {2, 4, 8})
        for (int g : {1, 4}) {
          c.waves_per_cu = w;
          c.chunks_per_grab = g;
          cand.push_back(c);
        }
    }
  return cand;
}

// Physics constants evaluated the way the reference's unit literals do
// (long double literal times a double unit, rounded to double;
// Interactions.ipp:19-25, Units.hpp:145-153) and its float literals.
inline void physicsConstants(FitArgs &a) {
  a.kMe = (double)(0.001L * 0.5109989461L);
  a.kK = ((double)(0.001L * 0.307075L)) * 10.0 * 10.0;
  a.kPlasma = (double)(1e-9L * 28.816L);
  a.kHighland = (double)(0.001L * 13.6L);
  const float c = 0.038f * 2;
  a.kHighlandLog = (double)c;
  const float conv = 2 * std::sqrt(2 * std::log(2.0f));
  a.kLandauConv = (double)conv;
}

// Device plane record: frame, and the MaterialSlab (MaterialSlab.ipp:15-20)
// and Material (Material.ipp:80-85, Material.hpp:102-104) quantities, only
// when the slab is valid (MaterialSlab.hpp:46-48).
inline DevPlane devPlane(const kf_plane &p) {
  DevPlane d;
  std::memset(&d, 0, sizeof d);
  for (int k = 0; k < 3; ++k) d.c[k] = p.center[k];
  for (int k = 0; k < 9; ++k) d.r[k] = p.rot[k];
  const bool valid = p.thickness > 0.0 && 0.0f < p.ar;
  d.has_material = valid ? 1 : 0;
  if (valid) {
    const double eps = 2 * DBL_EPSILON;
    d.thickness = p.thickness;
    d.thicknessInX0 = (eps < p.x0) ? (p.thickness / p.x0) : 0.0;
    d.meanExcitation = (16.0 * 1e-9) * std::pow(p.z, (double)0.9f);
    d.molarElectronDensity = p.z * p.molar_rho;
  }
  d.geo_id = p.geo_id;
  return d;
}

}  // namespace kfd
