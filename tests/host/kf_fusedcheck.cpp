// kf_fusedcheck.cpp -- CPU build of the fused fit program (TrackFit with the
// fixed-point smoother), for the tests: the same source the GPU runs, one
// track at a time.  Test infrastructure only: the library never loads it.
#include "kf_hostcheck.cpp"

namespace {

template <typename S, int FK>
void fusedTracks(Host &h, int32_t *redo, bool early = false) {
  using Fit = TrackFit<S, true, 1, false, false, FK, kKeepFirst>;
  std::vector<typename Fit::FxPair> sums((size_t)Fit::kFxN * KF_FUSED_BLOCK);
  for (int64_t i = 0; i < h.a.n; ++i) {
    Fit tf(h.a, i, nullptr, nullptr, nullptr, nullptr, 0u, i);
    tf.pls = h.planes.data();
    tf.fx = sums.data();
    tf.leaveEarly = early;
    redo[i] = tf.runFused() ? 0 : 1;
  }
}

}  // namespace

extern "C" {

// The fit of every track by the fused program, built for either field kind
// (0), the constant field (1) or the grid (2): params [6][n], cov [21][n],
// chi2, n_measured, status [n], and redo [n], nonzero for a track that it
// leaves to the RTS program (its params, cov and status are not set).
int kfh_fit_fused_kind(const kf_plane *planes, int32_t n_planes, const kfh_field *f,
                       const kf_tracks *tr, const kf_options *opt, int32_t field_kind,
                       double *params, double *cov, double *chi2, int32_t *n_measured,
                       uint32_t *status, int32_t *redo) {
  Host h(planes, n_planes, f, tr, opt, true);
  h.a.out_params = params;
  h.a.out_cov = cov;
  h.a.out_chi2 = chi2;
  h.a.out_nmeas = n_measured;
  h.a.out_status = status;
  h.a.out_ndf = nullptr;
  const bool mixed = opt->precision == KF_PRECISION_MIXED;
  if (mixed && field_kind == kFieldGrid)
    fusedTracks<float, kFieldGrid>(h, redo);
  else if (mixed && field_kind == kFieldConst)
    fusedTracks<float, kFieldConst>(h, redo);
  else if (mixed)
    fusedTracks<float, kFieldAny>(h, redo);
  else if (field_kind == kFieldGrid)
    fusedTracks<double, kFieldGrid>(h, redo);
  else if (field_kind == kFieldConst)
    fusedTracks<double, kFieldConst>(h, redo);
  else
    fusedTracks<double, kFieldAny>(h, redo);
  return 0;
}

int kfh_fit_fused(const kf_plane *planes, int32_t n_planes, const kfh_field *f,
                  const kf_tracks *tr, const kf_options *opt, double *params, double *cov,
                  double *chi2, int32_t *n_measured, uint32_t *status, int32_t *redo) {
  return kfh_fit_fused_kind(planes, n_planes, f, tr, opt, kFieldAny, params, cov, chi2,
                            n_measured, status, redo);
}

// As the kernel runs it: a track with a singular start covariance is left before
// the pass, its chi2 and n_measured not set either.
int kfh_fit_fused_early(const kf_plane *planes, int32_t n_planes, const kfh_field *f,
                        const kf_tracks *tr, const kf_options *opt, double *params, double *cov,
                        double *chi2, int32_t *n_measured, uint32_t *status, int32_t *redo) {
  Host h(planes, n_planes, f, tr, opt, true);
  h.a.out_params = params;
  h.a.out_cov = cov;
  h.a.out_chi2 = chi2;
  h.a.out_nmeas = n_measured;
  h.a.out_status = status;
  h.a.out_ndf = nullptr;
  if (opt->precision == KF_PRECISION_MIXED)
    fusedTracks<float, kFieldAny>(h, redo, true);
  else
    fusedTracks<double, kFieldAny>(h, redo, true);
  return 0;
}

// The square roots and their reciprocals of x [n] from estimates y of 1 / sqrt(x).
void kfh_roots(int64_t n, const double *x, const double *y, double *s, double *is) {
  for (int64_t i = 0; i < n; ++i) rootFromEven(x[i], y[i], s[i], is[i]);
}

// Whether a fit with this schedule sorts its tracks.
int kfh_sorts(const kf_schedule *s, int32_t fused, int64_t n_tracks, int64_t n_hits,
              int32_t max_states, int32_t n_cu) {
  return sortsByLength(*s, fused != 0, n_tracks, n_hits, max_states, n_cu) ? 1 : 0;
}
// The autotuner's candidates (at most `capacity` of them); their number.
int kfh_schedule_candidates(int32_t track_states, kf_schedule *out, int32_t capacity) {
  const std::vector<kf_schedule> c = scheduleCandidates(track_states != 0);
  for (size_t k = 0; k < c.size() && k < (size_t)capacity; ++k) out[k] = c[k];
  return (int)c.size();
}

// Whether each track is given to the RTS program from the start (nearWrap).
int kfh_near_wrap(const kf_plane *planes, int32_t n_planes, const kfh_field *f,
                  const kf_tracks *tr, const kf_options *opt, int32_t *pick) {
  Host h(planes, n_planes, f, tr, opt, true);
  for (int64_t i = 0; i < h.a.n; ++i) pick[i] = nearWrap(&h.a, i) ? 1 : 0;
  return 0;
}

}  // extern "C"
