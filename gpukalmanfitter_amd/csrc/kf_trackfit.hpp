// kf_trackfit.hpp -- the per-track Kalman fit program (one track per lane),
// shared by the fit kernels (kf_fit_kernels.hpp) and the chi2 adjoint
// (kf_adjoint.hip).
//
// The per-lane program is the reference's propagation loop (Propagator.ipp:
// 3-96): step -> navigator status -> Kalman actor -> aborters -> navigator
// target, until the Kalman aborter fires.  The loop is arranged so lanes
// re-converge before the expensive actor work: the inner loop runs the
// iterations in which the actor has nothing to do (no surface reached, no
// finalisation, target not reached), and only exits when a lane has a surface
// update, the smoother or the final perigee transport due.  Every lane still
// executes exactly the reference's per-iteration sequence.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "kf_device.hpp"
#include "kf_kernels.hpp"

namespace kfd {

// FWD = true: the forward kernel (start, steps, filter at every surface) that
// stops where the reference's actor would call finalize() and saves a carry
// record; FWD = false: the backward kernel (smoother, then propagation back to
// the perigee) that resumes from that record.
enum { kResumeNone = 0, kResumePreLoop = 1, kResumeInLoop = 2, kResumePostLoop = 3 };

// Whether a track of a fused fit is given to the RTS program from the start
// because one of its angles may come near the phi wrap, where the fixed-point
// smoother would leave it in the end (TrackFit::fxAngles): whether the interval
// that phi runs through from the perigee to the last plane of the sequence, widened
// for the start's errors, reaches +-pi.  The length is the straight line's and
// the turning rate the start's, q/p (d_z (d_x B_x + d_y B_y) / d_T^2 - B_z): an
// estimate, in float, and one that may be wrong either way, since both programs
// give the track's fit; a track that it misses is only fitted twice.
//
// Of tracks all facing phi = pi it picks 13-17 % (4.4-9.3 % are left in the end),
// spread over azimuth 0.8-1.3 % (0.3-0.9 %), and misses none of ten planes and
// 0.3 % facing pi, 0.05 % spread, of 8-40 planes of material.  Widened by three
// errors instead of two it picks a sixth more and misses as many.  Only tracks that
// start within kNearWrapPhi of pi are asked for.
//
// A call of its own, so that every kernel that asks has the same bits decide: the
// lanes that leave a track out and those that fit it must agree.
constexpr double kNearWrapPhi = 1.5;
__host__ __device__ __attribute__((noinline)) inline bool nearWrap(const FitArgs *args,
                                                                   int64_t i) {
  const FitArgs &a = *uniformArgs(args);
  const int64_t n = a.n;
  const double phi = a.start_params[2 * n + i];
  const int first = a.seq_first[i], size = a.seq_count[i];
  if (!(fabs(phi) > kNearWrapPhi) || size <= 0 || first < 0 || (int64_t)first + size > a.n_planes)
    return false;
  const float theta = (float)a.start_params[3 * n + i], qop = (float)a.start_params[4 * n + i];
  const float vPhi = (float)a.start_cov[sidx(2, 2) * n + i];
  const float vQop = (float)a.start_cov[sidx(4, 4) * n + i];
  const float x[3] = {(float)a.perigee[i], (float)a.perigee[n + i],
                      (float)(a.perigee[2 * n + i] + a.start_params[n + i])};
  const DevPlane &pl = a.planes[first + size - 1];
  const float nr[3] = {(float)pl.r[2], (float)pl.r[5], (float)pl.r[8]};
  const float v[3] = {(float)pl.c[0] - x[0], (float)pl.c[1] - x[1], (float)pl.c[2] - x[2]};
  float B[3];
  fieldNear(a.field, x, B);
#if defined(__HIP_DEVICE_COMPILE__)
  const float sp = __sinf((float)phi), cp = __cosf((float)phi), st = __sinf(theta),
              ct = __cosf(theta);
#else
  const float sp = sinf((float)phi), cp = cosf((float)phi), st = sinf(theta), ct = cosf(theta);
#endif
  const float rate = qop * (ct / st * (cp * B[0] + sp * B[1]) - B[2]);
  const float along = st * (cp * nr[0] + sp * nr[1]) + ct * nr[2];
  const float turn = rate * (dot3(nr, v) / along);
  const float wide = 0.005f + 2.0f * sqrtf(vPhi) + fabsf(turn) * (0.05f + 2.0f * sqrtf(vQop) / fabsf(qop));
  const float reach = (phi > 0.0) ? fmaxf((float)phi, (float)phi + turn) + wide
                                  : wide - fminf((float)phi, (float)phi + turn);
  return reach >= (float)kPi;
}

// L: lanes per track (1, 2 or 4; kf_device.hpp, lane groups).  The lanes of a
// group run this program on the same data; in the mixed mode the free
// transport matrix of each RK step is built column by column across them, and
// only the group's first lane writes to memory.
//
// KEEP: what a fit keeps of its measured states.
//  kKeepRecords  the per-state store, from which the backward kernel runs the
//                RTS smoother over all states, and the track-state records or
//                adjoint checkpoints where asked for;
//  kKeepStates   the store only (both record stores are null at compile time
//                and their writes not in the code);
//  kKeepCheckpoints  the adjoint's checkpoints only (no smoother follows);
//  kKeepFirst    only the smoothed state of the first measured surface is
//                wanted (it is what propagates to the perigee): the forward
//                pass carries a fixed-point smoother for it (below), nothing is
//                stored per state, and one kernel runs the whole fit (runFused).
enum { kKeepRecords = 0, kKeepStates = 1, kKeepFirst = 2, kKeepCheckpoints = 3 };
template <typename S, bool FWD, int L = 1, bool PS = false, bool OOL = false, int FK = kFieldAny,
          int KEEP = kKeepRecords>
struct TrackFit {
  static constexpr bool kRecords = KEEP == kKeepRecords;
  static constexpr bool kStore = KEEP == kKeepRecords || KEEP == kKeepStates;
  static constexpr bool kFirst = KEEP == kKeepFirst;
  static constexpr bool kMixed = sizeof(S) < sizeof(double);
  const FitArgs &a;
  const int64_t i;
  // index of this lane in its group, and whether it writes the track's
  // records and outputs
  uint32_t rank = 0;
  bool lead = true;
  KFD_INLINE void setRank(uint32_t r) {
    rank = r;
    lead = (r == 0);
  }

  // ---- stepper state (EigenStepper::State, EigenStepper.hpp:27-120) ----
  double pos[3], dir[3], p, t, q;
  int navDir;
  CStep ss;
  double pathAcc;
  // bound covariance (packed upper triangle).  S: in the mixed mode every
  // consumer of it between surfaces (the next sandwich, the stores) takes it
  // in float, so it is kept in float (half the registers)
  S cov[21];
  // free-from-bound Jacobian J (8x6).  Non-constant entries only:
  // A = J[0:3, 0:5], b = J[3, 4], G = J[4:7, 2:5]; J[3,5] = J[7,4] = 1, the
  // rest is zero between surfaces.
  S A[3][5];
  S b;
  S G[3][3];
  // propagation derivative (dir, dt/ds, k4, 0) of the last step; zero after
  // a Jacobian re-initialisation
  S k4d[3];
  S dtds;
  bool derivSet;
  bool stepFailed;

  // ---- navigation (DirectNavigator::State) ----
  int next, size, seqFirst;
  int cur;  // -1: none, -2: the perigee target, >= 0: plane-table index
  bool targetReached, navBreak;

  // ---- KalmanFitterResult ----
  int measured;
  int outliers;    // measured states the outlier finder left without an update
  int firstPlane;  // plane-table index of the first measured state
  // store slots (KF_SD_* / KF_SS_*).  PS = false: the slot of measured state
  // k is k.  PS = true (kf_schedule.store_by_plane): k + min(holes before
  // it, max_states - hits), i.e. its plane's position in the sequence
  // whenever the sequence fits max_states slots.  holes counts the planes
  // passed without a hit; slotLast / slotPrev are the slots of the last two
  // measured states.
  int holes, slotLast, slotPrev;
  bool smoothed, finished, result, smootherNaN;
  int64_t h0, h1;
  // hit search: while every match so far was the next hit in order and the
  // plane geo ids are distinct (inOrder), no hit before hitNext can match a
  // later plane, so the search starts at hitNext, whose data is loaded ahead
  // (pf*) while the track steps to the next surface
  int64_t hitNext;
  bool inOrder, pfValid;
  int32_t pfGeo;
  double pfM0, pfM1, pfV00, pfV01, pfV11;
  KFD_INLINE void prefetchHit() {
    pfValid = hitNext < h1;
    if (pfValid) {
      pfGeo = a.hit_geo_id[hitNext];
      pfM0 = a.hit_meas[hitNext];
      pfM1 = a.hit_meas[a.n_hits + hitNext];
      pfV00 = a.hit_cov[hitNext];
      pfV01 = a.hit_cov[a.n_hits + hitNext];
      pfV11 = a.hit_cov[2 * a.n_hits + hitNext];
    }
  }
  double chi2sum;
  double lc[3];  // perigee line point

  // quantities of the momentum used by every step, recomputed when p changes:
  // q/p, sqrt(1 + (m/p)^2) (dt/ds), and the transport's d(time)/d(q/p) per
  // unit step, m^2 q / (p sqrt(1 + (m/p)^2)) times q^2 = 1
  double cacheP = -1.0, cacheQ = 0.0, cacheQop = 0.0, cacheDtds = 0.0, cacheD37 = 0.0;
  KFD_INLINE void momentumCache() {
    if (p != cacheP || q != cacheQ) {
      cacheP = p;
      cacheQ = q;
      cacheQop = divD(q, p);
      const double mp = divD(a.mass, p);
      double is;
      rootD(1.0 + mp * mp, cacheDtds, is);
      cacheD37 = (a.mass * q) * (mp * is);
    }
  }
  // The direction and angles after the last update (or of the start
  // parameters): the angles at the next plane follow from the rotation
  // between the two directions (planeAngles).
  double refPhi = 0.0, refTheta = 0.0, refX = 0.0, refY = 0.0, refZ = 0.0;
  KFD_INLINE void setReference(const double par[6]) {
    refPhi = par[2];
    refTheta = par[3];
    refX = dir[0];
    refY = dir[1];
    refZ = dir[2];
  }
  // the last plane intersection computed by surfaceStatus (path length along
  // the direction, denominator n.d): navStatus and navTarget of one
  // iteration usually ask for the same plane; valid until pos, dir or navDir
  // change (moved())
  int pathPlane = -1;
  double pathLen = 0.0, pathDenom = 0.0;
  KFD_INLINE void moved() { pathPlane = -1; }
  // options read in every iteration
  double tol, negOverstep, outlierCut;
  int maxSteps;
  KFD_INLINE void loadOptions() {
    tol = inVgpr(a.tolerance);
    negOverstep = inVgpr(-a.overstep_limit);
    outlierCut = inVgpr(a.outlier_chi2_cut);
    maxSteps = inVgpr(a.max_steps);
  }

  // per-state stores of this wave's 64-track chunk (wave-uniform bases) and
  // this lane's slot in them
  double *tsd;
  S *tss;
  double *tsf;
  double *tsc;
  // the plane table: a copy in LDS (set by the kernel) or a.planes
  const DevPlane *pls;
  uint32_t lane;
  // slot of the forward -> backward hand-over record: the position within
  // the launch, so consecutive lanes use consecutive slots
  int64_t cpos;
  // slots of the hand-over buffer (its field stride)
  int64_t cslots;
  int32_t *ciBase;
  double *cdBase;

  KFD_INLINE TrackFit(const FitArgs &args, int64_t idx, double *d_base, S *s_base, double *f_base,
                      double *c_base, uint32_t ln, int64_t carry_slot = 0)
      : a(args), i(idx), tsd(d_base), tss(s_base), tsf(kRecords ? f_base : nullptr),
        tsc(kRecords || KEEP == kKeepCheckpoints ? c_base : nullptr), pls(args.planes), lane(ln), cpos(carry_slot), cslots(args.count),
        ciBase(args.carry_i), cdBase(args.carry_d) {}

  // The hand-over buffer of tracks fitted again after a fused fit.
  KFD_INLINE void redoSlots() {
    ciBase = a.redo_i;
    cdBase = a.redo_d;
    cslots = a.redo_lanes;
  }

  // ------------------------------------------------------------ storage ----
  // Element f of state k: base[(k * F + f) * 64 + lane] -- a 32-bit lane
  // offset from a wave-uniform base, so each access is one saddr load/store.
  KFD_INLINE static uint32_t slot(int k, int F, int f, uint32_t ln) {
    return (uint32_t)(((uint32_t)k * (uint32_t)F + (uint32_t)f) * 64u + ln);
  }
  KFD_INLINE double *recF(int k, int f) const { return tsf + slot(k, KF_TS_STRIDE, f, lane); }
  // The smoother stores tsd / tss in 16-byte groups per lane: the group of
  // element f (f a multiple of W = 16 / sizeof(element)) of state k at
  // base[(k * F + f) * 64 + lane * W].
  static constexpr int kW = 16 / (int)sizeof(S);
  KFD_INLINE static uint32_t gslot(int k, int F, int f, int W, uint32_t ln) {
    return (uint32_t)(((uint32_t)k * (uint32_t)F + (uint32_t)f) * 64u + ln * (uint32_t)W);
  }
  KFD_INLINE double *grpD(int k, int f) const { return tsd + gslot(k, KF_SD_N, f, 2, lane); }
  KFD_INLINE S *grpS(int k, int f) const { return tss + gslot(k, KF_SS_N, f, kW, lane); }
  // The forward kernel's store writes are non-temporal: the backward kernel
  // reads them back only after the whole forward launch (gigabytes later),
  // so they need not displace the hits and plane data in the caches
  // (measured: forward 2-3 %, backward 3 % faster on 1,048,576 tracks).
  typedef float v4f __attribute__((ext_vector_type(4)));
  typedef double v2d __attribute__((ext_vector_type(2)));
  KFD_INLINE static void st16(float *p, const float *v) {
    const v4f x = {v[0], v[1], v[2], v[3]};
    __builtin_nontemporal_store(x, (v4f *)p);
  }
  KFD_INLINE static void st16(double *p, const double *v) {
    const v2d x = {v[0], v[1]};
    __builtin_nontemporal_store(x, (v2d *)p);
  }
  // a store slot index kept in a padding element of the S store, bit for bit
  KFD_INLINE static float linkBits(int s, float) { return __builtin_bit_cast(float, s); }
  KFD_INLINE static double linkBits(int s, double) {
    return __builtin_bit_cast(double, (int64_t)s);
  }
  KFD_INLINE static int linkOf(float v) { return __builtin_bit_cast(int, v); }
  KFD_INLINE static int linkOf(double v) { return (int)__builtin_bit_cast(int64_t, v); }
  KFD_INLINE static void ld16(const float *p, float *v) {
    const float4 x = *(const float4 *)p;
    v[0] = x.x;
    v[1] = x.y;
    v[2] = x.z;
    v[3] = x.w;
  }
  KFD_INLINE static void ld16(const double *p, double *v) {
    const double2 x = *(const double2 *)p;
    v[0] = x.x;
    v[1] = x.y;
  }
  // six parameters at tsd element f (0 or 6) of state k
  KFD_INLINE void storePar(int k, int f, const double v[6]) const {
    if (!lead) return;
#pragma unroll
    for (int g = 0; g < 6; g += 2) st16(grpD(k, f + g), v + g);
  }
  KFD_INLINE void loadPar(int k, int f, double v[6]) const {
#pragma unroll
    for (int g = 0; g < 6; g += 2) ld16(grpD(k, f + g), v + g);
  }
  // n elements (a multiple of kW) at tss element f of state k
  template <int N>
  KFD_INLINE void storeS(int k, int f, const S v[N]) const {
    if (!lead) return;
#pragma unroll
    for (int g = 0; g < N; g += kW) st16(grpS(k, f + g), v + g);
  }
  template <int N>
  KFD_INLINE void loadS(int k, int f, S v[N]) const {
#pragma unroll
    for (int g = 0; g < N; g += kW) ld16(grpS(k, f + g), v + g);
  }
  KFD_INLINE double *recC(int k, int f) const { return tsc + slot(k, KF_CK_N, f, lane); }

  // Checkpoint k: the state right after the update and material of measured
  // surface k, from which the adjoint recomputes the next segment.
  KFD_INLINE void saveCheckpoint(int k, int64_t hit) const {
    if (!lead) return;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      *recC(k, KF_CK_POS + m) = pos[m];
      *recC(k, KF_CK_DIR + m) = dir[m];
    }
    *recC(k, KF_CK_P) = p;
    *recC(k, KF_CK_ACC) = ss.v[kAccuracy];
    *recC(k, KF_CK_ACT) = ss.v[kActor];
    int m = 0;
#pragma unroll
    for (int r = 0; r < 5; ++r)
#pragma unroll
      for (int c = r; c < 5; ++c, ++m) *recC(k, KF_CK_COV + m) = cov[sidx(r, c)];
    *recC(k, KF_CK_G + 0) = (double)G[0][0];
    *recC(k, KF_CK_G + 1) = (double)G[0][1];
    *recC(k, KF_CK_G + 2) = (double)G[1][0];
    *recC(k, KF_CK_G + 3) = (double)G[1][1];
    *recC(k, KF_CK_G + 4) = (double)G[2][1];
    *recC(k, KF_CK_NEXT) = (double)next;
    *recC(k, KF_CK_HIT) = (double)(hit - h0);
  }

  KFD_INLINE void loadCheckpoint(int k) {
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      pos[m] = *recC(k, KF_CK_POS + m);
      dir[m] = *recC(k, KF_CK_DIR + m);
    }
    p = *recC(k, KF_CK_P);
    t = 0.0;
    pathAcc = 0.0;
    ss.init(1.0 * fabs(a.max_step_size));
    ss.v[kAccuracy] = *recC(k, KF_CK_ACC);
    ss.v[kActor] = *recC(k, KF_CK_ACT);
    ss.dir = 1;
    navDir = 1;
    moved();
#pragma unroll
    for (int m = 0; m < 21; ++m) cov[m] = (S)0;
    int m = 0;
#pragma unroll
    for (int r = 0; r < 5; ++r)
#pragma unroll
      for (int c = r; c < 5; ++c, ++m) cov[sidx(r, c)] = *recC(k, KF_CK_COV + m);
    next = (int)*recC(k, KF_CK_NEXT);
    const DevPlane &pl = pls[seqFirst + next - 1];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      A[r][0] = (S)pl.r[3 * r + 0];
      A[r][1] = (S)pl.r[3 * r + 1];
      A[r][2] = A[r][3] = A[r][4] = (S)0;
      G[r][2] = (S)0;
    }
    b = (S)0;
    G[0][0] = (S)*recC(k, KF_CK_G + 0);
    G[0][1] = (S)*recC(k, KF_CK_G + 1);
    G[1][0] = (S)*recC(k, KF_CK_G + 2);
    G[1][1] = (S)*recC(k, KF_CK_G + 3);
    G[2][0] = (S)0;
    G[2][1] = (S)*recC(k, KF_CK_G + 4);
    derivSet = false;
    k4d[0] = k4d[1] = k4d[2] = (S)0;
    dtds = (S)0;
  }
  // public record: parameters + covariance at offset off
  template <typename T>
  KFD_INLINE void storeBoundF(int k, int off, const double par[6], const T c[21]) const {
    if (!lead) return;
#pragma unroll
    for (int m = 0; m < 6; ++m) *recF(k, off + m) = par[m];
#pragma unroll
    for (int m = 0; m < 21; ++m) *recF(k, off + 6 + m) = (double)c[m];
  }
  // packed index of Jacobian entry (r, c), r in {0, 1, 2, 3, 5}, c < 5
  KFD_INLINE static constexpr int jidx(int r, int c) { return ((r < 4) ? r : 4) * 5 + c; }

  // -------------------------------------------------------------- field ----
  // FK: the field kind the kernel was built for (kFieldConst and
  // kFieldGrid leave the other kind's code out of the step loop)
  // The grid cell of the last lookup; only in the fits' grid builds (the
  // either-kind builds and the adjoint are at the register limit, its 26
  // registers cost them 7 %).
  GridCell cell;
  KFD_INLINE void field(const double x[3], double B[3]) {
    if constexpr (FK == kFieldConst)
      fieldConst(a.field, B);
    else if constexpr (FK == kFieldGrid && !OOL)
      fieldGrid(a.field, x[0], x[1], x[2], B, cell);
    else
      fieldAt(a.field, x[0], x[1], x[2], B);
  }

  // ------------------------------------------------ Jacobian init (plane) ----
  // PlaneSurface::initJacobianToGlobal, PlaneSurface.ipp:122-156
  KFD_INLINE void initJacobianPlane(const DevPlane &pl, double cosT, double sinT, double cosP,
                                    double sinP) {
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      A[r][0] = (S)pl.r[3 * r + 0];
      A[r][1] = (S)pl.r[3 * r + 1];
      A[r][2] = (S)0;
      A[r][3] = (S)0;
      A[r][4] = (S)0;
    }
    b = (S)0;
    G[0][0] = (S)((-sinT) * sinP);
    G[0][1] = (S)(cosT * cosP);
    G[1][0] = (S)(sinT * cosP);
    G[1][1] = (S)(cosT * sinP);
    G[2][0] = (S)0;
    G[2][1] = (S)(-sinT);
    G[0][2] = G[1][2] = G[2][2] = (S)0;
    derivSet = false;
    k4d[0] = k4d[1] = k4d[2] = (S)0;
    dtds = (S)0;
  }

  // ------------------------------------------------------------- start ----
  // BoundParameters<LineSurface>(cov, params, &perigee) (SingleBound-
  // TrackParameters.hpp:48-60), EigenStepper::State ctor (EigenStepper.hpp:
  // 41-61) and LineSurface::initJacobianToGlobal (LineSurface.ipp:63-112).
  KFD_INLINE void start(const double pv[6]) {
    const double pabs = fabs(1.0 / pv[4]);
    const SinCos s3 = sinCosD(pv[3]), s2 = sinCosD(pv[2]);
    const double mom[3] = {pabs * s3.s * s2.c, pabs * s3.s * s2.s, pabs * s3.c};
    // LineSurface::localToGlobal: centre + (0,0,loc1) + loc0 * |z x mom|
    const double ra[3] = {0.0 - mom[1], mom[0] - 0.0, 0.0};
    const double ran = sqrt(ra[0] * ra[0] + ra[1] * ra[1] + ra[2] * ra[2]);
    const double raN[3] = {ra[0] / ran, ra[1] / ran, ra[2] / ran};
    const double locz[3] = {0.0 + lc[0], 0.0 + lc[1], pv[1] + lc[2]};
#pragma unroll
    for (int k = 0; k < 3; ++k) pos[k] = locz[k] + pv[0] * raN[k];
    const double charge = (pv[4] > 0.0) ? 1.0 : -1.0;
    double pc[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) pc[k] = pv[k];
    correctParams(pc);
    const double mn = sqrt(mom[0] * mom[0] + mom[1] * mom[1] + mom[2] * mom[2]);
#pragma unroll
    for (int k = 0; k < 3; ++k) dir[k] = mom[k] / mn;
    p = mn;
    q = charge;
    t = pc[5];
    setReference(pc);
    if (pc[3] != pv[3]) refX = refY = 0.0;  // theta was clamped: not the direction's
    navDir = 1;
    moved();
    ss.init(1.0 * fabs(a.max_step_size));
    pathAcc = 0.0;
    // line initJacobianToGlobal at (pos, dir) with the corrected parameters
    const double cosT = dir[2];
    const double sinT = sqrt(dir[0] * dir[0] + dir[1] * dir[1]);
    const double invSinT = 1.0 / sinT;
    const double cosP = dir[0] * invSinT, sinP = dir[1] * invSinT;
    const double mxr[3] = {0.0 * dir[2] - 1.0 * dir[1], 1.0 * dir[0] - 0.0 * dir[2],
                           0.0 * dir[1] - 0.0 * dir[0]};
    const double mxn = sqrt(mxr[0] * mxr[0] + mxr[1] * mxr[1] + mxr[2] * mxr[2]);
    const double mX[3] = {mxr[0] / mxn, mxr[1] / mxn, mxr[2] / mxn};
    const double mY[3] = {0.0, 0.0, 1.0};
    double mD[3];
    cross(mX, mY, mD);
    const double j42 = (-sinT) * sinP, j43 = cosT * cosP, j52 = sinT * cosP, j53 = cosT * sinP;
    const double j63 = (-sinT);
    const double ipdn = 1.0 / dot3(dir, mD);
    const double dPhi[3] = {j42, j52, 0.0};
    const double dTheta[3] = {j43, j53, j63};
    double dDPhiY[3], dDThetaY[3];
    cross(mY, dPhi, dDPhiY);
    cross(mY, dTheta, dDThetaY);
    const double xp = dot3(mX, dDPhiY), xt = dot3(mX, dDThetaY);
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      dDPhiY[r] = dDPhiY[r] - xp * mX[r];
      dDThetaY[r] = dDThetaY[r] - xt * mX[r];
    }
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      A[r][0] = (S)mX[r];
      A[r][1] = (S)mY[r];
      A[r][2] = (S)(dDPhiY[r] * pc[0] * ipdn);
      A[r][3] = (S)(dDThetaY[r] * pc[0] * ipdn);
      A[r][4] = (S)0;
    }
    b = (S)0;
    G[0][0] = (S)j42;
    G[0][1] = (S)j43;
    G[1][0] = (S)j52;
    G[1][1] = (S)j53;
    G[2][0] = (S)0;
    G[2][1] = (S)j63;
    G[0][2] = G[1][2] = G[2][2] = (S)0;
    derivSet = false;
    k4d[0] = k4d[1] = k4d[2] = (S)0;
    dtds = (S)0;
    stepFailed = false;
  }

  // Library sin/cos, atan2 and log: out of line with OOL (the chi2 adjoint's
  // segment recompute, see oolSinCos), inline in the fit kernels (measured
  // faster there: the calls on every surface cost more than the registers
  // they free).
  // The length that a direction is divided by, once per step and per plane.  In the
  // adjoint's builds without the lean of rootD: summed over 262,144 tracks whose
  // terms cancel it was 1.3 times the gradient's error against 64 bits (2.9e-13 ->
  // 1.9e-13, 2.2e-13 with library roots).  The other fits sum nothing over tracks; the
  // residual costs the mixed one 2 %.
  static constexpr bool kEvenRoots = OOL || KEEP == kKeepCheckpoints;
  KFD_INLINE static void rootOfDirection(double x, double &s, double &is) {
    if constexpr (kEvenRoots)
      rootEven(x, s, is);
    else
      rootD(x, s, is);
  }
  KFD_INLINE static SinCos sinCosD(double x) {
    if constexpr (!OOL) {
      return SinCos{sin(x), cos(x)};
    } else {
      return oolSinCos(x);
    }
  }
  KFD_INLINE static double atan2D(double y, double x) {
    if constexpr (!OOL) {
      return atan2(y, x);
    } else {
      return oolAtan2(y, x);
    }
  }
  KFD_INLINE static S logS(S x) {
    if constexpr (!OOL || kMixed) {
      return log(x);
    } else {
      return oolLog(x);
    }
  }

  // The step-size factor after a rejected trial (EigenStepper.ipp:274-283):
  // pow(tolerance / |2 err|, 0.25) clamped to [0.25, 4].  The fourth root is
  // taken as two square roots (each correctly rounded: within an ulp of the
  // pow, the same NaN, 0 and infinity cases); the inlined library pow was
  // ~200 instructions in the step loop and its temporaries raised the loop's
  // register peak (an out-of-line call of it, or of this, measured within
  // 1 % in the FP64 kernels and slower in the mixed ones).
  KFD_INLINE static double stepScale(double tol, double err) {
    double sc = sqrt(sqrt(tol / fabs(2.0 * err)));
    sc = (0.25 < sc) ? sc : 0.25;
    return (4.0 < sc) ? 4.0 : sc;
  }

  // -------------------------------------------------------------- step ----
  // EigenStepper::step, EigenStepper.ipp:226-332, with the transport of
  // transportMatrix (:50-124) applied to J directly.
  //
  // In a constant field the stages are polynomials of x -> x x w, w = q/p B,
  // on the direction: with v1 = d x w, v2 = v1 x w and v2 x w = -w^2 v1,
  //   k1 = v1,  k2 = v1 + h/2 v2,  k3 = (1 - c) v1 + h/2 v2,
  //   k4 = (1 - 2c) v1 + h (1 - c) v2,  c = (h w / 2)^2,
  // and the error estimate k1 - k2 - k3 + k4 is -c (v1 + h v2).
  KFD_INLINE bool step() {
    double B1[3], Bm[3], Bl[3];
    field(pos, B1);
    moved();
    momentumCache();
    const double qop = cacheQop;
    double k1[3], k2[3], k3[3], k4[3];
    double u1[3], u2[3], v2[3], w[3], w2 = 0.0, c = 0.0;  // constant field
    if constexpr (FK == kFieldConst) {
#pragma unroll
      for (int k = 0; k < 3; ++k) w[k] = qop * B1[k];
      w2 = dot3(w, w);
      cross(dir, B1, u1);
#pragma unroll
      for (int k = 0; k < 3; ++k) k1[k] = qop * u1[k];
      cross(u1, w, u2);
#pragma unroll
      for (int k = 0; k < 3; ++k) v2[k] = qop * u2[k];
    } else {
      cross(dir, B1, k1);
#pragma unroll
      for (int k = 0; k < 3; ++k) k1[k] = qop * k1[k];
    }
    double err = 0.0;
    unsigned nTrials = 0;
    for (;;) {
      const double h = ss.get();
      const double h2 = h * h;
      const double half_h = h * 0.5;
      if constexpr (FK == kFieldConst) {
        c = (0.25 * h2) * w2;
        double e1 = fabs(k1[0] + h * v2[0]);
#pragma unroll
        for (int k = 1; k < 3; ++k) e1 = e1 + fabs(k1[k] + h * v2[k]);
        err = h2 * (c * e1);
      } else {
        double p1[3], tv[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) p1[k] = pos[k] + half_h * dir[k] + (h2 * 0.125) * k1[k];
        field(p1, Bm);
#pragma unroll
        for (int k = 0; k < 3; ++k) tv[k] = dir[k] + half_h * k1[k];
        cross(tv, Bm, k2);
#pragma unroll
        for (int k = 0; k < 3; ++k) k2[k] = qop * k2[k];
#pragma unroll
        for (int k = 0; k < 3; ++k) tv[k] = dir[k] + half_h * k2[k];
        cross(tv, Bm, k3);
#pragma unroll
        for (int k = 0; k < 3; ++k) k3[k] = qop * k3[k];
#pragma unroll
        for (int k = 0; k < 3; ++k) p1[k] = pos[k] + h * dir[k] + (h2 * 0.5) * k3[k];
        field(p1, Bl);
#pragma unroll
        for (int k = 0; k < 3; ++k) tv[k] = dir[k] + h * k3[k];
        cross(tv, Bl, k4);
#pragma unroll
        for (int k = 0; k < 3; ++k) k4[k] = qop * k4[k];
        double e1 = 0.0;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const double e = k1[k] - k2[k] - k3[k] + k4[k];
          e1 = (k == 0) ? fabs(e) : e1 + fabs(e);
        }
        err = h2 * e1;
      }
      err = (err < 1e-20) ? 1e-20 : err;
      if (err <= tol) break;
      // std::min(std::max(0.25, x), 4.) with its NaN behaviour: a NaN error
      // estimate (h = DBL_MAX after an actor release) scales by 0.25
      ss.assign(ss.get() * stepScale(tol, err));
      const double hn = ss.get();
      if (hn * hn < a.step_size_cutoff * a.step_size_cutoff || nTrials > a.max_rk_trials) {
        stepFailed = true;
        return false;
      }
      nTrials++;
    }
    const double h = ss.get();
    // propagationTime, EigenStepper.ipp:36-47
    const double dt = cacheDtds;
    t = t + h * dt;
    const double h6 = h * (1.0 / 6.0);
    const double hh6 = h * h6;
    // b row of J <- D J
    b = b + (S)(h * cacheD37);
    if constexpr (FK == kFieldConst && !kMixed) {
      transportConst(w, u1, u2, h, h6, hh6, c);
    } else if constexpr (!kMixed) {
      transportColumns(B1, Bm, Bl, k1, k2, k3, h, h6, hh6, qop);
    } else {
      if constexpr (FK == kFieldConst) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          k2[k] = k1[k] + (0.5 * h) * v2[k];
          k3[k] = k2[k] - c * k1[k];
          Bm[k] = Bl[k] = B1[k];
        }
      }
      transport(B1, Bm, Bl, k1, k2, k3, h, qop);
    }
    if constexpr (FK == kFieldConst) {
      // the sums of the stages below, collected by v1 and v2
      const double f1 = hh6 * (3.0 - c), f2 = hh6 * h, g1 = h6 * (6.0 - 4.0 * c);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        pos[k] = pos[k] + h * dir[k] + (f1 * k1[k] + f2 * v2[k]);
        k4[k] = (1.0 - 2.0 * c) * k1[k] + (h * (1.0 - c)) * v2[k];
        dir[k] = dir[k] + (g1 * k1[k] + f1 * v2[k]);
      }
    } else {
      // h^2/6 and h/6 as products with 1/6 (within an ulp of the quotients)
#pragma unroll
      for (int k = 0; k < 3; ++k) pos[k] = pos[k] + h * dir[k] + hh6 * (k1[k] + k2[k] + k3[k]);
#pragma unroll
      for (int k = 0; k < 3; ++k)
        dir[k] = dir[k] + h6 * (k1[k] + 2.0 * (k2[k] + k3[k]) + k4[k]);
    }
    double dn, idn;
    rootOfDirection(dir[0] * dir[0] + dir[1] * dir[1] + dir[2] * dir[2], dn, idn);
#pragma unroll
    for (int k = 0; k < 3; ++k) dir[k] = dir[k] * idn;
    derivSet = true;
    dtds = (S)dt;
#pragma unroll
    for (int k = 0; k < 3; ++k) k4d[k] = (S)k4[k];
    if constexpr (kRecords) pathAcc = pathAcc + h;
    return true;
  }

  // J <- D J in a constant field, double: D's direction blocks are the
  // polynomials of step() applied to each column g of J's direction rows
  // (with v1 = g x w, v2 = v1 x w: dF g = h g + h^2/6 ((3 - c) v1 + h v2),
  // dG g = g + h/6 ((6 - 4c) v1 + h (3 - c) v2)), and the q/p column adds
  // their derivatives with respect to q/p at fixed d, in u1 = d x B and
  // u2 = u1 x w.  ~100 operations where building the 3x3 blocks from the four
  // stage matrices takes ~300.
  KFD_INLINE void transportConst(const double w[3], const double u1[3], const double u2[3],
                                 double h, double h6, double hh6, double c) {
    const double f1 = hh6 * (3.0 - c), f2 = hh6 * h, g1 = h6 * (6.0 - 4.0 * c);
#pragma unroll
    for (int col = 0; col < 3; ++col) {
      const double g[3] = {(double)G[0][col], (double)G[1][col], (double)G[2][col]};
      double v1[3], v2[3];
      cross(g, w, v1);
      cross(v1, w, v2);
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        A[r][2 + col] = A[r][2 + col] + (h * g[r] + (f1 * v1[r] + f2 * v2[r]));
        G[r][col] = g[r] + (g1 * v1[r] + f1 * v2[r]);
      }
    }
    const double a1 = hh6 * (3.0 - 3.0 * c), a2 = 2.0 * f2, b1 = h6 * (6.0 - 12.0 * c),
                 b2 = h * g1;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      A[r][4] = A[r][4] + (a1 * u1[r] + a2 * u2[r]);
      G[r][2] = G[r][2] + (b1 * u1[r] + b2 * u2[r]);
    }
  }

  // J <- D J in any field, double: the stage chain of the
  // direction block run on each column g of J's direction rows, with
  // w = q/p B of the stage: v1 = g x w1, v2 = (g + h/2 v1) x wm,
  // v3 = (g + h/2 v2) x wm, v4 = (g + h v3) x wl; the q/p column adds the
  // derivatives of the stages with respect to q/p.  ~210 operations where the
  // 3x3 blocks take ~300.  Lane groups run it whole on every lane: gathering a
  // column costs what computing it does.
  KFD_INLINE void transportColumns(const double B1[3], const double Bm[3], const double Bl[3],
                                   const double k1[3], const double k2[3], const double k3[3],
                                   double h, double h6, double hh6, double qop) {
    const double hh = 0.5 * h;
    double w1[3], wm[3], wl[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      w1[k] = qop * B1[k];
      wm[k] = qop * Bm[k];
      wl[k] = qop * Bl[k];
    }
#pragma unroll
    for (int col = 0; col < 3; ++col) {
      const double g[3] = {(double)G[0][col], (double)G[1][col], (double)G[2][col]};
      double v1[3], v2[3], v3[3], v4[3], x[3];
      cross(g, w1, v1);
#pragma unroll
      for (int k = 0; k < 3; ++k) x[k] = g[k] + hh * v1[k];
      cross(x, wm, v2);
#pragma unroll
      for (int k = 0; k < 3; ++k) x[k] = g[k] + hh * v2[k];
      cross(x, wm, v3);
#pragma unroll
      for (int k = 0; k < 3; ++k) x[k] = g[k] + h * v3[k];
      cross(x, wl, v4);
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const double m = v2[r] + v3[r];
        A[r][2 + col] = A[r][2 + col] + (h * g[r] + hh6 * (v1[r] + m));
        G[r][col] = g[r] + h6 * ((v1[r] + v4[r]) + 2.0 * m);
      }
    }
    // dk/d(q/p): L1 = d x B1, L2 = (d + h/2 k1 + h/2 qop L1) x Bm, ...
    double L1[3], L2[3], L3[3], L4[3], x[3];
    cross(dir, B1, L1);
#pragma unroll
    for (int k = 0; k < 3; ++k) x[k] = dir[k] + h * k1[k];  // qop L1 = k1
    cross(x, Bm, L2);
#pragma unroll
    for (int k = 0; k < 3; ++k) x[k] = dir[k] + hh * (k2[k] + qop * L2[k]);
    cross(x, Bm, L3);
#pragma unroll
    for (int k = 0; k < 3; ++k) x[k] = dir[k] + h * (k3[k] + qop * L3[k]);
    cross(x, Bl, L4);
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const double m = L2[r] + L3[r];
      A[r][4] = A[r][4] + hh6 * (L1[r] + m);
      G[r][2] = G[r][2] + h6 * ((L1[r] + L4[r]) + 2.0 * m);
    }
  }

  // J <- D J for the free transport matrix D of one RK step
  // (EigenStepper.ipp:50-124 builds D; its identity / zero blocks are used
  // implicitly): the mixed mode's, in float.
  KFD_INLINE void transport(const double Bfd[3], const double Bmd[3], const double Bld[3],
                            const double k1d[3], const double k2d[3], const double k3d[3],
                            double hd, double qopd) {
    const S h = (S)hd, qop = (S)qopd, half_h = (S)(hd * 0.5);
    S d[3], Bf[3], Bm[3], Bl[3], k1[3], k2[3], k3[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      d[k] = (S)dir[k];
      Bf[k] = (S)Bfd[k];
      Bm[k] = (S)Bmd[k];
      Bl[k] = (S)Bld[k];
      k1[k] = (S)k1d[k];
      k2[k] = (S)k2d[k];
      k3[k] = (S)k3d[k];
    }
    S dk1dL[3], dk2dL[3], dk3dL[3], dk4dL[3], tv[3], c1[3], c2[3];
    cross(d, Bf, dk1dL);
#pragma unroll
    for (int k = 0; k < 3; ++k) tv[k] = d[k] + half_h * k1[k];
    cross(tv, Bm, c1);
    cross(dk1dL, Bm, c2);
#pragma unroll
    for (int k = 0; k < 3; ++k) dk2dL[k] = c1[k] + (qop * half_h) * c2[k];
#pragma unroll
    for (int k = 0; k < 3; ++k) tv[k] = d[k] + half_h * k2[k];
    cross(tv, Bm, c1);
    cross(dk2dL, Bm, c2);
#pragma unroll
    for (int k = 0; k < 3; ++k) dk3dL[k] = c1[k] + (qop * half_h) * c2[k];
#pragma unroll
    for (int k = 0; k < 3; ++k) tv[k] = d[k] + h * k3[k];
    cross(tv, Bl, c1);
    cross(dk3dL, Bl, c2);
#pragma unroll
    for (int k = 0; k < 3; ++k) dk4dL[k] = c1[k] + (qop * h) * c2[k];

    // quotients: a float 1/6 constant is biased by 3e-8 relative, which
    // accumulates over the steps of a track
    const S h6 = sixthOf(h);
    const S hh6 = sixthOf(h * h);
    S dFdT[3][3], dGdT[3][3], dFdL[3], dGdL[3];
    if constexpr (L == 1) {
      // dk/dT matrices (row r, column c)
      S dk1dT[3][3] = {{(S)0, Bf[2], -Bf[1]}, {-Bf[2], (S)0, Bf[0]}, {Bf[1], -Bf[0], (S)0}};
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) dk1dT[r][c] = qop * dk1dT[r][c];
      S dk2dT[3][3], dk3dT[3][3], dk4dT[3][3];
      crossStep(dk1dT, half_h, Bm, qop, dk2dT);
      crossStep(dk2dT, half_h, Bm, qop, dk3dT);
      crossStep(dk3dT, h, Bl, qop, dk4dT);
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const S id = (r == c) ? (S)1 : (S)0;
          dFdT[r][c] = h * (id + h6 * (dk1dT[r][c] + dk2dT[r][c] + dk3dT[r][c]));
          dGdT[r][c] =
              id + h6 * (dk1dT[r][c] + (S)2.0 * (dk2dT[r][c] + dk3dT[r][c]) + dk4dT[r][c]);
        }
    } else {
      // lane groups: the columns of dF/dT and dG/dT are independent (column
      // c follows the chain dk1..dk4 of the unit vector e_c); each lane
      // builds the columns of its slots, c = rank + L * slot (the last
      // column again where that runs past it), and the group gathers them
      constexpr int kSlots = (3 + L - 1) / L;
      S colF[kSlots][3], colG[kSlots][3];
#pragma unroll
      for (int sl = 0; sl < kSlots; ++sl) {
        const uint32_t c = (rank + (uint32_t)(L * sl) < 3u) ? rank + (uint32_t)(L * sl) : 2u;
        const S e[3] = {(c == 0u) ? (S)1 : (S)0, (c == 1u) ? (S)1 : (S)0,
                        (c == 2u) ? (S)1 : (S)0};
        S k1c[3], k2c[3], k3c[3], k4c[3], col[3];
        // column c of dk1/dT = qop [B]x e_c: the unit-vector cross product
        // spelled out as the matrix of the single-lane path
        const S m1[3] = {e[1] * Bf[2] - e[2] * Bf[1], e[2] * Bf[0] - e[0] * Bf[2],
                         e[0] * Bf[1] - e[1] * Bf[0]};
#pragma unroll
        for (int k = 0; k < 3; ++k) k1c[k] = qop * m1[k];
#pragma unroll
        for (int k = 0; k < 3; ++k) col[k] = e[k] + half_h * k1c[k];
        cross(col, Bm, k2c);
#pragma unroll
        for (int k = 0; k < 3; ++k) k2c[k] = qop * k2c[k];
#pragma unroll
        for (int k = 0; k < 3; ++k) col[k] = e[k] + half_h * k2c[k];
        cross(col, Bm, k3c);
#pragma unroll
        for (int k = 0; k < 3; ++k) k3c[k] = qop * k3c[k];
#pragma unroll
        for (int k = 0; k < 3; ++k) col[k] = e[k] + h * k3c[k];
        cross(col, Bl, k4c);
#pragma unroll
        for (int k = 0; k < 3; ++k) k4c[k] = qop * k4c[k];
#pragma unroll
        for (int r = 0; r < 3; ++r) {
          colF[sl][r] = h * (e[r] + h6 * (k1c[r] + k2c[r] + k3c[r]));
          colG[sl][r] = e[r] + h6 * (k1c[r] + (S)2.0 * (k2c[r] + k3c[r]) + k4c[r]);
        }
      }
      // gather: column c from rank c % L, slot c / L
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        S f[kSlots], g[kSlots], fo[3], go[3];
#pragma unroll
        for (int sl = 0; sl < kSlots; ++sl) {
          f[sl] = colF[sl][r];
          g[sl] = colG[sl][r];
        }
        groupGather<L, 3>(f, fo);
        groupGather<L, 3>(g, go);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          dFdT[r][c] = fo[c];
          dGdT[r][c] = go[c];
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      dFdL[r] = hh6 * (dk1dL[r] + dk2dL[r] + dk3dL[r]);
      dGdL[r] = h6 * (dk1dL[r] + (S)2.0 * (dk2dL[r] + dk3dL[r]) + dk4dL[r]);
    }
    // J <- D J on the non-constant entries
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      S g[3] = {G[0][c], G[1][c], G[2][c]};
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        S fa = dFdT[r][0] * g[0] + dFdT[r][1] * g[1] + dFdT[r][2] * g[2];
        S ga = dGdT[r][0] * g[0] + dGdT[r][1] * g[1] + dGdT[r][2] * g[2];
        if (c == 2) {
          fa = fa + dFdL[r];
          ga = ga + dGdL[r];
        }
        A[r][2 + c] = A[r][2 + c] + fa;
        G[r][c] = ga;
      }
    }
  }

  // x / 6 in float, correctly rounded: the product with the rounded 1/6 and one
  // residual correction (Markstein's division theorem), 3 operations where the
  // library's quotient takes ~10
  KFD_INLINE static S sixthOf(S x) {
    if constexpr (kMixed) {
      const float q = x * (1.0f / 6.0f);
      return fmaf(fmaf(-6.0f, q, x), 1.0f / 6.0f, q);
    } else {
      return x / (S)6.0;
    }
  }

  // qop * cross_cols(I + hh * M, B)  (Helpers.hpp:168-176)
  KFD_INLINE static void crossStep(const S M[3][3], S hh, const S B[3], S qop, S out[3][3]) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      S col[3], r[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) col[k] = ((k == c) ? (S)1 : (S)0) + hh * M[k][c];
      cross(col, B, r);
#pragma unroll
      for (int k = 0; k < 3; ++k) out[k][c] = qop * r[k];
    }
  }

  // ------------------------------------------------ fixed-point smoother ----
  // The smoothed state of the first measured surface (x0, C0), from sums that
  // the forward pass accumulates.  With T the derivative of the current
  // predicted spatial parameters (loc0, loc1, phi, theta, q/p) with respect to
  // the filtered ones of state 0 -- T <- J T at a transport, T <- (I - K H) T
  // at an update -- the covariance of state 0 with the current state is
  // C_f0 T^T, and every later measurement (residual r, innovation S) adds
  //   lambda += T^T H^T S^-1 r,   Lambda += T^T H^T S^-1 H T;
  // at the end x0 = x_f0 + C_f0 lambda, C0 = C_f0 - C_f0 Lambda C_f0 (the
  // fixed-point smoother of Kalman filtering, e.g. Anderson and Moore, Optimal
  // Filtering, 1979, section 7.2).  In exact arithmetic it is the RTS
  // recursion's result for state 0; the time parameter never acts on the
  // spatial ones, so T is 5x5.  Per state ~210 multiply-adds and no memory,
  // against ~1,100 and 512 B written and read back for the RTS
  // step, whose 6x6 solve also loses more digits than the sums here.
  //
  // T, lambda and Lambda sit in LDS (kFxN 16-byte pairs per lane, stride
  // KF_FUSED_BLOCK: conflict-free 16-byte accesses), not in registers: they are
  // used once per surface.
  //
  // Where the RTS recursion's discrete behaviour could show -- a phi wrap or a
  // theta clamp of a smoothed state, a gain that is not finite, a covariance
  // that is not clearly positive definite -- the track is handed to the RTS
  // program instead (fxSafe, the redo list).
  struct alignas(16) FxPair {
    double a, b;
  };
  enum { kFxCol = 3, kFxSum = 15 };
  // The mixed mode's sums.  Its covariances are rounded to float between
  // surfaces, so J C_f J^T is not exactly the predicted covariance and the
  // identities above hold to 1e-7 only; the RTS gains G_k = C_f J^T C_p^-1 of
  // the rounded matrices still give state 0 as sums over the later states:
  // with P_k = G_0 G_1 ... G_(k-1),
  //   x0 = x_f0 + sum P_k (x_fk - x_pk),  C0 = C_f0 + sum P_k (C_fk - C_pk) P_k^T,
  // the recursion's result in exact arithmetic, whatever the matrices.  Per
  // state the ~1,100 multiply-adds of the RTS step (the same gain, from the
  // same numbers) and no memory.  P by rows of three pairs, then x0 and C0.
  enum { kFxRow = 3, kFxX0 = 18, kFxC0 = 21 };
  static constexpr bool kFxRts = kFirst && kMixed;
  static constexpr int kFxN = kMixed ? 32 : 23;
  FxPair *fx = nullptr;  // this lane's first pair
  bool fxOk = true;
  // the kernel's arguments where other waves of the launch fit the tracks near the
  // wrap (nearWrap), and whether this is one of them
  const FitArgs *picker = nullptr;
  bool elsewhere = false;
  // whether to leave a track with a singular start covariance before the pass (its
  // outputs are then not set at all), and whether this is one
  bool leaveEarly = false, left = false;
  S fxDiag[3];                          // kFxRts: (2,2), (3,3), (4,4) before the material update
  double fxLimit = kDblMax;  // total chi2 below which no smoothed angle can wrap (fxAngles)

  KFD_INLINE void fxLoad(int p, double &x, double &y) const {
    const FxPair v = fx[p * KF_FUSED_BLOCK];
    x = v.a;
    y = v.b;
  }
  KFD_INLINE void fxStore(int p, double x, double y) const { fx[p * KF_FUSED_BLOCK] = FxPair{x, y}; }
  // T column c: pairs 3c .. 3c + 2, the sixth element is lambda[c]
  KFD_INLINE void fxInit() const {
#pragma unroll
    for (int c = 0; c < 5; ++c)
#pragma unroll
      for (int g = 0; g < 3; ++g)
        fxStore(kFxCol * c + g, (c == 2 * g) ? 1.0 : 0.0, (c == 2 * g + 1) ? 1.0 : 0.0);
#pragma unroll
    for (int p = kFxSum; p < kFxN; ++p) fxStore(p, 0.0, 0.0);
  }
  // T <- J T (row 4 of J is e4; the time row does not enter)
  KFD_INLINE void fxTransport(const S jb[6][6]) const {
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      double t[6], n[4];
#pragma unroll
      for (int g = 0; g < 3; ++g) fxLoad(kFxCol * c + g, t[2 * g], t[2 * g + 1]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        double v = (double)jb[r][0] * t[0];
#pragma unroll
        for (int m = 1; m < 5; ++m) v = v + (double)jb[r][m] * t[m];
        n[r] = v;
      }
      fxStore(kFxCol * c, n[0], n[1]);
      fxStore(kFxCol * c + 1, n[2], n[3]);
    }
  }
  // a measurement with gain K, S^-1 (i00, i01, i11) and u = S^-1 r: the sums,
  // then T <- (I - K H) T
  KFD_INLINE void fxMeasure(const double K0[6], const double K1[6], double i00, double i01,
                            double i11, double u0, double u1) const {
    double a[5], b[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      double t[6];
#pragma unroll
      for (int g = 0; g < 3; ++g) fxLoad(kFxCol * c + g, t[2 * g], t[2 * g + 1]);
      a[c] = t[0];
      b[c] = t[1];
      t[5] = t[5] + (a[c] * u0 + b[c] * u1);
#pragma unroll
      for (int r = 0; r < 5; ++r) t[r] = t[r] - (K0[r] * a[c] + K1[r] * b[c]);
#pragma unroll
      for (int g = 0; g < 3; ++g) fxStore(kFxCol * c + g, t[2 * g], t[2 * g + 1]);
    }
    double l[16];
#pragma unroll
    for (int p = 0; p < 8; ++p) fxLoad(kFxSum + p, l[2 * p], l[2 * p + 1]);
    int m = 0;
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      const double w0 = i00 * a[c] + i01 * b[c], w1 = i01 * a[c] + i11 * b[c];
#pragma unroll
      for (int d = c; d < 5; ++d, ++m) l[m] = l[m] + (w0 * a[d] + w1 * b[d]);
    }
#pragma unroll
    for (int p = 0; p < 8; ++p) fxStore(kFxSum + p, l[2 * p], l[2 * p + 1]);
  }
  // packed index of Lambda (c, d)
  KFD_INLINE static constexpr int lidx(int c, int d) {
    return (c <= d) ? (c * 5 - (c * (c - 1)) / 2 + (d - c)) : (d * 5 - (d * (d - 1)) / 2 + (c - d));
  }
  // the filtered state 0, kept from its update to the end of the forward pass
  // in this position's column of the hand-over buffer: x_f0 (6), C_f0 (21)
  KFD_INLINE void fxKeepFirst(const double xf[6]) const {
    if (!lead) return;
#pragma unroll
    for (int m = 0; m < 6; ++m) cd(m) = xf[m];
#pragma unroll
    for (int m = 0; m < 21; ++m) cd(6 + m) = (double)cov[m];
  }
  // kFxRts: P = 1, x0 = x_f0, C0 = C_f0
  KFD_INLINE void fxRtsInit(const double xf[6]) const {
#pragma unroll
    for (int r = 0; r < 6; ++r)
#pragma unroll
      for (int g = 0; g < 3; ++g)
        fxStore(kFxRow * r + g, (r == 2 * g) ? 1.0 : 0.0, (r == 2 * g + 1) ? 1.0 : 0.0);
#pragma unroll
    for (int g = 0; g < 3; ++g) fxStore(kFxX0 + g, xf[2 * g], xf[2 * g + 1]);
#pragma unroll
    for (int g = 0; g < 11; ++g)
      fxStore(kFxC0 + g, (double)cov[2 * g], (g < 10) ? (double)cov[2 * g + 1] : 0.0);
  }
  // kFxRts: a later state with the transport J from the filtered covariance cf
  // of the state before, predicted x_p and C_p (cp), filtered x_f and C_f (cov)
  KFD_INLINE void fxRtsStep(const S J[6][6], const S cf[21], const S cp[21], const double xp[6],
                            const double xf[6]) {
    double X[6][6];
    {
      double cfd[21], cpd[21];
#pragma unroll
      for (int m = 0; m < 21; ++m) {
        cfd[m] = (double)cf[m];
        cpd[m] = (double)cp[m];
      }
      transported(J, cfd, X);
      fxOk = spdSolvePivots(cpd, X) && fxOk;
    }
    double P[6][6];
#pragma unroll
    for (int r = 0; r < 6; ++r) {
      double t[6];
#pragma unroll
      for (int g = 0; g < 3; ++g) fxLoad(kFxRow * r + g, t[2 * g], t[2 * g + 1]);
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        double v = t[0] * X[c][0];
#pragma unroll
        for (int m = 1; m < 6; ++m) v = v + t[m] * X[c][m];
        P[r][c] = v;
      }
#pragma unroll
      for (int g = 0; g < 3; ++g) fxStore(kFxRow * r + g, P[r][2 * g], P[r][2 * g + 1]);
    }
    double x0[6], c0[22], D[21];
#pragma unroll
    for (int g = 0; g < 3; ++g) fxLoad(kFxX0 + g, x0[2 * g], x0[2 * g + 1]);
#pragma unroll
    for (int g = 0; g < 11; ++g) fxLoad(kFxC0 + g, c0[2 * g], c0[2 * g + 1]);
#pragma unroll
    for (int m = 0; m < 21; ++m) D[m] = (double)cov[m] - (double)cp[m];
#pragma unroll
    for (int r = 0; r < 6; ++r) {
#pragma unroll
      for (int c = 0; c < 6; ++c) x0[r] = x0[r] + P[r][c] * (xf[c] - xp[c]);
      double w[6];  // row r of P (C_f - C_p)
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        double v = P[r][0] * D[sidx(0, c)];
#pragma unroll
        for (int m = 1; m < 6; ++m) v = v + P[r][m] * D[sidx(m, c)];
        w[c] = v;
      }
#pragma unroll
      for (int c = r; c < 6; ++c) {
        double v = w[0] * P[c][0];
#pragma unroll
        for (int m = 1; m < 6; ++m) v = v + w[m] * P[c][m];
        c0[sidx(r, c)] = c0[sidx(r, c)] + v;
      }
    }
#pragma unroll
    for (int g = 0; g < 3; ++g) fxStore(kFxX0 + g, x0[2 * g], x0[2 * g + 1]);
#pragma unroll
    for (int g = 0; g < 11; ++g) fxStore(kFxC0 + g, c0[2 * g], c0[2 * g + 1]);
  }
  KFD_INLINE void fxSmooth(double xs[6], double cs[21]) const {
    if constexpr (kFxRts) {
      double c0[22];
#pragma unroll
      for (int g = 0; g < 3; ++g) fxLoad(kFxX0 + g, xs[2 * g], xs[2 * g + 1]);
#pragma unroll
      for (int g = 0; g < 11; ++g) fxLoad(kFxC0 + g, c0[2 * g], c0[2 * g + 1]);
#pragma unroll
      for (int m = 0; m < 21; ++m) cs[m] = c0[m];
      correctParams(xs);
      return;
    }
    double x0[6], c0[21];
#pragma unroll
    for (int m = 0; m < 6; ++m) x0[m] = cd(m);
#pragma unroll
    for (int m = 0; m < 21; ++m) c0[m] = cd(6 + m);
    double lam[5], l[16];
#pragma unroll
    for (int c = 0; c < 5; ++c) {
      double t4;
      fxLoad(kFxCol * c + 2, t4, lam[c]);
    }
#pragma unroll
    for (int p = 0; p < 8; ++p) fxLoad(kFxSum + p, l[2 * p], l[2 * p + 1]);
#pragma unroll
    for (int r = 0; r < 6; ++r) {
      double v = c0[sidx(r, 0)] * lam[0];
#pragma unroll
      for (int m = 1; m < 5; ++m) v = v + c0[sidx(r, m)] * lam[m];
      xs[r] = x0[r] + v;
      double w[5];  // row r of C_f0 Lambda
#pragma unroll
      for (int c = 0; c < 5; ++c) {
        double q = c0[sidx(r, 0)] * l[lidx(0, c)];
#pragma unroll
        for (int m = 1; m < 5; ++m) q = q + c0[sidx(r, m)] * l[lidx(m, c)];
        w[c] = q;
      }
#pragma unroll
      for (int c = r; c < 6; ++c) {
        double q = w[0] * c0[sidx(0, c)];
#pragma unroll
        for (int m = 1; m < 5; ++m) q = q + w[m] * c0[sidx(m, c)];
        cs[sidx(r, c)] = c0[sidx(r, c)] - q;
      }
    }
    correctParams(xs);
  }
  // Whether the start covariance is positive definite with room to spare: the
  // pivots of the diagonally scaled matrix above the rounding of the mode.
  KFD_INLINE bool fxDefinite() const {
    const double low = kMixed ? 1e-5 : 1e-11;
    double sc[6], Lo[6][6], W[6][6];
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 6; ++k) sc[k] = scaleOf((double)cov[sidx(k, k)]);
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      double dj = (sc[j] * (double)cov[sidx(j, j)]) * sc[j];
#pragma unroll
      for (int k = 0; k < j; ++k) dj = dj - W[j][k] * Lo[j][k];
      ok = ok && dj > low;
      const double id = 1.0 / dj;
#pragma unroll
      for (int r = j + 1; r < 6; ++r) {
        double w = (sc[r] * (double)cov[sidx(r, j)]) * sc[j];
#pragma unroll
        for (int k = 0; k < j; ++k) w = w - W[r][k] * Lo[j][k];
        W[r][j] = w;
        Lo[r][j] = w * id;
      }
    }
    return ok;
  }
  // Whether the smoothed phi and theta of this state can pass their bounds.  A
  // smoothed state lies within sqrt(X) of the filtered one in units of the
  // filtered errors, X the chi2 that the later measurements add (it minimises
  // that distance squared plus a sum of squares, whose minimum is X), so the
  // angle stays a distance d away from its bound while X < d^2 / V: the total
  // chi2 must stay below the chi2 so far plus d^2 / V, for every state and both
  // angles; 2 % and 1e-6 cover rounding.  Not asked for state 0, whose smoothed
  // value is wrapped last, by both smoothers.
  KFD_INLINE void fxAngles(const double xf[6]) {
    const double dp = (kPi - 1e-6) - fabs(xf[2]), dt = (0.5 * kPi - 1e-6) - fabs(xf[3] - 0.5 * kPi);
    const double vp = (double)cov[sidx(2, 2)], vt = (double)cov[sidx(3, 3)];
    fxOk = fxOk && 0.0 < fmin(dp, dt) && 0.0 <= fmin(vp, vt) && vp + vt < kDblMax;
    // the smaller of dp^2 / vp and dt^2 / vt by one reciprocal, whose estimate is
    // far within the 2 % (variances of 0 set no limit: the state is exact)
    const double x = fmin((dp * dp) * vt, (dt * dt) * vp) * recipEstimate(vp * vt);
    fxLimit = fmin(fxLimit, chi2sum + x * (1.0 / (1.02 * 1.02)));
  }
  // Whether the RTS recursion over this track's states is free of wraps,
  // clamps and non-finite gains, so that its result for state 0 is this
  // smoother's.  False on NaN.
  KFD_INLINE bool fxSafe(const double xs[6], const double cs[21]) const {
    bool ok = fxOk && chi2sum < fxLimit;
#pragma unroll
    for (int m = 0; m < 6; ++m) ok = ok && fabs(xs[m]) < kDblMax;
#pragma unroll
    for (int m = 0; m < 21; ++m) ok = ok && fabs(cs[m]) < kDblMax;
    return ok;
  }

  // ------------------------------------------------- bound-state transport ----
  // detail::covarianceTransport (CovarianceEngine.hpp:269-290): derivative
  // correction J' = J - deriv sVec, bound Jacobian jb = jacToLocal J',
  // cov <- jb cov jb^T.  sVec is given; jacToLocal rows 0/1 are (u0, u1).
  KFD_INLINE void covarianceTransport(const double sVec[6], const double u0[3],
                                      const double u1[3], double cosT, double sinT,
                                      double invSinT, double cosP, double sinP, S jb[6][6]) {
    S dr[8];
#pragma unroll
    for (int k = 0; k < 3; ++k) dr[k] = derivSet ? (S)dir[k] : (S)0;
    // dtds and k4d are zero while derivSet is not
    dr[3] = dtds;
#pragma unroll
    for (int k = 0; k < 3; ++k) dr[4 + k] = k4d[k];
    const S l20 = (S)(-sinP * invSinT), l21 = (S)(cosP * invSinT);
    const S l30 = (S)(cosP * cosT), l31 = (S)(sinP * cosT), l32 = (S)(-sinT);
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      const S sv = (S)sVec[c];
      S jp[8];
#pragma unroll
      for (int r = 0; r < 3; ++r) jp[r] = ((c < 5) ? A[r][c] : (S)0) - dr[r] * sv;
      jp[3] = ((c == 4) ? b : ((c == 5) ? (S)1 : (S)0)) - dr[3] * sv;
#pragma unroll
      for (int r = 0; r < 3; ++r) jp[4 + r] = ((c >= 2 && c < 5) ? G[r][c - 2] : (S)0) - dr[4 + r] * sv;
      jp[7] = (c == 4) ? (S)1 : (S)0;
      jb[0][c] = (S)u0[0] * jp[0] + (S)u0[1] * jp[1] + (S)u0[2] * jp[2];
      jb[1][c] = (S)u1[0] * jp[0] + (S)u1[1] * jp[1] + (S)u1[2] * jp[2];
      jb[2][c] = l20 * jp[4] + l21 * jp[5];
      jb[3][c] = l30 * jp[4] + l31 * jp[5] + l32 * jp[6];
      jb[4][c] = jp[7];
      jb[5][c] = jp[3];
    }
    S cs[21];
#pragma unroll
    for (int m = 0; m < 21; ++m) cs[m] = cov[m];
    sandwich(jb, cs, cov);
  }

  // cn = jb c jb^T in S.  Row 4 of jb is e4 and column 5 is e5 exactly (the
  // q/p row and the time column of the transport), so those terms are
  // skipped; row r of jb c is formed and consumed at once.  The smoother
  // calls this with the stored operands to recompute the predicted
  // covariance bit for bit.
  template <typename Out>
  KFD_INLINE static void sandwich(const S jb[6][6], const S c[21], Out cn[21]) {
#pragma unroll
    for (int r = 0; r < 6; ++r) {
      S T[6];
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        if (r == 4) {
          T[k] = c[sidx(4, k)];
        } else {
          S s = jb[r][0] * c[sidx(0, k)];
#pragma unroll
          for (int m = 1; m < 5; ++m) s = s + jb[r][m] * c[sidx(m, k)];
          if (r == 5) s = s + c[sidx(5, k)];
          T[k] = s;
        }
      }
#pragma unroll
      for (int cc = r; cc < 6; ++cc) {
        S s;
        if (cc == 4) {
          s = T[4];
        } else {
          s = T[0] * jb[cc][0];
#pragma unroll
          for (int m = 1; m < 5; ++m) s = s + T[m] * jb[cc][m];
          if (cc == 5) s = s + T[5];
        }
        cn[sidx(r, cc)] = (Out)s;
      }
    }
  }

  // boundState on a plane (EigenStepper.ipp:516-540, CovarianceEngine.hpp:
  // 345-371) including the Jacobian re-initialisation on the plane.
  KFD_INLINE void boundStatePlane(const DevPlane &pl, double par[6], S jb[6][6]) {
    const double cosT = dir[2];
    double sinT, invSinT;
    rootD(dir[0] * dir[0] + dir[1] * dir[1], sinT, invSinT);
    const double cosP = dir[0] * invSinT, sinP = dir[1] * invSinT;
    const double u0[3] = {pl.r[0], pl.r[3], pl.r[6]};
    const double u1[3] = {pl.r[1], pl.r[4], pl.r[7]};
    const double nr[3] = {pl.r[2], pl.r[5], pl.r[8]};
    // PlaneSurface::derivativeFactors, PlaneSurface.ipp:191-204
    const double dp = nr[0] * dir[0] + nr[1] * dir[1] + nr[2] * dir[2];
    const double idp = recipD(dp);
    const double nv[3] = {nr[0] * idp, nr[1] * idp, nr[2] * idp};
    double sVec[6];
#pragma unroll
    for (int c = 0; c < 5; ++c)
      sVec[c] = nv[0] * (double)A[0][c] + nv[1] * (double)A[1][c] + nv[2] * (double)A[2][c];
    sVec[5] = 0.0;
    covarianceTransport(sVec, u0, u1, cosT, sinT, invSinT, cosP, sinP, jb);
    // bound parameters: global2parameters on the plane
    const double dd[3] = {pos[0] - pl.c[0], pos[1] - pl.c[1], pos[2] - pl.c[2]};
    par[0] = pl.r[0] * dd[0] + pl.r[3] * dd[1] + pl.r[6] * dd[2];
    par[1] = pl.r[1] * dd[0] + pl.r[4] * dd[1] + pl.r[7] * dd[2];
    planeAngles(sinT, par);
    par[5] = t;
    correctParams(par);
    // reinitializeJacobians on the plane (PlaneSurface.ipp:122-156)
    initJacobianPlane(pl, cosT, sinT, cosP, sinP);
  }

  // phi, theta and q/p of the direction at a plane (sinT = its transverse
  // length): the reference's conversions of the momentum vector, whose angles
  // are taken from those after the last update plus the arc tangents of the
  // rotation since, in the transverse plane and in theta.  Over a segment the
  // rotation is small, so each is a division (one shared reciprocal) and a
  // short series, ~50 instructions for both angles where two library arc
  // tangents take ~270; a rotation with a tangent above 1/16 (or no
  // reference, or a stopped particle) takes the library.  Agrees with it to
  // an ulp of the angle per segment.
  KFD_INLINE void planeAngles(double sinT, double par[6]) {
    const double n1 = refX * dir[1] - refY * dir[0], d1 = refX * dir[0] + refY * dir[1];
    double refS, refIS;
    rootD(refX * refX + refY * refY, refS, refIS);
    const double n2 = sinT * refZ - dir[2] * refS, d2 = dir[2] * refZ + sinT * refS;
    const double i12 = recipD(d1 * d2);
    const double r1 = n1 * (d2 * i12), r2 = n2 * (d1 * i12);
    if (0.0 < d1 && 0.0 < d2 && fabs(r1) <= 0.0625 && fabs(r2) <= 0.0625 && 0.0 < p) {
      par[2] = refPhi + atanSmall(r1);
      par[3] = refTheta + atanSmall(r2);
      par[4] = divD(q, p);
      return;
    }
    const double qop = q / p;
    const double pabs = fabs(1.0 / qop);
    const double mom[3] = {pabs * dir[0], pabs * dir[1], pabs * dir[2]};
    const double charge = copysign(1.0, qop);
    par[2] = atan2D(mom[1], mom[0]);
    par[3] = atan2D(sqrt(mom[0] * mom[0] + mom[1] * mom[1]), mom[2]);
    const double mn = sqrt(mom[0] * mom[0] + mom[1] * mom[1] + mom[2] * mom[2]);
    par[4] = ((fabs(charge) < 1e-4) ? 1.0 : charge) / mn;
  }

  // boundState on the perigee line (LineSurface.ipp:114-220); the Jacobians
  // are not re-initialised because propagation ends here.
  KFD_INLINE void boundStateLine(double par[6]) {
    const double cosT = dir[2];
    const double sinT = sqrt(dir[0] * dir[0] + dir[1] * dir[1]);
    const double invSinT = 1.0 / sinT;
    const double cosP = dir[0] * invSinT, sinP = dir[1] * invSinT;
    // reference frame: measY = z, measX = |z x dir|, measDepth = measX x measY
    const double mxr[3] = {0.0 * dir[2] - 1.0 * dir[1], 1.0 * dir[0] - 0.0 * dir[2],
                           0.0 * dir[1] - 0.0 * dir[0]};
    const double mxn = sqrt(mxr[0] * mxr[0] + mxr[1] * mxr[1] + mxr[2] * mxr[2]);
    const double mX[3] = {mxr[0] / mxn, mxr[1] / mxn, mxr[2] / mxn};
    const double mY[3] = {0.0, 0.0, 1.0};
    // LineSurface::derivativeFactors, LineSurface.ipp:145-182
    const double pc[3] = {pos[0] - lc[0], pos[1] - lc[1], pos[2] - lc[2]};
    const double long_c = mY[0] * dir[0] + mY[1] * dir[1] + mY[2] * dir[2];
    const double nvec[3] = {dir[0] - long_c * mY[0], dir[1] - long_c * mY[1], dir[2] - long_c * mY[2]};
    const double nrm = 1.0 / (1.0 - long_c * long_c);
    double sVec[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      double jc[3], jd[3];
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        jc[r] = (c < 5) ? (double)A[r][c] : 0.0;
        jd[r] = (c >= 2 && c < 5) ? (double)G[r][c - 2] : 0.0;
      }
      const double s_vec = nvec[0] * jc[0] + nvec[1] * jc[1] + nvec[2] * jc[2];
      double diff[3];
#pragma unroll
      for (int r = 0; r < 3; ++r) diff[r] = mY[r] * s_vec - jd[r];
      const double row = pc[0] * diff[0] + pc[1] * diff[1] + pc[2] * diff[2];
      sVec[c] = nrm * (s_vec - row);
    }
    S jb[6][6];
    covarianceTransport(sVec, mX, mY, cosT, sinT, invSinT, cosP, sinP, jb);
    const double qop = q / p;
    const double pabs = fabs(1.0 / qop);
    const double mom[3] = {pabs * dir[0], pabs * dir[1], pabs * dir[2]};
    const double charge = copysign(1.0, qop);
    // LineSurface::globalToLocal, LineSurface.ipp:200-220
    const double l3[3] = {pos[0] - lc[0], pos[1] - lc[1], pos[2] - lc[2]};
    double l0 = sqrt(l3[0] * l3[0] + l3[1] * l3[1]);
    const double cr[3] = {0.0 * mom[2] - 1.0 * mom[1], 1.0 * mom[0] - 0.0 * mom[2],
                          0.0 * mom[1] - 0.0 * mom[0]};
    const double sgn = (cr[0] * pc[0] + cr[1] * pc[1] + cr[2] * pc[2] < 0.0) ? -1.0 : 1.0;
    par[0] = l0 * sgn;
    par[1] = l3[2];
    par[2] = atan2D(mom[1], mom[0]);
    par[3] = atan2D(sqrt(mom[0] * mom[0] + mom[1] * mom[1]), mom[2]);
    const double mn = sqrt(mom[0] * mom[0] + mom[1] * mom[1] + mom[2] * mom[2]);
    par[4] = ((fabs(charge) < 1e-4) ? 1.0 : charge) / mn;
    par[5] = t;
    correctParams(par);
  }

  // EigenStepper::update from bound parameters on a plane
  // (boundParameters2freeParameters, coordinate_transformations.hpp:145-158,
  // then EigenStepper.ipp:554-564)
  KFD_INLINE void updateFromBound(const DevPlane &pl, const double par[6]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) pos[k] = (pl.r[3 * k] * par[0] + pl.r[3 * k + 1] * par[1]) + pl.c[k];
    const SinCos s3 = sinCosD(par[3]), s2 = sinCosD(par[2]);
    const double cT = s3.c, sT = s3.s;
    const double d0 = s2.c * sT, d1 = s2.s * sT, d2 = cT;
    const double idn = 1.0 / sqrt(d0 * d0 + d1 * d1 + d2 * d2);
    dir[0] = d0 * idn;
    dir[1] = d1 * idn;
    dir[2] = d2 * idn;
    moved();
    p = fabs(1.0 / par[4]);
    t = par[5];
  }

  // sin(d), cos(d) for |d| < 1/16 by their Taylor series to d^9 / d^10 (the
  // first omitted terms are below 2e-21)
  KFD_INLINE static void sinCosSmall(double d, double &s, double &c) {
    const double d2 = d * d;
    s = d * (1.0 - d2 * (1.0 / 6.0) *
                       (1.0 - d2 * (1.0 / 20.0) * (1.0 - d2 * (1.0 / 42.0) * (1.0 - d2 * (1.0 / 72.0)))));
    c = 1.0 - d2 * 0.5 *
                  (1.0 - d2 * (1.0 / 12.0) *
                             (1.0 - d2 * (1.0 / 30.0) *
                                        (1.0 - d2 * (1.0 / 56.0) * (1.0 - d2 * (1.0 / 90.0)))));
  }

  // updateFromBound after the gain-matrix update on a plane, while dir still
  // holds the predicted direction: cos and sin of the filtered angles follow
  // from those of the predicted ones (dir's components) by the angle-addition
  // theorems with the update d = filtered - predicted, in place of four
  // library calls; an update of 1/16 rad or more, or a direction within 1e-3
  // of the z axis, takes updateFromBound.  Agrees with it to a few ulp.
  KFD_INLINE void updateFromFiltered(const DevPlane &pl, const double xf[6], const double xp[6]) {
    double dphi = xf[2] - xp[2];  // modulo 2 pi (xf[2] is wrapped)
    if (dphi > kPi)
      dphi -= 2.0 * kPi;
    else if (dphi < -kPi)
      dphi += 2.0 * kPi;
    const double dth = xf[3] - xp[3];
    const double cosT = dir[2];
    double sinT, iS;
    rootD(dir[0] * dir[0] + dir[1] * dir[1], sinT, iS);
    if (!(fabs(dphi) < 0.0625 && fabs(dth) < 0.0625 && sinT > 1e-3)) {
      updateFromBound(pl, xf);
      return;
    }
    const double cosP = dir[0] * iS, sinP = dir[1] * iS;
    double sp, cp, st, ct;
    sinCosSmall(dphi, sp, cp);
    sinCosSmall(dth, st, ct);
    const double cPf = cosP * cp - sinP * sp, sPf = sinP * cp + cosP * sp;
    const double cTf = cosT * ct - sinT * st, sTf = sinT * ct + cosT * st;
#pragma unroll
    for (int k = 0; k < 3; ++k) pos[k] = (pl.r[3 * k] * xf[0] + pl.r[3 * k + 1] * xf[1]) + pl.c[k];
    const double d0 = cPf * sTf, d1 = sPf * sTf, d2 = cTf;
    double dn, idn;
    rootOfDirection(d0 * d0 + d1 * d1 + d2 * d2, dn, idn);
    dir[0] = d0 * idn;
    dir[1] = d1 * idn;
    dir[2] = d2 * idn;
    moved();
    p = fabs(1.0 / xf[4]);
    t = xf[5];
  }

  // ----------------------------------------------------------- navigation ----
  KFD_INLINE const DevPlane &plane(int idx) const { return pls[idx]; }

  // updateSingleSurfaceStatus on a plane, SteppingHelper.hpp:31-65 (+
  // PlanarHelper.hpp:28-49); returns 0 unreachable, 1 reachable, 2 on surface
  KFD_INLINE int surfaceStatus(int idx) {
    const double nd = (double)navDir;
    double denom, path;
    if (idx == pathPlane) {
      denom = pathDenom;
      path = pathLen;
    } else {
      // the plane's normal and centre read at once, and the quotient formed
      // whatever the denominator: one wait for the table instead of three
      const DevPlane &pl = plane(idx);
      const double nr[3] = {pl.r[2], pl.r[5], pl.r[8]};
      const double pc[3] = {pl.c[0], pl.c[1], pl.c[2]};
      const double d[3] = {nd * dir[0], nd * dir[1], nd * dir[2]};
      denom = dot3(d, nr);
      const double cm[3] = {pc[0] - pos[0], pc[1] - pos[1], pc[2] - pos[2]};
      const double quot = divD(dot3(nr, cm), denom);
      path = (denom != 0.0) ? quot : 0.0;
      pathPlane = idx;
      pathDenom = denom;
      pathLen = path;
    }
    if (denom != 0.0) {
      if (path * path < kOnSurfaceTolerance * kOnSurfaceTolerance) {
        ss.release(kActor);
        return 2;
      }
      const double pLimit = ss.v[kAborter];
      if (path > negOverstep && path * path < pLimit * pLimit) {
        ss.release(kActor);
        ss.update(nd * path, kActor);
        return 1;
      }
    }
    return 0;
  }

  // DirectNavigator::status, DirectNavigator.hpp:158-188
  KFD_INLINE void navStatus() {
    cur = -1;
    if (next != size) {
      const int sp = seqFirst + next;
      if (surfaceStatus(sp) == 2) {
        cur = sp;
        ++next;
        if (next != size) ss.release(kActor);
      }
    }
  }

  // DirectNavigator::target, DirectNavigator.hpp:197-225
  KFD_INLINE void navTarget() {
    cur = -1;
    if (next != size) {
      if (surfaceStatus(seqFirst + next) == 0) ++next;
    } else {
      navBreak = true;  // the perigee target is always set
    }
  }

  // PathLimitReached, StandardAborters.hpp:24-57
  // The limit is DBL_MAX, and an accumulated path is below 2^970 (a step whose
  // square overflows is refused), so DBL_MAX minus it rounds to DBL_MAX and the
  // update changes no number (a NaN: surfaceReached): only the builds that
  // record the path do it.
  KFD_INLINE bool pathLimit() {
    if (targetReached) return true;
    if constexpr (!kRecords) return false;
    const double distance = (double)navDir * kDblMax - pathAcc;
    ss.update(distance, kAborter);
    const bool reached = distance * distance < a.target_tolerance * a.target_tolerance;
    if (reached) targetReached = true;
    return reached;
  }

  // SurfaceReached on the perigee line, StandardAborters.hpp:86-132
  // (closest approach, LineSurface.ipp:229-262)
  KFD_INLINE bool surfaceReached() {
    if (targetReached) return true;
    if (cur == -2) {
      targetReached = true;
      return true;
    }
    const double nd = (double)navDir;
    const double d[3] = {nd * dir[0], nd * dir[1], nd * dir[2]};
    const double mab[3] = {lc[0] - pos[0], lc[1] - pos[1], lc[2] - pos[2]};
    const double eb[3] = {0.0, 0.0, 1.0};
    const double eaTeb = dot3(d, eb);
    const double denom = 1.0 - eaTeb * eaTeb;
    double distance = kDblMax;
    bool onSurface = false;
    if (denom * denom > kOnSurfaceTolerance * kOnSurfaceTolerance) {
      const double u = (dot3(mab, d) - dot3(mab, eb) * eaTeb) / denom;
      onSurface = u * u < kOnSurfaceTolerance * kOnSurfaceTolerance;
      distance = u;
    }
    if (onSurface) {
      cur = -2;
      targetReached = true;
    } else {
      ss.update(nd * distance, kAborter);
      // pathLimit's update follows and replaces a NaN by its limit
      if constexpr (!kRecords)
        if (distance != distance) ss.v[kAborter] = nd * kDblMax;
    }
    return onSurface;
  }

  KFD_INLINE bool kalmanAbort() const { return !result || finished; }
  KFD_INLINE bool finalizeCond() const {
    return (measured == (int)(h1 - h0) || (measured > 0 && navBreak)) && !smoothed && !finished;
  }

  // ------------------------------------------------------------- material ----
  // Actor::materialInteractor (KalmanFitter.hpp:405-449) with
  // PointwiseMaterialInteraction (.hpp:66-148, .ipp:14-53) and the RPP
  // formulas of Interactions.ipp (Bethe :150-176, Landau sigma :316-342,
  // Highland :501-546).  Only plane surfaces carry material (full update).
  // The formulas run in S: in the mixed mode the energy loss (~1e-4 of p)
  // and the noise variances need no more than float's 1e-7 relative; the
  // momentum itself is updated in double.
  KFD_INLINE void material(const DevPlane &pl) {
    if (!pl.has_material) return;
    const double momentum = p;
    const S qq = (S)q;
    const S qOverP = (S)(q / momentum);
    const S mass = (S)a.mass;
    const S nr[3] = {(S)pl.r[2], (S)pl.r[5], (S)pl.r[8]};
    const S d[3] = {(S)dir[0], (S)dir[1], (S)dir[2]};
    const S pcor = (S)1 / fabs(dot3(nr, d));
    const S thick = (S)pl.thickness * pcor;
    const S xOverX0 = (S)pl.thicknessInX0 * pcor;
    if (!((S)0 < thick)) return;
    // RelativisticQuantities, Interactions.ipp:27-52
    const S q2OverBeta2 = qq * qq + (mass * qOverP) * (mass * qOverP);
    const S mOverP = mass * fabs(qOverP / qq);
    const S pOverM = (S)1 / mOverP;
    const S beta2 = (S)1 / ((S)1 + mOverP * mOverP);
    const S betaGamma = pOverM;
    const S gamma = sqrt((S)1 + pOverM * pOverM);
    const S Ne = (S)pl.molarElectronDensity;
    const S eps = (S)0.5 * (S)a.kK * Ne * thick * q2OverBeta2;
    S Eloss = (S)0, vPhi = (S)0, vTheta = (S)0, vQop = (S)0;
    if (a.eloss) {
      const S I = (S)pl.meanExcitation;
      const S kMe = (S)a.kMe;
      S dhalf = (S)0;
      if (!(betaGamma < (S)10)) {
        const S plasma = (S)a.kPlasma * sqrt(Ne);
        dhalf = logS(betaGamma) + logS(plasma / I) - (S)0.5;
      }
      const S u = (S)2 * kMe * betaGamma * betaGamma;
      const S mfrac = kMe / mass;
      const S nom = (S)2 * kMe * betaGamma * betaGamma;
      const S den = (S)1 + (S)2 * gamma * mfrac + mfrac * mfrac;
      const S wmax = nom / den;
      const S running = (S)0.5 * logS(u / I) + (S)0.5 * logS(wmax / I) - beta2 - dhalf;
      Eloss = eps * running;
    }
    if (a.ms) {
      const S tt = sqrt(xOverX0 * q2OverBeta2);
      const S theta0 =
          (S)a.kHighland * fabs(qOverP / qq) * tt * ((S)1 + (S)a.kHighlandLog * logS(tt));
      const S dn = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
      const S sigmaPhi = theta0 * (dn / sqrt(d[0] * d[0] + d[1] * d[1]));
      vPhi = sigmaPhi * sigmaPhi;
      vTheta = theta0 * theta0;
    }
    if (a.eloss) {
      const S fwhm = (S)4 * eps;
      const S sigmaE = fwhm / (S)a.kLandauConv;
      const S pInv = qOverP / qq;
      const S sq = sqrt(q2OverBeta2) * pInv * pInv * sigmaE;
      vQop = sq * sq;
    }
    const double nextE =
        sqrt(a.mass * a.mass + momentum * momentum) - copysign((double)Eloss, (double)navDir);
    p = (a.mass < nextE) ? sqrt(nextE * nextE - a.mass * a.mass) : 0.0;
    const double mode = (navDir == 1) ? 1.0 : -1.0;
    double v;  // std::max(0, v) of updateVariance
    v = (double)cov[sidx(2, 2)] + copysign((double)vPhi, mode);
    cov[sidx(2, 2)] = (S)((0.0 < v) ? v : 0.0);
    v = (double)cov[sidx(3, 3)] + copysign((double)vTheta, mode);
    cov[sidx(3, 3)] = (S)((0.0 < v) ? v : 0.0);
    v = (double)cov[sidx(4, 4)] + copysign((double)vQop, mode);
    cov[sidx(4, 4)] = (S)((0.0 < v) ? v : 0.0);
  }

  // -------------------------------------------------------------- filter ----
  // Actor::filter (KalmanFitter.hpp:284-350) with GainMatrixUpdater
  // (GainMatrixUpdater.hpp:34-106).  FP64 mode: the reference's (I - K H) P
  // update.  Mixed mode: the Joseph form (I - K H) P (I - K H)^T + K V K^T,
  // which stays positive definite under the float-rounded predicted
  // covariance; each (i, j) pair is formed once, so the result is symmetric
  // by construction.  The 2x2 inversion and the update are double in both.
  KFD_INLINE bool filter(int sp) {
    // a copy in the fused builds (the smoother's LDS stores may alias the table in
    // LDS, and each would have the plane read again), but not in the mixed grid
    // one, whose registers it overfills (500,003 ragged tracks 2.27 -> 2.36 ms)
    using PlaneOrCopy =
        std::conditional_t<kFirst && (!kMixed || FK == kFieldConst), const DevPlane, const DevPlane &>;
    PlaneOrCopy pl = plane(sp);
    // the track's hit on this plane: first match in hit order (SurfaceFinder,
    // KalmanFitter.hpp:31-38); the loaded-ahead next hit, else a scan with
    // four independent geo-id loads per round trip
    int64_t hit = -1;
    double m0, m1, V00, V01, V11;
    if (inOrder && pfValid && pfGeo == pl.geo_id) {
      hit = hitNext;
      m0 = pfM0;
      m1 = pfM1;
      V00 = pfV00;
      V01 = pfV01;
      V11 = pfV11;
    } else {
      for (int64_t h = inOrder ? hitNext : h0; h < h1 && hit < 0; h += 4) {
        int32_t g[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) g[q] = (h + q < h1) ? a.hit_geo_id[h + q] : 0;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (hit < 0 && h + q < h1 && g[q] == pl.geo_id) hit = h + q;
      }
      if (hit < 0) {  // hole
        if constexpr (PS) ++holes;
        return true;
      }
      m0 = a.hit_meas[hit];
      m1 = a.hit_meas[a.n_hits + hit];
      V00 = a.hit_cov[hit];
      V01 = a.hit_cov[a.n_hits + hit];
      V11 = a.hit_cov[2 * a.n_hits + hit];
      // waited for here: left pending, every filter would wait before its gain
      // for all loads in flight, the next hit's among them
      waitLoads();
      inOrder = inOrder && hit == hitNext;
    }
    if (inOrder) {
      hitNext = hit + 1;
      prefetchHit();
    }
    if (measured >= a.max_states) return false;
    const int k = measured;
    int s = k;  // store slot
    if constexpr (PS) {
      const int slack = a.max_states - (int)(h1 - h0);
      s = k + ((holes < slack) ? holes : (slack > 0 ? slack : 0));
    }
    if (k == 0) firstPlane = sp;
    double xp[6];
    S jb[6][6];
    S cfPrev[21], cPred[21];  // kFxRts
    if constexpr (kFxRts) {
#pragma unroll
      for (int m = 0; m < 21; ++m) cfPrev[m] = cov[m];
      cfPrev[sidx(2, 2)] = fxDiag[0];
      cfPrev[sidx(3, 3)] = fxDiag[1];
      cfPrev[sidx(4, 4)] = fxDiag[2];
    }
    boundStatePlane(pl, xp, jb);
    if constexpr (kFxRts) {
#pragma unroll
      for (int m = 0; m < 21; ++m) cPred[m] = cov[m];
    }
    // predicted parameters and the transport Jacobian to the store, with the
    // slot of the state two measurements back (the smoother's look-ahead)
    if constexpr (kStore) {
      storePar(s, KF_SD_XP, xp);
      S jv[KF_SS_CF - KF_SS_J];
#pragma unroll
      for (int r = 0; r < 6; ++r)
#pragma unroll
        for (int c = 0; c < 5; ++c)
          if (r != 4) jv[jidx(r, c)] = jb[r][c];
      jv[KF_SS_LINK] = PS ? linkBits(slotPrev, (S)0) : (S)0;
#pragma unroll
      for (int m = KF_SS_LINK + 1; m < KF_SS_CF - KF_SS_J; ++m) jv[m] = (S)0;
      storeS<KF_SS_CF - KF_SS_J>(s, KF_SS_J, jv);
    } else if constexpr (kFirst && !kMixed) {
      if (k == 0)
        fxInit();
      else
        fxTransport(jb);
    }
    if (tsf && lead) {
      storeBoundF(k, KF_TS_PREDICTED, xp, cov);
#pragma unroll
      for (int r = 0; r < 6; ++r)
#pragma unroll
        for (int c = 0; c < 6; ++c) *recF(k, KF_TS_JACOBIAN + 6 * r + c) = (double)jb[r][c];
      *recF(k, KF_TS_PATH) = pathAcc;
      *recF(k, KF_TS_GEO_ID) = (double)pl.geo_id;
    }
    // gain-matrix update
    const double S00 = cov[sidx(0, 0)] + V00, S01 = cov[sidx(0, 1)] + V01;
    const double S10 = cov[sidx(1, 0)] + V01, S11 = cov[sidx(1, 1)] + V11;
    const double det = S00 * S11 - S01 * S10;
    const double idet = 1.0 / det;
    const double i00 = S11 * idet, i01 = -S01 * idet, i10 = -S10 * idet, i11 = S00 * idet;
    const double r0 = m0 - xp[0], r1 = m1 - xp[1];
    const double chi2 = r0 * (i00 * r0 + i01 * r1) + r1 * (i10 * r0 + i11 * r1);
    double xf[6];
    if constexpr (kFirst) {
      // the predicted covariance and the hit's are positive definite, and the
      // hit is not so much more precise that the update loses definiteness
      fxOk = fxOk && (S)0 < cov[sidx(0, 0)] && (S)0 < cov[sidx(1, 1)] && (S)0 < cov[sidx(2, 2)] &&
             (S)0 < cov[sidx(3, 3)] && (S)0 < cov[sidx(4, 4)] && (S)0 < cov[sidx(5, 5)] &&
             V00 > 1e-12 * S00 && V11 > 1e-12 * S11 &&
             V00 * V11 - V01 * V01 > 1e-12 * (V00 * V11);
    }
    // outlier finder: above the cut the state keeps its prediction (no
    // update, the covariance stays the predicted one) and stays out of the
    // chi2 sum and ndf; 0 disables it (the reference's void finder)
    if (outlierCut > 0.0 && chi2 > outlierCut) {
#pragma unroll
      for (int r = 0; r < 6; ++r) xf[r] = xp[r];
      ++outliers;
    } else {
    double K0[6], K1[6];
#pragma unroll
    for (int r = 0; r < 6; ++r) {
      K0[r] = cov[sidx(r, 0)] * i00 + cov[sidx(r, 1)] * i10;
      K1[r] = cov[sidx(r, 0)] * i01 + cov[sidx(r, 1)] * i11;
    }
#pragma unroll
    for (int r = 0; r < 6; ++r) xf[r] = xp[r] + (K0[r] * r0 + K1[r] * r1);
    if constexpr (kFirst && !kMixed) {
      if (k > 0) fxMeasure(K0, K1, i00, i01, i11, i00 * r0 + i01 * r1, i10 * r0 + i11 * r1);
    }
    // the update in place on cov: rows 0 and 1 of the result go to t01 first
    // (every entry reads the old rows 0 and 1), then rows 2..5 overwrite
    // cov, then rows 0 and 1 are written back
    double t01[11];
    if (kFxRts && 1e-6 * (S00 * S11) < det) {
      // the same matrix for the gain as computed here, (I - K H) P, with its
      // rows 0 and 1 as K V: no cancellation in them, and the other entries
      // cancel as in the Joseph form's first term.  First order in the error
      // of K, so only where the innovation is well conditioned (an error of K
      // below 1e-10, under the float rounding of the result); 42 operations
      // for ~200
#pragma unroll
      for (int c = 0; c < 6; ++c) t01[c] = K0[c] * V00 + K1[c] * V01;
#pragma unroll
      for (int c = 1; c < 6; ++c) t01[5 + c] = K0[c] * V01 + K1[c] * V11;
#pragma unroll
      for (int r = 2; r < 6; ++r)
#pragma unroll
        for (int c = r; c < 6; ++c)
          cov[sidx(r, c)] = (S)(cov[sidx(r, c)] - K0[r] * cov[sidx(0, c)] - K1[r] * cov[sidx(1, c)]);
    } else if constexpr (kMixed) {
      // B = (I - K H) P: columns 0 and 1 here, the other (r <= c) entries
      // where they are consumed
      double B0[6], B1[6];
#pragma unroll
      for (int r = 0; r < 6; ++r) {
        B0[r] = cov[sidx(r, 0)] - K0[r] * cov[sidx(0, 0)] - K1[r] * cov[sidx(1, 0)];
        B1[r] = cov[sidx(r, 1)] - K0[r] * cov[sidx(0, 1)] - K1[r] * cov[sidx(1, 1)];
      }
      auto joseph = [&](int r, int c) {
        const double brc = (c == 0) ? B0[r] : (c == 1) ? B1[r]
                                    : cov[sidx(r, c)] - K0[r] * cov[sidx(0, c)] - K1[r] * cov[sidx(1, c)];
        const double kv0 = V00 * K0[c] + V01 * K1[c];
        const double kv1 = V01 * K0[c] + V11 * K1[c];
        return (brc - B0[r] * K0[c] - B1[r] * K1[c]) + (K0[r] * kv0 + K1[r] * kv1);
      };
#pragma unroll
      for (int c = 0; c < 6; ++c) t01[c] = joseph(0, c);
#pragma unroll
      for (int c = 1; c < 6; ++c) t01[5 + c] = joseph(1, c);
#pragma unroll
      for (int r = 2; r < 6; ++r)
#pragma unroll
        for (int c = r; c < 6; ++c) cov[sidx(r, c)] = (S)joseph(r, c);
    } else {
      auto standard = [&](int r, int c) {
        const double ca = ((r == 0) ? 1.0 : 0.0) - K0[r];
        const double cb = ((r == 1) ? 1.0 : 0.0) - K1[r];
        double s = ca * cov[sidx(0, c)] + cb * cov[sidx(1, c)];
        if (r >= 2) s = s + cov[sidx(r, c)];
        return s;
      };
#pragma unroll
      for (int c = 0; c < 6; ++c) t01[c] = standard(0, c);
#pragma unroll
      for (int c = 1; c < 6; ++c) t01[5 + c] = standard(1, c);
#pragma unroll
      for (int r = 2; r < 6; ++r)
#pragma unroll
        for (int c = r; c < 6; ++c) cov[sidx(r, c)] = (S)standard(r, c);
    }
#pragma unroll
    for (int c = 0; c < 6; ++c) cov[sidx(0, c)] = (S)t01[c];
#pragma unroll
    for (int c = 1; c < 6; ++c) cov[sidx(1, c)] = (S)t01[5 + c];
    chi2sum = chi2sum + chi2;
    }
    if constexpr (kFirst)
      if (k > 0) fxAngles(xf);
    correctParams(xf);
    if constexpr (kStore) {
      storePar(s, KF_SD_XF, xf);
    } else if constexpr (kFxRts) {
      if (a.smoothing) {
        if (k == 0)
          fxRtsInit(xf);
        else
          fxRtsStep(jb, cfPrev, cPred, xp, xf);
        fxDiag[0] = cov[sidx(2, 2)];
        fxDiag[1] = cov[sidx(3, 3)];
        fxDiag[2] = cov[sidx(4, 4)];
      }
    } else if constexpr (kFirst) {
      if (k == 0) fxKeepFirst(xf);
    }
    if (tsf && lead) {
      storeBoundF(k, KF_TS_FILTERED, xf, cov);
      *recF(k, KF_TS_CHI2) = chi2;
    }
    // the filtered covariance and, after the material update, the three
    // diagonal entries in which the covariance the next transport starts
    // from differs from it
    S cm[KF_SS_N - KF_SS_CF];
    if constexpr (kStore) {
#pragma unroll
      for (int m = 0; m < 21; ++m) cm[m] = cov[m];
    }
    updateFromFiltered(pl, xf, xp);
    setReference(xf);
    material(pl);
    if constexpr (kStore) {
      cm[KF_SS_MD - KF_SS_CF + 0] = cov[sidx(2, 2)];
      cm[KF_SS_MD - KF_SS_CF + 1] = cov[sidx(3, 3)];
      cm[KF_SS_MD - KF_SS_CF + 2] = cov[sidx(4, 4)];
      storeS<KF_SS_N - KF_SS_CF>(s, KF_SS_CF, cm);
    }
    if (tsc) saveCheckpoint(k, hit);
    if constexpr (PS) {
      slotPrev = slotLast;
      slotLast = s;
    }
    ++measured;
    return true;
  }

  // -------------------------------------------------------------- smoother ----
  // The diagonal scale of spdSolve, ~1 / sqrt(c).  Any positive scale gives
  // the same solution in exact arithmetic (the factorisation works on the
  // scaled diagonal as computed, not on an assumed 1), so the GPU takes the
  // hardware's reciprocal square root without refinement (one instruction
  // instead of a correctly rounded square root and division); NaN for c < 0
  // and infinity for c = 0 as 1 / sqrt(c).
  KFD_INLINE static double scaleOf(double c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsq(c);
#else
    return 1.0 / sqrt(c);  // host build of the fit program
#endif
  }

  // X = C^-1 M for a symmetric positive-definite 6x6 C (packed) and six
  // right-hand sides, in place on M: LDL^T factorisation of the
  // diagonally scaled matrix S C S (S = diag(C)^-1/2, unit diagonal, so no
  // pivoting is needed), then forward substitution, scaling by D^-1 and back
  // substitution per column.  The reference inverts C explicitly (Eigen's
  // partial-pivoting LU on the host, cofactors on the device,
  // include/Utilities/Math.hpp:74-112); solving is ~3x cheaper and agrees to
  // rounding.  A non-positive diagonal entry gives NaNs (caught by the
  // smoother's NaN check, as the reference's).
  KFD_INLINE static void spdSolve(const double C[21], double M[6][6]) {
    double sc[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) sc[k] = scaleOf(C[sidx(k, k)]);
    // W[r][k] = Lo[r][k] D[k] (r > k), Lo below the diagonal, Dinv = 1 / D
    double Lo[6][6], W[6][6], Dinv[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      double dj = (sc[j] * C[sidx(j, j)]) * sc[j];
#pragma unroll
      for (int k = 0; k < j; ++k) dj = dj - W[j][k] * Lo[j][k];
      Dinv[j] = 1.0 / dj;
#pragma unroll
      for (int r = j + 1; r < 6; ++r) {
        double w = (sc[r] * C[sidx(r, j)]) * sc[j];
#pragma unroll
        for (int k = 0; k < j; ++k) w = w - W[r][k] * Lo[j][k];
        W[r][j] = w;
        Lo[r][j] = w * Dinv[j];
      }
    }
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      double y[6];
#pragma unroll
      for (int r = 0; r < 6; ++r) {
        double v = sc[r] * M[r][c];
#pragma unroll
        for (int k = 0; k < r; ++k) v = v - Lo[r][k] * y[k];
        y[r] = v;
      }
#pragma unroll
      for (int r = 0; r < 6; ++r) y[r] = y[r] * Dinv[r];
#pragma unroll
      for (int r = 5; r >= 0; --r) {
        double v = y[r];
#pragma unroll
        for (int k = r + 1; k < 6; ++k) v = v - Lo[k][r] * y[k];
        y[r] = v;
      }
#pragma unroll
      for (int r = 0; r < 6; ++r) M[r][c] = sc[r] * y[r];
    }
  }

  // X = J C_f (C_f symmetric); row 4 of J is e4 and column 5 is e5.
  KFD_INLINE static void transported(const S J[6][6], const double cf[21], double X[6][6]) {
#pragma unroll
    for (int r = 0; r < 6; ++r)
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        double s;
        if (r == 4) {
          s = cf[sidx(4, c)];
        } else {
          s = (double)J[r][0] * cf[sidx(0, c)];
#pragma unroll
          for (int m = 1; m < 5; ++m) s = s + (double)J[r][m] * cf[sidx(m, c)];
          if (r == 5) s = s + cf[sidx(5, c)];
        }
        X[r][c] = s;
      }
  }

  // spdSolve without the diagonal scaling (the pivots of L D L^T and what they
  // lose do not depend on it, 130 of 430 operations), for the fixed-point sums.
  // False where a pivot is not positive: such a track takes the RTS program,
  // whose scaled solver decides what its gain is.
  KFD_INLINE static bool spdSolvePivots(const double C[21], double M[6][6]) {
    double Lo[6][6], W[6][6], Dinv[6];
    bool ok = true;
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      double dj = C[sidx(j, j)];
#pragma unroll
      for (int k = 0; k < j; ++k) dj = dj - W[j][k] * Lo[j][k];
      ok = ok && 0.0 < dj;
      Dinv[j] = recipD(dj);
#pragma unroll
      for (int r = j + 1; r < 6; ++r) {
        double w = C[sidx(r, j)];
#pragma unroll
        for (int k = 0; k < j; ++k) w = w - W[r][k] * Lo[j][k];
        W[r][j] = w;
        Lo[r][j] = w * Dinv[j];
      }
    }
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      double y[6];
#pragma unroll
      for (int r = 0; r < 6; ++r) {
        double v = M[r][c];
#pragma unroll
        for (int k = 0; k < r; ++k) v = v - Lo[r][k] * y[k];
        y[r] = v;
      }
#pragma unroll
      for (int r = 5; r >= 0; --r) {
        double v = y[r] * Dinv[r];
#pragma unroll
        for (int k = r + 1; k < 6; ++k) v = v - Lo[k][r] * y[k];
        y[r] = v;
        M[r][c] = v;
      }
    }
    return ok;
  }

  // Filtered covariance of state k, in double.
  KFD_INLINE void loadFilteredCov(int k, double c[21]) const {
    S cm[KF_SS_N - KF_SS_CF];
    loadS<KF_SS_N - KF_SS_CF>(k, KF_SS_CF, cm);
#pragma unroll
    for (int m = 0; m < 21; ++m) c[m] = (double)cm[m];
  }

  // Stored operands of smoother step k: the Jacobian, predicted parameters
  // and link of state k + 1 (slot sn), the filtered covariance,
  // post-material diagonal and filtered parameters of state k (slot sk).
  struct SmoothIn {
    S j[25];
    S cf[21];
    S md[3];
    double xf[6];
    double xpn[6];
    int link;  // slot of state k - 1 (-1: none)
  };
  KFD_INLINE void loadSmoothIn(int sk, int sn, SmoothIn &in) const {
    S jv[KF_SS_CF - KF_SS_J], cm[KF_SS_N - KF_SS_CF];
    loadS<KF_SS_CF - KF_SS_J>(sn, KF_SS_J, jv);
    loadS<KF_SS_N - KF_SS_CF>(sk, KF_SS_CF, cm);
#pragma unroll
    for (int m = 0; m < 25; ++m) in.j[m] = jv[m];
    in.link = linkOf(jv[KF_SS_LINK]);
#pragma unroll
    for (int m = 0; m < 21; ++m) in.cf[m] = cm[m];
#pragma unroll
    for (int m = 0; m < 3; ++m) in.md[m] = cm[KF_SS_MD - KF_SS_CF + m];
    loadPar(sk, KF_SD_XF, in.xf);
    loadPar(sn, KF_SD_XP, in.xpn);
  }

  // One smoother step (GainMatrixSmoother.hpp:21-94): state k from its
  // stored operands `in` and the smoothed state k + 1 (xsn, csn), which it
  // overwrites with the smoothed state k.  False on a NaN gain.
  // G = (C_f J^T) C_p^-1, x_s = x_f + G (x_s' - x_p'), C_s = C_f - G (C_p - C_s') G^T,
  // in double in both modes.
  KFD_INLINE bool smoothStep(int k, const SmoothIn &in, double xsn[6], double csn[21]) {
    S J[6][6];
#pragma unroll
    for (int r = 0; r < 6; ++r)
#pragma unroll
      for (int c = 0; c < 6; ++c)
        J[r][c] = (r == 4 || c == 5) ? ((r == c) ? (S)1 : (S)0) : in.j[jidx(r, c)];
    // predicted covariance of state k + 1: the forward pass's transport of
    // the post-material covariance of state k, from the same operands
    double Cp[21];
    {
      S cm[21];
#pragma unroll
      for (int m = 0; m < 21; ++m) cm[m] = in.cf[m];
      cm[sidx(2, 2)] = in.md[0];
      cm[sidx(3, 3)] = in.md[1];
      cm[sidx(4, 4)] = in.md[2];
      sandwich(J, cm, Cp);
    }
    double cf[21];
#pragma unroll
    for (int m = 0; m < 21; ++m) cf[m] = (double)in.cf[m];
    // G^T = C_p^-1 (J C_f) (C_p symmetric)
    double G[6][6];
    {
      double X[6][6];
      transported(J, cf, X);
      spdSolve(Cp, X);
#pragma unroll
      for (int r = 0; r < 6; ++r)
#pragma unroll
        for (int c = 0; c < 6; ++c) G[r][c] = X[c][r];
    }
    bool nan = false;  // GainMatrixSmoother.hpp:63-66
#pragma unroll
    for (int r = 0; r < 6; ++r)
#pragma unroll
      for (int c = 0; c < 6; ++c) nan = nan || (G[r][c] != G[r][c]);
    if (nan) {
      smootherNaN = true;
      return false;
    }
    double dx[6];
#pragma unroll
    for (int r = 0; r < 6; ++r) dx[r] = xsn[r] - in.xpn[r];
#pragma unroll
    for (int r = 0; r < 6; ++r) {
      double s = G[r][0] * dx[0];
#pragma unroll
      for (int m = 1; m < 6; ++m) s = s + G[r][m] * dx[m];
      xsn[r] = in.xf[r] + s;
    }
    double Dm[21];
#pragma unroll
    for (int m = 0; m < 21; ++m) Dm[m] = Cp[m] - csn[m];
#pragma unroll
    for (int r = 0; r < 6; ++r) {
      double B1[6];  // row r of G (C_p - C_s')
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        double s = G[r][0] * Dm[sidx(0, c)];
#pragma unroll
        for (int m = 1; m < 6; ++m) s = s + G[r][m] * Dm[sidx(m, c)];
        B1[c] = s;
      }
#pragma unroll
      for (int c = r; c < 6; ++c) {
        double s = B1[0] * G[c][0];
#pragma unroll
        for (int m = 1; m < 6; ++m) s = s + B1[m] * G[c][m];
        csn[sidx(r, c)] = cf[sidx(r, c)] - s;
      }
    }
    correctParams(xsn);
    if (tsf) storeBoundF(k, KF_TS_SMOOTHED, xsn, csn);
    return true;
  }

  // The smoother over the stored states.  The operands of step k - 1 are
  // loaded while step k computes.  PS = false: the loop runs over k (state k
  // in slot k).  PS = true: it walks the store slots downwards from the last
  // one the sequence can use and smooths a state when it reaches its slot,
  // so the lanes whose tracks cross the same planes read the same store
  // chunk in the same iteration (a lane idles at the slots of its holes);
  // the walk ends after at most max_states iterations.
  KFD_INLINE bool smooth(double xs[6], double cs[21]) {
    const int n = measured;
    double xsn[6], csn[21];
    // last state: smoothed = filtered
    const int sl = PS ? slotLast : n - 1;  // its slot
    loadPar(sl, KF_SD_XF, xsn);
    loadFilteredCov(sl, csn);
    if (tsf) storeBoundF(n - 1, KF_TS_SMOOTHED, xsn, csn);
    SmoothIn cur;
    if constexpr (!PS) {
      if (n >= 2) loadSmoothIn(n - 2, n - 1, cur);
      for (int k = n - 2; k >= 0; --k) {
        SmoothIn nxt;
        loadSmoothIn((k > 0) ? k - 1 : 0, k, nxt);
        if (!smoothStep(k, cur, xsn, csn)) return false;
        cur = nxt;
      }
    } else {
      int sk = slotPrev;  // slot of state k
      if (n >= 2) loadSmoothIn(sk, sl, cur);
      int slot = ((size < a.max_states) ? size : a.max_states) - 1;
      int k = n - 2;
      for (; k >= 0 && slot >= 0; --slot) {
        if (slot != sk) continue;  // a hole of this track
        const int link = cur.link;
        SmoothIn nxt;
        loadSmoothIn((k > 0 && link >= 0 && link < sk) ? link : sk, sk, nxt);
        if (!smoothStep(k, cur, xsn, csn)) return false;
        cur = nxt;
        sk = link;
        --k;
      }
      if (k >= 0) {  // slots out of order: the store is inconsistent
        smootherNaN = true;
        return false;
      }
    }
#pragma unroll
    for (int m = 0; m < 6; ++m) xs[m] = xsn[m];
#pragma unroll
    for (int m = 0; m < 21; ++m) cs[m] = csn[m];
    return true;
  }

  // Actor::operator(), KalmanFitter.hpp:216-273, of the forward pass: filter
  // and the finalisation check; returns true where finalize() must run.
  KFD_INLINE bool actor() {
    if (cur >= 0 && !smoothed && !finished) {
      if (!filter(cur)) result = false;
    }
    if (finalizeCond()) {
      if (!a.smoothing) {
        finished = true;
      } else {
        return true;
      }
    }
    return false;
  }

  // The same of the backward pass: only the part after the finalisation can
  // act (smoothed is set).
  KFD_INLINE void actorPost() {
    if (smoothed && !finished && surfaceReached()) {
      double par[6];
      boundStateLine(par);
      writeFit(par, cov);
      finished = true;
    }
  }

  // Iterations of the propagation loop (Propagator.ipp:39-69) in which the
  // actor has nothing to do.  Stops where it has (true), or where the loop
  // ends: terminated by an aborter or after max_steps.
  template <bool F>
  KFD_INLINE bool cheapSteps(int &steps, bool &terminated) {
    while (steps < maxSteps) {
      step();
      navStatus();
      if (F && cur >= 0 && !smoothed && !finished) return true;
      if (F && finalizeCond()) return true;
      if (!F && smoothed && !finished && surfaceReached()) return true;
      if (kalmanAbort() || pathLimit()) {
        terminated = true;
        return false;
      }
      navTarget();
      ++steps;
    }
    return false;
  }

  // ------------------------------------------------------------- carry ----
  // Per-track hand-over record from the forward to the backward kernel.
  enum {
    kCI_resume = 0, kCI_steps, kCI_measured, kCI_first, kCI_next, kCI_flags, kCI_slotLast,
    kCI_slotPrev, kCI_N
  };
  enum { kCD_q = 0, kCD_J = 1, kCD_k4 = 26, kCD_dtds = 29, kCD_N = 30 };
  static_assert(kCI_N == KF_CARRY_I && kCD_N == KF_CARRY_D, "hand-over record layout");
  KFD_INLINE int32_t &ci(int f) const { return ciBase[(size_t)f * cslots + cpos]; }
  KFD_INLINE double &cd(int f) const { return cdBase[(size_t)f * cslots + cpos]; }

  KFD_INLINE void saveCarry(int resume, int steps, bool terminated) const {
    if (!lead) return;
    ci(kCI_resume) = resume;
    ci(kCI_steps) = steps;
    ci(kCI_measured) = measured;
    ci(kCI_first) = firstPlane;
    ci(kCI_next) = next;
    if constexpr (PS) {
      ci(kCI_slotLast) = slotLast;
      ci(kCI_slotPrev) = slotPrev;
    }
    ci(kCI_flags) = (result ? 1 : 0) | (stepFailed ? 2 : 0) | (navBreak ? 4 : 0) |
                    (terminated ? 8 : 0) | (derivSet ? 16 : 0);
    cd(kCD_q) = q;
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 5; ++c) cd(kCD_J + 5 * r + c) = (double)A[r][c];
    cd(kCD_J + 15) = (double)b;
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) cd(kCD_J + 16 + 3 * r + c) = (double)G[r][c];
#pragma unroll
    for (int k = 0; k < 3; ++k) cd(kCD_k4 + k) = (double)k4d[k];
    cd(kCD_dtds) = (double)dtds;
  }

  KFD_INLINE int loadCarry(int &steps, bool &terminated) {
    const int resume = ci(kCI_resume);
    steps = ci(kCI_steps);
    measured = ci(kCI_measured);
    firstPlane = ci(kCI_first);
    next = ci(kCI_next);
    if constexpr (PS) {
      slotLast = ci(kCI_slotLast);
      slotPrev = ci(kCI_slotPrev);
    }
    const int fl = ci(kCI_flags);
    result = (fl & 1) != 0;
    stepFailed = (fl & 2) != 0;
    navBreak = (fl & 4) != 0;
    terminated = (fl & 8) != 0;
    derivSet = (fl & 16) != 0;
    q = cd(kCD_q);
    return resume;
  }

  KFD_INLINE void loadCarryJacobian() {
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 5; ++c) A[r][c] = (S)cd(kCD_J + 5 * r + c);
    b = (S)cd(kCD_J + 15);
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) G[r][c] = (S)cd(kCD_J + 16 + 3 * r + c);
#pragma unroll
    for (int k = 0; k < 3; ++k) k4d[k] = (S)cd(kCD_k4 + k);
    dtds = (S)cd(kCD_dtds);
  }

  // ----------------------------------------------------------------- fit ----
  KFD_INLINE uint32_t statusBits(int steps, bool terminated) const {
    uint32_t status = 0;
    if (result && measured == (int)(h1 - h0)) status |= KF_STATUS_OK;
    if (smoothed) status |= KF_STATUS_SMOOTHED;
    if (finished) status |= KF_STATUS_FINISHED;
    if (!result) status |= KF_STATUS_RESULT_FAIL;
    if (stepFailed) status |= KF_STATUS_STEP_FAIL;
    if (!terminated && steps >= maxSteps) status |= KF_STATUS_MAX_STEPS;
    if (navBreak && measured != (int)(h1 - h0)) status |= KF_STATUS_NAV_BREAK;
    if (smootherNaN) status |= KF_STATUS_SMOOTHER_NAN;
    return status;
  }

  // The fitted parameters and covariance go out where they are computed (27
  // doubles that would otherwise stay in registers through the last steps).
  template <typename T>
  KFD_INLINE void writeFit(const double par[6], const T c[21]) const {
    if (!lead) return;
    if (a.out_params)
#pragma unroll
      for (int k = 0; k < 6; ++k) a.out_params[(size_t)k * a.n + i] = par[k];
    if (a.out_cov)
#pragma unroll
      for (int k = 0; k < 21; ++k) a.out_cov[(size_t)k * a.n + i] = (double)c[k];
  }
  // The end of a track: its status, and zeros where no fit came out.
  // `written`: writeFit has run.
  KFD_INLINE void writeFinal(uint32_t status, bool written) const {
    if (!written) {
      const double par[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      const double c[21] = {0.0};
      writeFit(par, c);
    }
    if (lead && a.out_status) a.out_status[i] = status;
  }

  KFD_INLINE void loadPerigee() {
#pragma unroll
    for (int k = 0; k < 3; ++k) lc[k] = a.perigee[(size_t)k * a.n + i];
  }

  KFD_INLINE void loadTrack() {
    loadOptions();
    h0 = a.hit_offset[i];
    h1 = a.hit_offset[i + 1];
    hitNext = h0;
    inOrder = a.unique_geo != 0;
    pfValid = false;
    seqFirst = a.seq_first[i];
    size = a.seq_count[i];
    loadPerigee();
    smoothed = finished = smootherNaN = false;
    cur = -1;
    targetReached = false;
  }

  // The forward pass: Propagator::propagate (Propagator.ipp:3-96) up to the
  // finalisation.  Returns where the finalisation is due (kResume*).
  KFD_INLINE int forwardPass(int &steps, bool &terminated, bool &bad) {
    loadTrack();
    double pv[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) pv[k] = a.start_params[(size_t)k * a.n + i];
#pragma unroll
    for (int k = 0; k < 21; ++k) cov[k] = a.start_cov[(size_t)k * a.n + i];
    measured = 0;
    outliers = 0;
    firstPlane = 0;
    holes = 0;
    slotLast = slotPrev = -1;
    result = true;
    chi2sum = 0.0;
    next = 0;
    navBreak = false;
    stepFailed = false;
    terminated = false;
    steps = 0;
    bad = size <= 0 || seqFirst < 0 || seqFirst + size > a.n_planes || h0 < 0 || h1 <= h0 ||
          h1 > a.n_hits || pv[4] == 0.0 || a.max_states < 1;
    if constexpr (kFirst)
      if (picker && !bad && fabs(pv[2]) > kNearWrapPhi && nearWrap(picker, i)) {
        elsewhere = true;
        return kResumeNone;
      }
    // A singular start covariance (leaveEarly): looked at after what does not wait for
    // the covariance, below (1,048,576 mixed tracks 1,758 -> 1,735 us), but here in the
    // mixed grid build, whose registers it overfills there (500,003 ragged ones
    // 2,306 -> 2,270 us)
    constexpr bool kLookFirst = kMixed && FK == kFieldGrid;
    if constexpr (kFirst && kLookFirst) {
      fxOk = bad || fxDefinite();
      if (leaveEarly && a.smoothing && !fxOk) {
        left = true;
        return kResumeNone;
      }
    }
    // Before the loop, in it and after it the actor is called from one place
    // (its code is most of the kernel): `at` says which of the three this is.
    int resume = kResumeNone;
    if (!bad) {
      prefetchHit();
      start(pv);
      if constexpr (kFirst && !kLookFirst) {
        fxOk = fxDefinite();
        if (leaveEarly && a.smoothing && !fxOk) {
          left = true;
          return kResumeNone;
        }
      }
      navStatus();
      int at = kResumePreLoop;
      for (;;) {
        if (actor()) {
          resume = at;
          break;
        }
        if (at == kResumePostLoop) break;
        bool more = !(kalmanAbort() || pathLimit());
        if (more) {
          navTarget();
          if (at == kResumeInLoop) ++steps;
          at = kResumeInLoop;
          more = cheapSteps<true>(steps, terminated);
        } else if (at == kResumeInLoop) {
          terminated = true;
        }
        if (!more) {
          at = kResumePostLoop;
          if (!terminated) navBreak = true;
        }
      }
    }
    if (lead) {
      if (a.out_chi2) a.out_chi2[i] = chi2sum;
      if (a.out_ndf) a.out_ndf[i] = 2 * (measured - outliers);
      if (a.out_nmeas) a.out_nmeas[i] = measured;
    }
    return resume;
  }

  // The state of the smoothed first surface (xs, cs), from which the
  // propagation back to the perigee starts.
  KFD_INLINE void fromSmoothed(const double xs[6], const double cs[21]) {
    updateFromBound(plane(firstPlane), xs);
#pragma unroll
    for (int m = 0; m < 21; ++m) cov[m] = (S)cs[m];
    navDir = -1;
    moved();
    ss.init(-1.0 * fabs(a.max_step_size));
    pathAcc = 0.0;
  }

  // The rest of the actor call that finalised, and the propagation back to
  // the perigee; the actor is called from one place, as in forwardPass.
  KFD_INLINE void backwardPass(int resume, int steps, bool terminated) {
    int at = resume;
    for (;;) {
      actorPost();
      if (at == kResumePostLoop) break;
      bool more = !(kalmanAbort() || pathLimit());
      if (more) {
        navTarget();
        if (at == kResumeInLoop) ++steps;
        at = kResumeInLoop;
        more = cheapSteps<false>(steps, terminated);
      } else if (at == kResumeInLoop) {
        terminated = true;
      }
      if (!more) {
        at = kResumePostLoop;
        if (!terminated) navBreak = true;
      }
    }
    writeFinal(statusBits(steps, terminated), finished);
  }

  // Forward kernel body (with the store).
  KFD_INLINE void runForward() {
    int steps;
    bool terminated, bad;
    const int resume = forwardPass(steps, terminated, bad);
    if (resume != kResumeNone) {
      saveCarry(resume, steps, terminated);
    } else {
      if (kStore && lead) ci(kCI_resume) = kResumeNone;
      writeFinal(bad ? KF_STATUS_BAD_INPUT : statusBits(steps, terminated), false);
    }
  }

  // Backward kernel body (with the store): Actor::finalize (KalmanFitter.hpp:
  // 360-393) and what follows it.
  KFD_INLINE void runBackward() {
    int steps = 0;
    bool terminated = false;
    loadTrack();
    const int resume = loadCarry(steps, terminated);
    if (resume == kResumeNone) return;
    smoothed = true;
    double xs[6], cs[21];
    if (smooth(xs, cs))
      fromSmoothed(xs, cs);
    else
      result = false;
    loadCarryJacobian();
    backwardPass(resume, steps, terminated);
  }

  // The whole fit with the fixed-point smoother (kKeepFirst).  False: the
  // track is left to the RTS program (its outputs are not final).
  KFD_INLINE bool runFused() {
    int steps;
    bool terminated, bad;
    const int resume = forwardPass(steps, terminated, bad);
    if (elsewhere) return true;
    if (left) return false;
    if (resume == kResumeNone) {
      writeFinal(bad ? KF_STATUS_BAD_INPUT : statusBits(steps, terminated), false);
      return true;
    }
    double xs[6], cs[21];
    fxSmooth(xs, cs);
    if (!fxSafe(xs, cs)) return false;
    smoothed = true;
    cur = -1;
    targetReached = false;
    loadPerigee();  // again: it need not stay in registers through the forward pass
    fromSmoothed(xs, cs);
    backwardPass(resume, steps, terminated);
    return true;
  }
};

}  // namespace kfd
