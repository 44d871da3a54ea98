// kf_api.hip -- C ABI of libkfmi.so (declared in include/kf_abi.h).
//
// A kf_ctx owns the device copies of the plane table and the field grid, the
// per-state store used by the smoother (grown on demand, never shrunk), and
// two HIP events that time the last fit kernel on its launch stream.
#include <hip/hip_runtime.h>
#include <rocprofiler-sdk-roctx/roctx.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>
#include <vector>

#include "../../include/kf_abi.h"
#include "kf_adjoint.hpp"
#include "kf_kernels.hpp"
#include "kf_setup.hpp"

// The fixed workspace of kf_fit_noalloc: one copy on every device the library
// runs on, held until the process ends.  Host code never uses this name as an
// address (on the host it is only a stand-in for the device symbol): the
// device address comes from hipGetSymbolAddress, once per device, in
// kf_ctx_create (noallocWorkspace below).
static __device__ __align__(256) unsigned char scratch[KF_NOALLOC_WORKSPACE_BYTES];

struct kf_ctx {
  int device = 0;
  char err[512] = {0};
  kfd::DevPlane *planes = nullptr;
  int32_t n_planes = 0;
  kfd::DevField field{};
  bool field_set = false;
  float *grid = nullptr;
  size_t grid_elems = 0;
  void *store = nullptr;  // per-state stores of the smoother (and track-state records)
  size_t store_bytes = 0;
  void *carry = nullptr;    // forward -> backward kernel hand-over, kept first states
  size_t carry_bytes = 0;
  void *redo = nullptr;     // fused fits: redo counters and list
  size_t redo_bytes = 0;
  bool redo_clean = false;  // its counters are zero (every complete fit leaves them so)
  void *adj = nullptr;      // chi2-adjoint buffers (step stack, plane adjoints, ...)
  size_t adj_bytes = 0;
  bool has_material = false;  // a plane of the table carries material
  bool unique_geo = false;    // the planes' geo ids are distinct
  uint64_t budget = KF_DEFAULT_MEMORY_BUDGET;  // per-batch working buffers
  hipEvent_t ev0 = nullptr, evm = nullptr, ev1 = nullptr;
  bool timed = false;
  bool phase_timed = false;  // the last call was not a graph replay or in slices
  bool one_kernel = false;   // the last call was one kernel: evm not recorded
  // scheduling (kf_schedule) and its buffers: track order, sort counters,
  // work-queue counters
  kf_schedule sched{};
  int n_cu = 0;
  void *sched_buf = nullptr;
  size_t sched_bytes = 0;
  // graph replay: the captured launch sequence and the arguments it holds
  hipStream_t cap_stream = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  std::vector<char> gkey;
  int64_t captures = 0;
};

namespace {

char g_create_err[512] = {0};

// Host-side profiler ranges around the entry points (the reference's
// PUSH_RANGE / POP_RANGE around KalmanFitter::fit, Utilities/Profiling.hpp:
// 12-26, KalmanFitter.hpp:728,758), shown by rocprofv3 --marker-trace; on
// when the environment holds KF_ROCTX=1 when the library first asks.
bool rangesOn() {
  static const bool on = [] {
    const char *v = std::getenv("KF_ROCTX");
    return v && v[0] == '1' && v[1] == 0;
  }();
  return on;
}
struct Range {
  bool on;
  explicit Range(const char *name) : on(rangesOn()) {
    if (on) roctxRangePushA(name);
  }
  ~Range() {
    if (on) roctxRangePop();
  }
  Range(const Range &) = delete;
  Range &operator=(const Range &) = delete;
};

// Device addresses of `scratch`, per device (resolved with that device
// current); g_ws_state: 0 unresolved, 1 resolved, < 0 the hipError_t of a
// failed resolution, negated.
constexpr int kMaxDevices = 64;
std::mutex g_ws_mu;
void *g_ws_ptr[kMaxDevices] = {};
int g_ws_state[kMaxDevices] = {};

// Resolves the workspace of `device` (the current device) once.
hipError_t noallocWorkspace(int device, void **out) {
  *out = nullptr;
  if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_ws_mu);
  if (g_ws_state[device] == 0) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      g_ws_state[device] = -(int)((e != hipSuccess) ? e : hipErrorInvalidSymbol);
    } else {
      g_ws_ptr[device] = p;
      g_ws_state[device] = 1;
    }
  }
  if (g_ws_state[device] < 0) return (hipError_t)(-g_ws_state[device]);
  *out = g_ws_ptr[device];
  return hipSuccess;
}

int fail(kf_ctx *ctx, int code, const char *fmt, ...) {
  char *buf = ctx ? ctx->err : g_create_err;
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, 512, fmt, ap);
  va_end(ap);
  return code;
}

// Grows a device buffer to at least `need` bytes (contents are not kept).
int grow(kf_ctx *ctx, void **buf, size_t *cap, size_t need, hipStream_t s, const char *what);

#define KF_HIP(ctx, call)                                                            \
  do {                                                                               \
    hipError_t e_ = (call);                                                          \
    if (e_ != hipSuccess)                                                            \
      return fail((ctx), KF_E_HIP, "%s failed: %s", #call, hipGetErrorString(e_));   \
  } while (0)

int grow(kf_ctx *ctx, void **buf, size_t *cap, size_t need, hipStream_t s, const char *what) {
  if (need <= *cap) return KF_OK;
  if (*buf) {
    KF_HIP(ctx, hipStreamSynchronize(s));
    KF_HIP(ctx, hipFree(*buf));
    *buf = nullptr;
    *cap = 0;
  }
  hipError_t e = hipMalloc(buf, need);
  if (e != hipSuccess) {
    *buf = nullptr;
    return fail(ctx, KF_E_NOMEM, "kf_fit: cannot allocate %zu bytes of %s: %s", need, what,
                hipGetErrorString(e));
  }
  *cap = need;
  return KF_OK;
}

// Whether the caller is capturing this stream (buffers can then not grow, and
// what is launched has not run when the call returns).
bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) == hipSuccess) return st != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return false;
}

}  // namespace

extern "C" {

int kf_abi_version(void) { return KF_ABI_VERSION; }

void kf_options_default(kf_options *o) {
  if (!o) return;
  std::memset(o, 0, sizeof *o);
  o->smoothing = 1;
  o->multiple_scattering = 1;
  o->energy_loss = 1;
  o->precision = KF_PRECISION_FP64;
  o->abs_pdg = 13;
  o->max_steps = 1000;
  o->max_rk_trials = 10000;
  o->max_states = 0;
  o->mass = 105.6583755 * 1e-3;
  o->tolerance = 1e-4;
  o->step_size_cutoff = 0.0;
  o->max_step_size = DBL_MAX;
  o->target_tolerance = 1e-4;
  o->overstep_limit = 0.01;
  o->outlier_chi2_cut = 0.0;
}

int kf_ctx_create(int device, kf_ctx **out) {
  if (!out) return fail(nullptr, KF_E_INVALID, "kf_ctx_create: out is NULL");
  *out = nullptr;
  int ndev = 0;
  hipError_t e = hipGetDeviceCount(&ndev);
  if (e != hipSuccess || ndev <= 0)
    return fail(nullptr, KF_E_HIP, "kf_ctx_create: no HIP device (%s)", hipGetErrorString(e));
  if (device < 0 || device >= ndev)
    return fail(nullptr, KF_E_INVALID, "kf_ctx_create: device %d out of range [0, %d)", device, ndev);
  kf_ctx *ctx = new (std::nothrow) kf_ctx();
  if (!ctx) return fail(nullptr, KF_E_NOMEM, "kf_ctx_create: out of host memory");
  ctx->device = device;
  e = hipSetDevice(device);
  if (e == hipSuccess) e = hipEventCreate(&ctx->ev0);
  if (e == hipSuccess) e = hipEventCreate(&ctx->ev1);
  if (e == hipSuccess) e = hipEventCreate(&ctx->evm);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&ctx->n_cu, hipDeviceAttributeMultiprocessorCount, device);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&ctx->cap_stream, hipStreamNonBlocking);
  if (e == hipSuccess) {
    void *ws = nullptr;
    e = noallocWorkspace(device, &ws);
  }
  kf_schedule_default(&ctx->sched);
  if (e != hipSuccess) {
    fail(nullptr, KF_E_HIP, "kf_ctx_create: %s", hipGetErrorString(e));
    delete ctx;
    return KF_E_HIP;
  }
  *out = ctx;
  return KF_OK;
}

int kf_ctx_destroy(kf_ctx *ctx) {
  if (!ctx) return KF_OK;
  (void)hipSetDevice(ctx->device);
  (void)hipDeviceSynchronize();
  if (ctx->planes) (void)hipFree(ctx->planes);
  if (ctx->grid) (void)hipFree(ctx->grid);
  if (ctx->store) (void)hipFree(ctx->store);
  if (ctx->carry) (void)hipFree(ctx->carry);
  if (ctx->redo) (void)hipFree(ctx->redo);
  if (ctx->adj) (void)hipFree(ctx->adj);
  if (ctx->ev0) (void)hipEventDestroy(ctx->ev0);
  if (ctx->ev1) (void)hipEventDestroy(ctx->ev1);
  if (ctx->evm) (void)hipEventDestroy(ctx->evm);
  if (ctx->gexec) (void)hipGraphExecDestroy(ctx->gexec);
  if (ctx->graph) (void)hipGraphDestroy(ctx->graph);
  if (ctx->cap_stream) (void)hipStreamDestroy(ctx->cap_stream);
  if (ctx->sched_buf) (void)hipFree(ctx->sched_buf);
  delete ctx;
  return KF_OK;
}

const char *kf_last_error(const kf_ctx *ctx) { return ctx ? ctx->err : g_create_err; }

int kf_set_geometry(kf_ctx *ctx, const kf_plane *planes, int32_t n_planes) {
  if (!ctx) return fail(nullptr, KF_E_INVALID, "kf_set_geometry: ctx is NULL");
  if (!planes || n_planes <= 0)
    return fail(ctx, KF_E_INVALID, "kf_set_geometry: need n_planes > 0 planes");
  std::vector<kfd::DevPlane> dp(n_planes);
  for (int i = 0; i < n_planes; ++i) dp[i] = kfd::devPlane(planes[i]);
  KF_HIP(ctx, hipSetDevice(ctx->device));
  if (ctx->planes && ctx->n_planes != n_planes) {
    KF_HIP(ctx, hipFree(ctx->planes));
    ctx->planes = nullptr;
  }
  if (!ctx->planes) KF_HIP(ctx, hipMalloc(&ctx->planes, sizeof(kfd::DevPlane) * n_planes));
  KF_HIP(ctx, hipMemcpy(ctx->planes, dp.data(), sizeof(kfd::DevPlane) * n_planes,
                        hipMemcpyHostToDevice));
  ctx->n_planes = n_planes;
  ctx->has_material = false;
  for (const kfd::DevPlane &d : dp) ctx->has_material = ctx->has_material || d.has_material;
  std::vector<int32_t> ids(n_planes);
  for (int i = 0; i < n_planes; ++i) ids[i] = planes[i].geo_id;
  std::sort(ids.begin(), ids.end());
  ctx->unique_geo = std::adjacent_find(ids.begin(), ids.end()) == ids.end();
  return KF_OK;
}

int kf_set_field_constant(kf_ctx *ctx, double bx, double by, double bz) {
  if (!ctx) return fail(nullptr, KF_E_INVALID, "kf_set_field_constant: ctx is NULL");
  const double scale = ctx->field_set ? ctx->field.scale : 1.0;
  ctx->field = kfd::DevField{};
  ctx->field.grid = 0;
  ctx->field.b[0] = bx;
  ctx->field.b[1] = by;
  ctx->field.b[2] = bz;
  ctx->field.scale = scale;
  ctx->field_set = true;
  return KF_OK;
}

int kf_set_field_grid(kf_ctx *ctx, const float *b, int32_t nx, int32_t ny, int32_t nz,
                      const double lo[3], const double hi[3]) {
  if (!ctx) return fail(nullptr, KF_E_INVALID, "kf_set_field_grid: ctx is NULL");
  if (!b || !lo || !hi || nx < 2 || ny < 2 || nz < 2)
    return fail(ctx, KF_E_INVALID, "kf_set_field_grid: need a >= 2x2x2 grid and bounds");
  for (int d = 0; d < 3; ++d)
    if (!(hi[d] > lo[d])) return fail(ctx, KF_E_INVALID, "kf_set_field_grid: hi <= lo on axis %d", d);
  const size_t elems = (size_t)nx * ny * nz * 3;
  KF_HIP(ctx, hipSetDevice(ctx->device));
  if (ctx->grid && ctx->grid_elems != elems) {
    KF_HIP(ctx, hipFree(ctx->grid));
    ctx->grid = nullptr;
  }
  if (!ctx->grid) KF_HIP(ctx, hipMalloc(&ctx->grid, elems * sizeof(float)));
  ctx->grid_elems = elems;
  KF_HIP(ctx, hipMemcpy(ctx->grid, b, elems * sizeof(float), hipMemcpyHostToDevice));
  const double scale = ctx->field_set ? ctx->field.scale : 1.0;
  ctx->field = kfd::DevField{};
  ctx->field.grid = 1;
  ctx->field.values = ctx->grid;
  ctx->field.n[0] = nx;
  ctx->field.n[1] = ny;
  ctx->field.n[2] = nz;
  const int n[3] = {nx, ny, nz};
  for (int d = 0; d < 3; ++d) {
    ctx->field.lo[d] = lo[d];
    ctx->field.hi[d] = hi[d];
    ctx->field.w[d] = (hi[d] - lo[d]) / (n[d] - 1);
    ctx->field.iw[d] = 1.0 / ctx->field.w[d];
  }
  ctx->field.scale = scale;
  ctx->field_set = true;
  return KF_OK;
}

int kf_set_field_scale(kf_ctx *ctx, double s) {
  if (!ctx) return fail(nullptr, KF_E_INVALID, "kf_set_field_scale: ctx is NULL");
  if (!ctx->field_set) return fail(ctx, KF_E_STATE, "kf_set_field_scale: no field set");
  ctx->field.scale = s;
  return KF_OK;
}

}  // extern "C"

namespace {

// Checks the batch and options and fills the kernel arguments shared by the
// fit and the adjoint (inputs, options, physics constants).
int setupArgs(kf_ctx *ctx, const kf_tracks *tr, const kf_options *opt, const char *who,
              kfd::FitArgs &a) {
  if (!ctx->planes) return fail(ctx, KF_E_STATE, "%s: no geometry (kf_set_geometry)", who);
  if (!ctx->field_set) return fail(ctx, KF_E_STATE, "%s: no field (kf_set_field_*)", who);
  if (tr->n_tracks < 0 || tr->n_hits < 0) return fail(ctx, KF_E_INVALID, "%s: negative size", who);
  if (tr->n_tracks > 0 && (!tr->start_params || !tr->start_cov || !tr->perigee ||
                           !tr->seq_first || !tr->seq_count || !tr->hit_offset))
    return fail(ctx, KF_E_INVALID, "%s: NULL per-track input array", who);
  if (tr->n_hits > 0 && (!tr->hit_geo_id || !tr->hit_meas || !tr->hit_cov))
    return fail(ctx, KF_E_INVALID, "%s: NULL hit array", who);
  if (opt->precision != KF_PRECISION_FP64 && opt->precision != KF_PRECISION_MIXED)
    return fail(ctx, KF_E_INVALID, "%s: unknown precision %d", who, opt->precision);
  if (opt->max_steps < 0 || opt->max_rk_trials < 0 || opt->max_states < 0 || !(opt->mass > 0.0) ||
      !(opt->overstep_limit >= 0.0) || !(opt->outlier_chi2_cut >= 0.0))
    return fail(ctx, KF_E_INVALID, "%s: invalid options", who);
  std::memset(&a, 0, sizeof a);
  a.n = tr->n_tracks;
  a.n_hits = tr->n_hits;
  a.start_params = tr->start_params;
  a.start_cov = tr->start_cov;
  a.perigee = tr->perigee;
  a.seq_first = tr->seq_first;
  a.seq_count = tr->seq_count;
  a.hit_offset = tr->hit_offset;
  a.hit_geo_id = tr->hit_geo_id;
  a.hit_meas = tr->hit_meas;
  a.hit_cov = tr->hit_cov;
  a.planes = ctx->planes;
  a.n_planes = ctx->n_planes;
  a.unique_geo = ctx->unique_geo ? 1 : 0;
  // byte copy: the padding of the field description is ctx's (zeroed), so
  // equal arguments give equal graph-replay keys
  std::memcpy(&a.field, &ctx->field, sizeof a.field);
  a.smoothing = opt->smoothing;
  a.ms = opt->multiple_scattering;
  a.eloss = opt->energy_loss;
  a.max_steps = opt->max_steps;
  a.max_rk_trials = (uint32_t)opt->max_rk_trials;
  a.max_states = opt->max_states > 0 ? opt->max_states : ctx->n_planes;
  a.mass = opt->mass;
  a.tolerance = opt->tolerance;
  a.step_size_cutoff = opt->step_size_cutoff;
  a.max_step_size = opt->max_step_size;
  a.target_tolerance = opt->target_tolerance;
  a.overstep_limit = opt->overstep_limit;
  a.outlier_chi2_cut = opt->outlier_chi2_cut;
  kfd::physicsConstants(a);
  return KF_OK;
}

constexpr size_t kCarryBytes = KF_CARRY_I * sizeof(int32_t) + KF_CARRY_D * sizeof(double);

// Working-buffer bytes per track of the recording fit: per-state stores and
// hand-over (the adjoint's forward pass: its checkpoints only).
size_t storeBytesPerTrack(const kfd::FitArgs &a, int precision, bool track_states,
                          bool checkpoints) {
  if (checkpoints) return (size_t)a.max_states * KF_CK_N * sizeof(double);
  const size_t s_size = (precision == KF_PRECISION_FP64) ? sizeof(double) : sizeof(float);
  size_t per_state = KF_SD_N * sizeof(double) + KF_SS_N * s_size;
  if (track_states) per_state += KF_TS_STRIDE * sizeof(double);
  return (size_t)a.max_states * per_state + kCarryBytes;
}

// Whether a fit runs on the fused kernel (kf_fit_kernels.hpp).
bool fitIsFused(bool track_states) { return !track_states; }

// Working-buffer bytes per track of the fused fit: the kept first state (FP64;
// the mixed mode has it in LDS) and the redo list.
size_t firstBytes(int precision) {
  return precision == KF_PRECISION_FP64 ? KF_FIRST_D * sizeof(double) : 0;
}
size_t fusedBytesPerTrack(int precision) { return firstBytes(precision) + sizeof(uint32_t); }

// Positions per slice: the largest multiple of 64 whose working set fits the
// budget (at least 64), or the whole batch.
int64_t sliceTracks(const kf_ctx *ctx, int64_t n, size_t bytes_per_track) {
  int64_t m = (int64_t)(ctx->budget / (bytes_per_track ? bytes_per_track : 1)) / 64 * 64;
  if (m < 64) m = 64;
  return m >= n ? n : m;
}

// Byte sizes of the working storage for slices of up to `slice` positions:
// the per-state stores (layout in kf_kernels.hpp), each 256-byte aligned, and
// the forward -> backward hand-over.
struct StoreLayout {
  size_t s_bytes, d_bytes, f_bytes, c_bytes, carry_bytes;
  size_t store() const { return s_bytes + d_bytes + f_bytes + c_bytes; }
};
StoreLayout storeLayout(int precision, bool track_states, bool checkpoints, int64_t slice,
                        int32_t max_states) {
  const size_t slots = ((size_t)slice + 63) / 64 * 64 * (size_t)max_states;
  const size_t s_size = (precision == KF_PRECISION_FP64) ? sizeof(double) : sizeof(float);
  StoreLayout L;
  L.s_bytes = checkpoints ? 0 : (slots * KF_SS_N * s_size + 255) / 256 * 256;
  L.d_bytes = checkpoints ? 0 : slots * KF_SD_N * sizeof(double);
  L.f_bytes = track_states ? slots * KF_TS_STRIDE * sizeof(double) : 0;
  L.c_bytes = checkpoints ? slots * KF_CK_N * sizeof(double) : 0;
  L.carry_bytes = checkpoints ? 0 : ((size_t)slice * kCarryBytes + 255) / 256 * 256;
  return L;
}

// Points the kernel arguments at stores carved from `store` and the
// hand-over buffer `carry`.
void carveStores(const StoreLayout &L, void *store, void *carry, bool track_states,
                 bool checkpoints, kfd::FitArgs &a) {
  char *base = (char *)store;
  a.tss = checkpoints ? nullptr : base;
  a.tsd = checkpoints ? nullptr : (double *)(base + L.s_bytes);
  a.tsf = track_states ? (double *)(base + L.s_bytes + L.d_bytes) : nullptr;
  a.tsc = checkpoints ? (double *)(base + L.s_bytes + L.d_bytes + L.f_bytes) : nullptr;
  // [field][count] of each slice (sliceCarry)
  a.carry_d = (double *)carry;
  a.carry_i = nullptr;
}

// The working storage for slices of up to `slice` positions, from the
// context's buffers (grown as needed).
int setupStores(kf_ctx *ctx, int precision, bool track_states, bool checkpoints, int64_t slice,
                hipStream_t s, kfd::FitArgs &a) {
  const StoreLayout L = storeLayout(precision, track_states, checkpoints, slice, a.max_states);
  int rc = grow(ctx, &ctx->store, &ctx->store_bytes, L.store(), s, "state store");
  if (rc != KF_OK) return rc;
  rc = grow(ctx, &ctx->carry, &ctx->carry_bytes, L.carry_bytes, s, "hand-over buffer");
  if (rc != KF_OK) return rc;
  carveStores(L, ctx->store, ctx->carry, track_states, checkpoints, a);
  return KF_OK;
}

// Working storage of a fused fit for slices of up to `slice` positions: the
// kept first states (carry), and for tracks that go to the RTS program the
// list, and store chunks with their hand-over (redo), the first `rts` of them
// for the waves near the wrap.
struct FusedLayout {
  StoreLayout store;   // of waves x 64 lanes
  size_t carry_bytes, list_bytes;
  int64_t lanes, rts;
  size_t redo_bytes() const { return list_bytes + store.carry_bytes; }
};
FusedLayout fusedLayout(int precision, int64_t slice, int32_t max_states, size_t budget) {
  FusedLayout F;
  // a chunk for every wave of the slice where the limit and the budget allow it;
  // else chunks of each kind, between the two the budget, one for handed-back tracks
  // at least
  const size_t one = storeLayout(precision, false, false, 64, max_states).store();
  const int64_t waves = (slice + 63) / 64, fit = std::max<int64_t>((int64_t)(budget / one), 1);
  if (waves <= std::min<int64_t>(fit, KF_RTS_WAVES)) {
    F.rts = waves;
    F.lanes = waves * 64;
  } else {
    F.rts = std::min<int64_t>(KF_RTS_WAVES, fit / 2);
    F.lanes = (F.rts + std::min<int64_t>(KF_REDO_WAVES, fit - F.rts)) * 64;
  }
  F.store = storeLayout(precision, false, false, F.lanes, max_states);
  F.carry_bytes = ((size_t)slice * firstBytes(precision) + 255) / 256 * 256;
  F.list_bytes = ((KF_REDO_LIST + (size_t)slice) * sizeof(uint32_t) + 255) / 256 * 256;
  return F;
}

void carveFused(const FusedLayout &F, void *store, void *carry, void *redo, kfd::FitArgs &a) {
  a.tss = store;
  a.tsd = (double *)((char *)store + F.store.s_bytes);
  a.tsf = a.tsc = nullptr;
  a.carry_d = (double *)carry;
  a.carry_i = nullptr;
  a.redo = (uint32_t *)redo;
  a.redo_d = (double *)((char *)redo + F.list_bytes);
  a.redo_i = (int32_t *)(a.redo_d + KF_CARRY_D * (size_t)F.lanes);
  a.redo_lanes = F.lanes;
  a.rts_waves = (int32_t)F.rts;
}

// The part of the budget that a fused fit's store chunks may take, and its slice:
// the positions whose kept states and list fit in what the chunks leave (64 at
// least).
size_t fusedStoreBudget(const kf_ctx *ctx) {
  return (size_t)std::min<uint64_t>(ctx->budget / 2, KF_REDO_STORE_BYTES);
}
int64_t fusedSlice(const kf_ctx *ctx, int precision, int64_t n, int32_t max_states) {
  const FusedLayout F = fusedLayout(precision, n, max_states, fusedStoreBudget(ctx));
  // (1,024: the rounding of the three buffers' parts)
  const uint64_t chunks = F.store.store() + F.store.carry_bytes + 1024;
  const uint64_t rest = ctx->budget > chunks ? ctx->budget - chunks : 0;
  const int64_t fit = (int64_t)(rest / fusedBytesPerTrack(precision)) / 64 * 64;
  return fit >= n ? n : std::max<int64_t>(fit, 64);
}

// The working storage of a fused fit, from the context's buffers (grown as
// needed); the redo counters are zeroed when the buffer is new or a call failed
// between the kernel that fills the list and the one that clears it.
int setupFused(kf_ctx *ctx, int precision, int64_t slice, hipStream_t s, kfd::FitArgs &a) {
  const size_t budget = fusedStoreBudget(ctx);
  FusedLayout F = fusedLayout(precision, slice, a.max_states, budget);
  auto held = [&] {
    return F.store.store() <= ctx->store_bytes && F.redo_bytes() <= ctx->redo_bytes;
  };
  // under capture, fewer chunks where the buffers hold no more
  if (ctx->store && !held() && capturing(s)) {
    const FusedLayout wanted = F;
    for (size_t b = ctx->store_bytes; b > 0 && !held(); b /= 2)
      F = fusedLayout(precision, slice, a.max_states, b);
    if (!held()) F = wanted;
  }
  int rc = grow(ctx, &ctx->store, &ctx->store_bytes, F.store.store(), s, "state store");
  if (rc != KF_OK) return rc;
  rc = grow(ctx, &ctx->carry, &ctx->carry_bytes, F.carry_bytes, s, "hand-over buffer");
  if (rc != KF_OK) return rc;
  if (F.redo_bytes() > ctx->redo_bytes) ctx->redo_clean = false;
  rc = grow(ctx, &ctx->redo, &ctx->redo_bytes, F.redo_bytes(), s, "redo buffers");
  if (rc != KF_OK) return rc;
  carveFused(F, ctx->store, ctx->carry, ctx->redo, a);
  if (!ctx->redo_clean) {
    KF_HIP(ctx, kfd_launch_redo_reset(a.redo, s));
    ctx->redo_clean = !capturing(s);  // captured: only a replay zeroes them
  }
  return KF_OK;
}

// Sets positions first .. first + count - 1 as the launch's range; the
// hand-over record is [30 doubles][count] followed by [8 ints][count] (a fused
// fit has its own, carveFused).
void sliceRange(kfd::FitArgs &a, int64_t first, int64_t count) {
  a.first = first;
  a.count = count;
  if (!a.redo && a.carry_d) a.carry_i = (int32_t *)(a.carry_d + KF_CARRY_D * (size_t)count);
}

// The whole fit of a batch: the length sort over all positions, then the
// positions slice by slice (each slice reuses the stores).  `between` is
// recorded between the two kernels when there is one slice.
hipError_t launchSlices(kfd::FitArgs a, const KfdLaunch &L, int precision, double *ts_out,
                        int64_t slice, hipEvent_t between, hipStream_t s) {
  hipError_t e = hipSuccess;
  if (L.sort_by_length) e = kfd_launch_sort(&a, &L, s);
  const bool one = slice >= a.n;
  for (int64_t first = 0; e == hipSuccess && first < a.n; first += slice) {
    sliceRange(a, first, (a.n - first < slice) ? a.n - first : slice);
    e = kfd_launch_fit(&a, precision, s, ts_out, one ? between : nullptr, &L);
  }
  return e;
}

// Checks the fit's arguments and fills the kernel arguments (inputs, options,
// outputs); makes ctx's device current.
int prepareFit(kf_ctx *ctx, const kf_tracks *tr, const kf_options *opt, const kf_results *res,
               const char *who, kfd::FitArgs &a) {
  if (!ctx) return fail(nullptr, KF_E_INVALID, "%s: ctx is NULL", who);
  if (!tr || !opt || !res) return fail(ctx, KF_E_INVALID, "%s: NULL tracks/options/results", who);
  int rc = setupArgs(ctx, tr, opt, who, a);
  if (rc != KF_OK) return rc;
  if (tr->n_tracks == 0) return KF_OK;
  if (!res->params || !res->cov || !res->status)
    return fail(ctx, KF_E_INVALID, "%s: results need params, cov and status", who);
  if (res->track_states && !res->n_measured)
    return fail(ctx, KF_E_INVALID, "%s: track_states needs results.n_measured", who);
  a.out_params = res->params;
  a.out_cov = res->cov;
  a.out_chi2 = res->chi2;
  a.out_ndf = res->ndf;
  a.out_nmeas = res->n_measured;
  a.out_status = res->status;
  KF_HIP(ctx, hipSetDevice(ctx->device));
  return KF_OK;
}

}  // namespace

extern "C" {

int kf_fit_noalloc(kf_ctx *ctx, const kf_tracks *tr, const kf_options *opt,
                   const kf_results *res, void *stream) {
  const Range range("kf_fit_noalloc");
  kfd::FitArgs a;
  int rc = prepareFit(ctx, tr, opt, res, "kf_fit_noalloc", a);
  if (rc != KF_OK || tr->n_tracks == 0) return rc;
  void *ws = nullptr;
  const hipError_t we = noallocWorkspace(ctx->device, &ws);
  if (we != hipSuccess)
    return fail(ctx, KF_E_HIP, "kf_fit_noalloc: workspace of device %d unavailable: %s",
                ctx->device, hipGetErrorString(we));
  const bool ts = res->track_states != nullptr;
  const bool fusedFit = fitIsFused(ts);
  // a fused fit: the redo store takes at most half of the workspace (one
  // chunk as a minimum)
  auto fused = [&](int64_t slice) {
    return fusedLayout(opt->precision, slice, a.max_states,
                       (size_t)KF_NOALLOC_WORKSPACE_BYTES / 2);
  };
  // the largest multiple of 64 positions whose storage fits the workspace
  auto fits = [&](int64_t slice) {
    if (fusedFit) {
      const FusedLayout F = fused(slice);
      return F.store.store() + F.carry_bytes + F.redo_bytes() <= (size_t)KF_NOALLOC_WORKSPACE_BYTES;
    }
    const StoreLayout L = storeLayout(opt->precision, ts, false, slice, a.max_states);
    return L.store() + L.carry_bytes <= (size_t)KF_NOALLOC_WORKSPACE_BYTES;
  };
  if (!fits(64)) {
    const StoreLayout L = storeLayout(opt->precision, ts, false, 64, a.max_states);
    return fail(ctx, KF_E_INVALID,
                "kf_fit_noalloc: one 64-track slice with %d states per track needs %zu bytes, "
                "the fixed workspace holds %llu (lower max_states)",
                a.max_states, L.store() + L.carry_bytes,
                (unsigned long long)KF_NOALLOC_WORKSPACE_BYTES);
  }
  int64_t lo = 64, hi = (a.n + 63) / 64 * 64;
  if (fits(hi)) {
    lo = hi;
  } else {
    while (hi - lo > 64) {  // fits(lo), !fits(hi)
      const int64_t mid = (lo + hi) / 128 * 64;
      if (fits(mid))
        lo = mid;
      else
        hi = mid;
    }
  }
  const int64_t slice = lo >= a.n ? a.n : lo;
  hipStream_t s = (hipStream_t)stream;
  KfdLaunch launch{};  // one thread per track, identity order
  hipError_t e = hipSuccess;
  KF_HIP(ctx, hipEventRecord(ctx->ev0, s));
  if (!fusedFit) {
    const StoreLayout L = storeLayout(opt->precision, ts, false, slice, a.max_states);
    carveStores(L, ws, (char *)ws + L.store(), ts, false, a);
  } else {
    const FusedLayout F = fused(slice);
    char *w = (char *)ws;
    carveFused(F, w, w + F.store.store(), w + F.store.store() + F.carry_bytes, a);
    // the workspace holds anything (an earlier call's slices)
    e = kfd_launch_redo_reset(a.redo, s);
  }
  if (e == hipSuccess)
    e = launchSlices(a, launch, opt->precision, res->track_states, slice,
                                    ctx->evm, s);
  if (e != hipSuccess)
    return fail(ctx, KF_E_HIP, "kf_fit_noalloc: launch failed: %s", hipGetErrorString(e));
  KF_HIP(ctx, hipEventRecord(ctx->ev1, s));
  ctx->timed = true;
  ctx->phase_timed = slice >= a.n;
  ctx->one_kernel = false;
  return KF_OK;
}

int kf_fit(kf_ctx *ctx, const kf_tracks *tr, const kf_options *opt, const kf_results *res,
           void *stream) {
  const Range range("kf_fit");
  kfd::FitArgs a;
  int rc = prepareFit(ctx, tr, opt, res, "kf_fit", a);
  if (rc != KF_OK || tr->n_tracks == 0) return rc;
  hipStream_t s = (hipStream_t)stream;
  const bool ts = res->track_states != nullptr;
  const bool fused = fitIsFused(ts);
  const int64_t slice =
      fused ? fusedSlice(ctx, opt->precision, a.n, a.max_states)
            : sliceTracks(ctx, a.n, storeBytesPerTrack(a, opt->precision, ts, false));
  rc = fused ? setupFused(ctx, opt->precision, slice, s, a)
             : setupStores(ctx, opt->precision, ts, false, slice, s, a);
  if (rc != KF_OK) return rc;
  const kf_schedule &sc = ctx->sched;
  KfdLaunch L{};
  L.lanes_per_track = sc.lanes_per_track;
  L.store_by_plane = sc.store_by_plane;
  bool sort = kfd::sortsByLength(sc, fused, tr->n_tracks, tr->n_hits, opt->max_states, ctx->n_cu);
  const size_t order_bytes = ((size_t)a.n * sizeof(int32_t) + 255) / 256 * 256;
  const size_t sched_bytes = order_bytes + 514 * sizeof(uint32_t);
  // the automatic sort is left out where its buffer cannot grow
  if (sort && sc.sort_by_length == KF_SORT_AUTO && sched_bytes > ctx->sched_bytes && capturing(s))
    sort = false;
  if (sort || sc.persistent) {
    rc = grow(ctx, &ctx->sched_buf, &ctx->sched_bytes, sched_bytes, s, "schedule buffers");
    if (rc != KF_OK) return rc;
    L.order = (int32_t *)ctx->sched_buf;
    L.sort_scratch = (uint32_t *)((char *)ctx->sched_buf + order_bytes);
    L.sort_by_length = sort;
    a.order = sort ? L.order : nullptr;
    a.queue = L.sort_scratch + 512;
    if (sc.persistent) {
      const int waves = sc.waves_per_cu * ctx->n_cu;
      L.persistent_blocks = (waves * 64 + KF_BLOCK - 1) / KF_BLOCK;
      a.persistent = 1;
      a.chunks_per_grab = sc.chunks_per_grab;
    }
  }
  hipError_t e = hipSuccess;
  if (sc.graph) {
    // key: every argument the captured launches hold
    std::vector<char> key(sizeof a + sizeof L + sizeof(int) + sizeof(void *) + sizeof slice);
    char *k = key.data();
    std::memcpy(k, &a, sizeof a);
    k += sizeof a;
    std::memcpy(k, &L, sizeof L);
    k += sizeof L;
    std::memcpy(k, &opt->precision, sizeof(int));
    k += sizeof(int);
    std::memcpy(k, &res->track_states, sizeof(void *));
    k += sizeof(void *);
    std::memcpy(k, &slice, sizeof slice);
    if (!ctx->gexec || key != ctx->gkey) {
      if (ctx->gexec) (void)hipGraphExecDestroy(ctx->gexec);
      if (ctx->graph) (void)hipGraphDestroy(ctx->graph);
      ctx->gexec = nullptr;
      ctx->graph = nullptr;
      ctx->gkey.clear();
      const Range capture("kf_fit: graph capture");
      KF_HIP(ctx, hipStreamSynchronize(s));
      KF_HIP(ctx, hipStreamBeginCapture(ctx->cap_stream, hipStreamCaptureModeThreadLocal));
      e = launchSlices(a, L, opt->precision, res->track_states, slice, nullptr, ctx->cap_stream);
      hipGraph_t g = nullptr;
      const hipError_t e2 = hipStreamEndCapture(ctx->cap_stream, &g);
      if (e == hipSuccess) e = e2;
      if (e != hipSuccess) {
        if (g) (void)hipGraphDestroy(g);
        return fail(ctx, KF_E_HIP, "kf_fit: graph capture failed: %s", hipGetErrorString(e));
      }
      ctx->graph = g;
      KF_HIP(ctx, hipGraphInstantiate(&ctx->gexec, g, nullptr, nullptr, 0));
      ctx->gkey = key;
      ++ctx->captures;
    }
    KF_HIP(ctx, hipEventRecord(ctx->ev0, s));
    e = hipGraphLaunch(ctx->gexec, s);
    ctx->phase_timed = false;
  } else {
    KF_HIP(ctx, hipEventRecord(ctx->ev0, s));
    // a fit that is one kernel has no second phase to time
    kfd::FitArgs whole = a;
    sliceRange(whole, 0, slice);
    ctx->one_kernel = fused && slice >= a.n && kfd::redoSlotPerTrack(whole);
    e = launchSlices(a, L, opt->precision, res->track_states, slice,
                     ctx->one_kernel ? nullptr : ctx->evm, s);
    ctx->phase_timed = slice >= a.n;
  }
  if (e != hipSuccess) {
    ctx->redo_clean = false;
    return fail(ctx, KF_E_HIP, "kf_fit: launch failed: %s", hipGetErrorString(e));
  }
  KF_HIP(ctx, hipEventRecord(ctx->ev1, s));
  ctx->timed = true;
  return KF_OK;
}

void kf_schedule_default(kf_schedule *s) {
  if (!s) return;
  s->sort_by_length = KF_SORT_AUTO;
  s->persistent = 0;
  s->waves_per_cu = 4;
  s->chunks_per_grab = 1;
  s->lanes_per_track = 1;
  s->graph = 0;
  s->store_by_plane = 0;
}

int kf_set_schedule(kf_ctx *ctx, const kf_schedule *s) {
  if (!ctx) return fail(nullptr, KF_E_INVALID, "kf_set_schedule: ctx is NULL");
  if (!s) return fail(ctx, KF_E_INVALID, "kf_set_schedule: schedule is NULL");
  if (s->lanes_per_track != 1 && s->lanes_per_track != 2 && s->lanes_per_track != 4)
    return fail(ctx, KF_E_INVALID, "kf_set_schedule: lanes_per_track must be 1, 2 or 4");
  if (s->store_by_plane != 0 && s->store_by_plane != 1)
    return fail(ctx, KF_E_INVALID, "kf_set_schedule: store_by_plane must be 0 or 1");
  if (s->store_by_plane && s->lanes_per_track > 1)
    return fail(ctx, KF_E_INVALID,
                "kf_set_schedule: store_by_plane runs with one lane per track");
  if (s->lanes_per_track > 1 && s->persistent)
    return fail(ctx, KF_E_INVALID,
                "kf_set_schedule: lanes_per_track > 1 runs on the one-shot grid (persistent = 0)");
  if (s->persistent && (s->waves_per_cu < 1 || s->waves_per_cu > 64 || s->chunks_per_grab < 1 ||
                        s->chunks_per_grab > 1024))
    return fail(ctx, KF_E_INVALID, "kf_set_schedule: waves_per_cu in [1, 64], chunks_per_grab in [1, 1024]");
  ctx->sched = *s;
  return KF_OK;
}

int kf_get_schedule(const kf_ctx *ctx, kf_schedule *s) {
  if (!ctx || !s) return KF_E_INVALID;
  *s = ctx->sched;
  return KF_OK;
}

int kf_autotune(kf_ctx *ctx, const kf_tracks *tracks, const kf_options *opt, const kf_results *res,
                void *stream, int32_t repeats, kf_schedule *best, double *best_ms) {
  const Range range("kf_autotune");
  if (!ctx) return fail(nullptr, KF_E_INVALID, "kf_autotune: ctx is NULL");
  if (!tracks || !opt || !res) return fail(ctx, KF_E_INVALID, "kf_autotune: NULL argument");
  if (repeats < 1) repeats = 1;
  const std::vector<kf_schedule> cand = kfd::scheduleCandidates(res->track_states != nullptr);
  const kf_schedule saved = ctx->sched;
  double best_t = 1e300;
  kf_schedule best_s = saved;
  for (const kf_schedule &c : cand) {
    int rc = kf_set_schedule(ctx, &c);
    if (rc == KF_OK) rc = kf_fit(ctx, tracks, opt, res, stream);  // warm-up / capture
    double t = 1e300;
    for (int r = 0; rc == KF_OK && r < repeats; ++r) {
      rc = kf_fit(ctx, tracks, opt, res, stream);
      if (rc == KF_OK) {
        const double ms = kf_last_kernel_ms(ctx);
        if (ms >= 0.0 && ms < t) t = ms;
      }
    }
    if (rc != KF_OK) {
      ctx->sched = saved;
      return rc;
    }
    if (t < best_t) {
      best_t = t;
      best_s = c;
    }
  }
  ctx->sched = best_s;
  if (best) *best = best_s;
  if (best_ms) *best_ms = best_t;
  return KF_OK;
}

int kf_chi2_gradient(kf_ctx *ctx, const kf_tracks *tr, const kf_options *opt, double *grad_planes,
                     double *grad_field_scale, double *chi2_sum, double *grad_raw,
                     uint32_t *track_flags, void *stream) {
  const Range range("kf_chi2_gradient");
  if (!ctx) return fail(nullptr, KF_E_INVALID, "kf_chi2_gradient: ctx is NULL");
  if (!tr || !opt || !grad_planes || !grad_field_scale)
    return fail(ctx, KF_E_INVALID, "kf_chi2_gradient: NULL tracks/options/outputs");
  if (opt->outlier_chi2_cut != 0.0)
    return fail(ctx, KF_E_INVALID,
                "kf_chi2_gradient: the outlier finder is not differentiated (outlier_chi2_cut "
                "must be 0)");
  kfd::FitArgs a;
  int rc = setupArgs(ctx, tr, opt, "kf_chi2_gradient", a);
  if (rc != KF_OK) return rc;
  a.smoothing = 0;  // the objective is the forward filter's chi2
  KF_HIP(ctx, hipSetDevice(ctx->device));
  hipStream_t s = (hipStream_t)stream;
  const int32_t max_seg = KF_ADJ_MAX_SEGMENT_STEPS;
  const size_t n = (size_t)tr->n_tracks;
  const size_t nplanes = (size_t)ctx->n_planes;
  // per slice position: stores, step stack, plane adjoints, scale adjoint
  const size_t adj_per_track = (size_t)max_seg * kfd::kSR_N * sizeof(double) +
                               nplanes * kfd::kPG_N * sizeof(double) + sizeof(double);
  const int64_t slice = sliceTracks(
      ctx, a.n, storeBytesPerTrack(a, KF_PRECISION_FP64, false, true) + adj_per_track);
  rc = setupStores(ctx, KF_PRECISION_FP64, false, true, slice, s, a);
  if (rc != KF_OK) return rc;
  const size_t sl = (size_t)(slice > 0 ? slice : 1);
  const size_t chunks = (sl + 63) / 64;
  // forward outputs of the batch that the sweep and the sums read (chi2,
  // n_measured) and flags; per slice: step stack, plane adjoints, field-scale
  // adjoints; the sums
  const size_t b_out = n * sizeof(double) + n * sizeof(int32_t);
  const size_t b_stack = chunks * 64 * (size_t)max_seg * kfd::kSR_N * sizeof(double);
  const size_t b_pg = nplanes * kfd::kPG_N * sl * sizeof(double);
  const size_t b_scale = sl * sizeof(double);
  const size_t b_flags = n * sizeof(uint32_t);
  // sums [n_planes + 2][12] followed by the reduction's partials
  const size_t b_sums = (nplanes + 2) * kfd::kPG_N * (1 + KF_ADJ_RED_SLICES) * sizeof(double);
  auto al = [](size_t x) { return (x + 255) / 256 * 256; };
  rc = grow(ctx, &ctx->adj, &ctx->adj_bytes,
            al(b_out) + al(b_stack) + al(b_pg) + al(b_scale) + al(b_flags) + al(b_sums), s,
            "adjoint buffers");
  if (rc != KF_OK) return rc;
  char *p = (char *)ctx->adj;
  a.out_chi2 = (double *)p;
  a.out_nmeas = (int32_t *)(a.out_chi2 + n);
  p += al(b_out);
  kfd::AdjArgs g;
  g.stack = (double *)p;
  p += al(b_stack);
  g.max_seg_steps = max_seg;
  g.max_seq = (int32_t)nplanes;
  g.plane_adj = (double *)p;
  p += al(b_pg);
  g.scale_adj = (double *)p;
  p += al(b_scale);
  g.status = track_flags ? track_flags : (uint32_t *)p;
  p += al(b_flags);
  double *sums = (double *)p;
  KF_HIP(ctx, hipEventRecord(ctx->ev0, s));
  // per slice: forward filter with checkpoints, then the reverse sweep and
  // its reduction onto the sums of the earlier slices
  hipError_t e = hipSuccess;
  if (n == 0) {
    sliceRange(a, 0, 0);
    e = hipEventRecord(ctx->evm, s);
    if (e == hipSuccess) e = kfd_launch_adjoint(&a, &g, sums, 0, s);
  }
  for (int64_t first = 0; e == hipSuccess && first < a.n; first += slice) {
    sliceRange(a, first, (a.n - first < slice) ? a.n - first : slice);
    e = kfd_launch_fit(&a, KF_PRECISION_FP64, s, nullptr,
                       slice >= a.n ? ctx->evm : nullptr, nullptr);
    if (e == hipSuccess) e = kfd_launch_adjoint(&a, &g, sums, first > 0, s);
  }
  ctx->phase_timed = slice >= a.n;
  ctx->one_kernel = false;
  if (e == hipSuccess)
    e = kfd_launch_adjoint_finish(&a, sums, grad_planes, grad_field_scale, chi2_sum, s);
  if (e == hipSuccess && grad_raw)
    e = hipMemcpyAsync(grad_raw, sums, nplanes * kfd::kPG_N * sizeof(double),
                       hipMemcpyDeviceToDevice, s);
  if (e != hipSuccess)
    return fail(ctx, KF_E_HIP, "kf_chi2_gradient: launch failed: %s", hipGetErrorString(e));
  KF_HIP(ctx, hipEventRecord(ctx->ev1, s));
  ctx->timed = true;
  return KF_OK;
}

int kf_set_memory_budget(kf_ctx *ctx, uint64_t bytes) {
  if (!ctx) return fail(nullptr, KF_E_INVALID, "kf_set_memory_budget: ctx is NULL");
  ctx->budget = bytes ? bytes : KF_DEFAULT_MEMORY_BUDGET;
  return KF_OK;
}

int64_t kf_intersect_scratch_bytes(int64_t n_rays, int64_t n_surfaces) {
  return (n_rays < 0 || n_surfaces < 0) ? 0 : kfd_intersect_scratch_bytes(n_rays, n_surfaces);
}

int kf_intersect(const kf_polygon_plane *surfaces, int64_t n_surfaces, const double *ray_pos,
                 const double *ray_dir, int64_t n_rays, int32_t bcheck, kf_intersection *hits,
                 int64_t capacity, int64_t *n_hits, void *work, void *stream) {
  const Range range("kf_intersect");
  if (n_surfaces < 0 || n_rays < 0 || capacity < 0)
    return fail(nullptr, KF_E_INVALID, "kf_intersect: negative size");
  if (n_surfaces > INT32_MAX || n_rays > INT32_MAX)
    return fail(nullptr, KF_E_INVALID, "kf_intersect: more than 2^31 - 1 rays or surfaces");
  if (!n_hits || !work || (n_rays > 0 && (!ray_pos || !ray_dir)) ||
      (n_surfaces > 0 && !surfaces) || (capacity > 0 && !hits))
    return fail(nullptr, KF_E_INVALID, "kf_intersect: NULL array");
  const hipError_t e = kfd_launch_intersect(surfaces, n_surfaces, ray_pos, ray_dir, n_rays,
                                            bcheck, hits, capacity, n_hits, work,
                                            (hipStream_t)stream);
  if (e != hipSuccess)
    return fail(nullptr, KF_E_HIP, "kf_intersect: launch failed: %s", hipGetErrorString(e));
  return KF_OK;
}

int64_t kf_graph_captures(const kf_ctx *ctx) { return ctx ? ctx->captures : 0; }

double kf_last_kernel_ms(const kf_ctx *ctx) {
  if (!ctx || !ctx->timed) return -1.0;
  if (hipEventSynchronize(ctx->ev1) != hipSuccess) return -1.0;
  float ms = 0.0f;
  if (hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1) != hipSuccess) return -1.0;
  return (double)ms;
}

int kf_last_phase_ms(const kf_ctx *ctx, double *forward_ms, double *backward_ms) {
  if (!ctx || !forward_ms || !backward_ms) return KF_E_INVALID;
  *forward_ms = *backward_ms = -1.0;
  if (!ctx->timed || !ctx->phase_timed) return KF_E_STATE;
  if (hipEventSynchronize(ctx->ev1) != hipSuccess) return KF_E_HIP;
  float f = 0.0f, b = 0.0f;
  if (ctx->one_kernel) {
    if (hipEventElapsedTime(&f, ctx->ev0, ctx->ev1) != hipSuccess) return KF_E_HIP;
    *forward_ms = (double)f;
    *backward_ms = 0.0;
    return KF_OK;
  }
  if (hipEventElapsedTime(&f, ctx->ev0, ctx->evm) != hipSuccess ||
      hipEventElapsedTime(&b, ctx->evm, ctx->ev1) != hipSuccess)
    return KF_E_HIP;
  *forward_ms = (double)f;
  *backward_ms = (double)b;
  return KF_OK;
}

}  // extern "C"
