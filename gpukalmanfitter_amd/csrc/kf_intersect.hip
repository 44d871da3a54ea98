// kf_intersect.hip -- batched intersection of rays with bounded planes
// (kf_intersect in include/kf_abi.h): the reference's intersection test
// (Run/GPU/IntersectGPUTest.cu:22-48, 116-172) over many rays.
//
// Work is split over (ray, surface chunk) pairs so that a launch fills the
// chip however few rays there are: a block takes 256 rays and one chunk of
// consecutive surfaces.  Every lane of a wave reads the same surface at the
// same time, so surface data comes through scalar loads into SGPRs (no LDS,
// no barriers).  Each pair first meets a bounding-sphere test (the ray's line
// against the sphere about the surface centre that holds the polygon, with a
// margin far above rounding): the full intersection runs only when a lane of
// the wave passes it, which for a detector mesh is a few percent of the
// surfaces.
//
// With more than a few rays a wave first drops surfaces for all its rays at
// once: each lane takes one surface and tests its sphere against the cone that
// holds the wave's 64 rays, so 64 surfaces cost ~35 instructions where 64
// sphere tests of one surface each cost ~900.  The cone is narrow when the
// rays point the same way, so they are taken in the order of their directions'
// cells (a counting sort, three short launches); the surfaces need no order.
// The cone passes every surface whose sphere test and full test a ray of it
// could pass, so the kept pairs do not change.  16,384 rays x 37,122
// triangles: 153 us a call (under the profiler the count pass 115, the write pass
// 20, five short launches 27) against 453 without, and 278 with boxes about 16
// surfaces in listed order instead of cones; 4,000 x 488 triangles 115 against
// 216.
//
// Output order is (ray, surface) without atomics: the count pass keeps, per
// (ray, chunk), the number of kept intersections and the first kIxSlots
// surface indices; an exclusive scan of the counts in (ray, chunk) order gives
// each (ray, chunk) its output offset; the write pass recomputes only the
// slotted surfaces (a (ray, chunk) with more than kIxSlots runs over its chunk
// again).
//
// This file is compiled without multiply-add contraction: every value is the
// correctly rounded result of the same operations, in the same order, as the
// reference formulation, so the kept pairs, paths and positions are
// bit-identical to an uncontracted FP64 build of it (double division on
// gfx950 is correctly rounded).
#include <hip/hip_runtime.h>

#include "../../include/kf_abi.h"
#include "kf_device.hpp"
#include "kf_scan.hpp"

namespace kfd {

constexpr int kIxBlock = 256;                // rays per block (count pass)
constexpr int kIxSlots = 8;                  // surface indices kept per (ray, chunk)
// sphere tests per group where a wave takes every surface: 4 keeps the kernel
// without cones at 42 VGPRs (8 waves per SIMD hide the scalar-load latency; 8
// tests per group need 98)
constexpr int kIxGroup = 4;
constexpr int64_t kIxTargetBlocks = 4096;    // count-pass blocks wanted (16 per CU)
// Rays are sorted by direction, and cones used, from two waves' worth of them
// and one ray to 32 surfaces on: with fewer all chunks run at once and the
// sort's launches (10 us) decide.  Plain and sorted: 37,122 triangles, 512
// rays 65 and 72 us, 1,500 rays 85 and 79; 16,000 triangles, 256 rays 68 and
// 73, 1,000 rays 76 and 71; 5,600 triangles, 128 rays 89 and 79.
constexpr int64_t kIxSortRays = 128, kIxSortSurfaces = 32;
constexpr int kIxCells = 64;                 // direction cells per axis of the unit square
constexpr int kIxBins = kIxCells * kIxCells;
// cosine of the half angle from which a wave's cone is used: past 60 degrees
// it passes most surfaces and only adds its own test
constexpr double kIxConeCos = 0.5;
constexpr int kIxList = 16;                  // candidates a lane collects before testing them
constexpr int64_t kIxMinChunk = 256;         // surfaces per chunk, lower bound
constexpr int64_t kIxMaxChunk = 8192;        // and upper bound
// bounding-sphere margin: relative on the radius^2, and on |centre|^2 and
// |ray origin|^2 (rounding of the full test is ~1e-15 of these)
constexpr double kIxRelMargin = 1e-6;
constexpr double kIxAbsMargin = 3e-12;

struct IxPlan {
  int64_t chunk;     // surfaces per chunk
  int64_t n_chunks;  // chunks (>= 1)
  int64_t pairs;     // n_rays * n_chunks
};

inline IxPlan ixPlan(int64_t n_rays, int64_t n_surfaces) {
  const int64_t ray_blocks = (n_rays + kIxBlock - 1) / kIxBlock;
  const int64_t want = ray_blocks > 0 ? (kIxTargetBlocks + ray_blocks - 1) / ray_blocks : 1;
  int64_t chunk = (n_surfaces + want - 1) / want;
  chunk = chunk < kIxMinChunk ? kIxMinChunk : (chunk > kIxMaxChunk ? kIxMaxChunk : chunk);
  chunk = (chunk + 63) / 64 * 64;  // whole waves of surfaces
  int64_t n_chunks = (n_surfaces + chunk - 1) / chunk;
  if (n_chunks < 1) n_chunks = 1;
  return {chunk, n_chunks, n_rays * n_chunks};
}

inline int64_t align256(int64_t b) { return (b + 255) / 256 * 256; }

// PlaneSurface::intersect (PlaneSurface.ipp:239-259) with
// PlanarHelper::intersectionEstimate (PlanarHelper.hpp:29-48) and the
// reference driver's selection: reachable (path^2 >= tolerance^2), path >= 0,
// inside the convex polygon when bcheck (BoundaryCheck::isInsidePolygon).
KFD_INLINE bool intersectKept(const kf_polygon_plane &s, const double p[3], const double d[3],
                              bool bcheck, double &path, double x[3]) {
  const double n[3] = {s.rot[2], s.rot[5], s.rot[8]};
  const double denom = d[0] * n[0] + d[1] * n[1] + d[2] * n[2];
  if (denom == 0.0) return false;  // unreachable
  const double cp[3] = {s.center[0] - p[0], s.center[1] - p[1], s.center[2] - p[2]};
  path = (n[0] * cp[0] + n[1] * cp[1] + n[2] * cp[2]) / denom;
  if (path * path < kOnSurfaceTolerance * kOnSurfaceTolerance) return false;  // on surface
  if (path < 0.0) return false;
#pragma unroll
  for (int k = 0; k < 3; ++k) x[k] = p[k] + path * d[k];
  if (!bcheck) return true;
  const double v[3] = {x[0] - s.center[0], x[1] - s.center[1], x[2] - s.center[2]};
  const double lu = s.rot[0] * v[0] + s.rot[3] * v[1] + s.rot[6] * v[2];
  const double lv = s.rot[1] * v[0] + s.rot[4] * v[1] + s.rot[7] * v[2];
  // the point is inside when it is on the same side of every edge
  // (signbit of the z component of edge x (point - edge start))
  const int nv =
      (s.n_vertices < 3) ? 3 : ((s.n_vertices > KF_POLY_MAX) ? KF_POLY_MAX : s.n_vertices);
  bool ref = false, inside = true;
  for (int i = 0; i < nv; ++i) {
    const int j = (i + 1 < nv) ? i + 1 : 0;
    const double e0 = s.vertices[2 * j] - s.vertices[2 * i];
    const double e1 = s.vertices[2 * j + 1] - s.vertices[2 * i + 1];
    const double q0 = lu - s.vertices[2 * i], q1 = lv - s.vertices[2 * i + 1];
    const bool side = signbit((e0 * q1) - (e1 * q0));
    if (i == 0) ref = side;
    inside = inside && (side == ref);
  }
  return inside;
}

// Per surface: centre and the squared radius of the sphere about it that
// holds every vertex, with the margin (|centre|^2 part included); negative
// where the polygon is not strictly convex or the rotation not orthonormal, so
// that the inside test could accept points outside the sphere (those surfaces
// are not dropped for lying behind a wave's rays).  Entries n_surfaces .. n_surfaces + kIxGroup - 1 are
// the zero padding.  Also zeroes the direction histogram.
__global__ void __launch_bounds__(256)
    kf_ix_spheres(const kf_polygon_plane *__restrict__ surfaces, int64_t n_surfaces,
                  double4 *__restrict__ spheres, int32_t *__restrict__ bins) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  for (int64_t b = i; bins && b < kIxBins; b += (int64_t)gridDim.x * 256) bins[b] = 0;
  if (i >= n_surfaces + kIxGroup) return;
  if (i >= n_surfaces) {
    spheres[i] = make_double4(0.0, 0.0, 0.0, 0.0);
    return;
  }
  const kf_polygon_plane &s = surfaces[i];
  const int nv =
      (s.n_vertices < 3) ? 3 : ((s.n_vertices > KF_POLY_MAX) ? KF_POLY_MAX : s.n_vertices);
  double r2 = 0.0;
  int left = 0, right = 0;
  for (int k = 0; k < nv; ++k) {
    const int n1 = (k + 1 < nv) ? k + 1 : 0, n2 = (n1 + 1 < nv) ? n1 + 1 : 0;
    const double u = s.vertices[2 * k], v = s.vertices[2 * k + 1];
    const double q = u * u + v * v;
    r2 = q > r2 ? q : r2;
    if (!bins) continue;  // the signs are read with the cones only
    // the turn from edge k to edge k + 1, against its rounding
    const double e0 = s.vertices[2 * n1] - u, e1 = s.vertices[2 * n1 + 1] - v;
    const double f0 = s.vertices[2 * n2] - s.vertices[2 * n1],
                 f1 = s.vertices[2 * n2 + 1] - s.vertices[2 * n1 + 1];
    const double x = e0 * f1, y = e1 * f0, tiny = 1e-9 * (fabs(x) + fabs(y));
    left += (x - y > tiny) ? 1 : 0;
    right += (y - x > tiny) ? 1 : 0;
  }
  const double cc =
      s.center[0] * s.center[0] + s.center[1] * s.center[1] + s.center[2] * s.center[2];
  const double w = r2 * (1.0 + kIxRelMargin) + kIxAbsMargin * cc;
  bool plain = left == nv || right == nv;
  if (bins)
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = a; b < 3; ++b)
        plain = plain && fabs(s.rot[a] * s.rot[b] + s.rot[3 + a] * s.rot[3 + b] +
                              s.rot[6 + a] * s.rot[6 + b] - (a == b ? 1.0 : 0.0)) < 1e-7;
  spheres[i] = make_double4(s.center[0], s.center[1], s.center[2],
                            plain ? w : -w);
}

// Cell of a direction: the octahedron's faces unfolded onto the unit square,
// cells numbered along a Hilbert curve, so that consecutive rays fill a compact
// patch (along a Z curve the median half angle of a wave's cone is 13 degrees
// instead of 11, and a tenth of the waves straddle one of its jumps).  Any
// value is a valid cell (0 for a direction that is not finite): the order
// only decides which rays share a wave.
KFD_INLINE int directionCell(const double *ray_dir, int64_t n_rays, int64_t r) {
  const float x = (float)ray_dir[r], y = (float)ray_dir[n_rays + r],
              z = (float)ray_dir[2 * n_rays + r];
  const float s = 1.0f / (fabsf(x) + fabsf(y) + fabsf(z));
  float u = x * s, v = y * s;
  if (z < 0.0f) {
    const float w = (1.0f - fabsf(v)) * (u < 0.0f ? -1.0f : 1.0f);
    v = (1.0f - fabsf(u)) * (v < 0.0f ? -1.0f : 1.0f);
    u = w;
  }
  int a = (int)((u * 0.5f + 0.5f) * (float)kIxCells), b = (int)((v * 0.5f + 0.5f) * (float)kIxCells);
  a = a < 0 ? 0 : (a > kIxCells - 1 ? kIxCells - 1 : a);
  b = b < 0 ? 0 : (b > kIxCells - 1 ? kIxCells - 1 : b);
  int m = 0;
#pragma unroll
  for (int q = kIxCells / 2; q > 0; q >>= 1) {
    const int ra = (a & q) ? 1 : 0, rb = (b & q) ? 1 : 0;
    m += q * q * ((3 * ra) ^ rb);
    a &= q - 1;
    b &= q - 1;
    if (rb == 0) {
      const int ta = ra ? q - 1 - b : b;
      b = ra ? q - 1 - a : a;
      a = ta;
    }
  }
  return m;
}

__global__ void __launch_bounds__(256)
    kf_ix_bin(const double *__restrict__ ray_dir, int64_t n_rays, int32_t *__restrict__ bins) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r < n_rays) atomicAdd(&bins[directionCell(ray_dir, n_rays, r)], 1);
}

// bins[b] <- rays in the bins before b (one block)
__global__ void __launch_bounds__(256) kf_ix_bin_offsets(int32_t *__restrict__ bins) {
  constexpr int kPer = kIxBins / 256;
  __shared__ int32_t part[256];
  int32_t v[kPer], sum = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    v[k] = bins[threadIdx.x * kPer + k];
    sum += v[k];
  }
  part[threadIdx.x] = sum;
  __syncthreads();
  for (int w = 1; w < 256; w <<= 1) {
    const int32_t add = (threadIdx.x >= (unsigned)w) ? part[threadIdx.x - w] : 0;
    __syncthreads();
    part[threadIdx.x] += add;
    __syncthreads();
  }
  int32_t run = part[threadIdx.x] - sum;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    bins[threadIdx.x * kPer + k] = run;
    run += v[k];
  }
}

__global__ void __launch_bounds__(256)
    kf_ix_order(const double *__restrict__ ray_dir, int64_t n_rays, int32_t *__restrict__ bins,
                int32_t *__restrict__ order) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r < n_rays) order[atomicAdd(&bins[directionCell(ray_dir, n_rays, r)], 1)] = (int32_t)r;
}

struct Ray {
  double p[3], d[3];
  double m[3];  // moment p x d
  double dd;    // |d|^2
  double pmdd;  // margin part of |p|^2, times |d|^2
};

KFD_INLINE Ray loadRay(const double *ray_pos, const double *ray_dir, int64_t n_rays, int64_t r) {
  Ray y;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    y.p[k] = ray_pos[(size_t)k * n_rays + r];
    y.d[k] = ray_dir[(size_t)k * n_rays + r];
  }
  y.m[0] = y.p[1] * y.d[2] - y.p[2] * y.d[1];
  y.m[1] = y.p[2] * y.d[0] - y.p[0] * y.d[2];
  y.m[2] = y.p[0] * y.d[1] - y.p[1] * y.d[0];
  y.dd = y.d[0] * y.d[0] + y.d[1] * y.d[1] + y.d[2] * y.d[2];
  y.pmdd = kIxAbsMargin * (y.p[0] * y.p[0] + y.p[1] * y.p[1] + y.p[2] * y.p[2]) * y.dd;
  return y;
}

// The ray's line passes within the sphere (or a component is not finite):
// |(c - p) x d|^2 <= R^2 |d|^2, with (c - p) x d = c x d - p x d.  Only a
// filter (the margin in R^2 is far above the rounding of either form), so
// it uses fused multiply-adds: 11 operations per pair.
KFD_INLINE bool sphereCandidate(const double4 &q, const Ray &y) {
  const double e0 = fma(q.y, y.d[2], fma(-q.z, y.d[1], -y.m[0]));
  const double e1 = fma(q.z, y.d[0], fma(-q.x, y.d[2], -y.m[1]));
  const double e2 = fma(q.x, y.d[1], fma(-q.y, y.d[0], -y.m[2]));
  const double lhs = fma(e0, e0, fma(e1, e1, e2 * e2));
  return !(fma(-fabs(q.w), y.dd, lhs) > y.pmdd);
}

// The value that lane j (the same for the whole wave) holds.
KFD_INLINE double laneValue(double v, int j) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, j);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), j);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
#else
  return v;
#endif
}
// Sum, minimum and maximum over a wave (every lane gets the result).
KFD_INLINE double waveSum(double v) {
#pragma unroll
  for (int w = 1; w < 64; w <<= 1) v += __shfl_xor(v, w, 64);
  return v;
}
KFD_INLINE double waveMin(double v) {
#pragma unroll
  for (int w = 1; w < 64; w <<= 1) v = fmin(v, __shfl_xor(v, w, 64));
  return v;
}
KFD_INLINE double waveMax(double v) {
#pragma unroll
  for (int w = 1; w < 64; w <<= 1) v = fmax(v, __shfl_xor(v, w, 64));
  return v;
}

// The cone that holds a wave's rays: about the axis u from the middle o of
// their origins (all within rho of it), half angle theta.  A point of a ray at
// height a = (x - o).u is within rho + (a + rho) tan(theta) of the axis, and
// a >= -rho; a sphere (c, R) it meets therefore has
//   |(c - o) x u| <= R + rho + (a_c + R + rho) tan(theta),  a_c >= -rho - R.
struct Cone {
  double o[3], u[3], tan, r0;  // r0: rho with its margin
  bool narrow;
};
KFD_INLINE Cone waveCone(const Ray &y) {
  Cone c;
  const double n = sqrt(y.dd), in = 1.0 / n;
  double m[3], mm = 0.0, rho = 0.0;
  bool finite = y.dd > 1e-200 && y.dd < 1e200;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    finite = finite && fabs(y.p[k]) < 1e100 && fabs(y.d[k] * in) <= 2.0;
    m[k] = waveSum(y.d[k] * in);
    c.o[k] = 0.5 * (waveMin(y.p[k]) + waveMax(y.p[k]));
    mm += m[k] * m[k];
  }
  const double im = 1.0 / sqrt(mm);
  double cosT = 0.0, big = 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    c.u[k] = m[k] * im;
    cosT += c.u[k] * (y.d[k] * in);
    rho += (y.p[k] - c.o[k]) * (y.p[k] - c.o[k]);
    big += fabs(y.p[k]);
  }
  cosT = waveMin(cosT) - 1e-9;
  // the sphere test allows 1.8e-6 |p| about the sphere
  c.r0 = waveMax(sqrt(rho) + 4e-6 * big);
  c.tan = sqrt(1.0 - cosT * cosT) / cosT;
  c.narrow = __all(finite) && cosT >= kIxConeCos && c.r0 < 1e100;
  return c;
}
// False only if no ray of the cone passes both tests of the surface.
KFD_INLINE bool coneCandidate(const double4 &q, const Cone &c) {
  const double v0 = q.x - c.o[0], v1 = q.y - c.o[1], v2 = q.z - c.o[2];
  const double x0 = v1 * c.u[2] - v2 * c.u[1], x1 = v2 * c.u[0] - v0 * c.u[2],
               x2 = v0 * c.u[1] - v1 * c.u[0];
  const double a = v0 * c.u[0] + v1 * c.u[1] + v2 * c.u[2];
  const double b2 = x0 * x0 + x1 * x1 + x2 * x2;
  // the radius, and what it takes to cover the rounding of the lines above
  const double r = (double)sqrtf((float)fabs(q.w)) * (1.0 + 1e-6) + c.r0 +
                   1e-9 * (fabs(v0) + fabs(v1) + fabs(v2));
  // (kf_ix_spheres: a surface with negative w is not dropped for lying behind)
  const double h = (signbit(q.w) ? fabs(a) : a) + r;
  const double lim = fma(h, c.tan, r);
  return !(h < 0.0 || b2 > lim * lim);
}

// Count pass: block (ray block, chunk); per (ray, chunk) the number of kept
// intersections and the first kIxSlots surface indices.  CONES: the rays come
// in the order of their directions, and each wave drops surfaces by its cone;
// rays past the end run as copies of the last one and count nothing.
template <bool CONES>
__global__ void __launch_bounds__(kIxBlock)
    kf_ix_count(const kf_polygon_plane *__restrict__ surfaces, const double4 *__restrict__ spheres,
                const int32_t *__restrict__ order, int64_t n_surfaces, int64_t chunk,
                int64_t n_chunks, const double *__restrict__ ray_pos,
                const double *__restrict__ ray_dir, int64_t n_rays, int bcheck,
                int32_t *__restrict__ counts, int32_t *__restrict__ slots) {
  const int64_t c = blockIdx.x % n_chunks;
  int64_t at = (blockIdx.x / n_chunks) * kIxBlock + threadIdx.x;
  if ((CONES ? at - (threadIdx.x & 63u) : at) >= n_rays) return;  // CONES: the whole wave
  const bool own = at < n_rays;
  if (!own) at = n_rays - 1;
  const int64_t r = CONES ? (int64_t)order[at] : at;
  const Ray y = loadRay(ray_pos, ray_dir, n_rays, r);
  const int64_t t = r * n_chunks + c, pairs = n_rays * n_chunks;
  // surface indices fit int32 (checked by the caller): 32-bit uniform loop
  const int s0 = (int)(c * chunk);
  const int s1 = (c + 1 == n_chunks) ? (int)n_surfaces : s0 + (int)chunk;
  int cnt = 0;
  auto test = [&](int i) {
    double path, x[3];
    if (intersectKept(surfaces[i], y.p, y.d, CONES || bcheck != 0, path, x)) {
      if (own && cnt < kIxSlots) slots[(int64_t)cnt * pairs + t] = i;
      ++cnt;
    }
  };
  if constexpr (CONES) {
    // A lane notes the surfaces whose sphere its line passes and tests them
    // later, in surface order: a surface is a candidate of a few of the 64
    // rays, so tested at once for the whole wave most lanes would idle through
    // a full test and the latency of its loads.
    __shared__ int32_t list[kIxList][kIxBlock];
    int n = 0;
    auto note = [&](int i) { list[n++][threadIdx.x] = i; };
    auto flush = [&](int room) {
      if (!__any(n > kIxList - room)) return;
      for (int k = 0; __any(k < n); ++k)
        if (k < n) test(list[k][threadIdx.x]);
      n = 0;
    };
    const Cone cone = waveCone(y);
    if (cone.narrow) {
      // 64 surfaces at a time, one per lane, against the cone; the sphere of
      // each that passes goes to every lane through scalar registers
      const int lane = (int)(threadIdx.x & 63u);
      double4 next = spheres[(s0 + lane < s1) ? s0 + lane : s1 - 1];
      for (int b0 = s0; b0 < s1; b0 += 64) {
        const double4 q = next;
        next = spheres[(b0 + 64 + lane < s1) ? b0 + 64 + lane : s1 - 1];
        uint64_t m = __ballot(b0 + lane < s1 && coneCandidate(q, cone));
        while (m) {
          const int j = __builtin_ctzll(m);
          m &= m - 1;
          const double4 w = make_double4(laneValue(q.x, j), laneValue(q.y, j), laneValue(q.z, j),
                                         laneValue(q.w, j));
          if (sphereCandidate(w, y)) note(b0 + j);
          flush(1);
        }
      }
    } else {
      for (int i0 = s0; i0 < s1; i0 += kIxGroup) {
#pragma unroll
        for (int j = 0; j < kIxGroup; ++j)
          if (sphereCandidate(spheres[i0 + j], y) && i0 + j < s1) note(i0 + j);
        flush(kIxGroup);
      }
    }
    flush(kIxList);
  } else if (!bcheck) {
    for (int i = s0; i < s1; ++i) test(i);
  } else {
    // groups of kIxGroup surfaces: the sphere tests first (their loads issued
    // together), then the full test of the candidates in surface order
    // (the sphere array is padded by kIxGroup entries: the loads past s1 stay
    // in bounds and their bits are masked off)
    for (int i0 = s0; i0 < s1; i0 += kIxGroup) {
      uint32_t m = 0;
#pragma unroll
      for (int j = 0; j < kIxGroup; ++j)
        if (sphereCandidate(spheres[i0 + j], y)) m |= 1u << j;
      if (s1 - i0 < kIxGroup) m &= (1u << (s1 - i0)) - 1u;
      if (m == 0) continue;
#pragma unroll 1
      for (int j = 0; j < kIxGroup; ++j)
        if ((m >> j) & 1u) test(i0 + j);
    }
  }
  if (own) counts[t] = cnt;
}

KFD_INLINE void writeHit(kf_intersection *h, int64_t r, int64_t i, double path,
                         const double x[3]) {
  h->ray = (int32_t)r;
  h->surface = (int32_t)i;
  h->path = path;
  h->position[0] = x[0];
  h->position[1] = x[1];
  h->position[2] = x[2];
}

// Write pass: one thread per (ray, chunk), in (ray, chunk) order.
__global__ void __launch_bounds__(256)
    kf_ix_write(const kf_polygon_plane *__restrict__ surfaces, const double4 *__restrict__ spheres,
                int64_t n_surfaces, int64_t chunk, int64_t n_chunks,
                const double *__restrict__ ray_pos, const double *__restrict__ ray_dir,
                int64_t n_rays, int bcheck, const int32_t *__restrict__ counts,
                const int32_t *__restrict__ slots, const int64_t *__restrict__ offsets,
                kf_intersection *__restrict__ hits, int64_t capacity) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t pairs = n_rays * n_chunks;
  if (t >= pairs) return;
  const int32_t cnt = counts[t];
  int64_t out = offsets[t];
  if (cnt == 0 || out >= capacity) return;
  const int64_t r = t / n_chunks, c = t - r * n_chunks;
  const Ray y = loadRay(ray_pos, ray_dir, n_rays, r);
  double path, x[3];
  if (cnt <= kIxSlots) {
    for (int k = 0; k < cnt && out < capacity; ++k) {
      const int64_t i = slots[(int64_t)k * pairs + t];
      if (intersectKept(surfaces[i], y.p, y.d, bcheck != 0, path, x))
        writeHit(hits + out++, r, i, path, x);
    }
    return;
  }
  const int64_t s0 = c * chunk;
  const int64_t s1 = (s0 + chunk < n_surfaces) ? s0 + chunk : n_surfaces;
  for (int64_t i = s0; i < s1 && out < capacity; ++i) {
    if (bcheck && !sphereCandidate(spheres[i], y)) continue;
    if (intersectKept(surfaces[i], y.p, y.d, bcheck != 0, path, x))
      writeHit(hits + out++, r, i, path, x);
  }
}

struct IxScratch {
  double4 *spheres;
  int32_t *bins, *order;  // the direction sort
  int32_t *counts, *slots;
  int64_t *offsets;
  void *scan;
  int64_t bytes;
};

// Scratch layout from `base` (nullptr: sizes only).
inline IxScratch ixScratch(void *base, int64_t n_rays, int64_t n_surfaces) {
  const IxPlan pl = ixPlan(n_rays, n_surfaces);
  IxScratch s;
  char *b = (char *)base;
  int64_t at = 0;
  s.spheres = (double4 *)(b + at);
  at += align256((n_surfaces + kIxGroup) * (int64_t)sizeof(double4));
  s.bins = (int32_t *)(b + at);
  at += align256(kIxBins * (int64_t)sizeof(int32_t));
  s.order = (int32_t *)(b + at);
  at += align256(n_rays * (int64_t)sizeof(int32_t));
  s.counts = (int32_t *)(b + at);
  at += align256(pl.pairs * (int64_t)sizeof(int32_t));
  s.slots = (int32_t *)(b + at);
  at += align256(pl.pairs * kIxSlots * (int64_t)sizeof(int32_t));
  s.offsets = (int64_t *)(b + at);
  at += align256((pl.pairs + 1) * (int64_t)sizeof(int64_t));
  s.scan = b + at;
  at += align256(kscan::scratchBytes(pl.pairs));
  s.bytes = at;
  return s;
}

}  // namespace kfd

extern "C" int64_t kfd_intersect_scratch_bytes(int64_t n_rays, int64_t n_surfaces) {
  return kfd::ixScratch(nullptr, n_rays, n_surfaces).bytes;
}

// Launches the sphere set-up, the direction sort, the count pass, the scan and the write pass;
// n_hits[0] = the total.
extern "C" hipError_t kfd_launch_intersect(const kf_polygon_plane *surfaces, int64_t n_surfaces,
                                           const double *ray_pos, const double *ray_dir,
                                           int64_t n_rays, int bcheck, kf_intersection *hits,
                                           int64_t capacity, int64_t *n_hits, void *scratch,
                                           hipStream_t s) {
  using namespace kfd;
  const IxPlan pl = ixPlan(n_rays, n_surfaces);
  const IxScratch sc = ixScratch(scratch, n_rays, n_surfaces);
  const bool sort = bcheck && n_rays >= kIxSortRays && n_surfaces > kIxMinChunk &&
                    n_rays * kIxSortSurfaces >= n_surfaces;
  hipLaunchKernelGGL(kf_ix_spheres, dim3((unsigned)((n_surfaces + kIxGroup + 255) / 256)),
                     dim3(256), 0, s, surfaces, n_surfaces, sc.spheres, sort ? sc.bins : nullptr);
  const int64_t ray_blocks = (n_rays + kIxBlock - 1) / kIxBlock;
  if (sort) {
    const dim3 rb((unsigned)ray_blocks);
    hipLaunchKernelGGL(kf_ix_bin, rb, dim3(256), 0, s, ray_dir, n_rays, sc.bins);
    hipLaunchKernelGGL(kf_ix_bin_offsets, dim3(1), dim3(256), 0, s, sc.bins);
    hipLaunchKernelGGL(kf_ix_order, rb, dim3(256), 0, s, ray_dir, n_rays, sc.bins, sc.order);
  }
  if (ray_blocks > 0)
    hipLaunchKernelGGL(HIP_KERNEL_NAME(sort ? kf_ix_count<true> : kf_ix_count<false>),
                       dim3((unsigned)(ray_blocks * pl.n_chunks)), dim3(kIxBlock), 0, s, surfaces,
                       (const double4 *)sc.spheres, (const int32_t *)sc.order, n_surfaces,
                       pl.chunk, pl.n_chunks, ray_pos, ray_dir, n_rays, bcheck, sc.counts,
                       sc.slots);
  hipError_t e = kscan::exclusiveScan(pl.pairs, sc.counts, sc.offsets, sc.scan, s);
  if (e != hipSuccess) return e;
  if (pl.pairs > 0 && capacity > 0)
    hipLaunchKernelGGL(kf_ix_write, dim3((unsigned)((pl.pairs + 255) / 256)), dim3(256), 0, s,
                       surfaces, (const double4 *)sc.spheres, n_surfaces, pl.chunk, pl.n_chunks,
                       ray_pos, ray_dir, n_rays, bcheck, (const int32_t *)sc.counts,
                       (const int32_t *)sc.slots, (const int64_t *)sc.offsets, hits, capacity);
  e = hipMemcpyAsync(n_hits, sc.offsets + pl.pairs, sizeof(int64_t), hipMemcpyDeviceToDevice, s);
  if (e != hipSuccess) return e;
  return hipGetLastError();
}
