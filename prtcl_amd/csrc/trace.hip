// Sphere tracer of a scene group on the device, the algorithm of the
// reference's SphereTracer::Trace (util/sphere_tracer.hpp:46-268):
//
// * cells of edge grid_diameter = 4 h (floor(x / grid_diameter)), in a dense
//   box around the group; a counting sort puts every particle in its cell,
//   ordered by host index inside a cell, and the occupied cells are
//   compacted into a list of cell centres;
// * one wavefront per pixel marches its ray (pinhole camera,
//   geometry/pinhole_camera.hpp:33-65). At every step the distance bound is
//   the minimum over all occupied cells of the rounded-box distance
//   |max(q, 0)| + min(max_k q_k, 0) - grid_diameter, q = |x - centre| -
//   grid_diameter. The reference evaluates every cell; here cells are
//   grouped by 4^3, a group's box bounds the distances of its cells from
//   below, and groups that cannot lower the minimum are skipped, so the
//   minimum is the same value at a fraction of the work. Below
//   grid_diameter the implicit function of the particles
//   in the 27 cells around the ray point (cubic spline with h =
//   grid_diameter / 2, divided by its Lipschitz constant and the particle
//   count) tightens the bound and gives the normal;
// * the pixel is 0 when the march ran out of steps, 0.3 when the ray left
//   (parameter beyond 10000 grid diameters), else -dot(ray, normal).
//
// Double precision throughout (PinholeCamera::Real), no contraction of
// multiply-adds, and every expression in the reference's order, so the image
// is that of the same arithmetic on the CPU.
#include "trace.hpp"

#include <cfloat>
#include <cmath>
#include <limits>
#include <stdexcept>
#include <type_traits>
#include <vector>

namespace prtcl_amd {
namespace {

constexpr int kTB = 256;

struct CellBox {
  int32_t ox, oy, oz, nx, ny, nz;
  double gd;
};

struct TraceParams {
  double O[3], v[3], p[3], hh[3];
  double f, pixel_size, sox, soy;
  double gd, half, phi0, L, alpha, h3, h4, grad_eps, max_parameter;
  int64_t width, height, max_steps;
};

__host__ __device__ inline double dot3(const double *a, const double *b) {
  return a[0] * b[0] + (a[1] * b[1] + a[2] * b[2]);
}

__host__ __device__ inline void normalized3(const double *a, double *out) {
  const double z = dot3(a, a);
  for (int k = 0; k < 3; ++k)
    out[k] = z > 0 ? a[k] / sqrt(z) : a[k];
}

__host__ __device__ inline double cpow(double x, int n) {
  double r = 1;
  for (; n > 0; --n)
    r *= x;
  return r;
}

// cubic spline, N = 3 (cubic_spline_kernel.hpp:43-78)
__host__ __device__ inline double evalq(double alpha, double q) {
  double r = 0;
  if (q < 1)
    r -= 4 * cpow(1 - q, 3);
  if (q < 2)
    r += cpow(2 - q, 3);
  return alpha * r;
}

__host__ __device__ inline double evaldq(double alpha, double q) {
  double r = 0;
  if (q < 1)
    r += 12 * cpow(1 - q, 2);
  if (q < 2)
    r -= 3 * cpow(2 - q, 2);
  return alpha * r;
}

// std::min / std::max of the reference, NaN behaviour included
__device__ inline double std_min(double a, double b) { return (b < a) ? b : a; }
__device__ inline double std_max(double a, double b) { return (a < b) ? b : a; }

__device__ inline bool cell_index(const CellBox &B, int32_t cx, int32_t cy, int32_t cz,
                                  int64_t *lin) {
  const int64_t x = static_cast<int64_t>(cx) - B.ox, y = static_cast<int64_t>(cy) - B.oy,
                z = static_cast<int64_t>(cz) - B.oz;
  if (x < 0 || y < 0 || z < 0 || x >= B.nx || y >= B.ny || z >= B.nz)
    return false;
  *lin = (z * B.ny + y) * B.nx + x;
  return true;
}

template <class T>
__global__ void k_tr_to_double(const T *src, double *dst, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kTB + threadIdx.x;
  if (i < n)
    dst[i] = static_cast<double>(src[i]);
}

// per block: min x, y, z and max x, y, z of its particles
__global__ __launch_bounds__(kTB) void k_tr_bbox(const double *x, int64_t n, double *part) {
  __shared__ double s[6][kTB];
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kTB + threadIdx.x;
  for (int k = 0; k < 3; ++k) {
    s[k][threadIdx.x] = i < n ? x[3 * i + k] : DBL_MAX;
    s[3 + k][threadIdx.x] = i < n ? x[3 * i + k] : -DBL_MAX;
  }
  __syncthreads();
  for (int w = kTB / 2; w > 0; w >>= 1) {
    if (static_cast<int>(threadIdx.x) < w)
      for (int k = 0; k < 3; ++k) {
        s[k][threadIdx.x] = fmin(s[k][threadIdx.x], s[k][threadIdx.x + w]);
        s[3 + k][threadIdx.x] = fmax(s[3 + k][threadIdx.x], s[3 + k][threadIdx.x + w]);
      }
    __syncthreads();
  }
  if (threadIdx.x < 6)
    part[6 * static_cast<int64_t>(blockIdx.x) + threadIdx.x] = s[threadIdx.x][0];
}

__global__ void k_tr_count(const double *x, int64_t n, CellBox B, uint32_t *count,
                           int64_t *lin_of) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kTB + threadIdx.x;
  if (i >= n)
    return;
  int64_t lin = -1;
  const double *p = x + 3 * i;
  if (isfinite(p[0]) && isfinite(p[1]) && isfinite(p[2])) {
    // inside the box, which was planned from the finite positions
    const int32_t cx = static_cast<int32_t>(floor(p[0] / B.gd));
    const int32_t cy = static_cast<int32_t>(floor(p[1] / B.gd));
    const int32_t cz = static_cast<int32_t>(floor(p[2] / B.gd));
    if (!cell_index(B, cx, cy, cz, &lin))
      lin = -1;
  }
  if (lin >= 0)
    atomicAdd(&count[lin], 1u);
  lin_of[i] = lin;  // -1: not placed (a non-finite position)
}

// exclusive scan of uint32 counts into uint32 starts, in tiles of kTB
// values per block (block sums scanned by one block, then added back)
__device__ uint32_t tr_block_scan(uint32_t v, uint32_t *total) {
  __shared__ uint32_t wsum[kTB / 64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  uint32_t x = v;
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, d, 64);
    if (lane >= d)
      x += y;
  }
  if (lane == 63)
    wsum[wv] = x;
  __syncthreads();
  uint32_t before = 0, all = 0;
  for (int k = 0; k < kTB / 64; ++k) {
    if (k < wv)
      before += wsum[k];
    all += wsum[k];
  }
  __syncthreads();
  *total = all;
  return before + x - v;
}

__global__ __launch_bounds__(kTB) void k_tr_scan_tiles(const uint32_t *in, int64_t n,
                                                       uint32_t *out, uint32_t *bsum) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kTB + threadIdx.x;
  uint32_t tot;
  const uint32_t ex = tr_block_scan(i < n ? in[i] : 0u, &tot);
  if (i < n)
    out[i] = ex;
  if (threadIdx.x == 0)
    bsum[blockIdx.x] = tot;
}

__global__ __launch_bounds__(kTB) void k_tr_scan_top(uint32_t *bsum, int64_t nb) {
  uint32_t carry = 0;
  for (int64_t base = 0; base < nb; base += kTB) {
    const int64_t i = base + threadIdx.x;
    uint32_t tot;
    const uint32_t ex = tr_block_scan(i < nb ? bsum[i] : 0u, &tot);
    if (i < nb)
      bsum[i] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0)
    bsum[nb] = carry;
}

__global__ void k_tr_scan_add(uint32_t *out, int64_t n, const uint32_t *bsum) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kTB + threadIdx.x;
  if (i < n)
    out[i] += bsum[blockIdx.x];
  if (i == n)
    out[n] = bsum[gridDim.x];  // the total after the last value
}

__global__ void k_tr_place(const int64_t *lin_of, int64_t n, const uint32_t *start,
                           uint32_t *cursor, uint32_t *ent) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kTB + threadIdx.x;
  if (i >= n)
    return;
  const int64_t lin = lin_of[i];
  if (lin >= 0)
    ent[start[lin] + atomicAdd(&cursor[lin], 1u)] = static_cast<uint32_t>(i);
}

// positions packed by cell, in host order inside every cell: the particle at
// (unordered) entry k goes to its cell's start plus the number of the cell's
// entries with a smaller host index
__global__ void k_tr_pack(const double *x, const int64_t *lin_of, const uint32_t *start,
                          const uint32_t *ent, int64_t n, double *ex) {
  const int64_t k = static_cast<int64_t>(blockIdx.x) * kTB + threadIdx.x;
  if (k >= n)
    return;
  const uint32_t i = ent[k];
  const int64_t c = lin_of[i];
  const uint32_t b = start[c], e = start[c + 1];
  uint32_t r = b;
  for (uint32_t m = b; m < e; ++m)
    r += ent[m] < i ? 1u : 0u;
  for (int d = 0; d < 3; ++d)
    ex[3 * static_cast<int64_t>(r) + d] = x[3 * static_cast<int64_t>(i) + d];
}

__global__ void k_tr_flags(const uint32_t *count, int64_t ncells, uint32_t *flag) {
  const int64_t c = static_cast<int64_t>(blockIdx.x) * kTB + threadIdx.x;
  if (c < ncells)
    flag[c] = count[c] > 0 ? 1u : 0u;
}

// centre of every occupied cell, in cell order (sphere_tracer.hpp:125-132)
// cells are grouped by kGroup^3 for the distance bound of the march
constexpr int kGroup = 4;

__global__ void k_tr_centres(const uint32_t *count, const uint32_t *occ, int64_t ncells,
                             CellBox B, double half, double *centres, uint32_t *gidx) {
  const int64_t c = static_cast<int64_t>(blockIdx.x) * kTB + threadIdx.x;
  if (c >= ncells || count[c] == 0)
    return;
  const int64_t x = c % B.nx, y = (c / B.nx) % B.ny, z = c / (static_cast<int64_t>(B.nx) * B.ny);
  const int64_t cp[3] = {x + B.ox, y + B.oy, z + B.oz};
  const int64_t k0 = occ[c];
  for (int k = 0; k < 3; ++k)
    centres[3 * k0 + k] = B.gd * static_cast<double>(cp[k]) + half;
  const int64_t gx = (B.nx + kGroup - 1) / kGroup, gy = (B.ny + kGroup - 1) / kGroup;
  gidx[k0] = static_cast<uint32_t>(((z / kGroup) * gy + y / kGroup) * gx + x / kGroup);
}

__global__ void k_tr_gcount(const uint32_t *gidx, int64_t nocc, uint32_t *gcount) {
  const int64_t k = static_cast<int64_t>(blockIdx.x) * kTB + threadIdx.x;
  if (k < nocc)
    atomicAdd(&gcount[gidx[k]], 1u);
}

// cell centres grouped (any order inside a group: only their minimum is used)
__global__ void k_tr_gplace(const uint32_t *gidx, const double *centres, int64_t nocc,
                            const uint32_t *gstart, uint32_t *gcursor, double *gcent) {
  const int64_t k = static_cast<int64_t>(blockIdx.x) * kTB + threadIdx.x;
  if (k >= nocc)
    return;
  const uint32_t g = gidx[k];
  const int64_t pos = gstart[g] + atomicAdd(&gcursor[g], 1u);
  for (int d = 0; d < 3; ++d)
    gcent[3 * pos + d] = centres[3 * k + d];
}

// the non-empty groups: box (centre relative to the cell box's origin, half
// extents) containing the boxes of half extent gd around the centres of all
// its cells, and the cell range
__global__ void k_tr_glist(const uint32_t *gcount, const uint32_t *gocc, const uint32_t *gstart,
                           int64_t ng, CellBox B, double half, float *gbox, uint32_t *grange) {
  const int64_t g = static_cast<int64_t>(blockIdx.x) * kTB + threadIdx.x;
  if (g >= ng || gcount[g] == 0)
    return;
  const int64_t gx = (B.nx + kGroup - 1) / kGroup, gy = (B.ny + kGroup - 1) / kGroup;
  const int64_t gc[3] = {g % gx, (g / gx) % gy, g / (gx * gy)};
  const int64_t o[3] = {B.ox, B.oy, B.oz};
  const int64_t j = gocc[g];
  for (int k = 0; k < 3; ++k) {
    const double c0 = static_cast<double>(o[k] + kGroup * gc[k]);
    const double lo = B.gd * c0 + half - B.gd;
    const double hi = B.gd * (c0 + (kGroup - 1)) + half + B.gd;
    gbox[6 * j + k] = static_cast<float>(0.5 * (lo + hi) - B.gd * static_cast<double>(o[k]));
    gbox[6 * j + 3 + k] = static_cast<float>(0.5 * (hi - lo));
  }
  grange[2 * j] = gstart[g];
  grange[2 * j + 1] = gstart[g + 1];
}

// the rounded-box distance of the reference (sphere_tracer.hpp:134-139) to
// the box of centre c and half extents e, minus gd
__device__ inline double box_sdf(const double *x, const double *c, const double *e, double gd) {
  double q[3], qm[3];
  for (int k = 0; k < 3; ++k) {
    q[k] = fabs(x[k] - c[k]) - e[k];
    qm[k] = std_max(q[k], 0.0);
  }
  const double mc = std_max(q[0], std_max(q[1], q[2]));
  return (sqrt(dot3(qm, qm)) + std_min(mc, 0.0)) - gd;
}

// FP32 estimate of box_sdf for a point and a centre relative to the same
// origin; within the march's margin of the exact value
__device__ inline float box_sdf_f32(const float *x, const float *c, const float *e, float gd) {
  const float q0 = fabsf(x[0] - c[0]) - e[0], q1 = fabsf(x[1] - c[1]) - e[1],
              q2 = fabsf(x[2] - c[2]) - e[2];
  const float m0 = fmaxf(q0, 0.0f), m1 = fmaxf(q1, 0.0f), m2 = fmaxf(q2, 0.0f);
  return sqrtf(m0 * m0 + m1 * m1 + m2 * m2) + fminf(fmaxf(q0, fmaxf(q1, q2)), 0.0f) - gd;
}

__device__ inline float wave_min_all(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    v = fminf(v, __shfl_xor(v, o, 64));
  return v;
}

__device__ inline double wave_std_min_all(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    v = std_min(v, __shfl_xor(v, o, 64));
  return v;
}

// orders a wavefront's own LDS writes before its later reads
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// particles listed at once by the march (one more round of 64 may be appended
// before a list that is too long is emptied)
constexpr int kNearCap = 448;
constexpr int kMarchWaves = kTB / 64;

// a / b, correctly rounded, with y = 1 / b correctly rounded: Markstein's
// iteration (IBM J. Res. Dev. 34, 1990), twice, so that the first quotient
// need not be faithful. For operands whose quotient is far from the range's
// ends, as distances over h and kernel sums over h^3 are.
struct Divisor {
  double b, y;
};
__device__ inline double divide(double a, const Divisor &d) {
  double q = a * d.y;
  q = fma(fma(-d.b, q, a), d.y, q);
  return fma(fma(-d.b, q, a), d.y, q);
}

// One wavefront per pixel. A ray of one lane would be a serial chain of up to
// 300 steps, each over every group, the cells of the near ones and up to
// 27 cells of particles, and the slowest ray would decide the time; here
// the 64 lanes share each step's groups, cells and particles. Near the surface
// the bound is divided by the particle count, so a ray that hits takes a
// hundred or more short steps; what bounds the kernel is the FP64 issue of
// those. Per such step:
//  * The particles within reach plus a skin are listed in LDS once, in the
//    reference's order (cells x outermost, then host order), and the list
//    serves every step that stays in the cell and within the skin. Values are
//    computed 64 at a time and subtracted one after the other, in order.
//  * The gradient is summed once, at the last step that summed particles: only
//    there does it reach the image.
//  * sdf = max(cell distance, phi): one cell's distance bounds the minimum over
//    the cells from above, so a phi above it needs no search. The last search's
//    cell gives that bound.
// The minimum over all cells is exact where it is needed: groups and cells are
// filtered by an FP32 distance with a margin of 32 roundings of the largest
// coordinate, and every cell that the filter leaves is evaluated in FP64. The
// minimum does not depend on the order.
// 400 x 300 pixels of 125,000 particles: 80.4 ms with one lane per pixel,
// 26.6 ms with one wavefront and a search, a walk over 27 cells and a gradient
// in every step, 10.3 ms now.
__global__ __launch_bounds__(kTB) void k_tr_march(
    TraceParams P, const float *__restrict__ gbox, const uint32_t *__restrict__ grange,
    const double *__restrict__ gcent, int64_t ngroups, const uint32_t *__restrict__ start,
    const double *__restrict__ ex, CellBox B, double *image, double *par) {
  __shared__ uint32_t s_idx[kMarchWaves][kNearCap + 64];
  __shared__ double s_val[kMarchWaves][4][64];
  const int wv = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const uint64_t below = (1ull << lane) - 1ull;
  uint32_t *idx = s_idx[wv];
  const float gdf = static_cast<float>(P.gd);
  const float ef[3] = {gdf, gdf, gdf};
  const double e3[3] = {P.gd, P.gd, P.gd};
  const double org[3] = {P.gd * B.ox, P.gd * B.oy, P.gd * B.oz};
  const double ext = P.gd * (B.nx > B.ny ? (B.nx > B.nz ? B.nx : B.nz)
                                         : (B.ny > B.nz ? B.ny : B.nz));
  const Divisor by_half{P.half, 1.0 / P.half}, by_h3{P.h3, 1.0 / P.h3}, by_h4{P.h4, 1.0 / P.h4};
  // w > 0 needs r < 2 half: a particle beyond reach + skin has none anywhere
  // within skin of the point that the list was made for
  const double skin = 0.25 * P.half;
  const double reach2 = (2 * P.half + skin) * (2 * P.half + skin) * (1 + 1e-9);
  const double skin2 = skin * skin * (1 - 1e-9);

  for (int64_t pid = static_cast<int64_t>(blockIdx.x) * kMarchWaves + wv;
       pid < P.width * P.height; pid += static_cast<int64_t>(gridDim.x) * kMarchWaves) {
    const int64_t ix = pid % P.width, iy = pid / P.width;

    // pinhole_camera.hpp:53-62
    double d[3];
    {
      const double px = (P.sox + static_cast<double>(ix)) * P.pixel_size;
      const double py = (P.soy + static_cast<double>(iy)) * P.pixel_size;
      double dir0[3];
      for (int k = 0; k < 3; ++k) {
        const double pp = ((P.O[k] + px * P.hh[k]) + py * P.v[k]) - P.f * P.p[k];
        dir0[k] = P.O[k] - pp;
      }
      normalized3(dir0, d);
    }

    double rx[3];           // the ray's point
    int32_t rc[3];          // its cell, where the particles are summed
    double sdf;             // least distance of the cells evaluated so far
    int64_t best_cell = -1; // the cell that gave it
    float xf[3], margin;

    // exact minimum over the cells [c0, c1) that the filter leaves into sdf
    // (a comparison with NaN leaves a cell in)
    auto group_cells = [&](uint32_t c0, uint32_t c1) {
      for (uint32_t c = c0; c < c1; c += 64) {
        const bool in = c + lane < c1;
        const double *cp = gcent + 3 * static_cast<int64_t>(in ? c + lane : c0);
        const double cc[3] = {cp[0], cp[1], cp[2]};
        const float cf[3] = {static_cast<float>(cc[0] - org[0]),
                             static_cast<float>(cc[1] - org[1]),
                             static_cast<float>(cc[2] - org[2])};
        const float lb = box_sdf_f32(xf, cf, ef, gdf);
        float bound = wave_min_all(in ? lb : 3.0e38f);
        bound = fminf(bound, static_cast<float>(sdf)) + 2.0f * margin;
        const bool keep = in && !(lb > bound);
        if (__ballot(keep) == 0ull)
          continue;
        double v = DBL_MAX;
        if (keep)
          v = std_min(v, box_sdf(rx, cc, e3, P.gd));
        const double m = wave_std_min_all(v);
        if (m < sdf) {
          sdf = m;
          best_cell = c + __ffsll(static_cast<long long>(__ballot(v == m))) - 1;
        }
      }
    };
    // the minimum over every occupied cell
    auto search = [&]() {
      double far = 0;
      for (int k = 0; k < 3; ++k) {
        xf[k] = static_cast<float>(rx[k] - org[k]);
        far = fmax(far, fabs(rx[k] - org[k]));
      }
      // 32 roundings of the largest term of either distance
      margin = 2e-6f * static_cast<float>(far + ext + P.gd);
      sdf = DBL_MAX;
      best_cell = -1;
      if (ngroups <= 0)
        return;
      // the group with the smallest estimate first
      float best = 3.0e38f;
      int64_t at = -1;
      for (int64_t g0 = 0; g0 < ngroups; g0 += 64) {
        const int64_t g = g0 + lane;
        const float lb =
            g < ngroups ? box_sdf_f32(xf, gbox + 6 * g, gbox + 6 * g + 3, gdf) : 3.0e38f;
        if (g < ngroups && (lb < best || at < 0)) {
          best = lb;
          at = g;
        }
      }
      const float m = wave_min_all(best);
      const uint64_t who = __ballot(at >= 0 && best == m);
      // NaN estimates (a ray point that is not finite): any group
      const int64_t first = __shfl(at, who ? __ffsll(static_cast<long long>(who)) - 1 : 0, 64);
      group_cells(grange[2 * first], grange[2 * first + 1]);
      for (int64_t g0 = 0; g0 < ngroups; g0 += 64) {
        const int64_t g = g0 + lane;
        const bool in = g < ngroups && g != first;
        const float lb =
            in ? box_sdf_f32(xf, gbox + 6 * g, gbox + 6 * g + 3, gdf) : 3.0e38f;
        uint64_t left = __ballot(in && !(lb > static_cast<float>(sdf) + 2.0f * margin));
        while (left) {
          const int l = __ffsll(static_cast<long long>(left)) - 1;
          left &= left - 1;
          // the bound may have come down since the ballot
          if (__shfl(lb, l, 64) > static_cast<float>(sdf) + 2.0f * margin)
            continue;
          group_cells(grange[2 * (g0 + l)], grange[2 * (g0 + l) + 1]);
        }
      }
    };

    int n = 0;                 // listed particles
    bool listed = false;       // the list serves the cell lc around lx
    int32_t lc[3] = {0, 0, 0};
    double lx[3] = {0, 0, 0};
    double acc[4];             // phi, and minus the gradient's sum
    int64_t count = 0;
    // subtracts the values of the listed particles in list order
    auto sum_list = [&](auto grad_tag) {
      constexpr bool kGrad = decltype(grad_tag)::value;
      constexpr int kVals = kGrad ? 4 : 1;
      wave_lds_sync();
      for (int m = 0; m < n; m += 64) {
        double w = 0, g[3] = {0, 0, 0};
        if (m + lane < n) {
          const double *xp = ex + 3 * static_cast<int64_t>(idx[m + lane]);
          double dv[3];
          for (int k = 0; k < 3; ++k)
            dv[k] = rx[k] - xp[k];
          const double r = sqrt(dot3(dv, dv));
          const double q = divide(fabs(r), by_half);
          w = divide(evalq(P.alpha, q), by_h3);
          if (kGrad && w > 0 && !(r < P.grad_eps)) {
            const double dr = -copysign(divide(evaldq(P.alpha, q), by_h4), r);
            const double s = dr / r;
            for (int k = 0; k < 3; ++k)
              g[k] = s * dv[k];
          }
        }
        const uint64_t hit = __ballot(w > 0);
        const int nh = __popcll(hit);
        if (w > 0) {
          const int at = __popcll(hit & below);
          s_val[wv][0][at] = w;
          if (kGrad)
            for (int k = 0; k < 3; ++k)
              s_val[wv][1 + k][at] = g[k];
        }
        wave_lds_sync();
        for (int k = 0; k < nh; ++k)
          for (int v = 0; v < kVals; ++v)
            acc[v] -= s_val[wv][v][k];
        count += nh;
        wave_lds_sync();
      }
    };
    // phi and the particle count (kGrad: the gradient too) at rx
    auto sum_particles = [&](auto grad_tag) {
      acc[0] = P.phi0;
      acc[1] = acc[2] = acc[3] = 0;
      count = 0;
      if (listed && rc[0] == lc[0] && rc[1] == lc[1] && rc[2] == lc[2]) {
        double m[3];
        for (int k = 0; k < 3; ++k)
          m[k] = rx[k] - lx[k];
        if (dot3(m, m) <= skin2) {
          sum_list(grad_tag);
          return;
        }
      }
      for (int k = 0; k < 3; ++k) {
        lc[k] = rc[k];
        lx[k] = rx[k];
      }
      listed = true;
      n = 0;
      // lane c < 27: the entries of cell c of the stencil
      uint32_t cb = 0, ce = 0;
      if (lane < 27) {
        int64_t lin;
        if (cell_index(B, rc[0] + lane / 9 - 1, rc[1] + lane / 3 % 3 - 1, rc[2] + lane % 3 - 1,
                       &lin)) {
          cb = start[lin];
          ce = start[lin + 1];
        }
      }
      uint64_t cells = __ballot(ce > cb);
      while (cells) {
        const int c = __ffsll(static_cast<long long>(cells)) - 1;
        cells &= cells - 1;
        const uint32_t b = __shfl(cb, c, 64), e = __shfl(ce, c, 64);
        for (uint32_t p0 = b; p0 < e; p0 += 64) {
          const uint32_t p = p0 + lane;
          bool ok = false;
          if (p < e) {
            const double *xp = ex + 3 * static_cast<int64_t>(p);
            double dv[3];
            for (int k = 0; k < 3; ++k)
              dv[k] = rx[k] - xp[k];
            ok = !(dot3(dv, dv) > reach2);
          }
          const uint64_t hit = __ballot(ok);
          if (ok)
            idx[n + __popcll(hit & below)] = p;
          n += __popcll(hit);
          if (n > kNearCap) {  // crowded: summed as it goes, not kept
            sum_list(grad_tag);
            n = 0;
            listed = false;
          }
        }
      }
      sum_list(grad_tag);
    };

    double t = 0, t_sum = -1;  // t_sum: the last step that summed particles
    bool done = false;         // broke out of the march
    for (int64_t step = 0; step < P.max_steps && !done; ++step) {
      for (int k = 0; k < 3; ++k)
        rx[k] = P.O[k] + t * d[k];
      bool exact = false;
      if (best_cell >= 0) {
        const double *cp = gcent + 3 * best_cell;
        const double cc[3] = {cp[0], cp[1], cp[2]};
        sdf = box_sdf(rx, cc, e3, P.gd);
      }
      if (best_cell < 0 || !(sdf < P.gd)) {
        search();
        exact = true;
      }
      if (sdf < P.gd) {
        for (int k = 0; k < 3; ++k)
          rc[k] = static_cast<int32_t>(floor(rx[k] / P.gd));
        sum_particles(std::false_type{});
        double phi = P.gd / 4;
        if (count > 0) {
          phi = acc[0] / (P.L * static_cast<double>(count));
          t_sum = t;
        }
        if (!exact && !(sdf <= phi))
          search();
        sdf = std_max(sdf, phi);
      }
      if (sdf < 1e-6) {
        done = true;
        break;
      }
      t += sdf;
      if (t >= P.max_parameter)
        done = true;
    }
    if (!done)
      t = P.max_parameter;  // ran out of steps
    double pix;
    if (t == P.max_parameter) {
      pix = 0;
    } else if (t > P.max_parameter) {
      pix = 0.3;
    } else {
      double normal[3] = {0, 0, 0};
      if (t_sum >= 0) {
        for (int k = 0; k < 3; ++k) {
          rx[k] = P.O[k] + t_sum * d[k];
          rc[k] = static_cast<int32_t>(floor(rx[k] / P.gd));
        }
        sum_particles(std::true_type{});
        const double s = P.L * static_cast<double>(count);
        for (int k = 0; k < 3; ++k)
          normal[k] = acc[1 + k] / s;
      }
      double dn[3], nn[3];
      normalized3(d, dn);
      normalized3(normal, nn);
      pix = -dot3(dn, nn);
    }
    if (lane == 0) {
      image[pid] = pix;
      if (par)
        par[pid] = t;
    }
  }
}

struct Dev {
  void *p = nullptr;
  explicit Dev(size_t bytes) { PRTCL_HIP_CHECK(hipMalloc(&p, bytes < 64 ? 64 : bytes)); }
  ~Dev() { (void)hipFree(p); }
  template <class U>
  U *as() const {
    return static_cast<U *>(p);
  }
};

unsigned blocks(int64_t n) { return static_cast<unsigned>((n + kTB - 1) / kTB); }

void scan_u32(hipStream_t st, const uint32_t *in, int64_t n, uint32_t *out) {
  // out has n + 1 entries; out[n] = total
  const int64_t nb = blocks(n + 1);
  Dev bsum(sizeof(uint32_t) * static_cast<size_t>(nb + 1));
  hipLaunchKernelGGL(k_tr_scan_tiles, dim3(static_cast<unsigned>(nb)), dim3(kTB), 0, st, in, n,
                     out, bsum.as<uint32_t>());
  hipLaunchKernelGGL(k_tr_scan_top, dim3(1), dim3(kTB), 0, st, bsum.as<uint32_t>(), nb);
  hipLaunchKernelGGL(k_tr_scan_add, dim3(static_cast<unsigned>(nb)), dim3(kTB), 0, st, out, n,
                     bsum.as<uint32_t>());
  PRTCL_HIP_CHECK(hipGetLastError());
  PRTCL_HIP_CHECK(hipStreamSynchronize(st));  // bsum is freed on return
}

}  // namespace

void trace_scene(SceneBase &sc, CtxResources &res, int group, const prtcl_hip_camera &cam,
                 double threshold, int32_t max_steps, double *image, double *parameter) {
  if (group != PRTCL_HIP_FLUID && group != PRTCL_HIP_BOUNDARY)
    throw std::invalid_argument("group must be PRTCL_HIP_FLUID or PRTCL_HIP_BOUNDARY");
  if (cam.width <= 0 || cam.height <= 0 || cam.width > (1 << 16) || cam.height > (1 << 16))
    throw std::invalid_argument("sensor width and height must be in 1..65536");
  if (max_steps < 0)
    throw std::invalid_argument("max_steps must not be negative");
  sc.ensure_resident();
  const prtcl_hip_scene_desc &d = sc.desc;
  hipStream_t st = res.stream;
  const int64_t n = group == PRTCL_HIP_FLUID ? d.n_fluid : d.n_boundary;

  TraceParams P{};
  // the model's smoothing_scale is a global of the scene's real type
  const double h = d.real_type == 1 ? d.smoothing_scale
                                    : static_cast<double>(static_cast<float>(d.smoothing_scale));
  P.gd = 4 * h;
  P.half = P.gd / 2;
  P.alpha = static_cast<double>(1.L / 4.L * (1.L / 3.141592653589793238462643383279502884L));
  P.h3 = cpow(P.half, 3);
  P.h4 = cpow(P.half, 4);
  P.phi0 = threshold * (evalq(P.alpha, std::abs(0.0) / P.half) / P.h3);
  P.L = -evaldq(P.alpha, 2.0 / 3.0) / P.h4;
  P.grad_eps = std::sqrt(std::numeric_limits<double>::epsilon());
  P.max_parameter = P.gd * 10000;
  P.width = cam.width;
  P.height = cam.height;
  P.max_steps = max_steps;
  // pinhole_camera.hpp:35-47
  normalized3(cam.up, P.v);
  normalized3(cam.principal, P.p);
  const double vp[3] = {P.v[1] * P.p[2] - P.v[2] * P.p[1], P.v[2] * P.p[0] - P.v[0] * P.p[2],
                        P.v[0] * P.p[1] - P.v[1] * P.p[0]};
  normalized3(vp, P.hh);
  P.pixel_size = 1.0 / static_cast<double>(cam.width);
  P.sox = -static_cast<double>(cam.width - 1) / 2;
  P.soy = -static_cast<double>(cam.height - 1) / 2;
  for (int k = 0; k < 3; ++k)
    P.O[k] = cam.origin[k];
  P.f = cam.focal_length;

  // positions in host order, as double
  const int64_t n3 = 3 * n;
  Dev x(sizeof(double) * static_cast<size_t>(n3));
  PRTCL_HIP_CHECK(hipStreamSynchronize(st));
  if (n > 0) {
    Dev raw(sizeof(double) * static_cast<size_t>(n3));
    sc.gather_device(group, PRTCL_HIP_F_POSITION, raw.p, static_cast<size_t>(n3));
    if (d.real_type == 1)
      hipLaunchKernelGGL(k_tr_to_double<double>, dim3(blocks(n3)), dim3(kTB), 0, st,
                         raw.as<const double>(), x.as<double>(), n3);
    else
      hipLaunchKernelGGL(k_tr_to_double<float>, dim3(blocks(n3)), dim3(kTB), 0, st,
                         raw.as<const float>(), x.as<double>(), n3);
    PRTCL_HIP_CHECK(hipGetLastError());
    PRTCL_HIP_CHECK(hipStreamSynchronize(st));
  }

  // the dense box of cells around the particles (one empty cell of margin)
  CellBox B{0, 0, 0, 1, 1, 1, P.gd};
  if (n > 0) {
    const int64_t nb = blocks(n);
    Dev part(sizeof(double) * 6 * static_cast<size_t>(nb));
    hipLaunchKernelGGL(k_tr_bbox, dim3(static_cast<unsigned>(nb)), dim3(kTB), 0, st,
                       x.as<const double>(), n, part.as<double>());
    std::vector<double> hp(6 * static_cast<size_t>(nb));
    PRTCL_HIP_CHECK(hipMemcpyAsync(hp.data(), part.p, sizeof(double) * hp.size(),
                                   hipMemcpyDeviceToHost, st));
    PRTCL_HIP_CHECK(hipStreamSynchronize(st));
    double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    for (int64_t b = 0; b < nb; ++b)
      for (int k = 0; k < 3; ++k) {
        lo[k] = std::min(lo[k], hp[6 * b + k]);
        hi[k] = std::max(hi[k], hp[6 * b + 3 + k]);
      }
    int32_t o[3], e[3];
    for (int k = 0; k < 3; ++k) {
      if (!(lo[k] <= hi[k]) || !std::isfinite(lo[k]) || !std::isfinite(hi[k])) {
        lo[k] = hi[k] = 0;  // no finite position: an empty box
      }
      const double a = std::floor(lo[k] / P.gd) - 1, b = std::floor(hi[k] / P.gd) + 1;
      if (a < -1e9 || b > 1e9 || b - a + 1 > 4096)
        throw std::invalid_argument("trace: the particles span more than 4096 cells per axis");
      o[k] = static_cast<int32_t>(a);
      e[k] = static_cast<int32_t>(b - a + 1);
    }
    if (static_cast<int64_t>(e[0]) * e[1] * e[2] > (int64_t(1) << 28))
      throw std::invalid_argument("trace: more than 2^28 cells around the particles");
    B = CellBox{o[0], o[1], o[2], e[0], e[1], e[2], P.gd};
  }
  const int64_t ncells = static_cast<int64_t>(B.nx) * B.ny * B.nz;

  Dev count(sizeof(uint32_t) * static_cast<size_t>(ncells + 1));
  Dev cursor(sizeof(uint32_t) * static_cast<size_t>(ncells + 1));
  Dev startb(sizeof(uint32_t) * static_cast<size_t>(ncells + 1));
  Dev occ(sizeof(uint32_t) * static_cast<size_t>(ncells + 1));
  Dev flag(sizeof(uint32_t) * static_cast<size_t>(ncells + 1));
  Dev lin_of(sizeof(int64_t) * static_cast<size_t>(n > 0 ? n : 1));
  Dev ent(sizeof(uint32_t) * static_cast<size_t>(n > 0 ? n : 1));
  Dev ex(sizeof(double) * static_cast<size_t>(n3 > 0 ? n3 : 1));
  PRTCL_HIP_CHECK(hipMemsetAsync(count.p, 0, sizeof(uint32_t) * (ncells + 1), st));
  PRTCL_HIP_CHECK(hipMemsetAsync(cursor.p, 0, sizeof(uint32_t) * (ncells + 1), st));
  if (n > 0)
    hipLaunchKernelGGL(k_tr_count, dim3(blocks(n)), dim3(kTB), 0, st, x.as<const double>(), n,
                       B, count.as<uint32_t>(), lin_of.as<int64_t>());
  PRTCL_HIP_CHECK(hipGetLastError());
  scan_u32(st, count.as<const uint32_t>(), ncells, startb.as<uint32_t>());
  uint32_t placed = 0;
  PRTCL_HIP_CHECK(hipMemcpyAsync(&placed, startb.as<uint32_t>() + ncells, sizeof(placed),
                                 hipMemcpyDeviceToHost, st));
  PRTCL_HIP_CHECK(hipStreamSynchronize(st));
  if (placed > 0) {
    hipLaunchKernelGGL(k_tr_place, dim3(blocks(n)), dim3(kTB), 0, st, lin_of.as<const int64_t>(),
                       n, startb.as<const uint32_t>(), cursor.as<uint32_t>(), ent.as<uint32_t>());
    hipLaunchKernelGGL(k_tr_pack, dim3(blocks(placed)), dim3(kTB), 0, st, x.as<const double>(),
                       lin_of.as<const int64_t>(), startb.as<const uint32_t>(),
                       ent.as<const uint32_t>(), static_cast<int64_t>(placed), ex.as<double>());
  }
  hipLaunchKernelGGL(k_tr_flags, dim3(blocks(ncells)), dim3(kTB), 0, st,
                     count.as<const uint32_t>(), ncells, flag.as<uint32_t>());
  PRTCL_HIP_CHECK(hipGetLastError());
  scan_u32(st, flag.as<const uint32_t>(), ncells, occ.as<uint32_t>());
  uint32_t nocc = 0;
  PRTCL_HIP_CHECK(hipMemcpyAsync(&nocc, occ.as<uint32_t>() + ncells, sizeof(nocc),
                                 hipMemcpyDeviceToHost, st));
  PRTCL_HIP_CHECK(hipStreamSynchronize(st));
  Dev centres(sizeof(double) * 3 * static_cast<size_t>(nocc > 0 ? nocc : 1));
  Dev gidx(sizeof(uint32_t) * static_cast<size_t>(nocc > 0 ? nocc : 1));
  hipLaunchKernelGGL(k_tr_centres, dim3(blocks(ncells)), dim3(kTB), 0, st,
                     count.as<const uint32_t>(), occ.as<const uint32_t>(), ncells, B, P.half,
                     centres.as<double>(), gidx.as<uint32_t>());
  // groups of kGroup^3 cells
  const int64_t ng = ((B.nx + kGroup - 1) / kGroup) * ((B.ny + kGroup - 1) / kGroup) *
                     ((B.nz + kGroup - 1) / kGroup);
  Dev gcount(sizeof(uint32_t) * static_cast<size_t>(ng + 1));
  Dev gcursor(sizeof(uint32_t) * static_cast<size_t>(ng + 1));
  Dev gstart(sizeof(uint32_t) * static_cast<size_t>(ng + 1));
  Dev gflag(sizeof(uint32_t) * static_cast<size_t>(ng + 1));
  Dev gocc(sizeof(uint32_t) * static_cast<size_t>(ng + 1));
  PRTCL_HIP_CHECK(hipMemsetAsync(gcount.p, 0, sizeof(uint32_t) * (ng + 1), st));
  PRTCL_HIP_CHECK(hipMemsetAsync(gcursor.p, 0, sizeof(uint32_t) * (ng + 1), st));
  if (nocc > 0)
    hipLaunchKernelGGL(k_tr_gcount, dim3(blocks(nocc)), dim3(kTB), 0, st,
                       gidx.as<const uint32_t>(), static_cast<int64_t>(nocc),
                       gcount.as<uint32_t>());
  PRTCL_HIP_CHECK(hipGetLastError());
  scan_u32(st, gcount.as<const uint32_t>(), ng, gstart.as<uint32_t>());
  Dev gcent(sizeof(double) * 3 * static_cast<size_t>(nocc > 0 ? nocc : 1));
  if (nocc > 0)
    hipLaunchKernelGGL(k_tr_gplace, dim3(blocks(nocc)), dim3(kTB), 0, st,
                       gidx.as<const uint32_t>(), centres.as<const double>(),
                       static_cast<int64_t>(nocc), gstart.as<const uint32_t>(),
                       gcursor.as<uint32_t>(), gcent.as<double>());
  hipLaunchKernelGGL(k_tr_flags, dim3(blocks(ng)), dim3(kTB), 0, st, gcount.as<const uint32_t>(),
                     ng, gflag.as<uint32_t>());
  PRTCL_HIP_CHECK(hipGetLastError());
  scan_u32(st, gflag.as<const uint32_t>(), ng, gocc.as<uint32_t>());
  uint32_t ngroups = 0;
  PRTCL_HIP_CHECK(hipMemcpyAsync(&ngroups, gocc.as<uint32_t>() + ng, sizeof(ngroups),
                                 hipMemcpyDeviceToHost, st));
  PRTCL_HIP_CHECK(hipStreamSynchronize(st));
  Dev gbox(sizeof(float) * 6 * static_cast<size_t>(ngroups > 0 ? ngroups : 1));
  Dev grange(sizeof(uint32_t) * 2 * static_cast<size_t>(ngroups > 0 ? ngroups : 1));
  hipLaunchKernelGGL(k_tr_glist, dim3(blocks(ng)), dim3(kTB), 0, st, gcount.as<const uint32_t>(),
                     gocc.as<const uint32_t>(), gstart.as<const uint32_t>(), ng, B, P.half,
                     gbox.as<float>(), grange.as<uint32_t>());

  const int64_t npx = cam.width * cam.height;
  Dev img(sizeof(double) * static_cast<size_t>(npx));
  Dev par(sizeof(double) * static_cast<size_t>(npx));
  // large sensors: each wavefront takes several pixels (2^32 threads at most)
  const int64_t mb = std::min<int64_t>((npx + kMarchWaves - 1) / kMarchWaves, int64_t(1) << 22);
  hipLaunchKernelGGL(k_tr_march, dim3(static_cast<unsigned>(mb)), dim3(kTB), 0, st, P,
                     gbox.as<const float>(), grange.as<const uint32_t>(),
                     gcent.as<const double>(), static_cast<int64_t>(ngroups),
                     startb.as<const uint32_t>(), ex.as<const double>(), B, img.as<double>(),
                     par.as<double>());
  PRTCL_HIP_CHECK(hipGetLastError());
  PRTCL_HIP_CHECK(hipMemcpyAsync(image, img.p, sizeof(double) * npx, hipMemcpyDeviceToHost, st));
  if (parameter)
    PRTCL_HIP_CHECK(hipMemcpyAsync(parameter, par.p, sizeof(double) * npx,
                                   hipMemcpyDeviceToHost, st));
  PRTCL_HIP_CHECK(hipStreamSynchronize(st));
}

}  // namespace prtcl_amd
