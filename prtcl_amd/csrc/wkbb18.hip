// WKBB18 implicit viscosity (Weiler et al. 2018) on the device: the 3x3
// block-diagonal system matrix and its inverse (wkbb18.hpp:194-270) and the
// preconditioned CG of cg_openmp.hpp:32-215 with the matrix-free product of
// wkbb18.hpp:342-390.
//
// Two product kernels share the CG engine:
//   * exact: walks the 27-cell grid with the reference predicate and
//     evaluates every pair term in the reference's FP32 operation order
//     (used by the wkbb18.* procedures);
//   * list: walks the step's fluid neighbour list with fused arithmetic and
//     applies the boundary part as a precomputed symmetric 3x3 matrix per
//     particle, B_i = sum_b k_ib gradW_ib x_ib^T (used by prtcl_hip_step).
// The CG scalars (dot products, alpha, beta, thresholds) are FP64 on the
// device; vectors are the scene's real type. The iteration logic follows the
// reference exactly: r = A x - b, p0 = -y0, break on |p.q| < tol and on
// |r.y|_prev < tol (absolute), stop when |r|^2 < max(tol^2 |b|^2, FLT_MIN),
// at most max_k + 1 iterations, the returned count is the loop counter.
#include "wkbb18.hpp"
#include "cg_ctl.hpp"
#include "exact_walk.hpp"
#include "scan8.hpp"

namespace prtcl_amd {

namespace {

template <class T>
__device__ __forceinline__ T cof3(const T *m, int i, int j) {
#pragma clang fp contract(off)
  const int i1 = (i + 1) % 3, i2 = (i + 2) % 3, j1 = (j + 1) % 3, j2 = (j + 2) % 3;
  return m[i1 + 3 * j1] * m[i2 + 3 * j2] - m[i1 + 3 * j2] * m[i2 + 3 * j1];
}

// inverse by adjugate / determinant, column-major (element (r,c) at r + 3c)
template <class T>
__device__ __forceinline__ void invert3(const T *m, T *out) {
#pragma clang fp contract(off)
  const T c00 = cof3(m, 0, 0), c10 = cof3(m, 1, 0), c20 = cof3(m, 2, 0);
  const T det = c00 * m[0] + (c10 * m[1] + c20 * m[2]);
  const T invdet = T(1) / det;
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c)
      out[r + 3 * c] = cof3(m, c, r) * invdet;
}

template <class T>
__device__ __forceinline__ T step_l(T eps, T x) {
  return (eps < x) ? T(1) : T(0);
}

template <class T>
struct RealEps;
template <>
struct RealEps<float> {
  static constexpr double value = 1.1920928955078125e-07;  // 2^-23
};
template <>
struct RealEps<double> {
  static constexpr double value = 2.220446049250313e-16;  // 2^-52
};

// Moore-Penrose pseudo-inverse of a 3x3 matrix m (column-major) into out, as
// invert_pm (eigen.hpp:266-276). The reference takes it from Eigen's complete
// orthogonal decomposition, whose rank counts the pivots above 3 eps of the
// largest; here a one-sided Jacobi SVD in FP64 (Hestenes rotations of the
// column pairs until they are orthogonal to working precision, at most 12
// sweeps) gives A V = B with orthogonal columns b_k = sigma_k u_k, and
// pinv(A) = sum over sigma_k > 3 eps sigma_max of v_k b_k^T / sigma_k^2.
//
// Fast path: sigma_min / sigma_max >= |det| / sigma_max^3 >= |det| / |A|_F^3,
// so |det| > 2 (3 eps) |A|_F^3 proves the matrix full rank under the
// threshold, and then the pseudo-inverse is the inverse (adjugate / det in
// FP64). Only the other matrices take the SVD.
template <class T>
__device__ void pinv3(const T *m, T *out) {
  double b[9], v[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
#pragma unroll
  for (int k = 0; k < 9; ++k)
    b[k] = static_cast<double>(m[k]);
  {
    double cof[9], fro2 = 0;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const int r1 = (r + 1) % 3, r2 = (r + 2) % 3, c1 = (c + 1) % 3, c2 = (c + 2) % 3;
        cof[r + 3 * c] = b[r1 + 3 * c1] * b[r2 + 3 * c2] - b[r1 + 3 * c2] * b[r2 + 3 * c1];
        fro2 += b[r + 3 * c] * b[r + 3 * c];
      }
    const double det = b[0] * cof[0] + b[1] * cof[1] + b[2] * cof[2];
    if (fabs(det) > 6.0 * RealEps<T>::value * fro2 * sqrt(fro2)) {
      const double id = 1.0 / det;
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int r = 0; r < 3; ++r)
          out[r + 3 * c] = static_cast<T>(cof[c + 3 * r] * id);  // adj(r, c) = cof(c, r)
      return;
    }
  }
  for (int sweep = 0; sweep < 12; ++sweep) {
    bool rotated = false;
#pragma unroll
    for (int pq = 0; pq < 3; ++pq) {
      const int p = pq == 2 ? 1 : 0, q = pq == 0 ? 1 : 2;
      double al = 0, be = 0, ga = 0;
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        al += b[r + 3 * p] * b[r + 3 * p];
        be += b[r + 3 * q] * b[r + 3 * q];
        ga += b[r + 3 * p] * b[r + 3 * q];
      }
      if (!(fabs(ga) > 1e-17 * sqrt(al * be)))
        continue;
      rotated = true;
      const double zeta = (be - al) / (2.0 * ga);
      const double t = copysign(1.0, zeta) / (fabs(zeta) + sqrt(1.0 + zeta * zeta));
      const double c = 1.0 / sqrt(1.0 + t * t), sn = c * t;
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const double bp = b[r + 3 * p], bq = b[r + 3 * q];
        b[r + 3 * p] = c * bp - sn * bq;
        b[r + 3 * q] = sn * bp + c * bq;
        const double vp = v[r + 3 * p], vq = v[r + 3 * q];
        v[r + 3 * p] = c * vp - sn * vq;
        v[r + 3 * q] = sn * vp + c * vq;
      }
    }
    if (!rotated)
      break;
  }
  double s2[3], smax2 = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    s2[k] = b[3 * k] * b[3 * k] + b[3 * k + 1] * b[3 * k + 1] + b[3 * k + 2] * b[3 * k + 2];
    smax2 = s2[k] > smax2 ? s2[k] : smax2;
  }
  const double thr = 3.0 * RealEps<T>::value;
  const double thr2 = thr * thr * smax2;
  double inv[3];
#pragma unroll
  for (int k = 0; k < 3; ++k)
    inv[k] = (s2[k] > thr2 && s2[k] > 0.0) ? 1.0 / s2[k] : 0.0;
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int r = 0; r < 3; ++r)
      out[r + 3 * c] = static_cast<T>(v[r] * b[c] * inv[0] + v[r + 3] * b[c + 3] * inv[1] +
                                      v[r + 6] * b[c + 6] * inv[2]);
}

// ---- correction.identity_gradient_correction (correction.hpp:133-158)
template <class T>
__global__ __launch_bounds__(kBlock) void k_corr_identity(SceneView<T> S) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= S.nf)
    return;
  T *L = S.gc + 9 * static_cast<size_t>(i);
#pragma unroll
  for (int k = 0; k < 9; ++k)
    L[k] = (k % 4 == 0) ? T(1) : T(0);
}

// ---- correction.compute_gradient_correction (correction.hpp:161-217):
// L_i = pinv(sum_f (m_j / rho_i) gradW_ij (x_j - x_i)^T), exact walk in the
// reference's FP32 operation order, or over the step's neighbour list
template <class T, bool kList, int kLanes>
__device__ __forceinline__ void corr_body(const SceneView<T> &S, const NbrList &L,
                                          unsigned lb) {
#pragma clang fp contract(off)
  const int i = static_cast<int>((lb * kBlock + threadIdx.x) / kLanes);
  const uint32_t sub = threadIdx.x % kLanes;
  const bool valid = i < S.nf;
  T M[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (valid) {
    const vec4_t<T> xi = S.xm[i];
    const T rhoi = S.rho[i];
    auto add = [&](const vec4_t<T> &pj, T f, T d0, T d1, T d2) {
      const T g[3] = {f * d0, f * d1, f * d2};
      const T e[3] = {pj.x - xi.x, pj.y - xi.y, pj.z - xi.z};
      const T k = pj.w / rhoi;
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int r = 0; r < 3; ++r)
          M[r + 3 * c] += k * (g[r] * e[c]);
    };
    const uint32_t info = kList ? L.info[i] : kListOverflow;
    if (kList && !(info & kListOverflow)) {
      list_gather_lanes<kLanes, 8>(
          L, pass_spans<kLanes>(L, S.nf, lb), static_cast<size_t>(S.nf), i, info, sub,
          [&](uint32_t j) { return S.xm[j]; },
          [&](const vec4_t<T> &pj) {
            const T d0 = xi.x - pj.x, d1 = xi.y - pj.y, d2 = xi.z - pj.z;
            add(pj, S.K.gradf(sqdist_exact(d0, d1, d2)), d0, d1, d2);
          });
    } else if (sub == 0) {
      nbrs_exact(S, xi, S.fcell[i], S.fstart, S.xm,
                 [&](uint32_t, T d0, T d1, T d2, T r2, const vec4_t<T> &pj) {
                   add(pj, S.K.gradf(r2), d0, d1, d2);
                 });
    }
  }
#pragma unroll
  for (int k = 0; k < 9; ++k)
    M[k] = lanes_sum<kLanes>(M[k]);
  if (valid && sub == 0)
    pinv3(M, S.gc + 9 * static_cast<size_t>(i));
}

template <class T, bool kList, int kLanes>
__global__ __launch_bounds__(kBlock) void k_corr(SceneView<T> S, NbrList L) {
  corr_body<T, kList, kLanes>(S, L, xcd_block(blockIdx.x, gridDim.x));
}

// L_i g with Eigen's fixed-size product order per row: l0 g0 + (l1 g1 + l2 g2)
template <class T>
__device__ __forceinline__ void apply_gc(const T *L, const T g[3], T out[3]) {
#pragma clang fp contract(off)
#pragma unroll
  for (int r = 0; r < 3; ++r)
    out[r] = L[r] * g[0] + (L[r + 3] * g[1] + L[r + 6] * g[2]);
}

// ---- wkbb18.compute_diagonal, exact (wkbb18.hpp:194-270); with kGC the
// gradient is L_i gradW (wkbb18_gc.hpp:236-262)
template <class T, bool kGC>
__global__ __launch_bounds__(kBlock) void k_diag_exact(SceneView<T> S) {
#pragma clang fp contract(off)
  const unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const int i = static_cast<int>(lb * kBlock + threadIdx.x);
  if (i >= S.nf)
    return;
  const vec4_t<T> xi = S.xm[i];
  const T rhoi = S.rho[i];
  const uint32_t cell = S.fcell[i];
  T Li[9];
  if (kGC) {
#pragma unroll
    for (int k = 0; k < 9; ++k)
      Li[k] = S.gc[9 * static_cast<size_t>(i) + k];
  }
  auto grad = [&](T f, T d0, T d1, T d2, T g[3]) {
    const T g0[3] = {f * d0, f * d1, f * d2};
    if (kGC) {
      apply_gc(Li, g0, g);
    } else {
      g[0] = g0[0];
      g[1] = g0[1];
      g[2] = g0[2];
    }
  };
  T D[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  nbrs_exact(S, xi, cell, S.fstart, S.xm, [&](uint32_t j, T d0, T d1, T d2, T r2,
                                                const vec4_t<T> &pj) {
    const T f = S.K.gradf(r2);
    T g[3];
    grad(f, d0, d1, d2, g);
    const T d[3] = {d0, d1, d2};
    const T k = ((T(10) * (S.mu_f / rhoi)) * (pj.w / S.rho[j])) / (r2 + S.hh001);
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int r = 0; r < 3; ++r)
        D[r + 3 * c] += k * (g[r] * d[c]);
  });
  nbrs_exact(S, xi, cell, S.bstart, S.bxV, [&](uint32_t, T d0, T d1, T d2, T r2,
                                                 const vec4_t<T> &pj) {
    const T f = S.K.gradf(r2);
    T g[3];
    grad(f, d0, d1, d2, g);
    const T d[3] = {d0, d1, d2};
    const T k = ((T(10) * (S.mu_b / rhoi)) * ((S.rho0 * pj.w) / rhoi)) / (r2 + S.hh001);
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int r = 0; r < 3; ++r)
        D[r + 3 * c] += k * (g[r] * d[c]);
  });
  T M[9];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int r = 0; r < 3; ++r)
      M[r + 3 * c] = ((r == c) ? T(1) : T(0)) - S.dt * D[r + 3 * c];
  invert3(M, S.sp + 9 * static_cast<size_t>(i));
}

// ---- product_s, exact (wkbb18.hpp:342-390): out = w - dt * l(w); with kGC
// every term is (s L_i) gradW (wkbb18_gc.hpp:362-390)
template <class T, bool kGC>
__device__ __forceinline__ void product_exact(const SceneView<T> &S, int i,
                                              const vec4_t<T> *__restrict__ w, int ws,
                                              T out[3]) {
#pragma clang fp contract(off)
  const vec4_t<T> xi = S.xm[i];
  const vec4_t<T> wi = w[static_cast<size_t>(ws) * i];
  const T rhoi = S.rho[i];
  const uint32_t cell = S.fcell[i];
  T l0 = 0, l1 = 0, l2 = 0;
  T Li[9];
  if (kGC) {
#pragma unroll
    for (int k = 0; k < 9; ++k)
      Li[k] = S.gc[9 * static_cast<size_t>(i) + k];
  }
  auto acc = [&](T s, T f, T d0, T d1, T d2) {
    if (kGC) {
      const T g[3] = {f * d0, f * d1, f * d2};
      T sl[9];
#pragma unroll
      for (int k = 0; k < 9; ++k)
        sl[k] = s * Li[k];
      T t[3];
      apply_gc(sl, g, t);
      l0 += t[0];
      l1 += t[1];
      l2 += t[2];
    } else {
      l0 += s * (f * d0);
      l1 += s * (f * d1);
      l2 += s * (f * d2);
    }
  };
  nbrs_exact(S, xi, cell, S.fstart, S.xm, [&](uint32_t j, T d0, T d1, T d2, T r2,
                                                const vec4_t<T> &pj) {
    const vec4_t<T> wj = w[static_cast<size_t>(ws) * j];
    const T f = S.K.gradf(r2);
    const T s = (((T(10) * (S.mu_f / rhoi)) * (pj.w / S.rho[j])) *
                 dot3_exact(wi.x - wj.x, wi.y - wj.y, wi.z - wj.z, d0, d1, d2)) /
                (r2 + S.hh001);
    acc(s, f, d0, d1, d2);
  });
  nbrs_exact(S, xi, cell, S.bstart, S.bxV, [&](uint32_t, T d0, T d1, T d2, T r2,
                                                 const vec4_t<T> &pj) {
    const T f = S.K.gradf(r2);
    const T s = (((T(10) * (S.mu_b / rhoi)) * ((S.rho0 * pj.w) / rhoi)) *
                 dot3_exact(wi.x, wi.y, wi.z, d0, d1, d2)) /
                (r2 + S.hh001);
    acc(s, f, d0, d1, d2);
  });
  out[0] = wi.x - S.dt * l0;
  out[1] = wi.y - S.dt * l1;
  out[2] = wi.z - S.dt * l2;
}

// ---- fast path: diagonal over the list, B_i, and (x, m/rho) packing
template <class T>
__device__ __forceinline__ T gradf_fast(const SceneView<T> &S, T r2) {
  // same closed form as the fused IISPH kernels: 3 alpha/h^4 (u^2 - t^2)/r
  const T h = S.K.h;
  const T inv_h = T(1) / h;
  const T rinv = T(1) / sqrt(r2);
  const T q = r2 * rinv * inv_h;
  const T t = T(2) - q;
  T u = T(2) - T(2) * q;
  u = u > T(0) ? u : T(0);
  const T ag3 = T(3) * S.K.alpha / (h * h * h * h);
  return r2 < S.K.eps * S.K.eps ? T(0) : ag3 * (u * u - t * t) * rinv;
}

// the boundary neighbours of particle i in a fused step, runs sub, sub + kLanes,
// ... of its cells (nothing for a particle whose list tells it has none):
// fn(d0, d1, d2, pj)
template <int kLanes, class T, class Fn>
__device__ __forceinline__ void boundary_lanes(const SceneView<T> &S, int i, uint32_t info,
                                               uint32_t sub, const vec4_t<T> &xi, Fn &&fn) {
  if (!list_has_boundary(info))
    return;
  const uint32_t cell = S.fcell[i];
  for (uint32_t r = sub; r < 9u; r += kLanes) {
    uint32_t b, e;
    run_bounds(S.grid, cell, S.bstart, static_cast<int>(r), &b, &e);
    for (uint32_t j = b; j < e; ++j) {
      const vec4_t<T> pj = S.bxV[j];
      const T d0 = xi.x - pj.x, d1 = xi.y - pj.y, d2 = xi.z - pj.z;
      if (sqdist_exact(d0, d1, d2) < S.thr2)
        fn(d0, d1, d2, pj);
    }
  }
}

// the symmetric boundary matrix B_i = sum_b k_ib gradW_ib x_ib^T (xx yy zz xy xz
// yz), this lane's share
template <int kLanes, class T>
__device__ __forceinline__ void boundary_matrix(const SceneView<T> &S, int i, uint32_t info,
                                                uint32_t sub, const vec4_t<T> &xi, T rhoi,
                                                T B[6]) {
  const T cb = T(10) * S.mu_b / rhoi * S.rho0 / rhoi;
  boundary_lanes<kLanes>(S, i, info, sub, xi, [&](T d0, T d1, T d2, const vec4_t<T> &pj) {
    const T r2 = d0 * d0 + d1 * d1 + d2 * d2;
    const T k = cb * pj.w * gradf_fast(S, r2) / (r2 + S.hh001);
    B[0] += k * d0 * d0;
    B[1] += k * d1 * d1;
    B[2] += k * d2 * d2;
    B[3] += k * d0 * d1;
    B[4] += k * d0 * d2;
    B[5] += k * d1 * d2;
  });
}

// (I - dt (D + B))^-1, or with kGC (I - dt L_i (D + B))^-1, to sp_i
template <class T, bool kGC>
__device__ __forceinline__ void store_diagonal(const SceneView<T> &S, int i, const T D[6],
                                               const T B[6]) {
  T M[9];
  const T dt = S.dt;
  const T Dt[6] = {D[0] + B[0], D[1] + B[1], D[2] + B[2], D[3] + B[3], D[4] + B[4], D[5] + B[5]};
  if (kGC) {
    const T Ds[9] = {Dt[0], Dt[3], Dt[4], Dt[3], Dt[1], Dt[5], Dt[4], Dt[5], Dt[2]};
    const T *Li = S.gc + 9 * static_cast<size_t>(i);
    T Lr[9];
#pragma unroll
    for (int k = 0; k < 9; ++k)
      Lr[k] = Li[k];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int r = 0; r < 3; ++r)
        M[r + 3 * c] = ((r == c) ? T(1) : T(0)) -
                       dt * (Lr[r] * Ds[3 * c] + Lr[r + 3] * Ds[1 + 3 * c] +
                             Lr[r + 6] * Ds[2 + 3 * c]);
  } else {
    M[0] = T(1) - dt * Dt[0];
    M[4] = T(1) - dt * Dt[1];
    M[8] = T(1) - dt * Dt[2];
    M[1] = M[3] = -dt * Dt[3];
    M[2] = M[6] = -dt * Dt[4];
    M[5] = M[7] = -dt * Dt[5];
  }
  invert3(M, S.sp + 9 * static_cast<size_t>(i));
}

// with kGC: M = I - dt L_i (D + B), and the product applies L_i to the summed
// vector (equal in real arithmetic to applying it per pair)
template <class T, bool kGC, int kLanes>
__global__ __launch_bounds__(kBlock) void k_diag_list(SceneView<T> S, NbrList L) {
  const unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const int i = static_cast<int>((lb * kBlock + threadIdx.x) / kLanes);
  const uint32_t sub = threadIdx.x % kLanes;
  const bool valid = i < S.nf;
  const vec4_t<T> xi = valid ? S.xm[i] : make4<vec4_t<T>>(T(0), T(0), T(0), T(0));
  const T rhoi = valid ? S.rho[i] : T(1);
  T D[6] = {0, 0, 0, 0, 0, 0};  // symmetric: xx yy zz xy xz yz
  T B[6] = {0, 0, 0, 0, 0, 0};
  if (valid) {
    auto add = [&](T k, T d0, T d1, T d2) {
      D[0] += k * d0 * d0;
      D[1] += k * d1 * d1;
      D[2] += k * d2 * d2;
      D[3] += k * d0 * d1;
      D[4] += k * d0 * d2;
      D[5] += k * d1 * d2;
    };
    const T cf = T(10) * S.mu_f / rhoi;
    struct P {
      vec4_t<T> x;
      T rho;
    };
    auto fluid = [&](const P &q) {
      const T d0 = xi.x - q.x.x, d1 = xi.y - q.x.y, d2 = xi.z - q.x.z;
      const T r2 = d0 * d0 + d1 * d1 + d2 * d2;
      add(cf * q.x.w / q.rho * gradf_fast(S, r2) / (r2 + S.hh001), d0, d1, d2);
    };
    auto load = [&](uint32_t j) { return P{S.xm[j], S.rho[j]}; };
    const uint32_t info = L.info[i];
    if (!(info & kListOverflow))
      list_gather_lanes<kLanes, 4>(L, pass_spans<kLanes>(L, S.nf, lb), static_cast<size_t>(S.nf),
                                   i, info, sub, load, fluid);
    else if (sub == 0)
      nbrs_exact(S, xi, S.fcell[i], S.fstart, S.xm,
                 [&](uint32_t j, T, T, T, T, const vec4_t<T> &) {
                   if (j != static_cast<uint32_t>(i))
                     fluid(load(j));
                 });
    boundary_matrix<kLanes>(S, i, info, sub, xi, rhoi, B);
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    D[k] = lanes_sum<kLanes>(D[k]);
    B[k] = lanes_sum<kLanes>(B[k]);
  }
  if (!valid || sub != 0)
    return;
  store_diagonal<T, kGC>(S, i, D, B);
  // B_i for the list product, (x_i, m_i / rho_i) for its gathers
  S.cb[i] = make4<vec4_t<T>>(B[0], B[1], B[2], T(0));
  S.G[i] = make4<vec4_t<T>>(B[3], B[4], B[5], T(0));
  const vec4_t<T> q = make4<vec4_t<T>>(xi.x, xi.y, xi.z, xi.w / rhoi);
  S.xq[i] = q;
  S.cxp[2 * static_cast<size_t>(i)] = q;
}

template <class T>
__device__ __forceinline__ T rsqrt_hw(T x);
template <>
__device__ __forceinline__ float rsqrt_hw<float>(float x) {
  return __builtin_amdgcn_rsqf(x);
}
template <>
__device__ __forceinline__ double rsqrt_hw<double>(double x) {
  return rsqrt(x);
}
template <class T>
__device__ __forceinline__ T rcp_hw(T x);
template <>
__device__ __forceinline__ float rcp_hw<float>(float x) {
  return __builtin_amdgcn_rcpf(x);
}
template <>
__device__ __forceinline__ double rcp_hw<double>(double x) {
  return 1.0 / x;
}

// one fluid pair of the list product: l += (m_j / rho_j) ((w_i - w_j) . d)
// f(r) / (r^2 + 0.01 h^2) d with d = x_i - x_j; xq = (x_i, m_i / rho_i),
// qx = (x_j, m_j / rho_j)
template <class T>
struct ProductPair {
  T inv_h, ag3, eps2, hh001;
  __device__ __forceinline__ explicit ProductPair(const SceneView<T> &S)
      : inv_h(T(1) / S.K.h), ag3(T(3) * S.K.alpha / (S.K.h * S.K.h * S.K.h * S.K.h)),
        eps2(S.K.eps * S.K.eps), hh001(S.hh001) {}
  __device__ __forceinline__ void operator()(const vec4_t<T> &xq, const vec4_t<T> &wi,
                                             const vec4_t<T> &qx, const vec4_t<T> &wj, T &l0,
                                             T &l1, T &l2) const {
    const T d0 = xq.x - qx.x, d1 = xq.y - qx.y, d2 = xq.z - qx.z;
    const T r2 = d0 * d0 + d1 * d1 + d2 * d2;
    const T rinv = rsqrt_hw(r2);
    const T qh = r2 * rinv * inv_h;
    const T t = T(2) - qh;
    T u = T(2) - T(2) * qh;
    u = u > T(0) ? u : T(0);
    const T f = r2 < eps2 ? T(0) : ag3 * (u * u - t * t) * rinv;
    const T s = qx.w * ((wi.x - wj.x) * d0 + (wi.y - wj.y) * d1 + (wi.z - wj.z) * d2) * f *
                rcp_hw(r2 + hh001);
    l0 += s * d0;
    l1 += s * d1;
    l2 += s * d2;
  }
};

// out = w_i - dt (10 mu_f / rho_i l + B_i w_i) from the fluid pair sum l
// and B_i = (bd: xx yy zz, bo: xy xz yz); with kGC L_i applies to the bracket
template <class T, bool kGC>
__device__ __forceinline__ void product_finish(const SceneView<T> &S, int i,
                                               const vec4_t<T> &wi, T l0, T l1, T l2,
                                               const vec4_t<T> &bd, const vec4_t<T> &bo,
                                               T out[3]) {
  const T cf = T(10) * S.mu_f / S.rho[i];
  const T b0 = bd.x * wi.x + bo.x * wi.y + bo.y * wi.z;
  const T b1 = bo.x * wi.x + bd.y * wi.y + bo.z * wi.z;
  const T b2 = bo.y * wi.x + bo.z * wi.y + bd.z * wi.z;
  if (kGC) {
    const T *Li = S.gc + 9 * static_cast<size_t>(i);
    const T u0 = cf * l0 + b0, u1 = cf * l1 + b1, u2 = cf * l2 + b2;
    out[0] = wi.x - S.dt * (Li[0] * u0 + Li[3] * u1 + Li[6] * u2);
    out[1] = wi.y - S.dt * (Li[1] * u0 + Li[4] * u1 + Li[7] * u2);
    out[2] = wi.z - S.dt * (Li[2] * u0 + Li[5] * u1 + Li[8] * u2);
  } else {
    out[0] = wi.x - S.dt * (cf * l0 + b0);
    out[1] = wi.y - S.dt * (cf * l1 + b1);
    out[2] = wi.z - S.dt * (cf * l2 + b2);
  }
}

// the list product at particle i (valid), complete in every one of its kLanes lanes
// with w at stride kStride: S.v, or the second half of the records S.cxp
template <class T, bool kGC, int kLanes, int kStride>
__device__ __forceinline__ void product_list(const SceneView<T> &S, const NbrList &L, unsigned lb,
                                             int i, bool valid, uint32_t sub,
                                             const vec4_t<T> *__restrict__ w,
                                             T out[3]) {
  T l0 = 0, l1 = 0, l2 = 0;
  vec4_t<T> wi = make4<vec4_t<T>>(T(0), T(0), T(0), T(0)), bd = wi, bo = wi;
  const vec4_t<T> xq = valid ? S.xq[i] : wi;  // (x_i, m_i / rho_i)
  const uint32_t info = valid ? L.info[i] : kListOverflow;
  if (valid)
    wi = w[kStride * static_cast<size_t>(i)];
  const ProductPair<T> pair(S);
  // (x_j, m_j / rho_j) and w_j
  auto use = [&](const vec4_t<T> &xj, const vec4_t<T> &wj) { pair(xq, wi, xj, wj, l0, l1, l2); };
  const Spans R = pass_spans<kLanes>(L, S.nf, lb);
  const size_t n = static_cast<size_t>(S.nf);
  const uint32_t live = (info & kListOverflow) ? 0u : info;
  if constexpr (kStride == 2) {
    list_gather_records<kLanes, 4>(L, R, n, i, live, sub, static_cast<uint32_t>(valid ? i : 0),
                                   S.cxp, use);
  } else {
    struct XW {
      vec4_t<T> x, w;
    };
    list_gather_lanes<kLanes, 4>(
        L, R, n, i, live, sub,
        [&](uint32_t j) { return XW{S.cxp[2 * static_cast<size_t>(j)], w[j]}; },
        [&](const XW &q) { use(q.x, q.w); });
  }
  if (valid) {
    if (sub == 0 && (info & kListOverflow))
      nbrs_exact(S, xq, S.fcell[i], S.fstart, S.xq,
                 [&](uint32_t j, T, T, T, T, const vec4_t<T> &) {
                   if (j != static_cast<uint32_t>(i))
                     use(S.xq[j], w[kStride * static_cast<size_t>(j)]);
                 });
    bd = S.cb[i];
    bo = S.G[i];
  }
  l0 = lanes_sum<kLanes>(l0);
  l1 = lanes_sum<kLanes>(l1);
  l2 = lanes_sum<kLanes>(l2);
  if (valid)
    product_finish<T, kGC>(S, i, wi, l0, l1, l2, bd, bo, out);
}

template <class T>
__device__ __forceinline__ T dot3r(const vec4_t<T> &a, const vec4_t<T> &b) {
#pragma clang fp contract(off)
  return a.x * b.x + (a.y * b.y + a.z * b.z);  // sum(cmul(l, r)) per item
}

template <class T>
__device__ __forceinline__ vec4_t<T> precond(const T *M, const vec4_t<T> &w) {
#pragma clang fp contract(off)
  vec4_t<T> y;
  y.x = M[0] * w.x + (M[3] * w.y + M[6] * w.z);
  y.y = M[1] * w.x + (M[4] * w.y + M[7] * w.z);
  y.z = M[2] * w.x + (M[5] * w.y + M[8] * w.z);
  y.w = T(0);
  return y;
}

// setup: x = v (guess), r = A x - b with b = v (the rhs of wkbb18.hpp:296-334
// is v - dt a_b with a_b = 0 because the boundary velocity is zero),
// y = P r, p = -y; partials of b.b, r.r, r.y
// the CG set-up of particle i from ax = A x0; acc = b.b, r.r, r.y
template <class T>
__device__ __forceinline__ void cg_start(const SceneView<T> &S, int i, const vec4_t<T> &v,
                                         const T ax[3], double acc[3]) {
  vec4_t<T> b = v;
  b.w = T(0);
  vec4_t<T> r;
  r.x = ax[0] - b.x;
  r.y = ax[1] - b.y;
  r.z = ax[2] - b.z;
  r.w = T(0);
  const vec4_t<T> y = precond(S.sp + 9 * static_cast<size_t>(i), r);
  S.cx[i] = b;
  S.cr[i] = r;
  S.cy[i] = y;
  S.cxp[2 * static_cast<size_t>(i) + 1] = make4<vec4_t<T>>(-y.x, -y.y, -y.z, T(0));
  acc[0] = static_cast<double>(dot3r<T>(b, b));
  acc[1] = static_cast<double>(dot3r<T>(r, r));
  acc[2] = static_cast<double>(dot3r<T>(r, y));
}

template <class T, bool kExact, bool kGC, int kLanes>
__global__ __launch_bounds__(kBlock) void k_cg_setup(SceneView<T> S, NbrList L, double *part) {
  const unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const int i = static_cast<int>((lb * kBlock + threadIdx.x) / kLanes);
  const uint32_t sub = threadIdx.x % kLanes;
  const bool valid = i < S.nf;
  double acc[3] = {0.0, 0.0, 0.0};
  T ax[3];
  if (kExact) {
    if (valid)
      product_exact<T, kGC>(S, i, S.v, 1, ax);
  } else {
    product_list<T, kGC, kLanes, 1>(S, L, lb, i, valid, sub, S.v, ax);
  }
  if (valid && sub == 0)
    cg_start(S, i, S.v[i], ax, acc);
  store_partials<3>(part, gridDim.x, acc, lb);
}

// k_diag_list and the list form of k_cg_setup in one walk over the list
// (fused steps): every pair term is the expression of the two kernels, in the
// same order, with (x_j, m_j / rho_j) formed from x_j, m_j and rho_j as the
// diagonal pass writes it, so the results equal those of the two kernels
// (lb: the block's logical index, nb: the scene's block count)
template <class T, bool kGC, int kLanes>
__device__ __forceinline__ void diag_setup_list_body(const SceneView<T> &S, const NbrList &L,
                                                     double *part, unsigned lb, unsigned nb) {
  const int i = static_cast<int>((lb * kBlock + threadIdx.x) / kLanes);
  const uint32_t sub = threadIdx.x % kLanes;
  const bool valid = i < S.nf;
  const vec4_t<T> zero4 = make4<vec4_t<T>>(T(0), T(0), T(0), T(0));
  const vec4_t<T> xi = valid ? S.xm[i] : zero4;
  const T rhoi = valid ? S.rho[i] : T(1);
  const vec4_t<T> wi = valid ? S.v[i] : zero4;  // the guess x0 = v
  const vec4_t<T> xqi = make4<vec4_t<T>>(xi.x, xi.y, xi.z, xi.w / rhoi);
  T D[6] = {0, 0, 0, 0, 0, 0};  // symmetric: xx yy zz xy xz yz
  T B[6] = {0, 0, 0, 0, 0, 0};
  T l0 = 0, l1 = 0, l2 = 0;
  if (valid) {
    const T cf = T(10) * S.mu_f / rhoi;
    const ProductPair<T> pair(S);
    struct P {
      vec4_t<T> x;  // (x_j, m_j)
      T rho;
      vec4_t<T> w;  // v_j
    };
    auto both = [&](const P &q) {
      const T d0 = xi.x - q.x.x, d1 = xi.y - q.x.y, d2 = xi.z - q.x.z;
      const T r2 = d0 * d0 + d1 * d1 + d2 * d2;
      const T k = cf * q.x.w / q.rho * gradf_fast(S, r2) / (r2 + S.hh001);
      D[0] += k * d0 * d0;
      D[1] += k * d1 * d1;
      D[2] += k * d2 * d2;
      D[3] += k * d0 * d1;
      D[4] += k * d0 * d2;
      D[5] += k * d1 * d2;
      pair(xqi, wi, make4<vec4_t<T>>(q.x.x, q.x.y, q.x.z, q.x.w / q.rho), q.w, l0, l1, l2);
    };
    auto load = [&](uint32_t j) { return P{S.xm[j], S.rho[j], S.v[j]}; };
    const uint32_t info = L.info[i];
    if (!(info & kListOverflow))
      list_gather_lanes<kLanes, 4>(L, pass_spans<kLanes>(L, S.nf, lb), static_cast<size_t>(S.nf),
                                   i, info, sub, load, both);
    else if (sub == 0)
      nbrs_exact(S, xi, S.fcell[i], S.fstart, S.xm,
                 [&](uint32_t j, T, T, T, T, const vec4_t<T> &) {
                   if (j != static_cast<uint32_t>(i))
                     both(load(j));
                 });
    boundary_matrix<kLanes>(S, i, info, sub, xi, rhoi, B);
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    D[k] = lanes_sum<kLanes>(D[k]);
    B[k] = lanes_sum<kLanes>(B[k]);
  }
  l0 = lanes_sum<kLanes>(l0);
  l1 = lanes_sum<kLanes>(l1);
  l2 = lanes_sum<kLanes>(l2);
  double acc[3] = {0.0, 0.0, 0.0};
  if (valid && sub == 0) {
    store_diagonal<T, kGC>(S, i, D, B);
    const vec4_t<T> bd = make4<vec4_t<T>>(B[0], B[1], B[2], T(0));
    const vec4_t<T> bo = make4<vec4_t<T>>(B[3], B[4], B[5], T(0));
    S.cb[i] = bd;
    S.G[i] = bo;
    S.xq[i] = xqi;
    S.cxp[2 * static_cast<size_t>(i)] = xqi;
    T ax[3];
    product_finish<T, kGC>(S, i, wi, l0, l1, l2, bd, bo, ax);
    cg_start(S, i, wi, ax, acc);
  }
  store_partials<3>(part, nb, acc, lb);
}

template <class T, bool kGC, int kLanes>
__global__ __launch_bounds__(kBlock) void k_diag_setup_list(SceneView<T> S, NbrList L,
                                                            double *part) {
  diag_setup_list_body<T, kGC, kLanes>(S, L, part, xcd_block(blockIdx.x, gridDim.x), gridDim.x);
}

// q = A p, partial p.q
template <class T, bool kExact, bool kGC, int kLanes>
__device__ __forceinline__ void cg_spmv_body(const SceneView<T> &S, const NbrList &L,
                                             double *part, unsigned lb, unsigned nb) {
  if (S.ctl->cg_done)
    return;
  const int i = static_cast<int>((lb * kBlock + threadIdx.x) / kLanes);
  const uint32_t sub = threadIdx.x % kLanes;
  const bool valid = i < S.nf;
  double acc[1] = {0.0};
  T q[3];
  if (kExact) {
    if (valid)
      product_exact<T, kGC>(S, i, S.cxp + 1, 2, q);
  } else {
    product_list<T, kGC, kLanes, 2>(S, L, lb, i, valid, sub, S.cxp + 1, q);
  }
  if (valid && sub == 0) {
    const vec4_t<T> qv = make4<vec4_t<T>>(q[0], q[1], q[2], T(0));
    S.cq[i] = qv;
    acc[0] = static_cast<double>(dot3r<T>(S.cxp[2 * static_cast<size_t>(i) + 1], qv));
  }
  store_partials<1>(part, nb, acc, lb);
}

template <class T, bool kExact, bool kGC, int kLanes>
__global__ __launch_bounds__(kBlock) void k_cg_spmv(SceneView<T> S, NbrList L, double *part) {
  cg_spmv_body<T, kExact, kGC, kLanes>(S, L, part, xcd_block(blockIdx.x, gridDim.x), gridDim.x);
}

// a particle's vectors of the update, loaded ahead of the scalars (whose partial
// sums are a chain of memory latencies of their own)
template <class T>
struct CgOwn {
  vec4_t<T> p, q, x, r;
  T M[9];
  __device__ __forceinline__ CgOwn(const SceneView<T> &S, int i) {
    if (i < S.nf) {
      p = S.cxp[2 * static_cast<size_t>(i) + 1];
      q = S.cq[i];
      x = S.cx[i];
      r = S.cr[i];
#pragma unroll
      for (int k = 0; k < 9; ++k)
        M[k] = S.sp[9 * static_cast<size_t>(i) + k];
    }
  }
};

// x += alpha p, r += alpha q, y = P r; partials r.r, r.y
template <class T>
__device__ __forceinline__ void cg_update_body(const SceneView<T> &S, const CgOwn<T> &o, T alpha,
                                               double *part, unsigned lb, unsigned nb) {
  const int i = static_cast<int>(lb * kBlock + threadIdx.x);
  double acc[2] = {0.0, 0.0};
  if (i < S.nf) {
    vec4_t<T> x = o.x, r = o.r;
    x.x += alpha * o.p.x;
    x.y += alpha * o.p.y;
    x.z += alpha * o.p.z;
    r.x += alpha * o.q.x;
    r.y += alpha * o.q.y;
    r.z += alpha * o.q.z;
    const vec4_t<T> y = precond(o.M, r);
    S.cx[i] = x;
    S.cr[i] = r;
    S.cy[i] = y;
    acc[0] = static_cast<double>(dot3r<T>(r, r));
    acc[1] = static_cast<double>(dot3r<T>(r, y));
  }
  store_partials<2>(part, nb, acc, lb);
}

// p = -y + beta p
template <class T>
__device__ __forceinline__ void cg_direction_body(const SceneView<T> &S, const vec4_t<T> &y,
                                                  vec4_t<T> p, T beta, unsigned lb) {
  const int i = static_cast<int>(lb * kBlock + threadIdx.x);
  if (i >= S.nf)
    return;
  p.x = -y.x + beta * p.x;
  p.y = -y.y + beta * p.y;
  p.z = -y.z + beta * p.z;
  S.cxp[2 * static_cast<size_t>(i) + 1] = p;
}

// The update and direction kernels of one scene. fold: without the two one-block
// kernels (cg_alpha_in_block, cg_beta_in_block): the block derives alpha from the
// npq partials of p.q (beta from the nb partials of r.r and r.y).
template <class T>
__device__ __forceinline__ void cg_update(const SceneView<T> &S, bool fold, const double *pq_part,
                                          unsigned npq, double *part, unsigned lb, unsigned nb) {
  const CgOwn<T> own(S, static_cast<int>(lb * kBlock + threadIdx.x));
  if (cg_done_for_block(S.ctl))
    return;
  double alpha;
  if (fold) {
    if (!cg_alpha_in_block(S.ctl, pq_part, npq, &alpha, lb))
      return;
  } else {
    alpha = S.ctl->cg_alpha;
  }
  cg_update_body(S, own, static_cast<T>(alpha), part, lb, nb);
}

template <class T>
__device__ __forceinline__ void cg_direction(const SceneView<T> &S, bool fold, const double *part,
                                             unsigned lb, unsigned nb) {
  const int i = static_cast<int>(lb * kBlock + threadIdx.x);
  vec4_t<T> y = make4<vec4_t<T>>(T(0), T(0), T(0), T(0)), p = y;
  if (i < S.nf) {
    y = S.cy[i];
    p = S.cxp[2 * static_cast<size_t>(i) + 1];
  }
  if (cg_done_for_block(S.ctl))
    return;
  double beta;
  if (fold) {
    if (!cg_beta_in_block(S.ctl, part, nb, &beta, lb))
      return;
  } else {
    beta = S.ctl->cg_beta;
  }
  cg_direction_body(S, y, p, static_cast<T>(beta), lb);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_cg_update(SceneView<T> S, int fold,
                                                      const double *pq_part, unsigned npq,
                                                      double *part) {
  cg_update(S, fold != 0, pq_part, npq, part, blockIdx.x, gridDim.x);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_cg_direction(SceneView<T> S, int fold,
                                                         const double *part) {
  cg_direction(S, fold != 0, part, blockIdx.x, gridDim.x);
}

// apply (wkbb18.hpp:401-413): vd = (x - v) H(t - t_birth - dt_fade), a = vd / dt
template <class T>
__device__ __forceinline__ void cg_apply_body(const SceneView<T> &S, unsigned lb) {
#pragma clang fp contract(off)
  const int i = static_cast<int>(lb * kBlock + threadIdx.x);
  if (i >= S.nf)
    return;
  const vec4_t<T> x = S.cx[i], v = S.v[i];
  const T H = step_l(T(0), (S.t - v.w) - S.fade);
  const vec4_t<T> vd = make4<vec4_t<T>>((x.x - v.x) * H, (x.y - v.y) * H, (x.z - v.z) * H, T(0));
  S.vd[i] = vd;
  S.a[i] = make4<vec4_t<T>>(vd.x / S.dt, vd.y / S.dt, vd.z / S.dt, T(0));
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_cg_apply(SceneView<T> S) {
  cg_apply_body(S, blockIdx.x);
}

// ---- batched WKBB18 (prtcl_hip_step over several scenes): the kernels above
// over the blocks of every scene of a table (B: group 0 the scenes without, group
// 1 those with the gradient correction), each block with its scene's view,
// list, CG partials and block counts, so every scene's sums and decisions are
// those of its single-scene step. A scene with cg_fold derives alpha and
// beta in its vector kernels, otherwise its one-block kernels do.
#define WK_BATCH_ENTRY(kF)                                                 \
  unsigned part_;                                                          \
  const uint32_t u = batch_block(B, kF, &part_);                           \
  const BatchEntry<T> &E = tab[u >> kBatchLocalBits];                      \
  const bool split = split_scene(E.S.nf);                                  \
  const unsigned lb = (u & kBatchLocalMask) * (split ? (kF) : 1u) + part_; \
  const unsigned nl = list_blocks(E.S.nf);                                 \
  const NbrList L{E.nidx, E.ninfo, E.nblk, E.nshift};                      \
  (void)L;                                                                 \
  if (lb >= ((kF) == 1u ? E.nblocks : nl))                                 \
  return

template <class T, bool kGC>
__global__ __launch_bounds__(kBlock) void k_diag_setup_b(const BatchEntry<T> *tab,
                                                         BatchBlocks B) {
  WK_BATCH_ENTRY(kListLanes);
  if (split)
    diag_setup_list_body<T, kGC, kListLanes>(E.S, L, E.cg_part, lb, nl);
  else
    diag_setup_list_body<T, kGC, 1>(E.S, L, E.cg_part, lb, nl);
}

// the gradient correction of wkbb18_gc scenes over the list
template <class T>
__global__ __launch_bounds__(kBlock) void k_corr_b(const BatchEntry<T> *tab, BatchBlocks B) {
  WK_BATCH_ENTRY(kListLanes);
  if (split)
    corr_body<T, true, kListLanes>(E.S, L, lb);
  else
    corr_body<T, true, 1>(E.S, L, lb);
}

// one block per scene
template <class T>
__global__ __launch_bounds__(kBlock) void k_cg_setup_fin_b(const BatchEntry<T> *tab) {
  const BatchEntry<T> &E = tab[blockIdx.x];
  cg_setup_fin_body(E.S.ctl, E.cg_part, list_blocks(E.S.nf), E.cg_tol, E.cg_max_k, E.cg_seq);
}

template <class T, bool kGC>
__global__ __launch_bounds__(kBlock) void k_cg_spmv_b(const BatchEntry<T> *tab, BatchBlocks B) {
  WK_BATCH_ENTRY(kListLanes);
  if (split)
    cg_spmv_body<T, false, kGC, kListLanes>(E.S, L, E.cg_part, lb, nl);
  else
    cg_spmv_body<T, false, kGC, 1>(E.S, L, E.cg_part, lb, nl);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_cg_alpha_b(const BatchEntry<T> *tab) {
  const BatchEntry<T> &E = tab[blockIdx.x];
  if (!E.cg_fold)
    cg_alpha_body(E.S.ctl, E.cg_part, list_blocks(E.S.nf));
}

// p.q partials at [0, nl), r.r and r.y at [nl, nl + 2 nb)
template <class T>
__global__ __launch_bounds__(kBlock) void k_cg_update_b(const BatchEntry<T> *tab,
                                                        BatchBlocks B) {
  WK_BATCH_ENTRY(1u);
  cg_update(E.S, E.cg_fold != 0, E.cg_part, nl, E.cg_part + nl, lb, E.nblocks);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_cg_beta_b(const BatchEntry<T> *tab) {
  const BatchEntry<T> &E = tab[blockIdx.x];
  if (!E.cg_fold)
    cg_beta_body(E.S.ctl, E.cg_part + list_blocks(E.S.nf), E.nblocks);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_cg_direction_b(const BatchEntry<T> *tab,
                                                           BatchBlocks B) {
  WK_BATCH_ENTRY(1u);
  cg_direction(E.S, E.cg_fold != 0, E.cg_part + nl, lb, E.nblocks);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_cg_apply_b(const BatchEntry<T> *tab,
                                                       BatchBlocks B) {
  WK_BATCH_ENTRY(1u);
  cg_apply_body(E.S, lb);
}

#undef WK_BATCH_ENTRY

}  // namespace

// a list kernel of one scene with its lanes per particle; the kernel's template
// arguments before the lanes are given in parentheses
#define WK_ARGS(...) __VA_ARGS__
#define WK_LIST(kern, targs, ...)                                                          \
  do {                                                                                     \
    if (split_scene(S.nf))                                                                 \
      hipLaunchKernelGGL((kern<WK_ARGS targs, kListLanes>), dim3(list_blocks(S.nf)),       \
                         dim3(kBlock), 0, st, S, ##__VA_ARGS__);                           \
    else                                                                                   \
      hipLaunchKernelGGL((kern<WK_ARGS targs, 1>), dim3(grid_blocks(S.nf)), dim3(kBlock), 0, \
                         st, S, ##__VA_ARGS__);                                            \
  } while (0)
#define WK_EXACT(kern, targs, ...)                                                           \
  hipLaunchKernelGGL((kern<WK_ARGS targs, 1>), dim3(grid_blocks(S.nf)), dim3(kBlock), 0, st, S, \
                     ##__VA_ARGS__)

template <class T>
void Wkbb18Ops<T>::diagonal(hipStream_t st, const SceneView<T> &S, const NbrList *L, bool gc) {
  if (S.nf <= 0)
    return;
  const dim3 gr(grid_blocks(S.nf)), bl(kBlock);
  if (L && gc)
    WK_LIST(k_diag_list, (T, true), *L);
  else if (L)
    WK_LIST(k_diag_list, (T, false), *L);
  else if (gc)
    hipLaunchKernelGGL((k_diag_exact<T, true>), gr, bl, 0, st, S);
  else
    hipLaunchKernelGGL((k_diag_exact<T, false>), gr, bl, 0, st, S);
}

template <class T>
void Wkbb18Ops<T>::setup(hipStream_t st, const SceneView<T> &S, const NbrList *L, bool gc,
                         double *part, double tol, int max_k, unsigned seq) {
  if (S.nf > 0) {
    if (L && gc)
      WK_LIST(k_cg_setup, (T, false, true), *L, part);
    else if (L)
      WK_LIST(k_cg_setup, (T, false, false), *L, part);
    else if (gc)
      WK_EXACT(k_cg_setup, (T, true, true), NbrList{}, part);
    else
      WK_EXACT(k_cg_setup, (T, true, false), NbrList{}, part);
  }
  hipLaunchKernelGGL(k_cg_setup_fin, dim3(1), dim3(kBlock), 0, st, S.ctl, part,
                     L ? list_blocks(S.nf) : grid_blocks(S.nf), tol, max_k, seq);
}

template <class T>
void Wkbb18Ops<T>::diagonal_setup(hipStream_t st, const SceneView<T> &S, const NbrList &L,
                                  bool gc, double *part, double tol, int max_k, unsigned seq) {
  if (S.nf > 0) {
    if (gc)
      WK_LIST(k_diag_setup_list, (T, true), L, part);
    else
      WK_LIST(k_diag_setup_list, (T, false), L, part);
  }
  hipLaunchKernelGGL(k_cg_setup_fin, dim3(1), dim3(kBlock), 0, st, S.ctl, part,
                     list_blocks(S.nf), tol, max_k, seq);
}

template <class T>
void Wkbb18Ops<T>::iteration_product(hipStream_t st, const SceneView<T> &S, const NbrList *L,
                                     bool gc, double *part) {
  if (S.nf <= 0)
    return;
  if (L && gc)
    WK_LIST(k_cg_spmv, (T, false, true), *L, part);
  else if (L)
    WK_LIST(k_cg_spmv, (T, false, false), *L, part);
  else if (gc)
    WK_EXACT(k_cg_spmv, (T, true, true), NbrList{}, part);
  else
    WK_EXACT(k_cg_spmv, (T, true, false), NbrList{}, part);
}

template <class T>
void Wkbb18Ops<T>::iteration_vectors(hipStream_t st, const SceneView<T> &S, const NbrList *L,
                                     double *part, bool split) {
  if (S.nf <= 0)
    return;
  const unsigned nb = grid_blocks(S.nf), nl = L ? list_blocks(S.nf) : nb;
  const dim3 gr(nb), bl(kBlock);
  // p.q partials at part[0, nl), r.r and r.y at part[nl, nl + 2 nb)
  const int fold = !split && nb <= kFusedCgBlocks ? 1 : 0;
  if (!fold)
    hipLaunchKernelGGL(k_cg_alpha, dim3(1), bl, 0, st, S.ctl, part, nl);
  hipLaunchKernelGGL(k_cg_update<T>, gr, bl, 0, st, S, fold, part, nl, part + nl);
  if (!fold)
    hipLaunchKernelGGL(k_cg_beta, dim3(1), bl, 0, st, S.ctl, part + nl, nb);
  hipLaunchKernelGGL(k_cg_direction<T>, gr, bl, 0, st, S, fold, part + nl);
}

template <class T>
void Wkbb18Ops<T>::correction(hipStream_t st, const SceneView<T> &S, const NbrList *L) {
  if (S.nf <= 0)
    return;
  if (L)
    WK_LIST(k_corr, (T, true), *L);
  else
    WK_EXACT(k_corr, (T, false), NbrList{});
}

template <class T>
void Wkbb18Ops<T>::identity_correction(hipStream_t st, const SceneView<T> &S) {
  if (S.nf > 0)
    hipLaunchKernelGGL(k_corr_identity<T>, dim3(grid_blocks(S.nf)), dim3(kBlock), 0, st, S);
}

template <class T>
void Wkbb18Ops<T>::apply(hipStream_t st, const SceneView<T> &S) {
  if (S.nf > 0)
    hipLaunchKernelGGL(k_cg_apply<T>, dim3(grid_blocks(S.nf)), dim3(kBlock), 0, st, S);
}

template <class T>
void Wkbb18Ops<T>::correction_batch(hipStream_t st, const BatchEntry<T> *tab,
                                    const BatchBlocks &B) {
  const BatchBlocks G = B.group(1);
  if (const unsigned n = G.launch(kListLanes))
    hipLaunchKernelGGL(k_corr_b<T>, dim3(n), dim3(kBlock), 0, st, tab, G);
}

template <class T>
void Wkbb18Ops<T>::diagonal_setup_batch(hipStream_t st, const BatchEntry<T> *tab,
                                        const BatchBlocks &B, unsigned nscenes) {
  if (nscenes == 0)
    return;
  const BatchBlocks P = B.group(0), G = B.group(1);
  if (const unsigned n = P.launch(kListLanes))
    hipLaunchKernelGGL((k_diag_setup_b<T, false>), dim3(n), dim3(kBlock), 0, st, tab, P);
  if (const unsigned n = G.launch(kListLanes))
    hipLaunchKernelGGL((k_diag_setup_b<T, true>), dim3(n), dim3(kBlock), 0, st, tab, G);
  hipLaunchKernelGGL(k_cg_setup_fin_b<T>, dim3(nscenes), dim3(kBlock), 0, st, tab);
}

template <class T>
void Wkbb18Ops<T>::iteration_batch(hipStream_t st, const BatchEntry<T> *tab, const BatchBlocks &B,
                                   unsigned nscenes, bool any_split) {
  const unsigned na = B.launch(1);
  if (na == 0)
    return;
  const BatchBlocks P = B.group(0), G = B.group(1);
  const dim3 bl(kBlock);
  if (const unsigned n = P.launch(kListLanes))
    hipLaunchKernelGGL((k_cg_spmv_b<T, false>), dim3(n), bl, 0, st, tab, P);
  if (const unsigned n = G.launch(kListLanes))
    hipLaunchKernelGGL((k_cg_spmv_b<T, true>), dim3(n), bl, 0, st, tab, G);
  if (any_split)
    hipLaunchKernelGGL(k_cg_alpha_b<T>, dim3(nscenes), bl, 0, st, tab);
  hipLaunchKernelGGL(k_cg_update_b<T>, dim3(na), bl, 0, st, tab, B);
  if (any_split)
    hipLaunchKernelGGL(k_cg_beta_b<T>, dim3(nscenes), bl, 0, st, tab);
  hipLaunchKernelGGL(k_cg_direction_b<T>, dim3(na), bl, 0, st, tab, B);
}

template <class T>
void Wkbb18Ops<T>::apply_batch(hipStream_t st, const BatchEntry<T> *tab, const BatchBlocks &B) {
  if (const unsigned n = B.launch(1))
    hipLaunchKernelGGL(k_cg_apply_b<T>, dim3(n), dim3(kBlock), 0, st, tab, B);
}

template struct Wkbb18Ops<float>;
template struct Wkbb18Ops<double>;

}  // namespace prtcl_amd
