// pt16 vorticity-preserving viscosity (pt16.hpp / pt16.prtcl) on the device.
// Every pair term walks the 27-cell grid with the reference predicate (the
// particle itself included, as CopyNeighbors) and is evaluated in the
// reference's FP32 operation order (this file is built without FMA
// contraction); matrices are 3x3 column-major, Eigen's fixed-size sums of
// three terms are x0 + (x1 + x2). In fused steps the CG products use the
// step's neighbour list instead: the pair coefficients m_j W_ij are written
// once per step and streamed by every product (the self term first, then
// the list order). The reference solves each system once per vector component,
// a `foreach dimension` loop of scalar CGOpenMP<T> solves (pt16.hpp:420-519,
// 608-760; cg_openmp.hpp:32-215). The three share the matrix and do not depend
// on each other, so here they run side by side: one product streams the
// coefficients once for all three and gathers one vector per neighbour, and each
// component keeps its own scalars, stop and iteration count (cg_ctl.hpp), with
// the values it has when solved alone. A solve is bound by the launches of its
// iterations and the gathers of the product: two steps of 125,000 particles, 58
// iterations of one component at a time against about 20 of three, 3.05 -> 2.31 ms.
#include "cg_ctl.hpp"
#include "exact_walk.hpp"
#include "nbrlist.hpp"
#include "pt16.hpp"

namespace prtcl_amd {

namespace {

// ---- list form (fused steps)
// index of the coefficient m_j W_ij of list entry e of particle i (chunks of
// 4 entries, so a lane reads 4 with one load and a wavefront's load is
// contiguous); written by the set-up, read by the products and the
// vorticity right-hand side of the same step
__device__ __forceinline__ size_t coef_index(size_t n, int i, uint32_t e) {
  return ((static_cast<size_t>(e / 4) * n + static_cast<size_t>(i)) * 4) + e % 4;
}

constexpr uint32_t kSelfEntry = 0xFFFFFFFEu;  // the particle itself
constexpr uint32_t kNoEntry = 0xFFFFFFFFu;    // a grid-walk neighbour (list overflowed)

// The fluid neighbours of particle i in a fused step, lane `sub` of kLanes:
// fn(rec, d0, d1, d2, r2, x_j, e) with rec = load(j), the neighbour's further
// fields, gathered ahead of the arithmetic; the particle itself first (lane 0,
// d = 0, e = kSelfEntry), then the list entries in list order (e = entry index); a
// particle whose list overflowed walks the grid (lane 0, itself included,
// e = kNoEntry).
template <int kLanes, class T, class Load, class Fn>
__device__ __forceinline__ void fluid_pairs_list(const SceneView<T> &S, const NbrList &L,
                                                 unsigned lb, int i, uint32_t sub,
                                                 const vec4_t<T> &xv, Load &&load, Fn &&fn) {
#pragma clang fp contract(off)
  const uint32_t info = L.info[i];
  if (info & kListOverflow) {
    if (sub == 0)
      nbrs_exact(S, xv, S.fcell[i], S.fstart, S.xm,
                 [&](uint32_t j, T d0, T d1, T d2, T r2, const vec4_t<T> &pj) {
                   fn(load(j), d0, d1, d2, r2, pj, kNoEntry);
                 });
    return;
  }
  if (sub == 0)
    fn(load(static_cast<uint32_t>(i)), T(0), T(0), T(0), T(0), xv, kSelfEntry);
  struct Rec {
    vec4_t<T> x;
    decltype(load(0u)) f;
  };
  uint32_t e = sub * kChunk;  // entries come in order, a lane's chunks kLanes apart
  list_gather_lanes<kLanes, 4>(
      L, pass_spans<kLanes>(L, S.nf, lb), static_cast<size_t>(S.nf), i, info, sub,
      [&](uint32_t j) { return Rec{S.xm[j], load(j)}; },
      [&](const Rec &q) {
        const T d0 = xv.x - q.x.x, d1 = xv.y - q.x.y, d2 = xv.z - q.x.z;
        fn(q.f, d0, d1, d2, d0 * d0 + (d1 * d1 + d2 * d2), q.x, e);
        ++e;
        if (kLanes > 1 && e % kChunk == 0u)
          e += (kLanes - 1) * kChunk;
      });
}

// fn(m_j W_ij, w_j) for the list entries of particle i (not overflowed), lane
// `sub` of kLanes: the coefficients of a chunk of 8 entries and its 8 gathers
// are issued before the arithmetic
template <int kLanes, class T, class Fn>
__device__ __forceinline__ void coef_pairs(const SceneView<T> &S, const NbrList &L, unsigned lb,
                                           int i, uint32_t sub, const vec4_t<T> *__restrict__ w,
                                           Fn &&fn) {
  const uint32_t info = L.info[i];
  const size_t n = static_cast<size_t>(S.nf);
  const Spans R = pass_spans<kLanes>(L, S.nf, lb);
  const uint32_t c0 = info & 0xFFu;
  const uint32_t c01 = c0 + ((info >> 8) & 0xFFu);
  const uint32_t c = list_count(info);
  const uint32_t d1 = R.b1 - R.b0, d2 = R.b2 - R.b1;
  const vec4_t<T> *__restrict__ coef = reinterpret_cast<const vec4_t<T> *>(S.pcoef);
  for (uint32_t g = sub; g * kChunk < c; g += kLanes) {
    const uint4 q = list_chunk(L, n, i, g);
    const vec4_t<T> ca = coef[(2 * static_cast<size_t>(g)) * n + i];
    vec4_t<T> cb = ca;
    if (g * kChunk + 4 < c)
      cb = coef[(2 * static_cast<size_t>(g) + 1) * n + i];
    vec4_t<T> wj[kChunk];
#pragma unroll
    for (int k = 0; k < static_cast<int>(kChunk); ++k) {
      const uint32_t e = g * kChunk + k;
      if (e < c)
        wj[k] = w[R.b0 + chunk_entry(q, k) + (e >= c0 ? d1 : 0u) + (e >= c01 ? d2 : 0u)];
    }
    __builtin_amdgcn_sched_barrier(0);
    const T cf[8] = {ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w};
#pragma unroll
    for (int k = 0; k < static_cast<int>(kChunk); ++k)
      if (g * kChunk + k < c)
        fn(cf[k], wj[k]);
  }
}

// ---- pt16.setup; with kList (fused steps) one list pass for the fluid sums
// that also writes the step's pair coefficients m_j W_ij
template <class T, bool kList, int kLanes>
__device__ __forceinline__ void pt16_setup_body(const SceneView<T> &S, const NbrList &L, T xi,
                                                unsigned lb) {
#pragma clang fp contract(off)
  const int i = static_cast<int>((lb * kBlock + threadIdx.x) / kLanes);
  const uint32_t sub = threadIdx.x % kLanes;
  const bool valid = i < S.nf;
  if (kLanes == 1 && !valid)
    return;
  const vec4_t<T> zero4 = make4<vec4_t<T>>(T(0), T(0), T(0), T(0));
  const vec4_t<T> xv = valid ? S.xm[i] : zero4;
  const vec4_t<T> vi = valid ? S.v[i] : zero4;
  const T rhoi = valid ? S.rho[i] : T(1);
  const uint32_t cell = valid ? S.fcell[i] : 0u;
  // same-group density and the smoothed density (pt16.prtcl:53-71), and the
  // velocity gradient sum_f m_j (v_j - v_i) gradW_ij^T / rho_i
  // (pt16.prtcl:76-88)
  T same = 0, prho = 0;
  T vg[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  auto grad_term = [&](const vec4_t<T> &vj, T d0, T d1, T d2, T r2, const vec4_t<T> &pj) {
    const T dv[3] = {vj.x - vi.x, vj.y - vi.y, vj.z - vi.z};
    const T f = S.K.gradf(r2);
    const T g[3] = {f * d0, f * d1, f * d2};
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int r = 0; r < 3; ++r)
        vg[r + 3 * c] += pj.w * (dv[r] * g[c]);
  };
  if (kList) {
    const size_t n = static_cast<size_t>(S.nf);
    if (valid) {
      fluid_pairs_list<kLanes>(
          S, L, lb, i, sub, xv, [&](uint32_t j) { return S.v[j]; },
          [&](const vec4_t<T> &vj, T d0, T d1, T d2, T r2, const vec4_t<T> &pj, uint32_t e) {
            const T w = S.K.w(r2);
            same += pj.w * w;
            prho += (pj.w / S.rho0) * w;
            if (e < kSelfEntry)
              S.pcoef[coef_index(n, i, e)] = pj.w * w;
            if (e != kSelfEntry)  // the particle's own term is zero
              grad_term(vj, d0, d1, d2, r2, pj);
          });
      if (sub == 0 && list_has_boundary(L.info[i]))
        nbrs_exact(S, xv, cell, S.bstart, S.bxV,
                   [&](uint32_t, T, T, T, T r2, const vec4_t<T> &pb) { prho += pb.w * S.K.w(r2); });
    }
    same = lanes_sum<kLanes>(same);
    prho = lanes_sum<kLanes>(prho);
#pragma unroll
    for (int k = 0; k < 9; ++k)
      vg[k] = lanes_sum<kLanes>(vg[k]);
    if (!valid || sub != 0)
      return;
    prho *= S.rho0;
  } else {
    nbrs_exact(S, xv, cell, S.fstart, S.xm,
               [&](uint32_t, T, T, T, T r2, const vec4_t<T> &pj) {
                 same += pj.w * S.K.w(r2);
               });
    nbrs_exact(S, xv, cell, S.fstart, S.xm,
               [&](uint32_t, T, T, T, T r2, const vec4_t<T> &pj) {
                 prho += (pj.w / S.rho0) * S.K.w(r2);
               });
    nbrs_exact(S, xv, cell, S.bstart, S.bxV,
               [&](uint32_t, T, T, T, T r2, const vec4_t<T> &pb) { prho += pb.w * S.K.w(r2); });
    prho *= S.rho0;
    nbrs_exact(S, xv, cell, S.fstart, S.xm,
               [&](uint32_t j, T d0, T d1, T d2, T r2, const vec4_t<T> &pj) {
                 grad_term(S.v[j], d0, d1, d2, r2, pj);
               });
  }
#pragma unroll
  for (int k = 0; k < 9; ++k)
    vg[k] /= rhoi;
  // spin, expansion and shear rate (pt16.prtcl:90-105)
  const T div = vg[0] + (vg[4] + vg[8]);
  T R[9], V[9], Sh[9];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      R[r + 3 * c] = (vg[r + 3 * c] - vg[c + 3 * r]) / T(2);
      V[r + 3 * c] = (div / T(3)) * ((r == c) ? T(1) : T(0));
      Sh[r + 3 * c] = ((vg[r + 3 * c] + vg[c + 3 * r]) / T(2)) - V[r + 3 * c];
    }
  // vorticity = 2 (R(2,1), R(0,2), R(1,0)); the target velocity gradient
  // without the spin: V unit_step_r(0, rho - rho0, -div) + xi S
  S.om[i] = make4<vec4_t<T>>(T(2) * R[2 + 3 * 1], T(2) * R[0 + 3 * 2], T(2) * R[1 + 3 * 0], T(0));
  const T step = ((T(0) <= rhoi - S.rho0) || (T(0) <= -div)) ? T(1) : T(0);
  T *G = S.tvg + 9 * static_cast<size_t>(i);
#pragma unroll
  for (int k = 0; k < 9; ++k)
    G[k] = V[k] * step + xi * Sh[k];
  S.psrho[i] = same;
  S.prho[i] = prho;
}

template <class T, bool kList, int kLanes>
__global__ __launch_bounds__(kBlock) void k_pt16_setup(SceneView<T> S, NbrList L, T xi) {
  pt16_setup_body<T, kList, kLanes>(S, L, xi,
                                    kList ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x);
}

// ---- vorticity diffusion rhs; with kList the coefficients m_j W_ij of the
// set-up are streamed and only w_j is gathered (the particle's own term is
// zero)
template <class T, bool kList, int kLanes>
__device__ __forceinline__ void pt16_omega_rhs_body(const SceneView<T> &S, const NbrList &L,
                                                    T xi, unsigned lb) {
#pragma clang fp contract(off)
  const int i = static_cast<int>((lb * kBlock + threadIdx.x) / kLanes);
  const uint32_t sub = threadIdx.x % kLanes;
  const bool valid = i < S.nf;
  if (kLanes == 1 && !valid)
    return;
  T a[3] = {0, 0, 0};
  if (valid) {
    const vec4_t<T> wi = S.om[i];
    if (kList && !(L.info[i] & kListOverflow)) {
      coef_pairs<kLanes>(S, L, lb, i, sub, S.om, [&](T c, const vec4_t<T> &wj) {
        a[0] += c * (wi.x - wj.x);
        a[1] += c * (wi.y - wj.y);
        a[2] += c * (wi.z - wj.z);
      });
    } else if (sub == 0) {
      nbrs_exact(S, S.xm[i], S.fcell[i], S.fstart, S.xm,
                 [&](uint32_t j, T, T, T, T r2, const vec4_t<T> &pj) {
                   const vec4_t<T> wj = S.om[j];
                   const T w = S.K.w(r2);
                   a[0] += (pj.w * (wi.x - wj.x)) * w;
                   a[1] += (pj.w * (wi.y - wj.y)) * w;
                   a[2] += (pj.w * (wi.z - wj.z)) * w;
                 });
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k)
    a[k] = lanes_sum<kLanes>(a[k]);
  if (valid && sub == 0)
    S.orhs[i] = make4<vec4_t<T>>(a[0] * xi, a[1] * xi, a[2] * xi, T(0));
}

template <class T, bool kList, int kLanes>
__global__ __launch_bounds__(kBlock) void k_pt16_omega_rhs(SceneView<T> S, NbrList L, T xi) {
  pt16_omega_rhs_body<T, kList, kLanes>(S, L, xi,
                                        kList ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x);
}

// ---- velocity reconstruction rhs
template <class T, bool kList, int kLanes>
__device__ __forceinline__ void pt16_vrec_rhs_body(const SceneView<T> &S, const NbrList &L,
                                                   unsigned lb) {
#pragma clang fp contract(off)
  const int i = static_cast<int>((lb * kBlock + threadIdx.x) / kLanes);
  const uint32_t sub = threadIdx.x % kLanes;
  const bool valid = i < S.nf;
  if (kLanes == 1 && !valid)
    return;
  T a[3] = {0, 0, 0};
  if (valid) {
    const vec4_t<T> xv = S.xm[i];
    T Gi[9];
#pragma unroll
    for (int k = 0; k < 9; ++k)
      Gi[k] = S.tvg[9 * static_cast<size_t>(i) + k];
    struct Grad {
      T g[9];
    };
    auto load = [&](uint32_t j) {
      Grad q;
#pragma unroll
      for (int k = 0; k < 9; ++k)
        q.g[k] = S.tvg[9 * static_cast<size_t>(j) + k];
      return q;
    };
    auto term = [&](const Grad &Gj, T d0, T d1, T d2, T r2, const vec4_t<T> &pj) {
      T M[9];
#pragma unroll
      for (int k = 0; k < 9; ++k)
        M[k] = Gi[k] + Gj.g[k];
      const T mh = pj.w * T(0.5);
      const T w = S.K.w(r2);
#pragma unroll
      for (int r = 0; r < 3; ++r)
        a[r] += (mh * (M[r] * d0 + (M[r + 3] * d1 + M[r + 6] * d2))) * w;
    };
    if (kList)
      fluid_pairs_list<kLanes>(S, L, lb, i, sub, xv, load,
                               [&](const Grad &Gj, T d0, T d1, T d2, T r2, const vec4_t<T> &pj,
                                   uint32_t e) {
                                 if (e != kSelfEntry)  // x_ii = 0: the own term is zero
                                   term(Gj, d0, d1, d2, r2, pj);
                               });
    else
      nbrs_exact(S, xv, S.fcell[i], S.fstart, S.xm,
                 [&](uint32_t j, T d0, T d1, T d2, T r2, const vec4_t<T> &pj) {
                   term(load(j), d0, d1, d2, r2, pj);
                 });
  }
#pragma unroll
  for (int k = 0; k < 3; ++k)
    a[k] = lanes_sum<kLanes>(a[k]);
  if (valid && sub == 0)
    S.vrhs[i] = make4<vec4_t<T>>(a[0], a[1], a[2], T(0));
}

template <class T, bool kList, int kLanes>
__global__ __launch_bounds__(kBlock) void k_pt16_vrec_rhs(SceneView<T> S, NbrList L) {
  pt16_vrec_rhs_body<T, kList, kLanes>(S, L,
                                       kList ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x);
}

// ---- spin: G += cross_product_matrix(0.5 w) (eigen.hpp:330-339)
template <class T>
__device__ __forceinline__ void pt16_spin_body(const SceneView<T> &S, unsigned lb) {
#pragma clang fp contract(off)
  const int i = static_cast<int>(lb * kBlock + threadIdx.x);
  if (i >= S.nf)
    return;
  const vec4_t<T> w = S.om[i];
  const T a0 = T(0.5) * w.x, a1 = T(0.5) * w.y, a2 = T(0.5) * w.z;
  T *G = S.tvg + 9 * static_cast<size_t>(i);
  // column-major (r, c) at r + 3c: [[0, -a2, a1], [a2, 0, -a0], [-a1, a0, 0]]
  const T C[9] = {T(0), a2, -a1, -a2, T(0), a0, a1, -a0, T(0)};
#pragma unroll
  for (int k = 0; k < 9; ++k)
    G[k] += C[k];
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_spin(SceneView<T> S) {
  pt16_spin_body(S, blockIdx.x);
}

// ---- the three scalar systems of a solve
// system diagonal coefficient and preconditioner of the reference:
//   (A x)_i = c_i x_i - sum_f (m_j W_ij) x_j, c = pt16_same_density (which 0)
//   or pt16_density (which 1); P y = y / (pt16_same_density_i - m_i W(0))

// A w at particle i in lane 0 of its kLanes lanes, w_i = wi; list form:
// c_i w_i - m_i W(0) w_i - sum_list (m_j W_ij) w_j
template <class T, bool kList, int kLanes>
__device__ __forceinline__ void product3(const SceneView<T> &S, const NbrList &L, int which,
                                         unsigned lb, int i, bool valid, uint32_t sub,
                                         const vec4_t<T> *__restrict__ w, const vec4_t<T> &wi,
                                         T out[3]) {
#pragma clang fp contract(off)
  out[0] = out[1] = out[2] = T(0);
  if (valid) {
    const bool listed = kList && !(L.info[i] & kListOverflow);
    if (sub == 0) {
      const vec4_t<T> xv = S.xm[i];
      const T c = which == 0 ? S.psrho[i] : S.prho[i];
      out[0] = c * wi.x;
      out[1] = c * wi.y;
      out[2] = c * wi.z;
      if (listed) {
        const T self = xv.w * S.K.w(T(0));
        out[0] -= self * wi.x;
        out[1] -= self * wi.y;
        out[2] -= self * wi.z;
      } else {
        nbrs_exact(S, xv, S.fcell[i], S.fstart, S.xm,
                   [&](uint32_t j, T, T, T, T r2, const vec4_t<T> &pj) {
                     const vec4_t<T> wj = w[j];
                     const T k = pj.w * S.K.w(r2);
                     out[0] -= k * wj.x;
                     out[1] -= k * wj.y;
                     out[2] -= k * wj.z;
                   });
      }
    }
    if (listed)
      coef_pairs<kLanes>(S, L, lb, i, sub, w, [&](T c, const vec4_t<T> &wj) {
#pragma clang fp contract(off)
        out[0] -= c * wj.x;
        out[1] -= c * wj.y;
        out[2] -= c * wj.z;
      });
  }
#pragma unroll
  for (int k = 0; k < 3; ++k)
    out[k] = lanes_sum<kLanes>(out[k]);
}

// x = guess, r = A x - b, y = P r, p = -y; partials b.b, r.r, r.y
template <class T, bool kList, int kLanes>
__device__ __forceinline__ void pt16_cg_setup_body(const SceneView<T> &S, const NbrList &L,
                                                   int which, double *part, unsigned lb,
                                                   unsigned nb) {
#pragma clang fp contract(off)
  const int i = static_cast<int>((lb * kBlock + threadIdx.x) / kLanes);
  const uint32_t sub = threadIdx.x % kLanes;
  const bool valid = i < S.nf;
  const vec4_t<T> *guess = which == 0 ? S.om : S.v;
  const vec4_t<T> zero4 = make4<vec4_t<T>>(T(0), T(0), T(0), T(0));
  const vec4_t<T> x0 = valid ? guess[i] : zero4;
  T ax[3];
  product3<T, kList, kLanes>(S, L, which, lb, i, valid, sub, guess, x0, ax);
  double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (valid && sub == 0) {
    const vec4_t<T> b = (which == 0 ? S.orhs : S.vrhs)[i];
    const T den = S.psrho[i] - S.xm[i].w * S.K.w(T(0));
    const T r[3] = {ax[0] - b.x, ax[1] - b.y, ax[2] - b.z};
    const T y[3] = {r[0] / den, r[1] / den, r[2] / den};
    const T bv[3] = {b.x, b.y, b.z};
    S.cx[i] = make4<vec4_t<T>>(x0.x, x0.y, x0.z, T(0));
    S.cr[i] = make4<vec4_t<T>>(r[0], r[1], r[2], T(0));
    S.cy[i] = make4<vec4_t<T>>(y[0], y[1], y[2], T(0));
    S.cxp[i] = make4<vec4_t<T>>(-y[0], -y[1], -y[2], T(0));
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      acc[k] = static_cast<double>(bv[k] * bv[k]);
      acc[3 + k] = static_cast<double>(r[k] * r[k]);
      acc[6 + k] = static_cast<double>(r[k] * y[k]);
    }
  }
  store_partials<9>(part, nb, acc, lb);
}

template <class T, bool kList, int kLanes>
__global__ __launch_bounds__(kBlock) void k_pt16_cg_setup(SceneView<T> S, NbrList L, int which,
                                                          double *part) {
  pt16_cg_setup_body<T, kList, kLanes>(S, L, which, part, xcd_block(blockIdx.x, gridDim.x),
                                       gridDim.x);
}

__global__ __launch_bounds__(kBlock) void k_pt16_cg_setup_fin(Ctl *c, const double *part,
                                                              unsigned nb, double tol, int max_k,
                                                              unsigned seq) {
  cg3_setup_fin_body(c, part, nb, tol, max_k, seq);
}

// q = A p, partials p.q
template <class T, bool kList, int kLanes>
__device__ __forceinline__ void pt16_cg_spmv_body(const SceneView<T> &S, const NbrList &L,
                                                  int which, double *part, unsigned lb,
                                                  unsigned nb) {
#pragma clang fp contract(off)
  if (S.ctl->cg_done)
    return;
  const int i = static_cast<int>((lb * kBlock + threadIdx.x) / kLanes);
  const uint32_t sub = threadIdx.x % kLanes;
  const bool valid = i < S.nf;
  const vec4_t<T> p = valid ? S.cxp[i] : make4<vec4_t<T>>(T(0), T(0), T(0), T(0));
  T q[3];
  product3<T, kList, kLanes>(S, L, which, lb, i, valid, sub, S.cxp, p, q);
  double acc[3] = {0.0, 0.0, 0.0};
  if (valid && sub == 0) {
    S.cq[i] = make4<vec4_t<T>>(q[0], q[1], q[2], T(0));
    acc[0] = static_cast<double>(p.x * q[0]);
    acc[1] = static_cast<double>(p.y * q[1]);
    acc[2] = static_cast<double>(p.z * q[2]);
  }
  store_partials<3>(part, nb, acc, lb);
}

template <class T, bool kList, int kLanes>
__global__ __launch_bounds__(kBlock) void k_pt16_cg_spmv(SceneView<T> S, NbrList L, int which,
                                                         double *part) {
  pt16_cg_spmv_body<T, kList, kLanes>(S, L, which, part, xcd_block(blockIdx.x, gridDim.x),
                                      gridDim.x);
}

// a particle's vectors of the update, loaded ahead of the scalars
template <class T>
struct Pt16Own {
  vec4_t<T> x, r, p, q;
  T den;
  __device__ __forceinline__ Pt16Own(const SceneView<T> &S, int i) {
    if (i < S.nf) {
      x = S.cx[i];
      r = S.cr[i];
      p = S.cxp[i];
      q = S.cq[i];
      den = S.psrho[i] - S.xm[i].w * S.K.w(T(0));
    }
  }
};

// x += alpha p, r += alpha q, y = P r of the components in `on`; partials r.r, r.y
template <class T>
__device__ __forceinline__ void pt16_update_body(const SceneView<T> &S, const Pt16Own<T> &o,
                                                 unsigned on, const double (&alpha)[3],
                                                 double *part, unsigned lb, unsigned nb) {
#pragma clang fp contract(off)
  const int i = static_cast<int>(lb * kBlock + threadIdx.x);
  double acc[6] = {0, 0, 0, 0, 0, 0};
  if (i < S.nf) {
    T x[3] = {o.x.x, o.x.y, o.x.z}, r[3] = {o.r.x, o.r.y, o.r.z}, y[3];
    const T p[3] = {o.p.x, o.p.y, o.p.z}, q[3] = {o.q.x, o.q.y, o.q.z};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if ((on >> k) & 1u) {
        const T a = static_cast<T>(alpha[k]);
        x[k] = x[k] + a * p[k];
        r[k] = r[k] + a * q[k];
      }
      y[k] = r[k] / o.den;
      acc[k] = static_cast<double>(r[k] * r[k]);
      acc[3 + k] = static_cast<double>(r[k] * y[k]);
    }
    S.cx[i] = make4<vec4_t<T>>(x[0], x[1], x[2], T(0));
    S.cr[i] = make4<vec4_t<T>>(r[0], r[1], r[2], T(0));
    S.cy[i] = make4<vec4_t<T>>(y[0], y[1], y[2], T(0));
  }
  store_partials<6>(part, nb, acc, lb);
}

// p = -y + beta p of the components in `on`
template <class T>
__device__ __forceinline__ void pt16_direction_body(const SceneView<T> &S, const vec4_t<T> &y,
                                                    const vec4_t<T> &p, unsigned on,
                                                    const double (&beta)[3], unsigned lb) {
#pragma clang fp contract(off)
  const int i = static_cast<int>(lb * kBlock + threadIdx.x);
  if (i >= S.nf)
    return;
  const T yv[3] = {y.x, y.y, y.z};
  T pv[3] = {p.x, p.y, p.z};
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if ((on >> k) & 1u)
      pv[k] = -yv[k] + static_cast<T>(beta[k]) * pv[k];
  S.cxp[i] = make4<vec4_t<T>>(pv[0], pv[1], pv[2], T(0));
}

// The update and direction kernels of one scene. fold: the block derives alpha
// (beta) from the partials of the kernel before it, npq (nb) blocks of it, and
// block 0 stores them; otherwise a one-block kernel has stored them.
template <class T>
__device__ __forceinline__ void pt16_update(const SceneView<T> &S, bool fold,
                                            const double *pq_part, unsigned npq, double *part,
                                            unsigned lb, unsigned nb) {
  Ctl *c = S.ctl;
  const Pt16Own<T> own(S, static_cast<int>(lb * kBlock + threadIdx.x));
  unsigned live = cg3_live(c);
  if (live == 0u)
    return;
  double alpha[3];
  if (fold) {
    live = cg3_alpha(c, pq_part, npq, live, lb == 0, alpha);
    if (live == 0u)
      return;
  } else {
#pragma unroll
    for (int k = 0; k < 3; ++k)
      alpha[k] = c->c3.alpha[k];
  }
  pt16_update_body(S, own, live, alpha, part, lb, nb);
}

template <class T>
__device__ __forceinline__ void pt16_direction(const SceneView<T> &S, bool fold,
                                               const double *part, unsigned lb, unsigned nb) {
  Ctl *c = S.ctl;
  const int i = static_cast<int>(lb * kBlock + threadIdx.x);
  vec4_t<T> y = make4<vec4_t<T>>(T(0), T(0), T(0), T(0)), p = y;
  if (i < S.nf) {
    y = S.cy[i];
    p = S.cxp[i];
  }
  unsigned live = cg3_live(c);
  if (live == 0u)
    return;
  double beta[3];
  if (fold) {
    live = cg3_beta(c, part, nb, live, lb == 0, beta);
    if (live == 0u)
      return;
  } else {
#pragma unroll
    for (int k = 0; k < 3; ++k)
      beta[k] = c->c3.beta[k];
  }
  pt16_direction_body(S, y, p, live, beta, lb);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_cg_update(SceneView<T> S, int fold,
                                                           const double *pq_part, unsigned npq,
                                                           double *part) {
  pt16_update(S, fold != 0, pq_part, npq, part, blockIdx.x, gridDim.x);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_cg_direction(SceneView<T> S, int fold,
                                                              const double *part) {
  pt16_direction(S, fold != 0, part, blockIdx.x, gridDim.x);
}

// one block: alpha and beta of a launch of more than kFusedCgBlocks blocks
__device__ __forceinline__ void pt16_alpha_body(Ctl *c, const double *part, unsigned nb) {
  const unsigned live = cg3_live(c);
  double alpha[3];
  if (live != 0u)
    cg3_alpha(c, part, nb, live, true, alpha);
}
__device__ __forceinline__ void pt16_beta_body(Ctl *c, const double *part, unsigned nb) {
  const unsigned live = cg3_live(c);
  double beta[3];
  if (live != 0u)
    cg3_beta(c, part, nb, live, true, beta);
}
__global__ __launch_bounds__(kBlock) void k_pt16_cg_alpha(Ctl *c, const double *part,
                                                          unsigned nb) {
  pt16_alpha_body(c, part, nb);
}
__global__ __launch_bounds__(kBlock) void k_pt16_cg_beta(Ctl *c, const double *part,
                                                         unsigned nb) {
  pt16_beta_body(c, part, nb);
}

// apply (pt16.hpp:491-502, 700-717): the vorticity (which 0) or the velocity
// (which 1) = x unit_step_l(0, (t - t_birth) - dt_fade) +
// old unit_step_r(0, dt_fade - (t - t_birth)); the control block keeps the last
// component's count, as after the reference's last solve
template <class T>
__device__ __forceinline__ void pt16_cg_apply_body(const SceneView<T> &S, int which,
                                                   unsigned lb) {
#pragma clang fp contract(off)
  const int i = static_cast<int>(lb * kBlock + threadIdx.x);
  if (i == 0)
    S.ctl->cg_iter = S.ctl->c3.iter[2];
  if (i >= S.nf)
    return;
  const T tb = S.v[i].w;
  const T age = S.t - tb;
  const T on = (T(0) < age - S.fade) ? T(1) : T(0);
  const T keep = (T(0) <= S.fade - age) ? T(1) : T(0);
  vec4_t<T> *f = (which == 0 ? S.om : S.v) + i;
  vec4_t<T> o = *f;
  const vec4_t<T> x = S.cx[i];
  o.x = x.x * on + o.x * keep;
  o.y = x.y * on + o.y * keep;
  o.z = x.z * on + o.z * keep;
  *f = o;
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_cg_apply(SceneView<T> S, int which) {
  pt16_cg_apply_body(S, which, blockIdx.x);
}

// ---- batched forms (prtcl_hip_step over several scenes, list forms): the
// bodies above over the blocks of every pt16 scene of a table (B: its blocks),
// each block with its scene's view, list, CG partials and block counts. The
// vorticity solve runs under sequence number cg_seq, the velocity solve under
// cg_seq + 1, each with the tolerance and cap of its system.
#define PT16_BATCH_ENTRY(kF)                                               \
  unsigned part_;                                                          \
  const uint32_t u = batch_block(B, kF, &part_);                           \
  const BatchEntry<T> &E = tab[u >> kBatchLocalBits];                      \
  const bool split = split_scene(E.S.nf);                                  \
  const unsigned lb = (u & kBatchLocalMask) * (split ? (kF) : 1u) + part_; \
  const NbrList L{E.nidx, E.ninfo, E.nblk, E.nshift};                      \
  (void)split;                                                             \
  (void)L;                                                                 \
  if (lb >= ((kF) == 1u ? E.nblocks : list_blocks(E.S.nf)))                \
  return

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_setup_b(const BatchEntry<T> *tab,
                                                         BatchBlocks B) {
  PT16_BATCH_ENTRY(kListLanes);
  if (split)
    pt16_setup_body<T, true, kListLanes>(E.S, L, static_cast<T>(E.pt16_xi), lb);
  else
    pt16_setup_body<T, true, 1>(E.S, L, static_cast<T>(E.pt16_xi), lb);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_omega_rhs_b(const BatchEntry<T> *tab,
                                                             BatchBlocks B) {
  PT16_BATCH_ENTRY(kListLanes);
  if (split)
    pt16_omega_rhs_body<T, true, kListLanes>(E.S, L, static_cast<T>(E.pt16_xi), lb);
  else
    pt16_omega_rhs_body<T, true, 1>(E.S, L, static_cast<T>(E.pt16_xi), lb);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_spin_b(const BatchEntry<T> *tab,
                                                        BatchBlocks B) {
  PT16_BATCH_ENTRY(1u);
  pt16_spin_body(E.S, lb);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_vrec_rhs_b(const BatchEntry<T> *tab,
                                                            BatchBlocks B) {
  PT16_BATCH_ENTRY(kListLanes);
  if (split)
    pt16_vrec_rhs_body<T, true, kListLanes>(E.S, L, lb);
  else
    pt16_vrec_rhs_body<T, true, 1>(E.S, L, lb);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_cg_setup_b(const BatchEntry<T> *tab,
                                                            BatchBlocks B, int which) {
  PT16_BATCH_ENTRY(kListLanes);
  const unsigned nl = list_blocks(E.S.nf);
  if (split)
    pt16_cg_setup_body<T, true, kListLanes>(E.S, L, which, E.cg_part, lb, nl);
  else
    pt16_cg_setup_body<T, true, 1>(E.S, L, which, E.cg_part, lb, nl);
}

// one block per scene
template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_cg_setup_fin_b(const BatchEntry<T> *tab,
                                                                int which) {
  const BatchEntry<T> &E = tab[blockIdx.x];
  cg3_setup_fin_body(E.S.ctl, E.cg_part, list_blocks(E.S.nf), E.pt16_tol[which],
                     E.pt16_max_k[which], E.cg_seq + static_cast<unsigned>(which));
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_cg_spmv_b(const BatchEntry<T> *tab,
                                                           BatchBlocks B, int which) {
  PT16_BATCH_ENTRY(kListLanes);
  const unsigned nl = list_blocks(E.S.nf);
  if (split)
    pt16_cg_spmv_body<T, true, kListLanes>(E.S, L, which, E.cg_part, lb, nl);
  else
    pt16_cg_spmv_body<T, true, 1>(E.S, L, which, E.cg_part, lb, nl);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_cg_alpha_b(const BatchEntry<T> *tab) {
  const BatchEntry<T> &E = tab[blockIdx.x];
  if (!E.cg_fold)
    pt16_alpha_body(E.S.ctl, E.cg_part, list_blocks(E.S.nf));
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_cg_beta_b(const BatchEntry<T> *tab) {
  const BatchEntry<T> &E = tab[blockIdx.x];
  if (!E.cg_fold)
    pt16_beta_body(E.S.ctl, E.cg_part + 3 * list_blocks(E.S.nf), E.nblocks);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_cg_update_b(const BatchEntry<T> *tab,
                                                             BatchBlocks B) {
  PT16_BATCH_ENTRY(1u);
  const unsigned nl = list_blocks(E.S.nf);
  pt16_update(E.S, E.cg_fold != 0, E.cg_part, nl, E.cg_part + 3 * nl, lb, E.nblocks);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_cg_direction_b(const BatchEntry<T> *tab,
                                                                BatchBlocks B) {
  PT16_BATCH_ENTRY(1u);
  pt16_direction(E.S, E.cg_fold != 0, E.cg_part + 3 * list_blocks(E.S.nf), lb, E.nblocks);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pt16_cg_apply_b(const BatchEntry<T> *tab,
                                                            BatchBlocks B, int which) {
  PT16_BATCH_ENTRY(1u);
  pt16_cg_apply_body(E.S, which, lb);
}

#undef PT16_BATCH_ENTRY

// a list kernel with the scene's lanes per particle, or its grid form
#define PT16_LAUNCH(kern, ...)                                                               \
  do {                                                                                       \
    const dim3 bl(kBlock);                                                                   \
    if (L && split_scene(S.nf))                                                              \
      hipLaunchKernelGGL((kern<T, true, kListLanes>), dim3(list_blocks(S.nf)), bl, 0, st, S, \
                         *L, ##__VA_ARGS__);                                                 \
    else if (L)                                                                              \
      hipLaunchKernelGGL((kern<T, true, 1>), dim3(grid_blocks(S.nf)), bl, 0, st, S, *L,      \
                         ##__VA_ARGS__);                                                     \
    else                                                                                     \
      hipLaunchKernelGGL((kern<T, false, 1>), dim3(grid_blocks(S.nf)), bl, 0, st, S,         \
                         NbrList{}, ##__VA_ARGS__);                                          \
  } while (0)

}  // namespace

template <class T>
void Pt16Ops<T>::setup_batch(hipStream_t st, const BatchEntry<T> *tab, const BatchBlocks &B) {
  if (const unsigned n = B.launch(kListLanes))
    hipLaunchKernelGGL(k_pt16_setup_b<T>, dim3(n), dim3(kBlock), 0, st, tab, B);
}

template <class T>
void Pt16Ops<T>::omega_rhs_batch(hipStream_t st, const BatchEntry<T> *tab, const BatchBlocks &B) {
  if (const unsigned n = B.launch(kListLanes))
    hipLaunchKernelGGL(k_pt16_omega_rhs_b<T>, dim3(n), dim3(kBlock), 0, st, tab, B);
}

template <class T>
void Pt16Ops<T>::spin_batch(hipStream_t st, const BatchEntry<T> *tab, const BatchBlocks &B) {
  if (const unsigned n = B.launch(1))
    hipLaunchKernelGGL(k_pt16_spin_b<T>, dim3(n), dim3(kBlock), 0, st, tab, B);
}

template <class T>
void Pt16Ops<T>::vrec_rhs_batch(hipStream_t st, const BatchEntry<T> *tab, const BatchBlocks &B) {
  if (const unsigned n = B.launch(kListLanes))
    hipLaunchKernelGGL(k_pt16_vrec_rhs_b<T>, dim3(n), dim3(kBlock), 0, st, tab, B);
}

template <class T>
void Pt16Ops<T>::cg_setup_batch(hipStream_t st, const BatchEntry<T> *tab, const BatchBlocks &B,
                                unsigned nscenes, int which) {
  if (nscenes == 0)
    return;
  if (const unsigned n = B.launch(kListLanes))
    hipLaunchKernelGGL(k_pt16_cg_setup_b<T>, dim3(n), dim3(kBlock), 0, st, tab, B, which);
  hipLaunchKernelGGL(k_pt16_cg_setup_fin_b<T>, dim3(nscenes), dim3(kBlock), 0, st, tab, which);
}

template <class T>
void Pt16Ops<T>::cg_iteration_batch(hipStream_t st, const BatchEntry<T> *tab,
                                    const BatchBlocks &B, unsigned nscenes, int which,
                                    bool any_split) {
  const unsigned nl = B.launch(kListLanes), n = B.launch(1);
  if (n == 0)
    return;
  const dim3 bl(kBlock);
  hipLaunchKernelGGL(k_pt16_cg_spmv_b<T>, dim3(nl), bl, 0, st, tab, B, which);
  if (any_split)
    hipLaunchKernelGGL(k_pt16_cg_alpha_b<T>, dim3(nscenes), bl, 0, st, tab);
  hipLaunchKernelGGL(k_pt16_cg_update_b<T>, dim3(n), bl, 0, st, tab, B);
  if (any_split)
    hipLaunchKernelGGL(k_pt16_cg_beta_b<T>, dim3(nscenes), bl, 0, st, tab);
  hipLaunchKernelGGL(k_pt16_cg_direction_b<T>, dim3(n), bl, 0, st, tab, B);
}

template <class T>
void Pt16Ops<T>::cg_apply_batch(hipStream_t st, const BatchEntry<T> *tab, const BatchBlocks &B,
                                int which) {
  if (const unsigned n = B.launch(1))
    hipLaunchKernelGGL(k_pt16_cg_apply_b<T>, dim3(n), dim3(kBlock), 0, st, tab, B, which);
}

template <class T>
void Pt16Ops<T>::setup(hipStream_t st, const SceneView<T> &S, const NbrList *L, T xi) {
  if (S.nf > 0)
    PT16_LAUNCH(k_pt16_setup, xi);
}

template <class T>
void Pt16Ops<T>::omega_rhs(hipStream_t st, const SceneView<T> &S, const NbrList *L, T xi) {
  if (S.nf > 0)
    PT16_LAUNCH(k_pt16_omega_rhs, xi);
}

template <class T>
void Pt16Ops<T>::vrec_rhs(hipStream_t st, const SceneView<T> &S, const NbrList *L) {
  if (S.nf > 0)
    PT16_LAUNCH(k_pt16_vrec_rhs);
}

template <class T>
void Pt16Ops<T>::spin(hipStream_t st, const SceneView<T> &S) {
  if (S.nf > 0)
    hipLaunchKernelGGL(k_pt16_spin<T>, dim3(grid_blocks(S.nf)), dim3(kBlock), 0, st, S);
}

template <class T>
void Pt16Ops<T>::cg_setup(hipStream_t st, const SceneView<T> &S, const NbrList *L, int which,
                          double *part, double tol, int max_k, unsigned seq) {
  if (S.nf > 0)
    PT16_LAUNCH(k_pt16_cg_setup, which, part);
  hipLaunchKernelGGL(k_pt16_cg_setup_fin, dim3(1), dim3(kBlock), 0, st, S.ctl, part,
                     L ? list_blocks(S.nf) : grid_blocks(S.nf), tol, max_k, seq);
}

template <class T>
void Pt16Ops<T>::cg_iteration(hipStream_t st, const SceneView<T> &S, const NbrList *L,
                              int which, double *part, bool split) {
  if (S.nf <= 0)
    return;
  PT16_LAUNCH(k_pt16_cg_spmv, which, part);
  const unsigned nb = grid_blocks(S.nf), nl = L ? list_blocks(S.nf) : nb;
  const dim3 gr(nb), bl(kBlock);
  // p.q partials at part[0, 3 nl), r.r and r.y at part[3 nl, 3 nl + 6 nb)
  double *part2 = part + 3 * static_cast<size_t>(nl);
  const bool fold = !split && nb <= kFusedCgBlocks;
  if (!fold)
    hipLaunchKernelGGL(k_pt16_cg_alpha, dim3(1), bl, 0, st, S.ctl, part, nl);
  hipLaunchKernelGGL(k_pt16_cg_update<T>, gr, bl, 0, st, S, fold ? 1 : 0, part, nl, part2);
  if (!fold)
    hipLaunchKernelGGL(k_pt16_cg_beta, dim3(1), bl, 0, st, S.ctl, part2, nb);
  hipLaunchKernelGGL(k_pt16_cg_direction<T>, gr, bl, 0, st, S, fold ? 1 : 0, part2);
}

template <class T>
void Pt16Ops<T>::cg_apply(hipStream_t st, const SceneView<T> &S, int which) {
  if (S.nf > 0)
    hipLaunchKernelGGL(k_pt16_cg_apply<T>, dim3(grid_blocks(S.nf)), dim3(kBlock), 0, st, S,
                       which);
}

template struct Pt16Ops<float>;
template struct Pt16Ops<double>;

}  // namespace prtcl_amd
