// Fused step kernels: the reference's step (density, gravity, explicit
// viscosity, integrate velocity, IISPH setup, IISPH iterations, integrate
// velocity / position) regrouped into the fewest neighbour passes.
//
// Regrouping (exact in real arithmetic; FP32 results differ from the
// reference's per-term evaluation by rounding only):
//   G_f = sum_f m_j gradW_ij, G_b = sum_b V_b gradW_ib,
//   c_i  = -(G_f + 1.4 rho0 G_b) / rho_i^2                    (iisph.hpp:197-249)
//   AA_i = dt^2 rho0/rho_i (c_i . (G_f + rho0 G_b) - m_i/rho_i^2 sum_f m_j |gradW|^2)
//   s_i  = (rho0 - rho_i) - dt rho0/rho_i (sum_f m_j (v_i - v_j).gradW + rho0 v_i.G_b)
//   a_i  = p_i c_i - sum_f m_j (p_j/rho_j^2) gradW_ij           (iisph.hpp:358-423)
//   Ap_i = dt^2 rho0/rho_i (a_i . (G_f + rho0 G_b) - sum_f m_j a_j.gradW_ij)
// so boundary particles are visited once per step (in the setup pass) and
// each IISPH iteration is two passes over fluid neighbours only. The setup
// pass records the fluid neighbours (self excluded, exact predicate) in a
// per-step list of 16-bit offsets (nbrlist.hpp), from which the IISPH passes
// gather the neighbours' fields through L2.
// A particle with more neighbours than the list holds is walked over the
// grid instead.
#include <limits>
#include <type_traits>

#include "fused.hpp"
#include "scan8.hpp"

namespace prtcl_amd {

namespace {

template <class T>
__device__ __forceinline__ T rsqrt_fast(T x);
template <>
__device__ __forceinline__ float rsqrt_fast<float>(float x) {
  return __builtin_amdgcn_rsqf(x);
}
template <>
__device__ __forceinline__ double rsqrt_fast<double>(double x) {
  return rsqrt(x);
}

template <class Fn>
__device__ __forceinline__ void runs(const GridDims &g, uint32_t cellc,
                                     const uint32_t *__restrict__ start, Fn &&fn) {
  const int cx = static_cast<int>(cellc & 0x7FFu);
  const int cy = static_cast<int>((cellc >> 11) & 0x7FFu);
  const int cz = static_cast<int>(cellc >> 22);
  const int x0 = cx > 0 ? cx - 1 : 0;
  const int x1 = cx + 1 < g.nx ? cx + 1 : g.nx - 1;
  for (int dz = -1; dz <= 1; ++dz) {
    const int z = cz + dz;
    if (z < 0 || z >= g.nz)
      continue;
    for (int dy = -1; dy <= 1; ++dy) {
      const int y = cy + dy;
      if (y < 0 || y >= g.ny)
        continue;
      const uint32_t row = static_cast<uint32_t>(g.nx) *
                           (static_cast<uint32_t>(y) +
                            static_cast<uint32_t>(g.ny) * static_cast<uint32_t>(z));
      fn(start[row + static_cast<uint32_t>(x0)], start[row + static_cast<uint32_t>(x1) + 1u]);
    }
  }
}

// W and grad-W factor of the cubic spline from r^2 with one reciprocal
// square root: q = r/h, W = aw ((2-q)^3 - 4 (1-q)^3_+),
// dW/dr = ag (12 (1-q)^2_+ - 3 (2-q)^2), gradW = (dW/dr / r) x_ij, and
// gradW = 0 below r = sqrt(eps) as the reference (kernel_facade.hpp:226).
//
// Neighbours satisfy r < 2h, so 2 - q >= 0 up to rounding; with
// t = 2 - q and u = max(2 - 2q, 0):  12 (1-q)^2_+ - 3 (2-q)^2 = 3 (u^2 - t^2).
// gradf_unscaled() returns (u^2 - t^2) / r; the caller multiplies the sum by
// ag3 = 3 alpha / h^4 once.
template <class T>
struct FastSpline {
  T inv_h, aw, ag, ag3, eps2;
  __device__ __forceinline__ void eval(T r2, T &w, T &f) const {
    const T rinv = rsqrt_fast<T>(fmax(r2, std::numeric_limits<T>::min()));
    const T r = r2 * rinv;
    const T q = r * inv_h;
    const T b2 = fmax(T(2) - q, T(0));
    const T b1p = fmax(T(1) - q, T(0));
    w = aw * (b2 * b2 * b2 - T(4) * b1p * b1p * b1p);
    const T dw = ag * (T(12) * b1p * b1p - T(3) * b2 * b2);
    f = r2 < eps2 ? T(0) : dw * rinv;
  }
  __device__ __forceinline__ T gradf(T r2) const { return ag3 * gradf_unscaled(r2); }
  __device__ __forceinline__ T gradf_unscaled(T r2) const {
    const T rinv = rsqrt_fast<T>(r2);  // r2 = 0 gives inf/NaN, masked below
    const T q = r2 * rinv * inv_h;
    const T t = T(2) - q;
    T u = T(2) - T(2) * q;
    u = u > T(0) ? u : T(0);
    const T d = (u * u - t * t) * rinv;
    return r2 < eps2 ? T(0) : d;
  }
};

template <class T>
__device__ __forceinline__ FastSpline<T> fast_spline(const SceneView<T> &S) {
  FastSpline<T> k;
  const T h = S.K.h;
  k.inv_h = T(1) / h;
  k.aw = S.K.alpha / (h * h * h);
  k.ag = S.K.alpha / (h * h * h * h);
  k.ag3 = T(3) * k.ag;
  k.eps2 = S.K.eps * S.K.eps;
  return k;
}

// the value of the wavefront's first lane in every lane, in scalar registers
template <class T>
__device__ __forceinline__ T scalar(T v) {
  int w[sizeof(T) / sizeof(int)];
  __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
  for (unsigned k = 0; k < sizeof(T) / sizeof(int); ++k)
    w[k] = __builtin_amdgcn_readfirstlane(w[k]);
  __builtin_memcpy(&v, w, sizeof(T));
  return v;
}

// fast_spline with the factors of eval() in scalar registers: the divisions leave
// them in vector registers, and the FP64 setup kernels then need 135 instead of 128,
// one wavefront per SIMD less (27,000 particles 24.6 -> 28.4 us)
template <class T>
__device__ __forceinline__ FastSpline<T> scalar_spline(const SceneView<T> &S) {
  FastSpline<T> k = fast_spline(S);
  k.inv_h = scalar(k.inv_h), k.aw = scalar(k.aw), k.ag = scalar(k.ag);
  k.eps2 = scalar(k.eps2);
  return k;
}

template <class T>
__device__ __forceinline__ T fade_step(const SceneView<T> &S, T t_birth) {
  return (T(0) < (S.t - t_birth) - S.fade) ? T(1) : T(0);
}

// Exact-predicate walk of particle i's 27-cell candidates in global memory:
// fn(j) for every fluid j != i with |x_i - x_j|^2 < r^2 (particles whose list
// overflowed).
template <class T, class Fn>
__device__ __forceinline__ void grid_walk(const SceneView<T> &S, int i, const vec4_t<T> &xi,
                                          Fn &&fn) {
  runs(S.grid, S.fcell[i], S.fstart, [&](uint32_t b, uint32_t e) {
    for (uint32_t j = b; j < e; ++j) {
      const vec4_t<T> pj = S.xm[j];
      if (j != static_cast<uint32_t>(i) &&
          sqdist_exact(xi.x - pj.x, xi.y - pj.y, xi.z - pj.z) < S.thr2)
        fn(j);
    }
  });
}

// the three x-runs of slab s (rows dz = s - 1, dy = -1..1) of a cell, in
// stencil order: fn(b, e); rows outside the box are skipped
template <class Fn>
__device__ __forceinline__ void slab_runs(const GridDims &g, uint32_t cellc,
                                          const uint32_t *__restrict__ start, int s, Fn &&fn) {
  const int cx = static_cast<int>(cellc & 0x7FFu);
  const int cy = static_cast<int>((cellc >> 11) & 0x7FFu);
  const int z = static_cast<int>(cellc >> 22) + s - 1;
  if (z < 0 || z >= g.nz)
    return;
  const int x0 = cx > 0 ? cx - 1 : 0;
  const int x1 = cx + 1 < g.nx ? cx + 1 : g.nx - 1;
#pragma unroll
  for (int dy = -1; dy <= 1; ++dy) {
    const int y = cy + dy;
    if (y < 0 || y >= g.ny)
      continue;
    const uint32_t row = static_cast<uint32_t>(g.nx) *
                         (static_cast<uint32_t>(y) +
                          static_cast<uint32_t>(g.ny) * static_cast<uint32_t>(z));
    fn(start[row + static_cast<uint32_t>(x0)], start[row + static_cast<uint32_t>(x1) + 1u]);
  }
}

// bounds of the three x-runs of slab s of a cell, loaded together (rows
// outside the box give empty runs)
__device__ __forceinline__ void slab_bounds(const GridDims &g, uint32_t cellc,
                                            const uint32_t *__restrict__ start, int s,
                                            uint32_t rb[3], uint32_t re[3]) {
  const int cx = static_cast<int>(cellc & 0x7FFu);
  const int cy = static_cast<int>((cellc >> 11) & 0x7FFu);
  const int z = static_cast<int>(cellc >> 22) + s - 1;
  const bool zok = z >= 0 && z < g.nz;
  const uint32_t x0 = static_cast<uint32_t>(cx > 0 ? cx - 1 : 0);
  const uint32_t x1 = static_cast<uint32_t>(cx + 1 < g.nx ? cx + 1 : g.nx - 1);
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const int y = cy + r - 1;
    const bool ok = zok && y >= 0 && y < g.ny;
    const uint32_t row = ok ? static_cast<uint32_t>(g.nx) *
                                  (static_cast<uint32_t>(y) +
                                   static_cast<uint32_t>(g.ny) * static_cast<uint32_t>(z))
                            : 0u;
    rb[r] = ok ? start[row + x0] : 0u;
    re[r] = ok ? start[row + x1 + 1u] : 0u;
  }
}

__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    const uint32_t u = __shfl_xor(v, o, kWave);
    v = u < v ? u : v;
  }
  return v;
}

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    const uint32_t u = __shfl_xor(v, o, kWave);
    v = u > v ? u : v;
  }
  return v;
}

// Spans of a block (all threads call it): span s runs from the first start
// to the last end of the slab-s runs of the block's particles. Written to R
// (LDS).
__device__ __forceinline__ void block_spans(const GridDims &g, const uint32_t *fstart,
                                            bool valid, uint32_t cell, BlockRanges &R) {
  __shared__ uint32_t lo[3], hi[3];
  if (threadIdx.x < 3) {
    lo[threadIdx.x] = 0xFFFFFFFFu;
    hi[threadIdx.x] = 0u;
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    uint32_t bm = 0xFFFFFFFFu, em = 0u;
    if (valid)
      slab_runs(g, cell, fstart, s, [&](uint32_t b, uint32_t e) {
        if (e > b) {
          bm = b < bm ? b : bm;
          em = e > em ? e : em;
        }
      });
    bm = wave_min_u32(bm);
    em = wave_max_u32(em);
    if (__lane_id() == 0) {
      atomicMin(&lo[s], bm);
      atomicMax(&hi[s], em);
    }
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const uint32_t b = lo[threadIdx.x], e = hi[threadIdx.x];
    R.base[threadIdx.x] = b < e ? b : 0u;
    R.len[threadIdx.x] = b < e ? e - b : 0u;
  }
  __syncthreads();
}

// IISPH iteration 1 of a solve without its neighbour passes (the loop of
// example.lua:409-421 over iisph.hpp:358-516): every pressure is 0 when the
// solve starts (iisph.hpp:282), so the pressure acceleration of iteration 1
// is zero, Ap = 0, and the relaxed Jacobi update and the aprde term need only
// the particle's own s and AA. The expressions are those of
// k_pressure_list_body with p_old = Ap = 0, so p and the aprde term are the
// ones the two passes give, bit for bit. Returns the particle's aprde term.
template <class T>
__device__ __forceinline__ double first_iteration(const SceneView<T> &S, int i,
                                                  const vec4_t<T> &xi, T rhoi, T si, T AA) {
  const T p_old = T(0), Ap = T(0);
  const T rcp = (fabs(AA) > T(1e-9)) ? T(1) / AA : T(0);
  const T upd = p_old + S.omega * (si - Ap) * rcp;
  const T pn = ((T(0) < upd) ? upd : T(0)) * ((T(1e-9) < fabs(AA)) ? T(1) : T(0));
  S.Ap[i] = Ap;
  S.p[i] = pn;
  S.pr[i] = pn / (rhoi * rhoi);
  S.xq[i] = make4<vec4_t<T>>(xi.x, xi.y, xi.z, xi.w * pn / (rhoi * rhoi));
  // the pressure acceleration of iteration 1 (read if the solve stops there)
  S.xa[S.xa_a(static_cast<size_t>(i))] = make4<vec4_t<T>>(T(0), T(0), T(0), T(0));
  return static_cast<double>((Ap - si) / S.rho0 * ((T(1e-9) < pn) ? T(1) : T(0)));
}

// ---------------------------------------------------------------------------
// setup pass: density + neighbour list + IISPH c, AA (+ s when the velocity
// of every neighbour is known without another pass, i.e. no explicit
// viscosity: the sort has stored v*_j = v_j + dt g H_j)
//
// Phase 1 tests the 27-cell candidates by their 16-bit positions (fixed_sqdist)
// and appends the accepted ones (entries relative to the slab's span) to this
// thread's column of an LDS table; phase 2 runs the exact predicate (where the
// 16 bits leave it open) and the pair sums over the compacted entries, so the
// lanes that reject a candidate do not wait for the kernel arithmetic of the
// ones that accept it. The table is written to the list row by row (coalesced).
//
// Bound by vector instructions (82 % busy; the loads' address work 62 %: 216 candidates
// and 30 pairs a particle). With candidates as 16-byte positions and
// 13 instructions, 65 a pair and five wavefronts per SIMD, 1M particles took 229
// us, 250,000 73 us, 16 scenes of 2,000 to 200,000 together 247 us; with 8-byte
// records and 9 instructions, the velocities integrated by the sort and six
// wavefronts 182, 54 and 223 (batches pay for the 8-lane search of their small
// scenes, nbrlist.hpp: 182 with one lane for each).
// ---------------------------------------------------------------------------
// the pair sums of the setup pass for one particle (or one lane's share)
template <class T, bool kWithSource>
struct SetupSums {
  const SceneView<T> &S;
  const FastSpline<T> K;
  vec4_t<T> xi;
  T vs0, vs1, vs2;
  // density, G_f, sum |gradW|^2 and the velocity-divergence sum of the source
  // term; density and G_b of the boundary
  T rho = 0, gf0 = 0, gf1 = 0, gf2 = 0, s2 = 0, dsum = 0;
  T rhob = 0, gb0 = 0, gb1 = 0, gb2 = 0;
  bool near_boundary = false;

  __device__ __forceinline__ SetupSums(const SceneView<T> &view, const vec4_t<T> &x,
                                       const vec4_t<T> &vi)
      : S(view), K(scalar_spline(view)), xi(x) {
    vs0 = vi.x, vs1 = vi.y, vs2 = vi.z;
  }
  // density self term W(0) = 4 alpha / h^3
  __device__ __forceinline__ T self() const { return xi.w * K.aw * T(4); }
  // neighbour (x_j, m_j) = pj with velocity vj (read only with kWithSource)
  __device__ __forceinline__ void pair(const vec4_t<T> &pj, const vec4_t<T> &vj) {
    const T d0 = xi.x - pj.x, d1 = xi.y - pj.y, d2 = xi.z - pj.z;
    add(pj, vj, d0, d1, d2, d0 * d0 + d1 * d1 + d2 * d2);
  }
  // the same for a candidate that fixed_sqdist has accepted: false (and nothing
  // added) where the exact predicate rejects it. The two forms of the squared
  // distance differ by a few roundings, far below the 1e-6 that decide here
  // whether the exact one is looked at; a NaN is.
  __device__ __forceinline__ bool pair_if(const vec4_t<T> &pj, const vec4_t<T> &vj) {
    const T d0 = xi.x - pj.x, d1 = xi.y - pj.y, d2 = xi.z - pj.z;
    const T r2 = d0 * d0 + d1 * d1 + d2 * d2;
    if (!(r2 < S.thr2 * T(0.999999)) && !(sqdist_exact(d0, d1, d2) < S.thr2))
      return false;
    add(pj, vj, d0, d1, d2, r2);
    return true;
  }
  // The kernel's factors are in every term: applied to the sums they save 1 % of the
  // pass (1M particles 182 -> 180 us), but the square of the gradient's leaves the FP32
  // range by itself, and the association shows, as 1e-4 of the pressure: the solve starts
  // from rho0 - rho, a difference of nearly equal numbers.
  __device__ __forceinline__ void add(const vec4_t<T> &pj, const vec4_t<T> &vj, T d0, T d1, T d2,
                                      T r2) {
    T w, f;
    K.eval(r2, w, f);
    rho += pj.w * w;
    const T g0 = f * d0, g1 = f * d1, g2 = f * d2;
    gf0 += pj.w * g0;
    gf1 += pj.w * g1;
    gf2 += pj.w * g2;
    s2 += pj.w * (g0 * g0 + g1 * g1 + g2 * g2);
    if (kWithSource) {
      const T u0 = vs0 - vj.x, u1 = vs1 - vj.y, u2 = vs2 - vj.z;
      dsum += pj.w * (u0 * g0 + u1 * g1 + u2 * g2);
    }
  }
  __device__ __forceinline__ vec4_t<T> load_v(uint32_t j) const {
    return kWithSource ? S.v[j] : make4<vec4_t<T>>(T(0), T(0), T(0), T(0));
  }
  // the boundary particles of slots [b, e)
  __device__ __forceinline__ void boundary(uint32_t b, uint32_t e) {
    for (uint32_t j = b; j < e; j += 4) {
      vec4_t<T> pk[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        pk[u] = S.bxV[min(j + u, e - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const vec4_t<T> pj = pk[u];
        const T d0 = xi.x - pj.x, d1 = xi.y - pj.y, d2 = xi.z - pj.z;
        const T r2 = sqdist_exact(d0, d1, d2);
        if (j + u >= e || !(r2 < S.thr2))
          continue;
        near_boundary = true;
        T w, f;
        K.eval(r2, w, f);
        rhob += pj.w * w;
        gb0 += pj.w * (f * d0);
        gb1 += pj.w * (f * d1);
        gb2 += pj.w * (f * d2);
      }
    }
  }
  // the particle's fields from the complete sums; returns its aprde term of
  // IISPH iteration 1 (S.first_iter)
  __device__ __forceinline__ double finish(int i) {
    const T rho0 = S.rho0;
    rho += rho0 * rhob;
    const T irho = T(1) / rho;
    const T irho2 = irho * irho;
    const T k14 = T(1.4) * rho0;
    const T c0 = -(gf0 + k14 * gb0) * irho2;
    const T c1 = -(gf1 + k14 * gb1) * irho2;
    const T c2 = -(gf2 + k14 * gb2) * irho2;
    const T gs0 = gf0 + rho0 * gb0, gs1 = gf1 + rho0 * gb1, gs2 = gf2 + rho0 * gb2;
    const T fac = S.dt * S.dt * rho0 * irho;
    const T AA = fac * ((c0 * gs0 + c1 * gs1 + c2 * gs2) - xi.w * irho2 * s2);
    S.rho[i] = rho;
    S.c[i] = make4<vec4_t<T>>(c0, c1, c2, T(0));
    S.G[i] = make4<vec4_t<T>>(gs0, gs1, gs2, T(0));
    S.AA[i] = AA;
    S.p[i] = T(0);
    S.pr[i] = T(0);
    S.xq[i] = make4<vec4_t<T>>(xi.x, xi.y, xi.z, T(0));
    S.xa[S.xa_x(static_cast<size_t>(i))] = xi;
    if (kWithSource) {
      const T src = (rho0 - rho) -
                    S.dt * rho0 * irho * (dsum + rho0 * (vs0 * gb0 + vs1 * gb1 + vs2 * gb2));
      S.s[i] = src;
      if (S.first_iter)
        return first_iteration(S, i, xi, rho, src, AA);
    } else {
      S.vd[i] = make4<vec4_t<T>>(gb0, gb1, gb2, T(0));  // G_b for the source pass
    }
    return 0.0;
  }
};

// wavefronts per SIMD of the setup pass (FP32: 80 registers)
template <class T>
constexpr int kSetupWaves = sizeof(T) == 4 ? 6 : 1;

struct SetupShared {
  // rows kNbrCap + 1 .. kNbrCap + 3 take the writes of a lane past its cap (52
  // rows: six blocks per CU)
  uint16_t lst[kNbrCap + 4][kBlock];
  BlockRanges sR;
};

template <class T, bool kWithSource>
__device__ __forceinline__ void k_setup_body(const SceneView<T> &S, const NbrList &L,
                                             unsigned lb, SetupShared &sh) {
  auto &lst = sh.lst;
  BlockRanges &sR = sh.sR;
  const unsigned t = threadIdx.x;
  const int i = static_cast<int>(lb * kBlock + t);
  const bool valid = i < S.nf;
  const uint32_t cell = valid ? S.fcell[i] : 0u;
  block_spans(S.grid, S.fstart, valid, cell, sR);
  if (t < 6)
    reinterpret_cast<uint32_t *>(L.blk + lb)[t] = t < 3 ? sR.base[t] : sR.len[t - 3];
  const Spans R = Spans::of(sR);
  const bool encodable = R.max_len() <= 0x10000u;

  const vec4_t<T> zero4 = make4<vec4_t<T>>(T(0), T(0), T(0), T(0));
  const vec4_t<T> xi = valid ? S.xm[i] : zero4;
  const vec4_t<T> vi = valid ? S.v[i] : zero4;
  const uint2 fi = valid ? S.xf[i] : make_uint2(0u, 0u);
  SetupSums<T, kWithSource> q(S, xi, vi);
  q.rho = q.self();
  constexpr uint32_t kRow = kBlock * sizeof(uint16_t);
  const uint32_t at0 = t * sizeof(uint16_t), top = at0 + (kNbrCap + 1u) * kRow;
  uint32_t at = at0;
  uint32_t cnt = 0;
  uint32_t cs[3] = {0u, 0u, 0u};  // entries per slab
  // candidate test of the slab-s runs; accepted entries are appended
  auto scan = [&](int s) {
    const uint32_t base = R.base(s);
    uint32_t rb[3], re[3];
    slab_bounds(S.grid, cell, S.fstart, s, rb, re);
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const uint32_t b = rb[r], e = re[r];
      const bool own = (s == 1) & (r == 1);  // the run holding particle i
      // eight candidates per trip from consecutive slots, loads issued
      // together. Branch-free append: every candidate is written to the next row
      // of this thread's column of the LDS table (at byte `at`), which advances
      // only for an accepted one. The table has 3 rows from kNbrCap + 1 on and the
      // row is clamped to kNbrCap + 1 at least every three candidates, so the writes
      // stay in the table and a count above kNbrCap still reads as overflow. Full
      // trips need no bound test; the last, partial trip of a run reads up
      // to 7 slots past it (the positions carry kRunPad slots of padding) and
      // rejects them. Only the run of the particle's own cell can hold the
      // particle itself.
      auto trip = [&](uint32_t j, auto tail_tag) {
        constexpr bool kTail = decltype(tail_tag)::value;
        struct alignas(8) Two {
          uint32_t xy0, z0, xy1, z1;
        };
        Two pk[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          pk[u] = *reinterpret_cast<const Two *>(S.xf + j + 2 * u);
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t lim = e - j;                          // u < lim: inside the run
        const uint32_t self = static_cast<uint32_t>(i) - j;  // u == self: the particle
        const uint32_t ent = j - base;                       // entry of candidate 0
        auto clamp = [&] { at = at < top ? at : top; };
        auto test = [&](int u, uint32_t xy, uint32_t z) {
          const bool ok = (!kTail | (static_cast<uint32_t>(u) < lim)) &
                          (!own | (static_cast<uint32_t>(u) != self)) &
                          (fixed_sqdist(fi.x, fi.y, xy, z) < kFixReach);
          *reinterpret_cast<uint16_t *>(reinterpret_cast<char *>(lst) + at) =
              static_cast<uint16_t>(ent + u);
          at += ok ? kRow : 0u;
        };
        test(0, pk[0].xy0, pk[0].z0);
        test(1, pk[0].xy1, pk[0].z1);
        test(2, pk[1].xy0, pk[1].z0);
        clamp();
        test(3, pk[1].xy1, pk[1].z1);
        if (!kTail || lim > 4u) {
          test(4, pk[2].xy0, pk[2].z0);
          test(5, pk[2].xy1, pk[2].z1);
          clamp();
          test(6, pk[3].xy0, pk[3].z0);
          test(7, pk[3].xy1, pk[3].z1);
        }
        clamp();
      };
      uint32_t j = b;
      for (; j + 8u <= e; j += 8u)
        trip(j, std::false_type{});
      if (j < e)
        trip(j, std::true_type{});
    }
  };
  bool over = !encodable;
  if (valid && !over) {
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      const uint32_t c0 = cnt;
      scan(s);
      cnt = (at - at0) / kRow;
      cs[s] = cnt - c0;
    }
    if (cnt > kNbrCap) {
      over = true;
    } else {
      const uint32_t c0 = cs[0], c01 = cs[0] + cs[1];
      const uint32_t d1 = R.b1 - R.b0, d2 = R.b2 - R.b1;
      auto slot = [&](uint32_t e) {
        return R.b0 + lst[e][t] + (e >= c0 ? d1 : 0u) + (e >= c01 ? d2 : 0u);
      };
      // groups of four: every gather of a group ahead of its arithmetic (the
      // last group repeats the last entry's gathers)
      uint64_t out = 0;  // entries that the exact predicate rejects
      for (uint32_t e = 0; e < cnt; e += 4) {
        vec4_t<T> px[4], pv[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
          const uint32_t j = slot(e + k < cnt ? e + k : cnt - 1u);
          px[k] = S.xm[j];
          pv[k] = q.load_v(j);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
          if (e + k < cnt && !q.pair_if(px[k], pv[k]))
            out |= 1ull << (e + k);
      }
      if (out != 0) {  // rare: candidates at the radius to within 1 in 4000
        uint32_t kept = 0, ks[3] = {0u, 0u, 0u};
        for (uint32_t e = 0; e < cnt; ++e)
          if (!((out >> e) & 1u)) {
            lst[kept++][t] = lst[e][t];
            ks[0] += e < c0 ? 1u : 0u;
            ks[1] += e >= c0 && e < c01 ? 1u : 0u;
            ks[2] += e >= c01 ? 1u : 0u;
          }
        cnt = kept;
#pragma unroll
        for (int s = 0; s < 3; ++s)
          cs[s] = ks[s];
      }
    }
  }
  // the rest is per particle; with S.first_iter the block then sums the
  // aprde terms of IISPH iteration 1 (every thread takes part)
  auto finish = [&]() -> double {
    const size_t nn = static_cast<size_t>(S.nf);
    uint32_t info;
    if (over) {
      // more neighbours than the list holds: all pair sums again over the grid
      q.rho = q.self();
      q.gf0 = q.gf1 = q.gf2 = q.s2 = q.dsum = T(0);
      grid_walk(S, i, xi, [&](uint32_t j) { q.pair(S.xm[j], q.load_v(j)); });
      info = kListOverflow;
    } else {
      // chunks of 8 entries, one 16-byte store per lane (1 KB per wavefront)
      for (uint32_t g = 0; g * kChunk < cnt; ++g) {
        uint32_t w[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint32_t e0 = g * kChunk + 2 * k;
          const uint32_t lo = e0 < cnt ? lst[e0][t] : 0u;
          const uint32_t hi = e0 + 1 < cnt ? lst[e0 + 1][t] : 0u;
          w[k] = lo | (hi << 16);
        }
        reinterpret_cast<uint4 *>(L.idx)[static_cast<size_t>(g) * nn + static_cast<size_t>(i)] =
            make_uint4(w[0], w[1], w[2], w[3]);
      }
      info = cs[0] | (cs[1] << 8) | (cs[2] << 16);
    }
    runs(S.grid, cell, S.bstart, [&](uint32_t b, uint32_t e) { q.boundary(b, e); });
    L.info[i] = info | (q.near_boundary && !over ? kListBoundary : 0u);
    return q.finish(i);
  };
  const double term = valid ? finish() : 0.0;
  if (kWithSource && S.first_iter) {
    const double bs = block_sum<kBlock>(term);
    if (t == 0)
      S.partials[lb] = bs;
  }
}

// The setup pass with 8 lanes per particle (scenes of up to kSplitMax
// particles, which do not fill the chip with one): the lanes share the
// candidates (scan8), the accepted neighbours and the boundary runs, and their
// sums are added in a fixed tree. Bound by its chain of dependent loads: run
// bounds, candidates of three slabs, neighbours. Measured, one lane -> eight:
// 2,048 particles 42 -> 13 us, 8,000: 42 -> 13, 59,000: 42 -> 31; with positions of
// 16 bytes 125,000: 50 -> 46, 250,000: 78 -> 82, 1M: 230 -> 294 (the lanes' idle slots
// cost more than the shorter chain gives).
template <class T, bool kWithSource>
__device__ __forceinline__ void k_setup8_body(const SceneView<T> &S, const NbrList &L,
                                              unsigned lb, Scan8Shared &sh) {
  const unsigned sub = threadIdx.x % kScanLanes, p = threadIdx.x / kScanLanes;
  const int i = static_cast<int>(lb * kScanParts + p);
  const bool valid = i < S.nf;
  const vec4_t<T> zero4 = make4<vec4_t<T>>(T(0), T(0), T(0), T(0));
  const vec4_t<T> xi = valid ? S.xm[i] : zero4;
  const vec4_t<T> vi = valid ? S.v[i] : zero4;
  const uint32_t cell = valid ? S.fcell[i] : 0u;
  Scan8 c = scan8<T, false>(S, L, lb, sh, i, valid, cell, xi);
  SetupSums<T, kWithSource> q(S, xi, vi);
  uint32_t rejected = 0;
  if (valid && !c.over) {
    const Spans R = Spans::of(sh.R);
    const uint32_t c0 = c.cs0, c01 = c.cs0 + c.cs1;
    const uint32_t d1 = R.b1 - R.b0, d2 = R.b2 - R.b1;
    for (uint32_t e0 = sub; e0 < c.cnt; e0 += 4u * kScanLanes) {
      vec4_t<T> px[4], pv[4];
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) {
        const uint32_t e = e0 + k * kScanLanes;
        if (e < c.cnt) {
          const uint32_t j =
              R.b0 + sh.lst[p][e] + (e >= c0 ? d1 : 0u) + (e >= c01 ? d2 : 0u);
          px[k] = S.xm[j];
          pv[k] = q.load_v(j);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) {
        const uint32_t e = e0 + k * kScanLanes;
        if (e < c.cnt && !q.pair_if(px[k], pv[k]))
          rejected |= 1u << (e / kScanLanes);
      }
    }
  } else if (valid && sub == 0) {
    grid_walk(S, i, xi, [&](uint32_t j) { q.pair(S.xm[j], q.load_v(j)); });
  }
  scan8_drop(sh, c, rejected);
  if (valid && S.nb > 0) {
    uint32_t b, e;
    run_bounds(S.grid, cell, S.bstart, static_cast<int>(sub), &b, &e);
    q.boundary(b, e);
    if (sub == 0) {
      run_bounds(S.grid, cell, S.bstart, 8, &b, &e);
      q.boundary(b, e);
    }
  }
  for (T *v : {&q.rho, &q.gf0, &q.gf1, &q.gf2, &q.s2, &q.rhob, &q.gb0, &q.gb1, &q.gb2})
    *v = lanes_sum<kScanLanes>(*v);
  if (kWithSource)
    q.dsum = lanes_sum<kScanLanes>(q.dsum);
  const uint64_t near = __ballot(q.near_boundary) >> ((threadIdx.x % kWave) & ~7u);
  double term = 0.0;
  if (valid) {
    scan8_write(L, sh, static_cast<size_t>(S.nf), i, c, (near & 0xFFu) != 0u);
    if (sub == 0) {
      q.rho += q.self();
      term = q.finish(i);
    }
  }
  if (kWithSource && S.first_iter) {
    const double bs = particle_sum<kScanLanes>(term);
    if (threadIdx.x == 0)
      S.partials[lb] = bs;
  }
}

template <class T, bool kWithSource>
__global__ __launch_bounds__(kBlock) void k_setup8(SceneView<T> S, NbrList L, SolveBegin B) {
  __shared__ Scan8Shared sh;
  k_setup8_body<T, kWithSource>(S, L, xcd_block(blockIdx.x, gridDim.x), sh);
  // no thread of the setup reads the control block
  if (B.seq != 0u && blockIdx.x == 0 && threadIdx.x == 0)
    begin_solve(S.ctl, B);
}

template <class T, bool kWithSource>
__global__ __launch_bounds__(kBlock, kSetupWaves<T>) void k_setup(SceneView<T> S, NbrList L, SolveBegin B) {
  __shared__ SetupShared sh;
  k_setup_body<T, kWithSource>(S, L, xcd_block(blockIdx.x, gridDim.x), sh);
  // no thread of the setup reads the control block
  if (B.seq != 0u && blockIdx.x == 0 && threadIdx.x == 0)
    begin_solve(S.ctl, B);
}

// does run r of particle i's boundary cells hold a particle within the radius
template <class T>
__device__ __forceinline__ bool boundary_in_run(const SceneView<T> &S, uint32_t cell,
                                                const vec4_t<T> &xi, int r) {
  uint32_t b, e;
  run_bounds(S.grid, cell, S.bstart, r, &b, &e);
  bool any = false;
  for (uint32_t j = b; j < e; ++j) {
    const vec4_t<T> pj = S.bxV[j];
    any = any || sqdist_exact(xi.x - pj.x, xi.y - pj.y, xi.z - pj.z) < S.thr2;
  }
  return any;
}

// The list of the procedures (8 lanes per particle). A procedure that walks
// it visits the particles of a grid walk in the same order, without the
// seven eighths of the candidates that the predicate rejects. Bound by the
// vector issue of the tests and appends.
template <class T>
__global__ __launch_bounds__(kBlock) void k_build_list(SceneView<T> S, NbrList L) {
  __shared__ Scan8Shared sh;
  const unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const int i = static_cast<int>(lb * kScanParts + threadIdx.x / kScanLanes);
  const unsigned sub = threadIdx.x % kScanLanes;
  const bool valid = i < S.nf;
  const vec4_t<T> xi =
      valid ? S.xm[i] : make4<vec4_t<T>>(T(0), T(0), T(0), T(0));
  const uint32_t cell = valid ? S.fcell[i] : 0u;
  const Scan8 c = scan8<T, true>(S, L, lb, sh, i, valid, cell, xi);
  bool near = false;
  if (valid && S.nb > 0)
    near = boundary_in_run(S, cell, xi, static_cast<int>(sub)) ||
           (sub == 0 && boundary_in_run(S, cell, xi, 8));
  const uint64_t m = __ballot(near) >> ((threadIdx.x % kWave) & ~7u);
  if (valid)
    scan8_write(L, sh, static_cast<size_t>(S.nf), i, c, (m & 0xFFu) != 0u);
}

// explicit viscosity (viscosity.hpp:171-240) over the list, then
// v* = v + dt (g + a_visc) H   (gravity.hpp:133, symplectic_euler.hpp:172-200)
template <class T, int kLanes>
__device__ __forceinline__ void k_viscosity_list_body(const SceneView<T> &S, const NbrList &L,
                                                      vec4_t<T> *vout, unsigned lb) {
  const int i = static_cast<int>((lb * kBlock + threadIdx.x) / kLanes);
  const uint32_t sub = threadIdx.x % kLanes;
  const bool valid = i < S.nf;
  const FastSpline<T> K = fast_spline(S);
  const vec4_t<T> zero4 = make4<vec4_t<T>>(T(0), T(0), T(0), T(0));
  const vec4_t<T> xi = valid ? S.xm[i] : zero4, vi = valid ? S.v[i] : zero4;
  const T rhoi = valid ? S.rho[i] : T(1);
  const uint32_t info = valid ? L.info[i] : 0u;
  const T cf = T(10) * S.mu_f / rhoi;
  T a0 = 0, a1 = 0, a2 = 0;
  struct Rec {
    vec4_t<T> x, v;
    T rho;
  };
  auto pair = [&](const Rec &q) {
    const vec4_t<T> &pj = q.x, &vj = q.v;
    const T d0 = xi.x - pj.x, d1 = xi.y - pj.y, d2 = xi.z - pj.z;
    const T r2 = d0 * d0 + d1 * d1 + d2 * d2;
    const T s = cf * (pj.w / q.rho) *
                ((vi.x - vj.x) * d0 + (vi.y - vj.y) * d1 + (vi.z - vj.z) * d2) /
                (r2 + S.hh001) * K.gradf(r2);
    a0 += s * d0;
    a1 += s * d1;
    a2 += s * d2;
  };
  auto load = [&](uint32_t j) { return Rec{S.xm[j], S.v[j], S.rho[j]}; };
  if (valid && !(info & kListOverflow))
    list_gather_lanes<kLanes, 4>(L, pass_spans<kLanes>(L, S.nf, lb), static_cast<size_t>(S.nf), i, info, sub,
                                 load, pair);
  else if (valid && sub == 0)
    grid_walk(S, i, xi, [&](uint32_t j) { pair(load(j)); });
  const T cb = T(10) * S.mu_b / rhoi * S.rho0 / rhoi;
  // the bounds of the lane's runs together and four candidates in flight (pass of 8,000
  // particles, 16,000 at the walls: 14.2 -> 12.1 us)
  auto wall = [&](uint32_t b, uint32_t e) {
    for (uint32_t j = b; j < e; j += 4) {
      vec4_t<T> pk[4];
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u)
        pk[u] = S.bxV[min(j + u, e - 1)];
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) {
        const vec4_t<T> pj = pk[u];
        const T d0 = xi.x - pj.x, d1 = xi.y - pj.y, d2 = xi.z - pj.z;
        const T r2e = sqdist_exact(d0, d1, d2);
        if (j + u >= e || !(r2e < S.thr2))
          continue;
        const T r2 = d0 * d0 + d1 * d1 + d2 * d2;
        const T s = cb * pj.w * (vi.x * d0 + vi.y * d1 + vi.z * d2) / (r2 + S.hh001) *
                    K.gradf(r2);
        a0 += s * d0;
        a1 += s * d1;
        a2 += s * d2;
      }
    }
  };
  if (list_has_boundary(info)) {
    if (kLanes == 1) {
      runs(S.grid, S.fcell[i], S.bstart, wall);
    } else {
      constexpr uint32_t kRuns = (9 + kLanes - 1) / kLanes;
      uint32_t b[kRuns], e[kRuns];
      const uint32_t cell = S.fcell[i];
#pragma unroll
      for (uint32_t q = 0; q < kRuns; ++q) {
        b[q] = e[q] = 0u;
        if (sub + q * kLanes < 9u)
          run_bounds(S.grid, cell, S.bstart, static_cast<int>(sub + q * kLanes), &b[q], &e[q]);
      }
#pragma unroll
      for (uint32_t q = 0; q < kRuns; ++q)
        wall(b[q], e[q]);
    }
  }
  a0 = lanes_sum<kLanes>(a0);
  a1 = lanes_sum<kLanes>(a1);
  a2 = lanes_sum<kLanes>(a2);
  if (!valid || sub != 0)
    return;
  const T H = fade_step(S, vi.w);
  T g0, g1, g2;
  step_gravity(S, xi.x, xi.y, xi.z, g0, g1, g2);
  vout[i] = make4<vec4_t<T>>(vi.x + S.dt * (g0 + a0) * H, vi.y + S.dt * (g1 + a1) * H,
                             vi.z + S.dt * (g2 + a2) * H, vi.w);
}

template <class T, int kLanes>
__global__ __launch_bounds__(kBlock) void k_viscosity_list(SceneView<T> S, NbrList L,
                                                           vec4_t<T> *vout) {
  k_viscosity_list_body<T, kLanes>(S, L, vout, xcd_block(blockIdx.x, gridDim.x));
}

// v* = v + dt a_axial(x) H (gravity.hpp:189-215, symplectic_euler.hpp:172-200)
// for steps with axial gravity and no explicit viscosity
template <class T>
__device__ __forceinline__ void k_gravity_v_body(const SceneView<T> &S, vec4_t<T> *vout,
                                                 unsigned lb) {
  const int i = static_cast<int>(lb * kBlock + threadIdx.x);
  if (i >= S.nf)
    return;
  const vec4_t<T> xi = S.xm[i], vi = S.v[i];
  const T H = fade_step(S, vi.w);
  T g0, g1, g2;
  step_gravity(S, xi.x, xi.y, xi.z, g0, g1, g2);
  vout[i] = make4<vec4_t<T>>(vi.x + S.dt * g0 * H, vi.y + S.dt * g1 * H,
                             vi.z + S.dt * g2 * H, vi.w);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_gravity_v(SceneView<T> S, vec4_t<T> *vout) {
  k_gravity_v_body(S, vout, blockIdx.x);
}

// source term s from the integrated velocities (explicit-viscosity path)
template <class T, int kLanes>
__device__ __forceinline__ void k_source_list_body(const SceneView<T> &S, const NbrList &L,
                                                   unsigned lb) {
  const int i = static_cast<int>((lb * kBlock + threadIdx.x) / kLanes);
  const uint32_t sub = threadIdx.x % kLanes;
  const bool valid = i < S.nf;
  const FastSpline<T> K = fast_spline(S);
  const vec4_t<T> zero4 = make4<vec4_t<T>>(T(0), T(0), T(0), T(0));
  const vec4_t<T> xi = valid ? S.xm[i] : zero4, vi = valid ? S.v[i] : zero4;
  const vec4_t<T> gb = valid ? S.vd[i] : zero4;
  const uint32_t info = valid ? L.info[i] : 0u;
  T dsum = 0;
  struct Rec {
    vec4_t<T> x, v;
  };
  auto pair = [&](const Rec &q) {
    const T d0 = xi.x - q.x.x, d1 = xi.y - q.x.y, d2 = xi.z - q.x.z;
    const T f = K.gradf(d0 * d0 + d1 * d1 + d2 * d2);
    dsum += q.x.w * f * ((vi.x - q.v.x) * d0 + (vi.y - q.v.y) * d1 + (vi.z - q.v.z) * d2);
  };
  auto load = [&](uint32_t j) { return Rec{S.xm[j], S.v[j]}; };
  if (valid && !(info & kListOverflow))
    list_gather_lanes<kLanes, 4>(L, pass_spans<kLanes>(L, S.nf, lb), static_cast<size_t>(S.nf), i, info, sub,
                                 load, pair);
  else if (valid && sub == 0)
    grid_walk(S, i, xi, [&](uint32_t j) { pair(load(j)); });
  dsum = lanes_sum<kLanes>(dsum);
  double term = 0.0;
  if (valid && sub == 0) {
    const T rhoi = S.rho[i];
    const T rho0 = S.rho0;
    const T src = (rho0 - rhoi) -
                  S.dt * rho0 / rhoi * (dsum + rho0 * (vi.x * gb.x + vi.y * gb.y + vi.z * gb.z));
    S.s[i] = src;
    if (S.first_iter)
      term = first_iteration(S, i, xi, rhoi, src, S.AA[i]);
  }
  if (S.first_iter) {  // IISPH iteration 1: the block's aprde partial
    const double bs = particle_sum<kLanes>(term);
    if (threadIdx.x == 0)
      S.partials[lb] = bs;
  }
}

template <class T, int kLanes>
__global__ __launch_bounds__(kBlock) void k_source_list(SceneView<T> S, NbrList L) {
  k_source_list_body<T, kLanes>(S, L, xcd_block(blockIdx.x, gridDim.x));
}

// The end of IISPH iteration `it` with the sum aprde (example.lua:418-419): stop when
// it >= min_it and aprde / nprde < tol, or at max_it. store: this thread writes
// and reports it.
__device__ __forceinline__ bool iteration_decision(Ctl *c, double aprde, int it, bool store) {
  const double rel = aprde / static_cast<double>(c->nprde);
  const bool converged = it >= c->min_it && rel < c->tol;
  const bool done = converged || it >= c->max_it;
  if (store) {
    c->aprde = aprde;
    c->iters = it;
    c->rel = rel;
    if (done) {
      c->done = 1;
      c->converged = converged ? 1 : 0;
    }
    publish_progress(c);
  }
  return done;
}

// The same decision in the first pass of the next iteration: every block sums the
// partials of the pressure pass before it (the sum of k_pressure_finalize_body, bit
// for bit) and derives the decision, block 0 stores it. One launch fewer per
// iteration, 2.5 us and the gap before it, for about 1 us in the pass; the blocks
// read all partials, so it is for launches of up to kFoldBlocks blocks (1,000 blocks
// read 8 MB from L2; 4,000 would read 128 MB), and not for batches, which fill the
// chip: there the pass went from 20 to 32 us. A block reads `done` once: block 0 of
// this launch may set it meanwhile, and a block that sees it set would decide the
// same. iters_next, staged by the pressure pass, is not written here.
// False: the solve is done.
constexpr unsigned kFoldBlocks = 1024;
__host__ __device__ inline bool fold_scene(int nf) { return list_blocks(nf) <= kFoldBlocks; }
__device__ __forceinline__ bool fold_iteration(const Ctl *c, const double *partials,
                                               unsigned nparts, bool store) {
  __shared__ double ws[kBlock / kWave];
  __shared__ int flag;
  static_assert(kBlock / kWave == 4, "four wave sums");
  const double part = wave_sum(strided_sum<kBlock>(partials, nparts));
  if (threadIdx.x % kWave == 0)
    ws[threadIdx.x / kWave] = part;
  if (threadIdx.x == 0)
    flag = c->done;
  __syncthreads();
  if (flag != 0)
    return false;
  // block_sum's order
  return !iteration_decision(const_cast<Ctl *>(c), (ws[0] + ws[2]) + (ws[1] + ws[3]),
                             c->iters_next, store && threadIdx.x == 0);
}

// IISPH pressure acceleration over the list: a_i = p_i c_i - sum m_j pr_j gradW
template <class T, int kLanes>
__device__ __forceinline__ void k_accel_list_body(const SceneView<T> &S, const NbrList &L,
                                                  unsigned lb, bool fold) {
  if (!fold && S.ctl->done)
    return;
  const int i = static_cast<int>((lb * kBlock + threadIdx.x) / kLanes);
  const uint32_t sub = threadIdx.x % kLanes;
  const bool valid = i < S.nf;
  const Spans R = pass_spans<kLanes>(L, S.nf, lb);
  const FastSpline<T> K = fast_spline(S);
  const vec4_t<T> zero4 = make4<vec4_t<T>>(T(0), T(0), T(0), T(0));
  const vec4_t<T> xi = valid ? S.xm[i] : zero4;
  const uint32_t info = valid ? L.info[i] : kListOverflow;
  // own fields loaded ahead of the walk so their latency overlaps it
  const vec4_t<T> ci = valid ? S.c[i] : zero4;
  const T pi = valid ? S.p[i] : T(0);
  if (fold && !fold_iteration(S.ctl, S.partials, list_blocks(S.nf), lb == 0))
    return;
  T a0 = 0, a1 = 0, a2 = 0;
  auto pair = [&](const vec4_t<T> &qj) {  // (x_j, m_j p_j / rho_j^2)
    const T d0 = xi.x - qj.x, d1 = xi.y - qj.y, d2 = xi.z - qj.z;
    const T s = qj.w * K.gradf_unscaled(d0 * d0 + d1 * d1 + d2 * d2);
    a0 += s * d0;
    a1 += s * d1;
    a2 += s * d2;
  };
  if (!(info & kListOverflow))
    list_gather_lanes<kLanes, 8>(
        L, R, static_cast<size_t>(S.nf), i, info, sub, [&](uint32_t j) { return S.xq[j]; }, pair);
  if (valid && sub == 0 && (info & kListOverflow))
    grid_walk(S, i, xi, [&](uint32_t j) { pair(S.xq[j]); });
  a0 = lanes_sum<kLanes>(a0);
  a1 = lanes_sum<kLanes>(a1);
  a2 = lanes_sum<kLanes>(a2);
  if (!valid || sub != 0)
    return;
  const vec4_t<T> ai = make4<vec4_t<T>>(pi * ci.x - K.ag3 * a0, pi * ci.y - K.ag3 * a1,
                                        pi * ci.z - K.ag3 * a2, T(0));
  // the pressure pass gathers it from here; the integration copies it to a
  S.xa[S.xa_a(static_cast<size_t>(i))] = ai;
}

template <class T, int kLanes>
__global__ __launch_bounds__(kBlock) void k_accel_list(SceneView<T> S, NbrList L, int fold) {
  k_accel_list_body<T, kLanes>(S, L, xcd_block(blockIdx.x, gridDim.x), fold != 0);
}

// IISPH relaxed Jacobi update over the list, FP64 aprde reduction and the
// device-side convergence decision (example.lua:409-421)
template <class T, int kLanes>
__device__ __forceinline__ void k_pressure_list_body(const SceneView<T> &S, const NbrList &L,
                                                     unsigned lb) {
  if (S.ctl->done)
    return;
  if (lb == 0 && threadIdx.x == 0)
    S.ctl->iters_next = S.ctl->iters + 1;
  struct XA {
    vec4_t<T> x, a;  // (x, m) and (a, 0) of a neighbour
  };
  const int i = static_cast<int>((lb * kBlock + threadIdx.x) / kLanes);
  const uint32_t sub = threadIdx.x % kLanes;
  const bool valid = i < S.nf;
  const Spans R = pass_spans<kLanes>(L, S.nf, lb);
  const FastSpline<T> K = fast_spline(S);
  const vec4_t<T> zero4 = make4<vec4_t<T>>(T(0), T(0), T(0), T(0));
  const vec4_t<T> xi = valid ? S.xm[i] : zero4;
  const uint32_t info = valid ? L.info[i] : kListOverflow;
  // own fields loaded ahead of the walk so their latency overlaps it
  const vec4_t<T> ai = valid ? S.xa[S.xa_a(static_cast<size_t>(i))] : zero4;
  const vec4_t<T> gs = valid ? S.G[i] : zero4;
  const T rhoi = valid ? S.rho[i] : T(1), AA = valid ? S.AA[i] : T(0);
  const T si = valid ? S.s[i] : T(0), p_old = valid ? S.p[i] : T(0);
  T sum = 0;
  auto pair = [&](const XA &q) {
    const T d0 = xi.x - q.x.x, d1 = xi.y - q.x.y, d2 = xi.z - q.x.z;
    sum += q.x.w * K.gradf_unscaled(d0 * d0 + d1 * d1 + d2 * d2) *
           (q.a.x * d0 + q.a.y * d1 + q.a.z * d2);
  };
  list_gather_records<kLanes, 4>(
      L, R, static_cast<size_t>(S.nf), i, (info & kListOverflow) ? 0u : info, sub,
      static_cast<uint32_t>(valid ? i : 0), S.xa,
      [&](const vec4_t<T> &x, const vec4_t<T> &a) { pair(XA{x, a}); });
  if (valid && sub == 0 && (info & kListOverflow))
    grid_walk(S, i, xi, [&](uint32_t j) {
      pair(XA{S.xa[S.xa_x(j)], S.xa[S.xa_a(j)]});
    });
  sum = lanes_sum<kLanes>(sum);
  double term = 0.0;
  if (valid && sub == 0) {
    const T Ap = S.dt * S.dt * S.rho0 / rhoi *
                 ((ai.x * gs.x + ai.y * gs.y + ai.z * gs.z) - K.ag3 * sum);
    const T rcp = (fabs(AA) > T(1e-9)) ? T(1) / AA : T(0);
    const T upd = p_old + S.omega * (si - Ap) * rcp;
    const T pn = ((T(0) < upd) ? upd : T(0)) * ((T(1e-9) < fabs(AA)) ? T(1) : T(0));
    S.Ap[i] = Ap;
    S.p[i] = pn;
    S.pr[i] = pn / (rhoi * rhoi);
    S.xq[i] = make4<vec4_t<T>>(xi.x, xi.y, xi.z, xi.w * pn / (rhoi * rhoi));
    term = static_cast<double>((Ap - si) / S.rho0 * ((T(1e-9) < pn) ? T(1) : T(0)));
  }
  const double bs = particle_sum<kLanes>(term);
  if (threadIdx.x == 0)
    S.partials[lb] = bs;
}

template <class T, int kLanes>
__global__ __launch_bounds__(kBlock) void k_pressure_list(SceneView<T> S, NbrList L) {
  k_pressure_list_body<T, kLanes>(S, L, xcd_block(blockIdx.x, gridDim.x));
}

// Sum of the block partials in block order (FP64, fixed tree) and the
// convergence decision, in a kernel of its own. half: the partials are of half
// the particles of a list pass's block (k_setup8) and are added in pairs first.
__device__ __forceinline__ void k_pressure_finalize_body(Ctl *c, const double *partials,
                                                        unsigned nparts, bool half = false) {
  if (c->done)
    return;
  double part = 0.0;
  if (half) {
    for (unsigned k = 2u * threadIdx.x; k < nparts; k += 2u * kBlock)
      part += partials[k] + (k + 1u < nparts ? partials[k + 1u] : 0.0);
  } else {
    part = strided_sum<kBlock>(partials, nparts);
  }
  const double acc = block_sum<kBlock>(part);
  if (threadIdx.x == 0)
    iteration_decision(c, acc, c->iters + 1, true);
}

__global__ __launch_bounds__(kBlock) void k_pressure_finalize(Ctl *c, const double *partials,
                                                              unsigned nparts, bool half) {
  k_pressure_finalize_body(c, partials, nparts, half);
}

template <class T>
__device__ __forceinline__ void max_speed_atomic(Ctl *ctl, T s);
template <>
__device__ __forceinline__ void max_speed_atomic<float>(Ctl *ctl, float s) {
  atomicMax(&ctl->max_speed_bits_f, __float_as_uint(s));
}
template <>
__device__ __forceinline__ void max_speed_atomic<double>(Ctl *ctl, double s) {
  atomicMax(&ctl->max_speed_bits_d, static_cast<unsigned long long>(__double_as_longlong(s)));
}

// v += dt a H (pressure acceleration), x += dt v, running max |v|; seq > 0:
// only once solve seq is done (integrate_now)
template <class T>
__device__ __forceinline__ void k_integrate_body(SceneView<T> S, unsigned lb, unsigned seq) {
  if (seq != 0u && !integrate_now(S.ctl, seq))
    return;
  const int i = static_cast<int>(lb * kBlock + threadIdx.x);
  T speed = T(0);
  bool bad = false;
  if (i < S.nf) {
    vec4_t<T> v = S.v[i];
    const vec4_t<T> a = S.xa[S.xa_a(static_cast<size_t>(i))];
    S.a[i] = a;  // the acceleration field after the step, as the reference's
    const T H = fade_step(S, v.w);
    v.x += S.dt * a.x * H;
    v.y += S.dt * a.y * H;
    v.z += S.dt * a.z * H;
    vec4_t<T> x = S.xm[i];
    x.x += S.dt * v.x;
    x.y += S.dt * v.y;
    x.z += S.dt * v.z;
    S.v[i] = v;
    S.xm[i] = x;
    speed = sqrt(v.x * v.x + v.y * v.y + v.z * v.z);
    bad = !(isfinite(x.x) && isfinite(x.y) && isfinite(x.z) && isfinite(speed));
    if (bad)
      speed = T(0);
  }
  speed = block_max<kBlock>(speed);
  if (threadIdx.x == 0)
    S.partials[lb] = static_cast<double>(speed);
  if (bad)
    S.ctl->nonfinite = 1;
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_integrate(SceneView<T> S, unsigned seq) {
  k_integrate_body<T>(S, blockIdx.x, seq);
}

// running maximum speed (symplectic_euler.hpp:250-268) from the block maxima;
// seq > 0: after the integration of solve seq's step, which it marks taken
template <class T>
__device__ __forceinline__ void k_speed_finalize_body(Ctl *c, const double *partials,
                                                      unsigned nparts, unsigned seq) {
  if (seq != 0u && !integrate_now(c, seq))
    return;
  const double m = block_max<kBlock>(strided_max<kBlock>(partials, nparts, 0.0));
  if (threadIdx.x == 0) {
    max_speed_atomic<T>(c, static_cast<T>(m));
    if (seq != 0u)
      c->integrated = seq;
    publish_step_end(c);
  }
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_speed_finalize(Ctl *c, const double *partials,
                                                           unsigned nparts, unsigned seq) {
  k_speed_finalize_body<T>(c, partials, nparts, seq);
}

// ---- batched wrappers (prtcl_hip_step over several scenes): the setup and list
// passes take the body that the block's scene takes alone (split_scene)
// the two setup bodies share their LDS, so the large scenes' blocks keep
// their six per CU
union SetupPool {
  SetupShared setup;
  Scan8Shared scan;
};

// this block's entry E, list L and local block lb in the units of its pass (kF
// blocks for each block of a split scene); returns from the kernel for a block
// past the scene's particles
#define BATCH_PASS_ENTRY(kF, total)                                                       \
  unsigned part;                                                                          \
  const uint32_t u = batch_block(B, kF, &part);                                           \
  const BatchEntry<T> &E = tab[u >> kBatchLocalBits];                                     \
  const bool split = split_scene(E.S.nf);                                                 \
  const unsigned lb = (u & kBatchLocalMask) * (split ? (kF) : 1u) + part;                 \
  if (lb >= total(E.S.nf))                                                                \
    return;                                                                               \
  const NbrList L{E.nidx, E.ninfo, E.nblk, E.nshift}

constexpr unsigned kSetupParts = kBlock / kScanParts;  // setup blocks per block of a split scene
constexpr unsigned kListParts = kListLanes;

template <class T, bool kWithSource>
__global__ __launch_bounds__(kBlock, kSetupWaves<T>) void k_setup_b(const BatchEntry<T> *tab, BatchBlocks B) {
  __shared__ SetupPool sh;
  BATCH_PASS_ENTRY(kSetupParts, setup_blocks);
  if (split)
    k_setup8_body<T, kWithSource>(E.S, L, lb, sh.scan);
  else
    k_setup_body<T, kWithSource>(E.S, L, lb, sh.setup);
}

// scenes with explicit viscosity or axial gravity: after the setup without the
// source term, v* (explicit viscosity and gravity, or the axial gravity
// alone) into vtmp, then the source term and iteration 1 from v* (the three
// launches of FusedOps::setup for such a scene)
template <class T>
__global__ __launch_bounds__(kBlock) void k_vstar_b(const BatchEntry<T> *tab, BatchBlocks B) {
  BATCH_PASS_ENTRY(kListParts, list_blocks);
  if (!E.explicit_visc)
    k_gravity_v_body(E.S, E.vtmp, lb);  // blocks past the particles find none
  else if (split)
    k_viscosity_list_body<T, kListLanes>(E.S, L, E.vtmp, lb);
  else
    k_viscosity_list_body<T, 1>(E.S, L, E.vtmp, lb);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_source_b(const BatchEntry<T> *tab, BatchBlocks B) {
  BATCH_PASS_ENTRY(kListParts, list_blocks);
  SceneView<T> S2 = E.S;
  S2.v = E.vtmp;  // the integrated velocities
  if (split)
    k_source_list_body<T, kListLanes>(S2, L, lb);
  else
    k_source_list_body<T, 1>(S2, L, lb);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_accel_b(const BatchEntry<T> *tab, BatchBlocks B) {
  BATCH_PASS_ENTRY(kListParts, list_blocks);
  if (split)
    k_accel_list_body<T, kListLanes>(E.S, L, lb, false);
  else
    k_accel_list_body<T, 1>(E.S, L, lb, false);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_pressure_b(const BatchEntry<T> *tab, BatchBlocks B) {
  BATCH_PASS_ENTRY(kListParts, list_blocks);
  if (split)
    k_pressure_list_body<T, kListLanes>(E.S, L, lb);
  else
    k_pressure_list_body<T, 1>(E.S, L, lb);
}

// one block per scene
template <class T>
__global__ __launch_bounds__(kBlock) void k_pressure_finalize_b(const BatchEntry<T> *tab) {
  const BatchEntry<T> &E = tab[blockIdx.x];
  k_pressure_finalize_body(E.S.ctl, E.S.partials, list_blocks(E.S.nf));
}

// iteration 1's convergence step for the scenes whose solve it could end
template <class T>
__global__ __launch_bounds__(kBlock) void k_first_finalize_b(const BatchEntry<T> *tab) {
  const BatchEntry<T> &E = tab[blockIdx.x];
  // partials of the setup, or of the source pass of the three-launch setup
  if (!E.first_preset)
    k_pressure_finalize_body(E.S.ctl, E.S.partials,
                             E.split_setup ? list_blocks(E.S.nf) : setup_blocks(E.S.nf),
                             !E.split_setup && split_scene(E.S.nf));
}

// guarded: each scene's integration only once its solve (E.seq) is done;
// scenes whose step ends with the WKBB18 path are left to it
template <class T>
__global__ __launch_bounds__(kBlock) void k_integrate_b(const BatchEntry<T> *tab,
                                                        const uint32_t *pmap, int guarded) {
  const uint32_t u = pmap[xcd_block(blockIdx.x, gridDim.x)];
  const BatchEntry<T> &E = tab[u >> kBatchLocalBits];
  if (E.viscous)
    return;
  k_integrate_body<T>(E.S, u & kBatchLocalMask, guarded ? E.seq : 0u);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_speed_finalize_b(const BatchEntry<T> *tab,
                                                             int guarded) {
  const BatchEntry<T> &E = tab[blockIdx.x];
  if (E.viscous)
    return;
  k_speed_finalize_body<T>(E.S.ctl, E.S.partials, E.nblocks, guarded ? E.seq : 0u);
}

}  // namespace

template <class T>
void FusedOps<T>::build_list(hipStream_t st, const SceneView<T> &S, const NbrList &L) {
  if (S.nf > 0)
    hipLaunchKernelGGL(k_build_list<T>, dim3(grid_blocks(S.nf, kScanParts)), dim3(kBlock), 0, st,
                       S, L);
}

template <class T>
void FusedOps<T>::setup(hipStream_t st, const SceneView<T> &S, const NbrList &L,
                        bool explicit_viscosity, vec4_t<T> *vtmp, const SolveBegin &B) {
  if (S.nf <= 0)
    return;
  const dim3 gr(setup_blocks(S.nf)), bl(kBlock);
  const bool split = split_scene(S.nf);
  // the one-pass setup reads velocities that the sort has integrated with a
  // uniform g (GravityKick); explicit viscosity or a position-dependent (axial)
  // gravity integrate them after the list is built
  if (!explicit_viscosity && !S.axial) {
    if (split)
      hipLaunchKernelGGL((k_setup8<T, true>), gr, bl, 0, st, S, L, B);
    else
      hipLaunchKernelGGL((k_setup<T, true>), gr, bl, 0, st, S, L, B);
    return;
  }
  if (split)
    hipLaunchKernelGGL((k_setup8<T, false>), gr, bl, 0, st, S, L, B);
  else
    hipLaunchKernelGGL((k_setup<T, false>), gr, bl, 0, st, S, L, B);
  const dim3 gl(list_blocks(S.nf));
  if (!explicit_viscosity)
    hipLaunchKernelGGL(k_gravity_v<T>, dim3(grid_blocks(S.nf)), bl, 0, st, S, vtmp);
  else if (split)
    hipLaunchKernelGGL((k_viscosity_list<T, kListLanes>), gl, bl, 0, st, S, L, vtmp);
  else
    hipLaunchKernelGGL((k_viscosity_list<T, 1>), gl, bl, 0, st, S, L, vtmp);
  // the integrated velocities replace v once every thread has read the old ones
  SceneView<T> S2 = S;
  S2.v = vtmp;
  if (split)
    hipLaunchKernelGGL((k_source_list<T, kListLanes>), gl, bl, 0, st, S2, L);
  else
    hipLaunchKernelGGL((k_source_list<T, 1>), gl, bl, 0, st, S2, L);
}

template <class T>
void FusedOps<T>::accel(hipStream_t st, const SceneView<T> &S, const NbrList &L, bool fold) {
  if (S.nf <= 0)
    return;
  const dim3 gr(list_blocks(S.nf)), bl(kBlock);
  if (split_scene(S.nf))
    hipLaunchKernelGGL((k_accel_list<T, kListLanes>), gr, bl, 0, st, S, L, fold ? 1 : 0);
  else
    hipLaunchKernelGGL((k_accel_list<T, 1>), gr, bl, 0, st, S, L, fold ? 1 : 0);
}

template <class T>
void FusedOps<T>::pressure(hipStream_t st, const SceneView<T> &S, const NbrList &L, bool last) {
  if (S.nf <= 0)
    return;
  const unsigned nb = list_blocks(S.nf);
  if (split_scene(S.nf))
    hipLaunchKernelGGL((k_pressure_list<T, kListLanes>), dim3(nb), dim3(kBlock), 0, st, S, L);
  else
    hipLaunchKernelGGL((k_pressure_list<T, 1>), dim3(nb), dim3(kBlock), 0, st, S, L);
  if (last)
    hipLaunchKernelGGL(k_pressure_finalize, dim3(1), dim3(kBlock), 0, st, S.ctl, S.partials, nb,
                       false);
}

template <class T>
bool FusedOps<T>::folds(int nf) {
  return fold_scene(nf);
}

// a = the acceleration of the last pressure-acceleration pass
template <class T>
__global__ __launch_bounds__(kBlock) void k_copy_accel(SceneView<T> S) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < S.nf)
    S.a[i] = S.xa[S.xa_a(static_cast<size_t>(i))];
}

template <class T>
void FusedOps<T>::finish_first_iteration(hipStream_t st, const SceneView<T> &S,
                                         bool explicit_viscosity) {
  // written by the setup, or by the source pass of the three-launch setup
  const bool three = explicit_viscosity || S.axial;
  if (S.nf > 0)
    hipLaunchKernelGGL(k_pressure_finalize, dim3(1), dim3(kBlock), 0, st, S.ctl, S.partials,
                       three ? list_blocks(S.nf) : setup_blocks(S.nf),
                       !three && split_scene(S.nf));
}

template <class T>
void FusedOps<T>::finish_first_iteration_batch(hipStream_t st, const BatchEntry<T> *tab,
                                               unsigned nscenes) {
  if (nscenes > 0)
    hipLaunchKernelGGL(k_first_finalize_b<T>, dim3(nscenes), dim3(kBlock), 0, st, tab);
}

template <class T>
void FusedOps<T>::copy_accel(hipStream_t st, const SceneView<T> &S) {
  if (S.nf > 0)
    hipLaunchKernelGGL(k_copy_accel<T>, dim3(grid_blocks(S.nf)), dim3(kBlock), 0, st, S);
}

template <class T>
void FusedOps<T>::integrate(hipStream_t st, const SceneView<T> &S, unsigned seq) {
  if (S.nf <= 0)
    return;
  const unsigned nb = grid_blocks(S.nf);
  hipLaunchKernelGGL(k_integrate<T>, dim3(nb), dim3(kBlock), 0, st, S, seq);
  hipLaunchKernelGGL(k_speed_finalize<T>, dim3(1), dim3(kBlock), 0, st, S.ctl, S.partials, nb,
                     seq);
}

template <class T>
void FusedOps<T>::setup_batch(hipStream_t st, const BatchEntry<T> *tab, const BatchBlocks &B) {
  const dim3 bl(kBlock);
  const BatchBlocks B1 = B.group(0), B3 = B.group(1);
  if (const unsigned n = B1.launch(kSetupParts))
    hipLaunchKernelGGL((k_setup_b<T, true>), dim3(n), bl, 0, st, tab, B1);
  if (const unsigned n = B3.launch(kSetupParts)) {
    hipLaunchKernelGGL((k_setup_b<T, false>), dim3(n), bl, 0, st, tab, B3);
    const dim3 gl(B3.launch(kListParts));
    hipLaunchKernelGGL(k_vstar_b<T>, gl, bl, 0, st, tab, B3);
    hipLaunchKernelGGL(k_source_b<T>, gl, bl, 0, st, tab, B3);
  }
}

template <class T>
void FusedOps<T>::accel_batch(hipStream_t st, const BatchEntry<T> *tab, const BatchBlocks &B) {
  if (const unsigned n = B.launch(kListParts))
    hipLaunchKernelGGL(k_accel_b<T>, dim3(n), dim3(kBlock), 0, st, tab, B);
}

template <class T>
void FusedOps<T>::pressure_batch(hipStream_t st, const BatchEntry<T> *tab, const BatchBlocks &B,
                                 unsigned nscenes) {
  const unsigned n = B.launch(kListParts);
  if (n == 0)
    return;
  hipLaunchKernelGGL(k_pressure_b<T>, dim3(n), dim3(kBlock), 0, st, tab, B);
  hipLaunchKernelGGL(k_pressure_finalize_b<T>, dim3(nscenes), dim3(kBlock), 0, st, tab);
}

template <class T>
void FusedOps<T>::integrate_batch(hipStream_t st, const BatchEntry<T> *tab, const uint32_t *pmap,
                                  unsigned npblocks, unsigned nscenes, bool guarded) {
  if (npblocks == 0)
    return;
  const int g = guarded ? 1 : 0;
  hipLaunchKernelGGL(k_integrate_b<T>, dim3(npblocks), dim3(kBlock), 0, st, tab, pmap, g);
  hipLaunchKernelGGL(k_speed_finalize_b<T>, dim3(nscenes), dim3(kBlock), 0, st, tab, g);
}

template struct FusedOps<float>;
template struct FusedOps<double>;

}  // namespace prtcl_amd
