// FP64 control of the preconditioned CG of cg_openmp.hpp:32-215 on the
// device, shared by every solver that uses it (WKBB18's 3-vector system, the
// scalar systems of pt16): per-block partial sums of the dot products, the
// set-up scalars, alpha with the |p.q| < tol break, beta with the
// |r.y|_prev < tol break and ok(k, |r|^2), all in one block reading the
// partials in block order (deterministic), and the progress word the host
// polls.
#pragma once

#include "device_common.hpp"
#include "scene.hpp"

namespace prtcl_amd {
namespace {

// The block sums of K values at once, in every thread: a wave sum each, one
// barrier, and the four wave sums added as block_sum adds them,
// (w0 + w2) + (w1 + w3).
template <int K>
__device__ __forceinline__ void block_sums(double (&v)[K]) {
  static_assert(kBlock / kWave == 4, "four wave sums");
  __shared__ double ws[K][4];
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
#pragma unroll
  for (int k = 0; k < K; ++k)
    v[k] = wave_sum(v[k]);
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < K; ++k)
      ws[k][w] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < K; ++k)
    v[k] = (ws[k][0] + ws[k][2]) + (ws[k][1] + ws[k][3]);
  __syncthreads();  // a later call writes ws again
}

// per-block partial sums of K FP64 dot products, stored at the block's logical
// index b (the partials are summed in logical block order)
template <int K>
__device__ __forceinline__ void store_partials(double *partials, unsigned nblocks,
                                               const double (&v)[K], unsigned b) {
  double s[K];
#pragma unroll
  for (int k = 0; k < K; ++k)
    s[k] = v[k];
  block_sums(s);
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < K; ++k)
      partials[k * nblocks + b] = s[k];
}

// the sums of K arrays of n partials (array k at p + k n), each in block order,
// in every thread of the block; a thread's share is that of strided_sum, with
// the loads of all arrays in flight together
template <int K>
__device__ __forceinline__ void sum_partials(const double *p, unsigned n, double (&out)[K]) {
  constexpr unsigned kBatch = K > 4 ? 4 : 8;
#pragma unroll
  for (int k = 0; k < K; ++k)
    out[k] = 0.0;
  for (unsigned k0 = threadIdx.x; k0 < n; k0 += kBatch * kBlock) {
    double t[kBatch][K];
#pragma unroll
    for (unsigned u = 0; u < kBatch; ++u) {
      const unsigned i = k0 + u * kBlock;
#pragma unroll
      for (int k = 0; k < K; ++k)
        t[u][k] = p[static_cast<size_t>(k) * n + (i < n ? i : n - 1)];
    }
#pragma unroll
    for (unsigned u = 0; u < kBatch; ++u)
      if (k0 + u * kBlock < n)
#pragma unroll
        for (int k = 0; k < K; ++k)
          out[k] += t[u][k];
  }
  block_sums(out);
}

__device__ __forceinline__ void publish_cg(Ctl *c) {
  if (c->host_mirror) {
    const unsigned long long w = (static_cast<unsigned long long>(c->seq) << 32) |
                                 (static_cast<unsigned long long>(c->cg_done ? 1u : 0u) << 31) |
                                 static_cast<unsigned long long>(static_cast<unsigned>(c->cg_iter));
    __hip_atomic_store(c->host_mirror + 2, w, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

__device__ __forceinline__ void cg_setup_fin_body(Ctl *c, const double *part, unsigned nb,
                                                  double tol, int max_k, unsigned seq) {
  double sums[3];
  sum_partials(part, nb, sums);
  const double bb = sums[0], rr = sums[1], ry = sums[2];
  if (threadIdx.x == 0) {
    c->cg_tol = tol;
    c->cg_max_k = max_k;
    c->cg_b_nsq = bb;
    // thr = max(tol^2 |b|^2, FLT_MIN)   (cg_openmp.hpp:74)
    const double thr = tol * tol * bb;
    c->cg_thr = thr > 1.1754943508222875e-38 ? thr : 1.1754943508222875e-38;
    c->cg_r_nsq = rr;
    c->cg_ry = ry;
    c->cg_iter = 0;
    c->cg_done = 0;  // ok(0) holds: k < min_k = 1
    c->seq = seq;
    publish_cg(c);
  }
}

__global__ __launch_bounds__(kBlock) void k_cg_setup_fin(Ctl *c, const double *part,
                                                         unsigned nb, double tol, int max_k,
                                                         unsigned seq) {
  cg_setup_fin_body(c, part, nb, tol, max_k, seq);
}

// |p.q| < tol breaks (cg_openmp.hpp:147); alpha = (r.y) / (p.q)
__device__ __forceinline__ void cg_alpha_body(Ctl *c, const double *part, unsigned nb) {
  if (c->cg_done)
    return;
  double sums[1];
  sum_partials(part, nb, sums);
  const double pq = sums[0];
  if (threadIdx.x == 0) {
    c->cg_ry_prev = c->cg_ry;
    c->cg_pq = pq;
    if (fabs(pq) < c->cg_tol) {
      c->cg_done = 1;
      publish_cg(c);
    } else {
      c->cg_alpha = c->cg_ry_prev / pq;
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_cg_alpha(Ctl *c, const double *part, unsigned nb) {
  cg_alpha_body(c, part, nb);
}

// |r.y|_prev < tol breaks (:187); beta; ++k; ok(k, |r|^2) (:100-111)
__device__ __forceinline__ void cg_beta_body(Ctl *c, const double *part, unsigned nb) {
  if (c->cg_done)
    return;
  double sums[2];
  sum_partials(part, nb, sums);
  const double rr = sums[0], ry = sums[1];
  if (threadIdx.x == 0) {
    c->cg_r_nsq = rr;
    c->cg_ry = ry;
    if (fabs(c->cg_ry_prev) < c->cg_tol) {
      c->cg_done = 1;
    } else {
      c->cg_beta = ry / c->cg_ry_prev;
      const int k = c->cg_iter + 1;
      c->cg_iter = k;
      if (k > c->cg_max_k || rr < c->cg_thr)
        c->cg_done = 1;
    }
    publish_cg(c);
  }
}

__global__ __launch_bounds__(kBlock) void k_cg_beta(Ctl *c, const double *part, unsigned nb) {
  cg_beta_body(c, part, nb);
}

// The same decisions inside the vector kernels of an iteration, for
// launches of at most kFusedCgBlocks blocks: every block sums all partials of
// the kernel before it (in the order of the one-block kernels, so every
// block derives the same scalars and decisions), and block
// 0 writes them to the control block. The iteration count the stop test
// needs is staged in cg_iter_next beside alpha, so no value a block reads is
// written in the same kernel except cg_done, which a block reads once
// (cg_done_for_block): a block that sees it set would have decided the same.
// (kFusedCgBlocks: scene.hpp)

// cg_done as one value for the whole block. Block 0 of a folded kernel may
// set it while the wavefronts of another block start, so each wavefront
// reading it itself could see different values; a block that split would
// reduce with missing wavefronts. Thread 0 reads it for the block.
__device__ __forceinline__ bool cg_done_for_block(const Ctl *c) {
  __shared__ int flag;
  if (threadIdx.x == 0)
    flag = c->cg_done;
  __syncthreads();
  const bool done = flag != 0;
  __syncthreads();  // a later call writes flag again
  return done;
}

// k_cg_alpha in every block of the update kernel: false when the solve
// breaks (|p.q| < tol), else alpha
// (lb: the block's logical index; block 0 writes the control block)
__device__ __forceinline__ bool cg_alpha_in_block(Ctl *c, const double *pq_part, unsigned nb,
                                                  double *alpha, unsigned lb = blockIdx.x) {
  double sums[1];
  sum_partials(pq_part, nb, sums);
  const double pq = sums[0];
  const double ry_prev = c->cg_ry;
  const bool brk = fabs(pq) < c->cg_tol;
  if (lb == 0 && threadIdx.x == 0) {
    c->cg_ry_prev = ry_prev;
    c->cg_pq = pq;
    c->cg_iter_next = c->cg_iter + 1;
    if (brk) {
      c->cg_done = 1;
      publish_cg(c);
    } else {
      c->cg_alpha = ry_prev / pq;
    }
  }
  *alpha = brk ? 0.0 : ry_prev / pq;
  return !brk;
}

// k_cg_beta in every block of the direction kernel (r.r partials at part,
// r.y at part + nb): false when the solve is done, else beta
__device__ __forceinline__ bool cg_beta_in_block(Ctl *c, const double *part, unsigned nb,
                                                 double *beta, unsigned lb = blockIdx.x) {
  double sums[2];
  sum_partials(part, nb, sums);
  const double rr = sums[0], ry = sums[1];
  const double ry_prev = c->cg_ry_prev;
  const bool brk = fabs(ry_prev) < c->cg_tol;
  const double b = brk ? 0.0 : ry / ry_prev;
  const int k = c->cg_iter_next;
  const bool done = brk || k > c->cg_max_k || rr < c->cg_thr;
  if (lb == 0 && threadIdx.x == 0) {
    c->cg_r_nsq = rr;
    c->cg_ry = ry;
    if (!brk) {
      c->cg_beta = b;
      c->cg_iter = k;
    }
    if (done)
      c->cg_done = 1;
    publish_cg(c);
  }
  *beta = b;
  return !done;
}

// ---- three scalar systems solved side by side (pt16: the components of a
// vector field): each has its own scalars, decisions and iteration count
// (Ctl::c3) with the rules above, so each is the solve it would be alone. Set-up
// partials: b.b, r.r, r.y of the components at [0, 9 nb); p.q at [0, 3 nb); r.r,
// r.y at [0, 6 nb). cg_iter counts the iterations run, cg_done is set when every
// component is done.
__device__ __forceinline__ void publish_cg3(Ctl *c) {
  if (c->host_mirror)  // the last component's own count, before the progress word
    __hip_atomic_store(c->host_mirror + kMirrorCg3, static_cast<unsigned long long>(c->c3.iter[2]),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  publish_cg(c);
}

__device__ __forceinline__ void cg3_setup_fin_body(Ctl *c, const double *part, unsigned nb,
                                                   double tol, int max_k, unsigned seq) {
  double sums[9];
  sum_partials(part, nb, sums);
  if (threadIdx.x == 0) {
    c->cg_tol = tol;
    c->cg_max_k = max_k;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double thr = tol * tol * sums[k];
      c->c3.thr[k] = thr > 1.1754943508222875e-38 ? thr : 1.1754943508222875e-38;
      c->c3.ry[k] = sums[6 + k];
      c->c3.iter[k] = 0;
      c->c3.done[k] = 0;
    }
    c->cg_iter = 0;
    c->cg_done = 0;
    c->seq = seq;
    publish_cg3(c);
  }
}

// the components not yet done, one value for the whole block (0: all done):
// block 0 of a folded kernel may set a flag while other blocks start, and a
// block that sees it set would decide the same itself
__device__ __forceinline__ unsigned cg3_live(const Ctl *c) {
  __shared__ unsigned live;
  if (threadIdx.x == 0)
    live = c->cg_done ? 0u
                      : (c->c3.done[0] ? 0u : 1u) | (c->c3.done[1] ? 0u : 2u) |
                            (c->c3.done[2] ? 0u : 4u);
  __syncthreads();
  const unsigned r = live;
  __syncthreads();
  return r;
}

// alpha of every live component; the components that go on. write: this block
// stores them
__device__ __forceinline__ unsigned cg3_alpha(Ctl *c, const double *pq_part, unsigned nb,
                                              unsigned live, bool write, double (&alpha)[3]) {
  double pq[3];
  sum_partials(pq_part, nb, pq);
  unsigned on = live;
  double ry_prev[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    ry_prev[k] = c->c3.ry[k];
    alpha[k] = 0.0;
    if (!((live >> k) & 1u))
      continue;
    if (fabs(pq[k]) < c->cg_tol)
      on &= ~(1u << k);
    else
      alpha[k] = ry_prev[k] / pq[k];
  }
  if (write && threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if (!((live >> k) & 1u))
        continue;
      c->c3.ry_prev[k] = ry_prev[k];
      c->c3.iter_next[k] = c->c3.iter[k] + 1;
      if ((on >> k) & 1u)
        c->c3.alpha[k] = alpha[k];
      else
        c->c3.done[k] = 1;
    }
    if (on == 0u) {
      c->cg_done = 1;
      publish_cg3(c);
    }
  }
  return on;
}

// beta of every live component; the components that go on
__device__ __forceinline__ unsigned cg3_beta(Ctl *c, const double *part, unsigned nb,
                                             unsigned live, bool write, double (&beta)[3]) {
  double sums[6];
  sum_partials(part, nb, sums);
  unsigned on = live;
  int prog = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    beta[k] = 0.0;
    if (!((live >> k) & 1u))
      continue;
    const double ry_prev = c->c3.ry_prev[k];
    const bool brk = fabs(ry_prev) < c->cg_tol;
    const int it = c->c3.iter_next[k];
    const bool done = brk || it > c->cg_max_k || sums[k] < c->c3.thr[k];
    if (!brk)
      beta[k] = sums[3 + k] / ry_prev;
    if (done)
      on &= ~(1u << k);
    if (write && threadIdx.x == 0) {
      c->c3.ry[k] = sums[3 + k];
      if (!brk) {
        c->c3.beta[k] = beta[k];
        c->c3.iter[k] = it;
      }
      if (done)
        c->c3.done[k] = 1;
    }
    prog = it > prog ? it : prog;
  }
  if (write && threadIdx.x == 0) {
    c->cg_iter = prog;
    if (on == 0u)
      c->cg_done = 1;
    publish_cg3(c);
  }
  return on;
}

}  // namespace
}  // namespace prtcl_amd
