// Candidate search of a neighbour list with 8 lanes per particle: lane l
// takes candidate l of every 8, so a particle's 27 cells (about 216
// candidates) are 27 loads per lane, ten of them in flight at a time,
// instead of a serial chain of 216 tests in one lane. The accepted
// candidates are appended in ascending slot order, so the list is the one
// that a single lane per particle builds.
#pragma once

#include <type_traits>

#include "nbrlist.hpp"

namespace prtcl_amd {

constexpr int kScanLanes = 8;
constexpr int kScanParts = kBlock / kScanLanes;  // particles per block
constexpr uint32_t kScanRow = 64;                // list entries kept per particle
static_assert((1 << kSpanShiftScan) == kScanParts, "one span table per block of the scan");
static_assert(kNbrCap + 1 < kScanRow, "a full list and one more must fit a row");

struct alignas(16) Scan8Shared {
  uint16_t lst[kScanParts][kScanRow];  // accepted candidates, relative to their span
  uint32_t rb[kScanParts][9], re[kScanParts][9];
  uint32_t lo[3], hi[3];
  BlockRanges R;
};

// the result for the lane's particle: entries in lst[p][0, cnt), cs per slab
struct Scan8 {
  uint32_t cnt, cs0, cs1, cs2;
  bool over;  // more neighbours than the list holds, or a span beyond 16 bits
};

// bounds of x-run r (0..8, stencil order) of a cell; empty outside the box
__device__ __forceinline__ void run_bounds(const GridDims &g, uint32_t cellc,
                                           const uint32_t *__restrict__ start, int r,
                                           uint32_t *b, uint32_t *e) {
  const int cx = static_cast<int>(cellc & 0x7FFu);
  const int y = static_cast<int>((cellc >> 11) & 0x7FFu) + r % 3 - 1;
  const int z = static_cast<int>(cellc >> 22) + r / 3 - 1;
  const bool ok = z >= 0 && z < g.nz && y >= 0 && y < g.ny;
  const uint32_t x0 = static_cast<uint32_t>(cx > 0 ? cx - 1 : 0);
  const uint32_t x1 = static_cast<uint32_t>(cx + 1 < g.nx ? cx + 1 : g.nx - 1);
  const uint32_t row = ok ? static_cast<uint32_t>(g.nx) *
                                (static_cast<uint32_t>(y) +
                                 static_cast<uint32_t>(g.ny) * static_cast<uint32_t>(z))
                          : 0u;
  const uint32_t lo = start[row + x0], hi = start[row + x1 + 1u];
  *b = ok ? lo : 0u;
  *e = ok ? hi : 0u;
}

// makes the rows written by other lanes of the wavefront readable
__device__ __forceinline__ void scan8_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Candidates of particle i = 32 lb + threadIdx.x / 8 (every thread of the block
// calls it; valid: i < nf). kSelf: by the exact predicate, the particle itself
// included; otherwise by their 16-bit positions, without the particle: the caller
// applies the exact predicate and drops what it rejects (scan8_drop). Writes the
// block's span table.
template <class T, bool kSelf>
__device__ __forceinline__ Scan8 scan8(const SceneView<T> &S, const NbrList &L, unsigned lb,
                                       Scan8Shared &sh, int i, bool valid, uint32_t cell,
                                       const vec4_t<T> &xi) {
  const unsigned t = threadIdx.x;
  const unsigned sub = t % kScanLanes, p = t / kScanLanes;
  const unsigned lane = t % kWave;
  if (t < 3) {
    sh.lo[t] = 0xFFFFFFFFu;
    sh.hi[t] = 0u;
  }
  __syncthreads();
  // lane l of a particle fetches the bounds of run l, lane 0 also run 8; the
  // smallest start and largest end of each run over the wavefront's
  // particles go to the span of the run's slab
  auto bounds = [&](int r) {
    uint32_t b = 0u, e = 0u;
    if (valid)
      run_bounds(S.grid, cell, S.fstart, r, &b, &e);
    sh.rb[p][r] = b;
    sh.re[p][r] = e;
    if (e > b) {
      atomicMin(&sh.lo[r / 3], b);
      atomicMax(&sh.hi[r / 3], e);
    }
  };
  bounds(static_cast<int>(sub));
  if (sub == 0)
    bounds(8);
  __syncthreads();
  if (t < 3) {
    const uint32_t b = sh.lo[t], e = sh.hi[t];
    sh.R.base[t] = b < e ? b : 0u;
    sh.R.len[t] = b < e ? e - b : 0u;
  }
  __syncthreads();
  if (t < 6)
    reinterpret_cast<uint32_t *>(L.blk + lb)[t] = t < 3 ? sh.R.base[t] : sh.R.len[t - 3];
  const Spans R = Spans::of(sh.R);

  Scan8 out{0u, 0u, 0u, 0u, R.max_len() > 0x10000u};
  if (out.over)  // the same for every thread of the block
    return out;
  uint32_t cnt = 0;
  const unsigned group = lane & ~7u;
  // candidate j, appended in lane order where it is accepted
  auto append = [&](uint32_t base, uint32_t j, bool ok) {
    const uint32_t m = static_cast<uint32_t>(__ballot(ok) >> group) & 0xFFu;
    const uint32_t at = cnt + static_cast<uint32_t>(__popc(m & ((1u << sub) - 1u)));
    if (ok && at < kScanRow)
      sh.lst[p][at] = static_cast<uint16_t>(j - base);
    cnt += static_cast<uint32_t>(__popc(m));
  };
  // the positions that candidates are tested by
  using Pos = std::conditional_t<kSelf, vec4_t<T>, uint2>;
  const uint2 fi = !kSelf && valid ? S.xf[i] : make_uint2(0u, 0u);
  auto load = [&](uint32_t j) {
    if constexpr (kSelf)
      return S.xm[j];
    else
      return S.xf[j];
  };
  auto near = [&](uint32_t j, const Pos &pj) {
    if constexpr (kSelf)
      return sqdist_exact(xi.x - pj.x, xi.y - pj.y, xi.z - pj.z) < S.thr2;
    else
      return (j != static_cast<uint32_t>(i)) &
             (fixed_sqdist(fi.x, fi.y, pj.x, pj.y) < kFixReach);
  };
  // The three runs of a slab as one sequence of candidates: lane l takes the
  // candidates l, l + 8, ... of it, kIn loads in flight (a lane past the end
  // reads slot 0). A fluid at rest has about 72 candidates a slab.
  constexpr uint32_t kIn = sizeof(Pos) <= 16 ? 10u : 5u;
  uint32_t c_end[3];
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    const uint32_t base = R.base(s);
    const uint32_t b0 = sh.rb[p][3 * s], b1 = sh.rb[p][3 * s + 1], b2 = sh.rb[p][3 * s + 2];
    const uint32_t n0 = sh.re[p][3 * s] - b0;
    const uint32_t n01 = n0 + (sh.re[p][3 * s + 1] - b1);
    const uint32_t tot = n01 + (sh.re[p][3 * s + 2] - b2);
    const uint32_t o1 = b1 - n0, o2 = b2 - n01;
    for (uint32_t q0 = sub; __ballot(q0 < tot) != 0ull; q0 += kIn * kScanLanes) {
      Pos pk[kIn];
      uint32_t jk[kIn];
#pragma unroll
      for (uint32_t u = 0; u < kIn; ++u) {
        const uint32_t q = q0 + u * kScanLanes;
        jk[u] = q < tot ? q + (q < n0 ? b0 : (q < n01 ? o1 : o2)) : 0u;
        pk[u] = load(jk[u]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (uint32_t u = 0; u < kIn; ++u) {
        const bool in = q0 + u * kScanLanes < tot;
        if (__ballot(in) != 0ull)
          append(base, jk[u], in & near(jk[u], pk[u]));
      }
    }
    c_end[s] = cnt;
  }
  out.cnt = cnt;
  out.cs0 = c_end[0];
  out.cs1 = c_end[1] - c_end[0];
  out.cs2 = c_end[2] - c_end[1];
  out.over = cnt > kNbrCap;
  scan8_sync();
  return out;
}

// Drops entries of the rows: bit m of a lane's `rejected` is entry 8 m + lane of its
// particle (every lane of the wavefront calls it; rarely is there any).
__device__ __forceinline__ void scan8_drop(Scan8Shared &sh, Scan8 &c, uint32_t rejected) {
  if (__ballot(rejected != 0u) == 0ull)
    return;
  const unsigned sub = threadIdx.x % kScanLanes, p = threadIdx.x / kScanLanes;
  const unsigned group = (threadIdx.x % kWave) & ~7u;
  uint64_t out = 0;
#pragma unroll
  for (int m = 0; m < static_cast<int>(kScanRow / kScanLanes); ++m)
    out |= ((__ballot((rejected >> m) & 1u) >> group) & 0xFFull) << (8 * m);
  uint32_t kept = 0, ks0 = 0, ks1 = 0;
  if (sub == 0 && out != 0)
    for (uint32_t e = 0; e < c.cnt; ++e)
      if (!((out >> e) & 1u)) {
        sh.lst[p][kept++] = sh.lst[p][e];
        ks0 += e < c.cs0 ? 1u : 0u;
        ks1 += e >= c.cs0 && e < c.cs0 + c.cs1 ? 1u : 0u;
      }
  scan8_sync();
  kept = __shfl(kept, static_cast<int>(group), kWave);
  ks0 = __shfl(ks0, static_cast<int>(group), kWave);
  ks1 = __shfl(ks1, static_cast<int>(group), kWave);
  if (out != 0) {
    c.cnt = kept;
    c.cs0 = ks0;
    c.cs1 = ks1;
    c.cs2 = kept - ks0 - ks1;
  }
}

// the list of particle i to memory: lane l writes chunk l
__device__ __forceinline__ void scan8_write(const NbrList &L, const Scan8Shared &sh, size_t n,
                                            int i, const Scan8 &c, bool boundary) {
  const unsigned sub = threadIdx.x % kScanLanes, p = threadIdx.x / kScanLanes;
  if (!c.over && sub * kChunk < c.cnt)
    reinterpret_cast<uint4 *>(L.idx)[static_cast<size_t>(sub) * n + static_cast<size_t>(i)] =
        reinterpret_cast<const uint4 *>(sh.lst[p])[sub];
  if (sub == 0)
    L.info[i] = c.over ? kListOverflow
                       : (c.cs0 | (c.cs1 << 8) | (c.cs2 << 16) |
                          (boundary ? kListBoundary : 0u));
}

}  // namespace prtcl_amd
