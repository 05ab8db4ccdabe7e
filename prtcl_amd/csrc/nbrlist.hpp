// Per-step fluid neighbour list of the fused step, built by the setup pass
// and walked by every later neighbour pass of the step.
//
// The 27-cell stencil of a particle is 9 x-runs (rows dy, dz = -1..1, cells
// x-1..x+1). Slots are in cell order, x fastest, so the three runs of one dz
// ("slab") of every particle of a block of kBlock consecutive slots lie in
// one slot interval, the block's span of that slab: from the first run start
// to the last run end over the block's particles (about three rows of
// particles). A list entry is the neighbour's offset from the span start of
// its slab (16 bits), so the list costs 2 bytes per pair; the global slot is
// span base + entry. (Staging the spans in LDS instead of gathering through L2 is
// slower in full launches: 250,000 particles, setup 72.6 against 68.3 us,
// pressure acceleration 17.3 against 14.8, pressure 29.9 against 23.7; 1M, setup
// 321 against 229.)
//
// Layout: chunks of 8 entries; entry e of particle i at
// idx[((e / 8) * n + i) * 8 + e % 8], so one 16-byte load per lane fetches 8
// entries and a wavefront's load is 1 KB contiguous. Entries are ordered by
// slab; info[i] holds the entry count of each slab (8 bits each),
// kListBoundary where a boundary particle is in reach, and kListOverflow when the particle has
// more than kNbrCap neighbours or a span of its block exceeds 16 bits (its
// passes then walk the grid with the exact predicate instead).
#pragma once

#include <type_traits>

#include "scene.hpp"

namespace prtcl_amd {

constexpr uint32_t kListOverflow = 1u << 31;
// set where a boundary particle is within the radius, so later passes skip
// the boundary walk of the others (an overflowed particle always walks)
constexpr uint32_t kListBoundary = 1u << 24;
__device__ __forceinline__ bool list_has_boundary(uint32_t info) {
  return (info & (kListBoundary | kListOverflow)) != 0u;
}
struct BlockRanges {
  uint32_t base[3];  // first slot of the span of slab s (dz = s - 1)
  uint32_t len[3];   // its length (0: no particle of the block has that layer)
  uint32_t spare[2];
};

// slots per span table: a block's 256, or the 32 of a block that searches with
// 8 lanes per particle (scan8.hpp)
constexpr uint32_t kSpanShiftBlock = 8, kSpanShiftScan = 5;

struct NbrList {
  uint16_t *idx;
  uint32_t *info;
  BlockRanges *blk;  // one per 1 << shift slots
  uint32_t shift;
  uint32_t zero = 0;  // no byte left unset: the list is part of a graph's key
};
static_assert(std::has_unique_object_representations_v<NbrList>, "no padding");

// The span table of one block in registers (selected by slab without
// indexing, so it never lives in scratch memory).
struct Spans {
  uint32_t b0, b1, b2, l0, l1, l2;
  __device__ __forceinline__ static Spans of(const BlockRanges &R) {
    return Spans{R.base[0], R.base[1], R.base[2], R.len[0], R.len[1], R.len[2]};
  }
  __device__ __forceinline__ uint32_t base(int s) const { return s == 0 ? b0 : (s == 1 ? b1 : b2); }
  __device__ __forceinline__ uint32_t max_len() const {
    return l0 > l1 ? (l0 > l2 ? l0 : l2) : (l1 > l2 ? l1 : l2);
  }
};

// the span table of particle i's list
__device__ __forceinline__ Spans list_spans(const NbrList &L, int i) {
  return Spans::of(L.blk[i >> L.shift]);
}

constexpr uint32_t kChunk = 8;  // list entries per 16-byte chunk

// the 8 entries of chunk g of particle i
__device__ __forceinline__ uint4 list_chunk(const NbrList &L, size_t n, int i, uint32_t g) {
  return reinterpret_cast<const uint4 *>(L.idx)[static_cast<size_t>(g) * n +
                                                static_cast<size_t>(i)];
}

// entry k (0..7) of a chunk
__device__ __forceinline__ uint32_t chunk_entry(const uint4 &q, int k) {
  const uint32_t w = k < 2 ? q.x : (k < 4 ? q.y : (k < 6 ? q.z : q.w));
  return (k & 1) ? (w >> 16) : (w & 0xFFFFu);
}

// entries of a (not overflowed) list: the sum of its three slab counts
__device__ __forceinline__ uint32_t list_count(uint32_t info) {
  return (info & 0xFFu) + ((info >> 8) & 0xFFu) + ((info >> 16) & 0xFFu);
}

// Walks the list entries of particle i (not overflowed) in list order, one chunk
// (8 entries) at a time, with the memory traffic of a chunk issued before its
// arithmetic: the chunk, then the gathers (v[k] = load(j_k)) of kGroup entries,
// then use(v[k]) in order. R is the span table of i's list: the slot of entry e is
// b0 + entry + [e >= c0] (b1 - b0) + [e >= c01] (b2 - b1). The next
// chunk is fetched while the current one is in flight. kGroup < 8 keeps fewer
// gathered values live (more waves per SIMD) for wide records.
template <int kGroup = 8, class Load, class Use>
__device__ __forceinline__ void list_gather(const NbrList &L, const Spans &R, size_t n, int i,
                                            uint32_t info, Load &&load, Use &&use) {
  static_assert(kChunk % kGroup == 0, "group must divide the chunk");
  const uint32_t c0 = info & 0xFFu;
  const uint32_t c01 = c0 + ((info >> 8) & 0xFFu);
  const uint32_t c = c01 + ((info >> 16) & 0xFFu);
  const uint32_t d1 = R.b1 - R.b0, d2 = R.b2 - R.b1;
  using V = decltype(load(0u));
  uint4 q = c > 0 ? list_chunk(L, n, i, 0) : make_uint4(0u, 0u, 0u, 0u);
  for (uint32_t g = 0; g * kChunk < c; ++g) {
    const uint4 cur = q;
    if ((g + 1) * kChunk < c)
      q = list_chunk(L, n, i, g + 1);
#pragma unroll
    for (int h = 0; h < static_cast<int>(kChunk); h += kGroup) {
      V v[kGroup];
#pragma unroll
      for (int k = 0; k < kGroup; ++k) {
        const uint32_t e = g * kChunk + h + k;
        if (e < c)
          v[k] = load(R.b0 + chunk_entry(cur, h + k) + (e >= c0 ? d1 : 0u) +
                      (e >= c01 ? d2 : 0u));
      }
      // keep every gather of the group ahead of the arithmetic (the
      // scheduler would otherwise consume each gather before issuing the
      // next one)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < kGroup; ++k)
        if (g * kChunk + h + k < c)
          use(v[k]);
    }
  }
}

// ---- several lanes per particle (small scenes)
//
// A small scene does not fill the chip with one lane per particle (65,536
// particles are one wavefront per SIMD), and a pass takes as long as one lane's
// chain of list chunks and gathers. Up to kSplitMax particles each pass gives a
// particle kListLanes lanes: lane l takes chunks l, l + kListLanes, ... (a mean
// list of 30 entries is four chunks, one per lane) and the lanes' sums are added
// in a fixed tree. Measured per launch, one lane -> four, accel pass: 2,048
// particles 5.9 -> 3.7 us, 8,000: 6.3 -> 3.9, 59,000: 5.5 -> 5.2, 125,000: 7.2 ->
// 7.3, 250,000: 13.6 -> 13.6; pressure pass 8.1 -> 4.7, 8.3 -> 4.9, 8.0 -> 7.1,
// 10.0 -> 10.4, 20.7 -> 21.3. The rule depends on the scene alone, so that a
// scene's results are the same alone and in a batch. At the line a scene of 59,000
// particles still gains (10 steps 1.71 -> 1.51 ms, FP64 27,000 1.90 -> 1.39); a batch,
// which fills the chip anyway, pays for the search's idle lanes (16 scenes of 2,000
// to 200,000 particles: setup 182 -> 221 us, pressure passes 59.3 -> 56.6).
constexpr int kSplitMax = 65536;
constexpr int kListLanes = 4;
__host__ __device__ inline bool split_scene(int nf) { return nf <= kSplitMax; }
// threads of a list pass
__host__ __device__ inline long list_threads(int nf) {
  return split_scene(nf) ? static_cast<long>(nf) * kListLanes : nf;
}
// blocks of a list pass and of the setup pass (scan8.hpp where split)
__host__ __device__ inline unsigned list_blocks(int nf) { return grid_blocks(list_threads(nf)); }
__host__ __device__ inline unsigned setup_blocks(int nf) {
  return split_scene(nf) ? grid_blocks(nf, 1 << kSpanShiftScan) : grid_blocks(nf);
}
__host__ __device__ inline uint32_t list_shift(int nf) {
  return split_scene(nf) ? kSpanShiftScan : kSpanShiftBlock;
}

// The blocks of 256 particles of a batch's scenes: words (scene, local block)
// in four runs, two groups (0, 1: one, 2, 3: the other) of one-lane scenes and
// of split scenes. A list or setup pass launches `factor` blocks for each block
// of a split scene; each run is spread over the XCDs in contiguous parts.
struct BatchBlocks {
  const uint32_t *map;
  unsigned n[4];
  __host__ unsigned launch(unsigned factor) const {
    return n[0] + n[2] + factor * (n[1] + n[3]);
  }
  __host__ BatchBlocks group(int g) const {
    return BatchBlocks{map + (g ? n[0] + n[1] : 0u),
                       {g ? 0u : n[0], g ? 0u : n[1], g ? n[2] : 0u, g ? n[3] : 0u}};
  }
};
static_assert(std::has_unique_object_representations_v<BatchBlocks>, "no padding (graph keys)");
// the word of this block and its part (0 .. factor - 1) of a split scene's block
__device__ __forceinline__ uint32_t batch_block(const BatchBlocks &B, unsigned factor,
                                                unsigned *part) {
  unsigned x = blockIdx.x;
  const uint32_t *m = B.map;
  uint32_t word = 0;
  *part = 0;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const unsigned f = (s & 1) ? factor : 1u;
    const unsigned cnt = f * B.n[s];
    if (x < cnt) {
      const unsigned l = xcd_block(x, cnt);
      *part = l % f;
      word = m[l / f];
      break;
    }
    x -= cnt;
    m += B.n[s];
  }
  return word;
}

// the span table of a wavefront of a fused list pass with kLanes lanes per
// particle (block lb of the pass), uniform over the wavefront: one lane per
// particle goes with a table per block, four with a table per 32 particles
template <int kLanes>
__device__ __forceinline__ Spans pass_spans(const NbrList &L, int nf, unsigned lb) {
  if (kLanes == 1)
    return Spans::of(L.blk[lb]);
  static_assert(kWave / kListLanes <= (1 << kSpanShiftScan), "one table per wavefront");
  const int first = __builtin_amdgcn_readfirstlane(
      static_cast<int>((lb * kBlock + (threadIdx.x & ~63u)) / kLanes));
  return Spans::of(L.blk[first < nf ? first >> kSpanShiftScan : 0]);
}

// list_gather for lane `sub` of kLanes lanes of particle i
template <int kLanes, int kGroup, class Load, class Use>
__device__ __forceinline__ void list_gather_lanes(const NbrList &L, const Spans &R, size_t n, int i,
                                                  uint32_t info, uint32_t sub, Load &&load,
                                                  Use &&use) {
  if (kLanes == 1) {
    list_gather<kGroup>(L, R, n, i, info, load, use);
    return;
  }
  const uint32_t c0 = info & 0xFFu;
  const uint32_t c01 = c0 + ((info >> 8) & 0xFFu);
  const uint32_t c = c01 + ((info >> 16) & 0xFFu);
  const uint32_t d1 = R.b1 - R.b0, d2 = R.b2 - R.b1;
  using V = decltype(load(0u));
  for (uint32_t g = sub; g * kChunk < c; g += kLanes) {
    const uint4 q = list_chunk(L, n, i, g);
#pragma unroll
    for (int h = 0; h < static_cast<int>(kChunk); h += kGroup) {
      V v[kGroup];
#pragma unroll
      for (int k = 0; k < kGroup; ++k) {
        const uint32_t e = g * kChunk + h + k;
        if (e < c)
          v[k] = load(R.b0 + chunk_entry(q, h + k) + (e >= c0 ? d1 : 0u) + (e >= c01 ? d2 : 0u));
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < kGroup; ++k)
        if (g * kChunk + h + k < c)
          use(v[k]);
    }
  }
}

// the value of the lane beside (lane ^ 1; every lane of the wavefront calls it)
template <class V>
__device__ __forceinline__ V pair_swap(const V &v) {
  static_assert(sizeof(V) % sizeof(int) == 0, "whole words");
  int w[sizeof(V) / sizeof(int)];
  __builtin_memcpy(w, &v, sizeof(V));
#pragma unroll
  for (unsigned k = 0; k < sizeof(V) / sizeof(int); ++k)
    w[k] = __builtin_amdgcn_update_dpp(0, w[k], 0xB1, 0xF, 0xF, true);  // quad_perm 1 0 3 2
  V r;
  __builtin_memcpy(&r, w, sizeof(V));
  return r;
}

// list_gather_lanes for records of two adjacent values: use(rec[2 j], rec[2 j + 1])
// for the entries j of the lane. A gather is bound by the cache lines that its
// lanes touch, and the two values of a record lie in one line: so two lanes load
// the two values of the even lane's record together, then those of the odd lane's,
// and exchange what is the other's. Every lane of the wavefront calls it (info 0: no
// entries); a lane without an entry left loads record `idle`. Pressure pass of 1M
// particles 87 -> 79 us, of a batch 37.5 -> 34.5, CG product of 250,000 22.2 -> 20.5.
// With four lanes per particle it pays only for 32-byte values (FP64, 27,000: 7.4 ->
// 6.5 us; FP32, 2,048: 4.2 -> 4.7, 59,000: 6.8 -> 6.9): launches of latency rather than
// of cache lines.
template <int kLanes, int kGroup, class V, class Use>
__device__ __forceinline__ void list_gather_records(const NbrList &L, const Spans &R, size_t n,
                                                    int i, uint32_t info, uint32_t sub,
                                                    uint32_t idle, const V *__restrict__ rec,
                                                    Use &&use) {
  if constexpr (kLanes > 1 && sizeof(V) == 16) {
    struct Two {
      V a, b;
    };
    list_gather_lanes<kLanes, kGroup>(
        L, R, n, i, info, sub,
        [&](uint32_t j) {
          return Two{rec[2 * static_cast<size_t>(j)], rec[2 * static_cast<size_t>(j) + 1]};
        },
        [&](const Two &q) { use(q.a, q.b); });
    return;
  }
  const uint32_t c0 = info & 0xFFu;
  const uint32_t c01 = c0 + ((info >> 8) & 0xFFu);
  const uint32_t c = c01 + ((info >> 16) & 0xFFu);
  const uint32_t d1 = R.b1 - R.b0, d2 = R.b2 - R.b1;
  const bool odd = (threadIdx.x & 1u) != 0u;
  const V *__restrict__ half = rec + (odd ? 1 : 0);
  const uint4 none = make_uint4(0u, 0u, 0u, 0u);
  uint4 q = sub * kChunk < c ? list_chunk(L, n, i, sub) : none;
  for (uint32_t g = sub; __ballot(g * kChunk < c) != 0ull; g += kLanes) {
    const uint4 cur = q;
    if ((g + kLanes) * kChunk < c)
      q = list_chunk(L, n, i, g + kLanes);
#pragma unroll
    for (int h = 0; h < static_cast<int>(kChunk); h += kGroup) {
      V r1[kGroup], r2[kGroup];
      if (__ballot(g * kChunk + h < c) == 0ull)
        break;
#pragma unroll
      for (int k = 0; k < kGroup; ++k) {
        const uint32_t e = g * kChunk + h + k;
        const uint32_t j =
            e < c ? R.b0 + chunk_entry(cur, h + k) + (e >= c0 ? d1 : 0u) + (e >= c01 ? d2 : 0u)
                  : idle;
        const uint32_t p = pair_swap(j);
        r1[k] = half[2 * static_cast<size_t>(odd ? p : j)];  // the even lane's neighbour
        r2[k] = half[2 * static_cast<size_t>(odd ? j : p)];  // the odd lane's
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < kGroup; ++k) {
        const V s1 = pair_swap(r1[k]), s2 = pair_swap(r2[k]);
        if (g * kChunk + h + k < c)
          use(odd ? s2 : r1[k], odd ? r2[k] : s1);
      }
    }
  }
}

// the sum over a particle's kLanes lanes, in every one of them (all lanes of
// the wavefront call it)
template <int kLanes, class T>
__device__ __forceinline__ T lanes_sum(T v) {
#pragma unroll
  for (int o = 1; o < kLanes; o <<= 1)
    v += __shfl_xor(v, o, kWave);
  return v;
}

// The sum over a block of a value that the first of every kLanes lanes holds
// (valid in thread 0; all threads of the block call it, once per kernel). With
// several lanes neighbouring particles are added first, so that the sums of two
// blocks of 32 particles (8 lanes) add up to exactly the sum of the block of 64
// (4 lanes) that they make.
template <int kLanes>
__device__ __forceinline__ double particle_sum(double v) {
  if (kLanes == 1)
    return block_sum<kBlock>(v);
  static_assert(kBlock / kWave == 4, "four wavefronts per block");
  __shared__ double ws[kBlock / kWave];
#pragma unroll
  for (int o = kLanes; o < kWave; o <<= 1)
    v += __shfl_xor(v, o, kWave);
  if (threadIdx.x % kWave == 0)
    ws[threadIdx.x / kWave] = v;
  __syncthreads();
  return (ws[0] + ws[1]) + (ws[2] + ws[3]);
}

}  // namespace prtcl_amd
