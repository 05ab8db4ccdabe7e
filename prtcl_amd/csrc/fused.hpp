// Launchers of the fused step kernels (fused.hip).
#pragma once

#include "nbrlist.hpp"

namespace prtcl_amd {

// Launch schedule of a step. All schedules give bit-identical results.
struct FusedSchedule {
  // bits 0-2 of a mask chose LDS-staged passes, which are slower than the
  // gathers through L2 at every size; they are accepted, reported back and
  // change nothing
  int unused = 0;
  // each IISPH iteration is replayed from a captured hipGraph unless eager
  bool eager = false;
  // the CG iterations (WKBB18, pt16) launch their one-block alpha and beta
  // kernels even where the vector kernels can derive the scalars themselves
  bool cg_split = false;
  // the WKBB18 diagonal and the CG set-up of a fused step in two list walks
  // instead of one
  bool wk_split = false;
  // IISPH iteration 1 in its own two neighbour passes instead of folded into
  // the setup pass (the fold needs no neighbours: every pressure starts at 0)
  bool first_split = false;
  int mask() const {
    return unused | (eager ? 8 : 0) | (cg_split ? 16 : 0) | (wk_split ? 32 : 0) |
           (first_split ? 64 : 0);
  }
  static FusedSchedule from_mask(int m) {
    FusedSchedule s;
    s.unused = m & 7;
    s.eager = (m & 8) != 0;
    s.cg_split = (m & 16) != 0;
    s.wk_split = (m & 32) != 0;
    s.first_split = (m & 64) != 0;
    return s;
  }
};

// The schedule in force: a forced mask (>= 0), or the default. Graph replay of
// the iteration measured no faster than eager launches on this stack: eager
// unless a forced mask clears bit 3.
struct ScheduleChoice {
  int forced = -1;
  FusedSchedule current() const { return FusedSchedule::from_mask(forced >= 0 ? forced : 8); }
  void force(int mask) { forced = mask; }
};

template <class T>
struct FusedOps {
  // the neighbour list alone, for the procedures: every particle includes
  // itself, at its place in slot order
  static void build_list(hipStream_t st, const SceneView<T> &S, const NbrList &L);
  // density, neighbour list, IISPH c / AA / s; with explicit viscosity or axial
  // gravity also the integrated velocity, into vtmp (otherwise S.v holds it)
  // B.seq != 0: the first kernel also begins solve B (one launch fewer)
  static void setup(hipStream_t st, const SceneView<T> &S, const NbrList &L,
                    bool explicit_viscosity, vec4_t<T> *vtmp,
                    const SolveBegin &B = SolveBegin{});
  // the pressure acceleration goes to the second half of S.xa only
  // fold: the pass first ends the iteration before it, whose pressure pass had
  // last = false (only where folds(nf)); last: with the iteration's end
  static void accel(hipStream_t st, const SceneView<T> &S, const NbrList &L, bool fold = false);
  static void pressure(hipStream_t st, const SceneView<T> &S, const NbrList &L, bool last = true);
  static bool folds(int nf);
  // the convergence step of IISPH iteration 1, whose pressures and aprde
  // partials the setup (with S.first_iter) has written (batched: for the
  // scenes without first_preset)
  static void finish_first_iteration(hipStream_t st, const SceneView<T> &S,
                                     bool explicit_viscosity);
  static void finish_first_iteration_batch(hipStream_t st, const BatchEntry<T> *tab,
                                           unsigned nscenes);
  // v += dt a H, x += dt v, with a from S.xa, also stored to S.a; seq > 0:
  // enqueued ahead of the host's knowledge that IISPH solve seq is done, it
  // integrates only once that solve is done, and only once (integrate_now)
  static void integrate(hipStream_t st, const SceneView<T> &S, unsigned seq = 0);
  // S.a from S.xa (before a procedure kernel reads the acceleration)
  static void copy_accel(hipStream_t st, const SceneView<T> &S);
  // the same passes over every scene of a batch; group 0 of B are the scenes with
  // the one-launch setup, group 1 those with the three-launch setup (entry
  // flag explicit_visc: explicit viscosity, else axial gravity)
  static void setup_batch(hipStream_t st, const BatchEntry<T> *tab, const BatchBlocks &B);
  static void accel_batch(hipStream_t st, const BatchEntry<T> *tab, const BatchBlocks &B);
  static void pressure_batch(hipStream_t st, const BatchEntry<T> *tab, const BatchBlocks &B,
                             unsigned nscenes);
  // guarded: each scene as integrate() with seq = its solve's sequence
  static void integrate_batch(hipStream_t st, const BatchEntry<T> *tab, const uint32_t *pmap,
                              unsigned npblocks, unsigned nscenes, bool guarded = false);
};

}  // namespace prtcl_amd
