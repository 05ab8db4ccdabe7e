"""The passes that give a particle several lanes (scenes of up to 65,536
particles), those that give it one, and the procedures' list, at the sizes where they
change: groups of 32 and 64 particles with remainders, and the line between them.
Bars: density is one pair sum in another order (2e-5 of the field's scale, as for
the single procedures), position after one step as for whole steps (1e-5)."""

import os

import numpy as np
import pytest

from prtcl_amd import scenes

pytestmark = pytest.mark.gpu

SPLIT = 65536  # kSplitMax


def _block(n, seed=4, jitter=1e-3, **kw):
    """n particles of a jittered block in a box, moving."""
    s = 0.025
    side = int(np.ceil(n ** (1 / 3)))
    box = scenes.box_boundary(side + 4, side + 4, side + 4, s)
    fx = scenes.fluid_block((side, side, side), (1, 1, 1), s, jitter, scenes.stream_base(seed, n))
    v = np.random.default_rng(n).uniform(-0.2, 0.2, (n, 3))
    sc = scenes._finish(f"block{n}", s, fx[:n], box, 1, v=v, **kw)
    sc.permute_every = 0
    return sc


def _close(gpu, ref, rtol, what):
    scale = float(np.max(np.abs(ref)))
    err = float(np.max(np.abs(np.asarray(gpu, np.float64) - ref))) / scale
    assert err <= rtol, f"{what}: {err:.3e} > {rtol:.1e}"


@pytest.mark.parametrize("n,jitter", [(n, 1e-3) for n in (1, 31, 32, 33, 64, 65, 255, 257, 1025,
                                                         SPLIT, SPLIT + 1)] +
                         [(n, 0.0) for n in (343, SPLIT + 1)])
def test_step_sizes_vs_oracle(hip_ctx, oracle_lib, n, jitter):
    """Without jitter most particles have six neighbours at exactly the radius, which
    the 16-bit candidate test leaves to the exact predicate."""
    from prtcl_amd import hip
    sc = _block(n, jitter=jitter)
    o = oracle_lib.OracleScene(sc, fp64_reductions=True, permute_every=0)
    g = hip.HipScene(hip_ctx, sc)
    o.prepare()
    g.prepare()
    o.step()
    g.step(1)
    _close(g.download("fluid", "density"), o.get("fluid", "density"), 2e-5, "density")
    _close(g.download("fluid", "position"), o.get("fluid", "position"), 1e-5, "position")
    g.destroy()


@pytest.mark.parametrize("n", [31, 33, 65, 257])
@pytest.mark.parametrize("iv", [1, 2, 3], ids=["wkbb18", "wkbb18_gc", "pt16"])
def test_viscous_step_sizes_vs_oracle(hip_ctx, oracle_lib, iv, n):
    """The CG of implicit viscosity with several lanes per particle (pt16: its three
    components side by side). Both sides stop at a relative residual of 1e-4, if
    need be one iteration apart: velocity to ten times that."""
    from prtcl_amd import hip
    sc = _block(n, implicit_viscosity=iv, fluid_viscosity=10.0, boundary_viscosity=10.0,
                wkbb18_maximum_error=1e-4, pt16_vorticity_maximum_error=1e-4,
                pt16_velocity_maximum_error=1e-4)
    o = oracle_lib.OracleScene(sc, fp64_reductions=True, permute_every=0)
    g = hip.HipScene(hip_ctx, sc)
    o.prepare()
    g.prepare()
    o.step()
    g.step(1)
    _close(g.download("fluid", "velocity"), o.get("fluid", "velocity"), 1e-3, "velocity")
    _close(g.download("fluid", "position"), o.get("fluid", "position"), 1e-5, "position")
    g.destroy()


def test_batch_of_both_kinds_equals_alone(hip_ctx):
    """One launch over scenes with several lanes per particle and one beyond the
    line, whose blocks differ in size: each as it is alone."""
    from prtcl_amd import hip
    out = []
    for together in (True, False):
        hs = [hip.HipScene(hip_ctx, _block(n)) for n in (300, SPLIT + 1, 33, SPLIT)]
        for h in hs:
            h.prepare()
        for _ in range(2):
            if together:
                hip_ctx.step(hs, 1)
            else:
                for h in hs:
                    h.step(1)
        out.append([(h.step_info(), h.download("fluid", "velocity"),
                     h.download("fluid", "pressure")) for h in hs])
        for h in hs:
            h.destroy()
    for (ia, va, pa), (ib, vb, pb) in zip(*out):
        assert ia == ib
        np.testing.assert_array_equal(va, vb)
        np.testing.assert_array_equal(pa, pb)


@pytest.mark.parametrize("group", ["fluid", "boundary"])
@pytest.mark.parametrize("n", [8192, 8193, 70001])
def test_grid_follows_uploaded_box(hip_ctx, oracle_lib, n, group):
    """The bounding box of an upload, on the host up to 8,192 particles and on the
    device beyond: after an upload far from the first one every neighbour is found, and
    a particle without a finite position does not move the box."""
    from prtcl_amd import hip
    rng = np.random.default_rng(n)
    sc = scenes.tiny(4)
    fx = rng.uniform(0.0, 0.6, (n if group == "fluid" else 500, 3)).astype(np.float32)
    bx = rng.uniform(0.0, 0.6, (n if group == "boundary" else 500, 3)).astype(np.float32)
    sc = scenes._finish("cloud", 0.025, fx, bx, 1)
    sc.permute_every = 0
    o = oracle_lib.OracleScene(sc, fp64_reductions=True, permute_every=0)
    g = hip.HipScene(hip_ctx, sc)
    o.prepare()
    g.prepare()
    moved = (fx if group == "fluid" else bx) * np.float32([1.0, -2.0, 0.5]) + np.float32(3.0)
    q = 1 if group == "fluid" else 0
    for x in (o, g):
        (x.set if x is o else x.upload)(group, "position", moved)
        x.update() if x is o else x.run("neighborhood.update")
    oo, oi = o.neighbors(q, q)
    go, gi = g.neighbors(q, q)
    np.testing.assert_array_equal(oo, go)
    np.testing.assert_array_equal(oi, gi)
    bad = moved.copy()
    bad[n // 2] = [np.nan, np.inf, -np.inf]
    g.upload(group, "position", bad)
    g.run("neighborhood.update")
    go, gi = g.neighbors(q, q)
    keep = [np.delete(gi[go[i]:go[i + 1]], np.flatnonzero(gi[go[i]:go[i + 1]] == n // 2))
            for i in (0, n // 2 - 1, n - 1)]
    for i, k in zip((0, n // 2 - 1, n - 1), keep):
        ref = oi[oo[i]:oo[i + 1]]
        np.testing.assert_array_equal(k, ref[ref != n // 2])
    g.destroy()


@pytest.mark.parametrize("dims", [(4, 3, 3), (16, 16, 16), (16, 16, 17), (40, 40, 40), (32, 32, 64),
                                  (40, 40, 41), (61, 40, 40)])
def test_sort_over_scan_tiles(hip_ctx, oracle_lib, dims):
    """The cell scan in one launch up to 16 tiles of 4,096 cells and in two beyond, with
    whole and partial last tiles; sorted three times, so counts left over would show."""
    from prtcl_amd import hip
    r = 0.05
    rng = np.random.default_rng(dims[2])
    hi = (np.array(dims) - 3 + 0.5) * r
    fx = rng.uniform(0.5 * r, hi, (700, 3)).astype(np.float32)
    bx = np.array([[0.5 * r] * 3, hi], np.float32)
    sc = scenes._finish("tiles", r / 2, fx, bx, 1)
    sc.permute_every = 0
    o = oracle_lib.OracleScene(sc, fp64_reductions=True, permute_every=0)
    g = hip.HipScene(hip_ctx, sc)
    o.prepare()
    g.prepare()
    for _ in range(3):
        fx = rng.uniform(0.5 * r, hi, (700, 3)).astype(np.float32)
        o.set("fluid", "position", fx)
        o.update()
        g.upload("fluid", "position", fx)
        g.run("neighborhood.update")
        oo, oi = o.neighbors(1, 1)
        go, gi = g.neighbors(1, 1)
        np.testing.assert_array_equal(oo, go)
        np.testing.assert_array_equal(oi, gi)
    g.destroy()


@pytest.mark.parametrize("spacing", [1.0, 0.6], ids=["list", "overflow"])
def test_procedures_follow_the_positions(hip_ctx, oracle_lib, spacing):
    """A procedure between two changes of the positions reads a list that an
    earlier one built; after an upload, an update or an integration it must see
    the new positions (lists that overflow walk the grid)."""
    from prtcl_amd import hip
    s = 0.025
    fx = scenes.fluid_block((9, 9, 9), (3, 3, 3), spacing * s, 1e-4, scenes.stream_base(9, 0))
    sc = scenes._finish("moving", s, fx, scenes.box_boundary(15, 15, 15, s), 1)
    sc.permute_every = 0
    o = oracle_lib.OracleScene(sc, fp64_reductions=True, permute_every=0)
    g = hip.HipScene(hip_ctx, sc)
    o.prepare()
    g.prepare()

    def same(what):
        for x in (o, g):
            x.run("density.compute_density")
        _close(g.download("fluid", "density"), o.get("fluid", "density"), 2e-5, what)

    same("first")
    moved = fx[:, [1, 2, 0]] + np.float32(0.3 * s)
    g.upload("fluid", "position", moved)
    g.run("neighborhood.update")
    o.set("fluid", "position", moved)
    o.update()
    same("after an upload")
    v = np.random.default_rng(1).uniform(-5, 5, fx.shape).astype(np.float32)
    g.upload("fluid", "velocity", v)
    o.set("fluid", "velocity", v)
    for x in (o, g):
        x.run("symplectic_euler.integrate_position")
    g.run("neighborhood.update")
    o.update()
    same("after an integration")
    g.destroy()


KINDS = {
    "plain": {},
    "explicit": dict(explicit_viscosity=True, fluid_viscosity=0.05, boundary_viscosity=0.05),
    "axial": dict(axial_gravity=True, gravity_center=(0.5, 0.5, 0.5)),
    "wkbb18": dict(implicit_viscosity=1, fluid_viscosity=10.0, boundary_viscosity=10.0),
    "wkbb18_gc": dict(implicit_viscosity=2, fluid_viscosity=10.0, boundary_viscosity=10.0),
    "pt16": dict(implicit_viscosity=3, fluid_viscosity=10.0, boundary_viscosity=10.0),
}


@pytest.mark.parametrize("kind,real", [(k, "f32") for k in KINDS] + [("plain", "f64"),
                                                                     ("wkbb18", "f64")])
def test_one_lane_steps_keep_their_bits(hip_ctx, kind, real):
    """Two steps just above the line, at 48 of the particles, against the recorded bits
    of the passes that evaluate every pair term with its factors, in slot order and
    one lane per particle. The pressure solve starts from rho0 - rho, a difference of
    nearly equal numbers: sums in another association differ by 1e-7 in density and
    1e-4 in pressure, so a change of the arithmetic shows here and in no tolerance."""
    from prtcl_amd import hip
    ref = np.load(os.path.join(os.path.dirname(__file__), "golden", "one_lane.npz"))
    g = hip.HipScene(hip_ctx, _block(SPLIT + 1, **KINDS[kind]), real_type=int(real == "f64"))
    g.prepare()
    g.step(2)
    at = np.linspace(0, SPLIT, 48).astype(int)
    for f in ("density", "iisph_diagonal_element", "iisph_source_term", "pressure", "position",
              "velocity"):
        np.testing.assert_array_equal(g.download("fluid", f)[at], ref[f"{kind}.{real}.{f}"], f)
    g.destroy()


def test_diagonal_of_a_lone_particle_at_small_scale(hip_ctx):
    """Without neighbours every pair sum is 0 and so is the diagonal, at every smoothing
    scale whose kernel is in range (the square of the gradient's factor alone is not,
    here 8e41)."""
    from prtcl_amd import hip
    h = 4e-6
    x = np.array([[0, 0, 0], [50 * h, 0, 0]], np.float32)
    sc = scenes._finish("lone", h, x, np.zeros((0, 3), np.float32), 1, v=np.zeros((2, 3)))
    g = hip.HipScene(hip_ctx, sc)
    g.prepare()
    g.step(1)
    np.testing.assert_array_equal(g.download("fluid", "iisph_diagonal_element"), [0, 0])
    g.destroy()


def test_step_far_from_the_origin(hip_ctx):
    """A scene of 64-bit positions 786,432 radii from the origin has the lists, and so
    the bits, that it has at the origin. (All lengths are multiples of 2^-22 and the
    shift is one of the cell edge, 2^-4, so that every difference is exact; beyond 2^18
    radii a candidate position counted from the origin leaves 32 bits, every candidate
    is accepted, and the overflowed lists walk the grid in another order.)"""
    from prtcl_amd import hip
    s = 2.0 ** -5
    rng = np.random.default_rng(8)
    fx = scenes.fluid_block((9, 9, 9), (1, 1, 1), s, 0.0, None).astype(np.float64)
    fx = np.round((fx + rng.uniform(-1e-3, 1e-3, fx.shape)) * 2.0 ** 22) / 2.0 ** 22
    bx = scenes.box_boundary(12, 12, 12, s).astype(np.float64)
    out = []
    for shift in (0.0, 3.0 * 2.0 ** 14, -3.0 * 2.0 ** 14):
        sc = scenes._finish("far", s, fx + shift, bx + shift, 1,
                            v=rng.uniform(-0.2, 0.2, fx.shape) if not out else v)
        v = sc.fluid_v
        sc.permute_every = 0
        g = hip.HipScene(hip_ctx, sc, real_type=1)
        g.prepare()
        g.step(1)
        out.append([g.download("fluid", f) for f in ("density", "iisph_diagonal_element",
                                                     "pressure", "velocity")])
        g.destroy()
    for far in out[1:]:
        for a, b in zip(out[0], far):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n", [343, SPLIT + 1])
@pytest.mark.parametrize("far", [5.0, -5.0, 1e4])
def test_step_outside_the_planned_box(hip_ctx, oracle_lib, n, far):
    """Particles that have left the cell box are candidates of each other in its border
    cells. Eight radii apart their 16-bit positions agree, which the exact predicate has
    to see, also where they are more than a list holds; those within the radius are found."""
    from prtcl_amd import hip
    sc = _block(n, seed=6)
    r = sc.radius
    g = hip.HipScene(hip_ctx, sc)
    g.prepare()  # plans the box
    x = sc.fluid_x.copy()
    k = np.arange(70)
    x[:70] = far
    x[:60, 0] += (8 * r * k[:60]).astype(np.float32)       # a row, all alike in 16 bits
    x[60:70, 1] += (0.9 * r * k[:10]).astype(np.float32)   # a chain of neighbours
    x[60:70, 2] += np.float32(20 * r)
    sc.fluid_x = x
    g.upload("fluid", "position", x)
    o = oracle_lib.OracleScene(sc, fp64_reductions=True, permute_every=0)
    o.prepare()
    o.step()
    g.step(1)
    rho, ref = g.download("fluid", "density"), o.get("fluid", "density")
    np.testing.assert_allclose(rho[:70], ref[:70], rtol=2e-5)
    _close(rho, ref, 2e-5, "density")
    g.destroy()


@pytest.mark.parametrize("iv,n", [(0, n) for n in (1, 2, 3, 257, SPLIT + 1)] +
                         [(3, n) for n in (2, 3, 257, SPLIT + 1)])
def test_step_after_updates_vs_oracle(hip_ctx, oracle_lib, iv, n):
    """An update of all fields exchanges the vector that holds the 16-bit positions with
    the nine-component fields; after one, two and three of them a step finds room. (The
    preconditioner of pt16 divides a lone particle by 0.)"""
    from prtcl_amd import hip
    kw = dict(KINDS["pt16"], pt16_vorticity_maximum_error=1e-4,
              pt16_velocity_maximum_error=1e-4) if iv else {}
    sc = _block(n, **kw)
    o = oracle_lib.OracleScene(sc, fp64_reductions=True, permute_every=0)
    g = hip.HipScene(hip_ctx, sc)
    o.prepare()
    g.prepare()
    for _ in range(3):
        o.step()
        g.run("neighborhood.update")
        g.step(1)
    _close(g.download("fluid", "density"), o.get("fluid", "density"), 6e-5, "density")
    _close(g.download("fluid", "position"), o.get("fluid", "position"), 3e-5, "position")
    g.destroy()


def _tight(kind):
    """The kind with solves that stop at 1e-4, as in test_viscous_step_sizes_vs_oracle."""
    return dict(KINDS[kind], wkbb18_maximum_error=1e-4, pt16_vorticity_maximum_error=1e-4,
                pt16_velocity_maximum_error=1e-4)


def _one_step_vs_oracle(hip_ctx, oracle_lib, sc, bars, real_type=0):
    from prtcl_amd import hip
    o = oracle_lib.OracleScene(sc, fp64_reductions=True, permute_every=0)
    g = hip.HipScene(hip_ctx, sc, real_type=real_type)
    o.prepare()
    g.prepare()
    o.step()
    g.step(1)
    for f, bar in bars.items():
        _close(g.download("fluid", f), o.get("fluid", f), bar, f)
    g.destroy()


BARS = {"density": 2e-5, "position": 1e-5, "velocity": 1e-3}


@pytest.mark.parametrize("kind", [k for k in KINDS if k != "plain"])
def test_one_lane_kinds_vs_oracle(hip_ctx, oracle_lib, kind):
    """Every kind of step just above the line, where its passes give a particle one lane."""
    print(f"case: {SPLIT + 1} particles, {kind}", flush=True)
    _one_step_vs_oracle(hip_ctx, oracle_lib, _block(SPLIT + 1, **_tight(kind)), BARS)


@pytest.mark.parametrize("kind", KINDS)
def test_one_lane_overflow_vs_oracle(hip_ctx, oracle_lib, kind):
    """A block at 0.6 spacings (about 200 neighbours) beside an ordinary one, above the
    line: its particles run past the rows of the setup's table and walk the grid in
    every pass, beside lanes that do not. Bars of the same block alone
    (test_dense_block_list_overflow and its viscous form, in test_gpu_parity), and its
    two iterations: further ones diverge in it, the pressure grows from 1e8 to 1e10 by
    the twentieth, and a difference of 1e-6 grows with it to 1e-4, in the oracle's FP32
    as well."""
    s, side = 0.025, 41
    fx = np.concatenate([
        scenes.fluid_block((side, side, side), (1, 1, 1), s, 1e-4,
                           scenes.stream_base(3, 0))[:SPLIT + 1 - 1000],
        scenes.fluid_block((10, 10, 10), (10, 10, (side + 6) / 0.6), 0.6 * s, 1e-4,
                           scenes.stream_base(9, 0))])
    v = np.random.default_rng(5).uniform(-0.2, 0.2, fx.shape)
    sc = scenes._finish("dense", s, fx, scenes.box_boundary(side + 4, side + 4, side + 20, s), 1,
                        v=v, **_tight(kind))
    sc.permute_every = 0
    sc.iisph_max_iterations = 2
    print(f"case: {len(fx)} particles, 1000 of them dense, {kind}", flush=True)
    bars = {"density": 2e-5, "position": 1e-5}
    if "implicit_viscosity" in KINDS[kind]:
        bars = {"density": 1e-3, "position": 1e-5, "velocity": 5e-3}
    if kind == "pt16":
        # the velocity itself is what its solves stop at 1e-4 of, an iteration apart if
        # need be: ten times that of the block's speed, which moves it by 0.28 m of the
        # 1.5 m that the position is measured by, is 2e-4 there
        bars["position"] = 2e-4
    _one_step_vs_oracle(hip_ctx, oracle_lib, sc, bars)


@pytest.mark.parametrize("kind", ["plain", "wkbb18"])
@pytest.mark.parametrize("n", [2, 31, 32, 33, 64, 65, 257, SPLIT, SPLIT + 1])
def test_fp64_step_sizes_vs_oracle(hip_ctx, oracle_lib, n, kind):
    """The 64-bit forms (32-byte records, gathered by lane pairs with several lanes too)
    against the oracle, whose FP32 sums set the bars."""
    _one_step_vs_oracle(hip_ctx, oracle_lib, _block(n, **_tight(kind)), BARS, real_type=1)
