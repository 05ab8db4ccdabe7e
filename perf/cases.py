"""Performance cases of the SPH step path: what a program that uses this library has it do.

A program keeps its scenes on the device, sets the particles it wants advanced
(a rollout from a stored state, a state that host code has changed), advances
them by k time steps per call (the request of the served workload is k = 10),
and reads the particles back for a frame or for its own use. Setting the state
in every pass also makes all passes the same work. Every case goes through the
C ABI as prtcl_amd/hip.py binds it. The kinds:

  step        position and velocity in, k whole steps of one scene
              (prtcl_hip_step), position, velocity, density and pressure out
  batch       the same for several independent scenes in one call, position
              and velocity out
  serve       one request per scene through the request loop (submit, tick
              until nothing is pending, poll), position and velocity out
  procedures  the step of the reference's Lua loop procedure by procedure, the
              convergence test on the host, as host code that drops this
              library in for the reference's schemes runs it
  trace       one image of a scene by the sphere tracer, as the scripts render
              one per frame

Host buffers are page-locked and kept, as a program that moves particles back
and forth would. Host order stays the upload order
(permute_every = 0), so results can be compared particle by particle.
"""

from __future__ import annotations

import ctypes
import math
import random

import numpy as np
import torch

from prtcl_amd import hip, scenes

VISCOSITY = {"none": 0, "explicit": 0, "wkbb18": 1, "wkbb18_gc": 2, "pt16": 3}
STEP_FIELDS = ("position", "velocity", "density", "pressure")
PROC_FIELDS = ("position", "velocity", "acceleration", "density", "pressure")


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def _step(name, n, tank, spacing=0.01, viscosity="none", real="f32", speed=0.0, at="corner",
          k=10):
    return {"name": name, "kind": "step", "nx": n[0], "ny": n[1], "nz": n[2], "tx": tank[0],
            "ty": tank[1], "tz": tank[2], "spacing": spacing, "viscosity": viscosity,
            "real": real, "speed": speed, "at": at, "k": k}


def _many(name, kind, count, lo, hi, viscous, mix, k=10):
    return {"name": name, "kind": kind, "count": count, "lo": lo, "hi": hi, "viscous": viscous,
            "mix": mix, "k": k}


def listed():
    return [
        # the smallest scene of the batched workload on its own: nothing but
        # launches and latency
        _step("small_2k", (14, 11, 13), (28, 22, 26), speed=0.5),
        # the reference's dam break at the size its script runs on a CPU
        # (20^3 particles, explicit viscosity)
        _step("dambreak_8k", (20, 20, 20), (80, 40, 40), spacing=0.025, viscosity="explicit"),
        # a middling scene of the served workload, odd in every axis
        _step("dambreak_59k", (47, 41, 31), (94, 82, 62), speed=0.5),
        # the headline scene: 100^3 particles in a 4 x 2 x 2 m box
        _step("dambreak_1m", (100, 100, 100), (400, 200, 200)),
        # a double-precision run, as a check of a production run would be made
        _step("fp64_27k", (30, 29, 31), (60, 58, 62), real="f64"),
        # the highly viscous column collapsing on a floor (implicit WKBB18)
        _step("viscous_250k", (50, 50, 100), (100, 100, 150), viscosity="wkbb18",
              at="middle"),
        # the gradient-corrected scheme of the reference's second script
        _step("viscous_gc_48k", (37, 43, 30), (74, 86, 60), viscosity="wkbb18_gc",
              speed=0.5),
        # vorticity-preserving viscosity (pt16) on half the viscous column
        _step("pt16_125k", (50, 50, 50), (100, 100, 100), viscosity="pt16", at="middle",
              k=2),
        # independent scenes of the batched workload in one call
        _many("batch_16", "batch", 16, 2000, 200000, 0.0, 3),
        # a moment of the served stream: requests for scenes of mixed sizes,
        # some of them viscous
        _many("serve_12", "serve", 12, 5000, 200000, 0.3, 4),
        # the drop-in use: one call per procedure, host-side loop
        {"name": "procedures_64k", "kind": "procedures", "nx": 40, "ny": 40, "nz": 40, "tx": 80,
         "ty": 80, "tz": 80, "spacing": 0.01, "viscosity": "explicit", "real": "f32",
         "speed": 0.0, "at": "corner", "k": 2},
        # one frame of a scene at a preview's resolution
        {"name": "trace_125k", "kind": "trace", "nx": 50, "ny": 50, "nz": 50, "tx": 100,
         "ty": 100, "tz": 100, "spacing": 0.01, "viscosity": "none", "real": "f32",
         "speed": 0.0, "at": "corner", "width": 400, "height": 300, "steps": 300},
    ]


def _block(rng, lo, hi):
    """lattice of about N particles, N log-uniform, aspects 0.5..2, and a tank
    of 1.5 to 4 times its extent"""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    r = [rng.uniform(0.5, 2.0) for _ in range(3)]
    s = (n / (r[0] * r[1] * r[2])) ** (1.0 / 3.0)
    dims = [max(3, int(round(a * s))) for a in r]
    while dims[0] * dims[1] * dims[2] > hi:
        dims[dims.index(max(dims))] -= 1
    return dims, [max(int(d * rng.uniform(1.5, 3.0)), d + 2) for d in dims]


def _motion(rng):
    """a block at rest or in motion, in the corner of its tank or free of its walls"""
    return {"speed": rng.choice([0.0, 0.5]), "at": rng.choice(["corner", "corner", "middle"])}


def draw(rng):
    kind = rng.choice(["step", "step", "step", "step", "viscous", "viscous", "batch", "serve",
                       "procedures", "trace"])
    if kind == "step":
        real = rng.choice(["f32", "f32", "f32", "f64"])
        v = rng.choice(["none", "none", "explicit"])
        n, t = _block(rng, 2000, 200000 if real == "f64" else 900000 if v == "none" else 400000)
        c = _step("", n, t, viscosity=v, real=real, k=rng.choice([1, 5, 10]), **_motion(rng))
    elif kind == "viscous":
        v = rng.choice(["wkbb18", "wkbb18", "wkbb18_gc", "pt16"])
        n, t = _block(rng, 5000, 250000 if v == "wkbb18" else 120000)
        c = _step("", n, t, viscosity=v, k=rng.choice([1, 2] if v == "pt16" else [1, 5, 10]),
                  **_motion(rng))
    elif kind == "batch":
        c = _many("", "batch", rng.randint(3, 16), 2000, rng.choice([20000, 100000]), 0.0,
                  rng.randrange(1000))
    elif kind == "serve":
        c = _many("", "serve", rng.randint(3, 10), 5000, rng.choice([50000, 100000]),
                  rng.choice([0.0, 0.3]), rng.randrange(1000), k=rng.choice([2, 10]))
    elif kind == "procedures":
        n, t = _block(rng, 2000, 64000)
        c = dict(_step("", n, t, viscosity=rng.choice(["none", "explicit"]),
                       k=rng.choice([1, 2]), **_motion(rng)), kind="procedures")
    else:
        n, t = _block(rng, 2000, 125000)
        c = dict(_step("", n, t), kind="trace", width=rng.randint(64, 400),
                 height=rng.randint(48, 300), steps=rng.choice([100, 300]))
        del c["k"]
    del c["name"]
    return c


def _members(case):
    """(n, tank, viscous mu) of every scene of a batch: sizes are the case's,
    particle data the seed's"""
    out = []
    for i in range(case["count"]):
        rng = random.Random("%d/%d" % (case["mix"], i))
        n, _ = _block(rng, case["lo"], case["hi"])
        mu = rng.uniform(1.0, 100.0) if rng.random() < case["viscous"] else 0.0
        out.append((n, [2 * d for d in n], mu))
    return out


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _scene(n, tank, spacing, viscosity, speed, at, seed, mu=None):
    """A fluid block one spacing above the floor of a closed single-layer box,
    in its corner or in the middle. The lattice is 1 % wider than the spacing
    and jittered by 3 % of it: a block that has just settled off the walls,
    whose pressure solves take the 2 to 6 iterations that they take in a
    running dam break (a block exactly at the spacing bursts off the walls,
    with solves at the iteration cap). With a speed the block slides and falls
    at about that speed and carries a divergence-free wave."""
    seed &= 0x7FFFFFFF
    wide = 1.01
    off = [((t - d) // 2 if at == "middle" and k < 2 else 1) / wide
           for k, (t, d) in enumerate(zip(tank, n))]
    x = scenes.fluid_block(tuple(n), off, spacing * wide, 0.03 * spacing,
                           scenes.stream_base(seed, 0))
    nf = x.shape[0]
    v = np.zeros((nf, 3), np.float32)
    if speed:
        u = 0.9 + 0.2 * scenes.uniform(scenes.stream_base(seed, 1), 0, 3)
        phase = x * (2.0 * math.pi / spacing / np.asarray(n))
        v = speed * (u * (0.6, -0.4, -0.8) + 0.5 * np.sin(phase[:, [1, 2, 0]]))
        v = np.ascontiguousarray(v, np.float32)
    h = float(np.float32(spacing))
    if mu is None:
        mu = {"explicit": 0.01, "wkbb18": 50.0, "wkbb18_gc": 50.0}.get(viscosity, 0.0)
    return scenes.Scene(
        name="case", spacing=spacing, fluid_x=x, fluid_v=v,
        fluid_m=np.full(nf, np.float32(h * h * h * 1000.0), np.float32),
        time_of_birth=np.full(nf, -1.0, np.float32),
        boundary_x=scenes.box_boundary(tank[0] + 1, tank[1] + 1, tank[2] + 1, spacing),
        smoothing_scale=h, explicit_viscosity=viscosity == "explicit",
        implicit_viscosity=VISCOSITY[viscosity], fluid_viscosity=mu, boundary_viscosity=mu,
        permute_every=0)


def _scenes(case, seed):
    if case["kind"] in ("batch", "serve"):
        return [_scene(n, t, 0.01, "wkbb18" if mu else "none", 0.5, "corner", seed * 64 + i, mu)
                for i, (n, t, mu) in enumerate(_members(case))]
    return [_scene((case["nx"], case["ny"], case["nz"]), (case["tx"], case["ty"], case["tz"]),
                   case["spacing"], case["viscosity"], case["speed"], case["at"], seed)]


def _camera(case):
    """The block seen from above one of its corners."""
    s = case["spacing"]
    ext = [s * case[a] for a in ("nx", "ny", "nz")]
    far = 1.7 * max(ext)
    eye = [ext[0] * 0.5 - far, ext[1] * 0.5 - 0.8 * far, ext[2] * 0.5 + 0.7 * far]
    look = [ext[k] * 0.5 - eye[k] for k in range(3)]
    return hip.camera(eye, look, [0.0, 0.0, 1.0], 1.0, case["width"], case["height"])


class _State:
    pass


def prepare(case, seed):
    st = _State()
    st.case = case
    st.ctx = hip.Context(0)
    real = 1 if case.get("real") == "f64" else 0
    st.hs = []
    for sc in _scenes(case, seed):
        h = hip.HipScene(st.ctx, sc, real_type=real)
        h.prepare()
        st.hs.append(h)
    st.ctx.synchronize()
    dt = torch.float64 if real else torch.float32
    fields = {"procedures": PROC_FIELDS, "step": STEP_FIELDS, "trace": ()}.get(
        case["kind"], ("position", "velocity"))
    st.out, st.start = [], []
    for h in st.hs:
        st.start.append({f: torch.from_numpy(a).to(dt).pin_memory() for f, a in (
            ("position", h.scene.fluid_x), ("velocity", h.scene.fluid_v))})
        st.out.append({f: torch.empty((h.nf, 3) if hip.FIELD_COMPONENTS[hip.FIELDS[f]] == 3
                                      else (h.nf,), dtype=dt, pin_memory=True) for f in fields})
    if case["kind"] == "trace":
        st.cam = _camera(case)
        st.out = {f: torch.empty((case["height"], case["width"]), dtype=torch.float64,
                                 pin_memory=True) for f in ("image", "parameter")}
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _set(h, start):
    for f, t in start.items():
        h.ctx.check(h.L.prtcl_hip_upload_field(h.ctx.h, h.id, hip.FLUID, hip.FIELDS[f],
                                               t.data_ptr(), t.numel()), f)


def _fetch(h, out):
    for f, t in out.items():
        h.ctx.check(h.L.prtcl_hip_download_field(h.ctx.h, h.id, hip.FLUID, hip.FIELDS[f],
                                                 t.data_ptr(), t.numel()), f)


def _procedure_step(h, explicit):
    """share/scripts/prtcl-lua.example.lua:363-462, one procedure per call."""
    h.run("neighborhood.update")
    h.run("density.compute_density")
    h.run("gravity.initialize_acceleration")
    if explicit:
        h.run("viscosity.accumulate_acceleration")
    h.run("symplectic_euler.integrate_velocity_with_hard_fade")
    h.run("iisph.setup")
    nprde = h.get_global("iisph_nprde")
    for it in range(1, h.scene.iisph_max_iterations + 1):
        h.run("iisph.iteration_pressure_acceleration")
        h.set_global("iisph_aprde", 0.0)
        h.run("iisph.iteration_pressure")
        rel = h.get_global("iisph_aprde") / nprde
        if it >= h.scene.iisph_min_iterations and rel < h.scene.iisph_tolerance:
            break
    h.run("symplectic_euler.integrate_velocity_with_hard_fade")
    h.run("symplectic_euler.integrate_position")


def run(st):
    case = st.case
    kind = case["kind"]
    if kind == "trace":
        h, cam = st.hs[0], st.cam
        st.ctx.check(h.L.prtcl_hip_scene_trace(
            st.ctx.h, h.id, hip.FLUID, ctypes.byref(cam), 0.5, case["steps"],
            st.out["image"].data_ptr(), st.out["parameter"].data_ptr()), "trace")
        return st.out
    for h, start in zip(st.hs, st.start):
        _set(h, start)
    if kind == "procedures":
        for _ in range(case["k"]):
            _procedure_step(st.hs[0], case["viscosity"] == "explicit")
    elif kind == "serve":
        for h in st.hs:
            st.ctx.submit(h, case["k"])
        while st.ctx.pending()[0]:
            st.ctx.tick()
        st.ctx.poll()
    else:
        st.ctx.step(st.hs, case["k"])
    for h, out in zip(st.hs, st.out):
        _fetch(h, out)
    return st.out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _step_work(n, viscosity, real_bytes):
    """Bytes and operations of one whole step of n particles. Bytes: x, m, v
    and the birth time in, x, v, density and pressure out, and what every
    global dependency inside the step makes a pass write and read once (p and
    a of each of two IISPH iterations, one vector per iteration of the
    implicit solves). Operations: about 30 neighbours, 60 per pair for
    the set-up sums, 45 per pair for the second IISPH iteration, about 30 per
    pair and CG iteration."""
    words = 8 + 8 + 2 * 8
    flops = n * 30.0 * (60 + 45)
    if viscosity == "explicit":
        words += 8
        flops += n * 30.0 * 30
    if viscosity in ("wkbb18", "wkbb18_gc"):
        words += 5 * 12
        flops += n * 30.0 * (40 + 5 * 30)
    if viscosity == "pt16":
        words += 8 * 12
        flops += n * 30.0 * (80 + 8 * 6)
    return words * real_bytes * float(n), flops


def work(case):
    kind = case["kind"]
    rb = 8 if case.get("real") == "f64" else 4
    if kind in ("batch", "serve"):
        b = f = 0.0
        for n, _, mu in _members(case):
            nf = n[0] * n[1] * n[2]
            sb, sf = _step_work(nf, "wkbb18" if mu else "none", rb)
            b += case["k"] * sb + 48.0 * nf
            f += case["k"] * sf
        return {"bytes": b, "flops": f}
    nf = case["nx"] * case["ny"] * case["nz"]
    if kind == "trace":
        # the positions, one image and one parameter; a ray near the surface
        # sums a few hundred particles in each of about ten steps, and a third
        # of the rays come near it
        px = case["width"] * case["height"]
        return {"bytes": 12.0 * nf + 16.0 * px, "flops": px / 3.0 * 10 * 300 * 30}
    sb, sf = _step_work(nf, case["viscosity"], rb)
    moved = 6 + (11 if kind == "procedures" else 8)  # state in, fields out
    return {"bytes": case["k"] * sb + rb * moved * float(nf), "flops": case["k"] * sf}


def tolerance(case):
    """About four times what the outputs are measured to be off the same pass
    in 64 bits. The pressure is the loosest of them (its solve stops at 0.1 %
    density error); pt16's solves stop at 10 %, where a product that rounds
    otherwise can end an iteration earlier."""
    kind, v = case["kind"], case.get("viscosity")
    if kind == "trace":
        return {"rel": 1e-9, "max": 1e-6}
    if case.get("real") == "f64":
        return {"rel": 1e-12, "max": 1e-11}
    if kind in ("batch", "serve"):
        return {"rel": 1e-4, "max": 3e-3}
    if kind == "procedures":
        return {"rel": 1e-4, "max": 1e-3}
    if v == "pt16":
        return {"rel": 0.03, "max": 0.5}
    if v in ("wkbb18", "wkbb18_gc"):
        return {"rel": 5e-3, "max": 0.2}
    return {"rel": 1.5e-3, "max": 0.05}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

ALPHA = 1.0 / (4.0 * math.pi)


def _near(x, y, r, same):
    """Neighbours of every x among y within r, padded: (index [n, k], mask)."""
    n, dev = x.shape[0], x.device
    lo = torch.minimum(x.min(0).values, y.min(0).values) - 2 * r
    hi = torch.maximum(x.max(0).values, y.max(0).values) + 2 * r
    dim = [int(v) + 1 for v in ((hi - lo) / r).ceil().tolist()]
    lin = torch.tensor([1, dim[0], dim[0] * dim[1]], device=dev, dtype=torch.long)
    cx = (((x - lo) / r).floor().long() * lin).sum(1)
    cy = (((y - lo) / r).floor().long() * lin).sum(1)
    cs, order = torch.sort(cy)
    ys = y[order]
    start = torch.searchsorted(cs, torch.arange(dim[0] * dim[1] * dim[2] + 1, device=dev))
    me = torch.arange(n, device=dev)
    got_i, got_j = [], []
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            row = cx + dy * dim[0] + dz * dim[0] * dim[1]
            b, e = start[row - 1], start[row + 2]
            for u in range(int((e - b).max())):
                live = torch.nonzero(b + u < e).flatten()
                j = b[live] + u
                d = x[live] - ys[j]
                ok = (d * d).sum(1) < r * r
                if same:
                    ok &= order[j] != me[live]
                got_i.append(live[ok])
                got_j.append(order[j[ok]])
    if not got_i:
        return torch.zeros((n, 1), dtype=torch.long, device=dev), torch.zeros(
            (n, 1), dtype=torch.bool, device=dev)
    i, p = torch.sort(torch.cat(got_i), stable=True)
    j = torch.cat(got_j)[p]
    cnt = torch.bincount(i, minlength=n)
    k = max(1, int(cnt.max()))
    pos = torch.arange(i.numel(), device=dev) - (torch.cumsum(cnt, 0) - cnt)[i]
    idx = torch.zeros((n, k), dtype=torch.long, device=dev)
    mask = torch.zeros((n, k), dtype=torch.bool, device=dev)
    idx[i, pos] = j
    mask[i, pos] = True
    return idx, mask


def _kernel(r2, h, mask):
    """W and the factor f of gradW = f x_ij (cubic spline of support 2 h)."""
    r = r2.sqrt()
    q = r / h
    a, b = (2 - q).clamp(min=0), (1 - q).clamp(min=0)
    w = ALPHA / h ** 3 * (a ** 3 - 4 * b ** 3)
    f = ALPHA / h ** 4 * (12 * b * b - 3 * a * a) / torch.where(r > 0, r, torch.ones_like(r))
    f = torch.where(r < math.sqrt(np.finfo(np.float32).eps), torch.zeros_like(f), f)
    zero = torch.zeros_like(w)
    return torch.where(mask, w, zero), torch.where(mask, f, zero)


def _cg(product, precond, b, x, tol, max_k):
    """Preconditioned CG with the reference's conventions: r = A x - b,
    absolute breaks, stop at |r|^2 < tol^2 |b|^2, at most max_k + 1 steps."""
    r = product(x) - b
    thr = max(tol * tol * float((b * b).sum()), float(np.finfo(np.float32).tiny))
    y = precond(r)
    p, ry, rr, k = -y, float((r * y).sum()), float((r * r).sum()), 0
    while k < 1 or (k <= max_k and not rr < thr):
        prev, q = ry, product(p)
        pq = float((p * q).sum())
        if abs(pq) < tol:
            break
        x, r = x + prev / pq * p, r + prev / pq * q
        y = precond(r)
        ry, rr = float((r * y).sum()), float((r * r).sum())
        if abs(prev) < tol:
            break
        p = -y + ry / prev * p
        k += 1
    return x


class _Exact:
    """One scene in 64 bits, advanced by whole steps."""

    def __init__(self, sc):
        dev = torch.device("cuda")

        def to(a):
            return torch.from_numpy(np.asarray(a, np.float64)).to(dev)

        def f(v):
            return float(np.float32(v))

        self.sc, self.h, self.r = sc, f(sc.smoothing_scale), sc.radius
        self.x, self.v, self.m = to(sc.fluid_x), to(sc.fluid_v), to(sc.fluid_m)
        self.bx = to(sc.boundary_x)
        self.dt, self.rho0, self.omega = f(sc.time_step), f(sc.rest_density), f(
            sc.iisph_relaxation)
        self.mu, self.mub = f(sc.fluid_viscosity), f(sc.boundary_viscosity)
        self.g = to([f(v) for v in sc.gravity])
        j, ok = _near(self.bx, self.bx, self.r, False)
        d = self.bx[:, None] - self.bx[j]
        self.V = 1.0 / _kernel((d * d).sum(2), self.h, ok)[0].sum(1)
        self.a = torch.zeros_like(self.x)

    def step(self):
        h, dt, rho0, m, mu, mub = self.h, self.dt, self.rho0, self.m, self.mu, self.mub
        j, ok = _near(self.x, self.x, self.r, True)
        d = self.x[:, None] - self.x[j]
        r2 = (d * d).sum(2)
        W, f = _kernel(r2, h, ok)
        mj = m[j]
        b, okb = _near(self.x, self.bx, self.r, False)
        db = self.x[:, None] - self.bx[b]
        r2b = (db * db).sum(2)
        Wb, fb = _kernel(r2b, h, okb)
        Vb = self.V[b]
        W0 = 4 * ALPHA / h ** 3
        rho = m * W0 + (mj * W).sum(1) + rho0 * (Vb * Wb).sum(1)
        hh = 0.01 * h * h

        def dot(p, q):
            return (p * q).sum(-1)

        acc = self.g.expand_as(self.v)
        if self.sc.explicit_viscosity:
            s = (10 * mu / rho[:, None] * mj / rho[j] * dot(self.v[:, None] - self.v[j], d) /
                 (r2 + hh) * f)
            sb = (10 * mub / rho[:, None] * rho0 * Vb / rho[:, None] *
                  dot(self.v[:, None], db) / (r2b + hh) * fb)
            acc = acc + (s[..., None] * d).sum(1) + (sb[..., None] * db).sum(1)
        v = self.v + dt * acc

        # iisph.setup
        Gf = ((mj * f)[..., None] * d).sum(1)
        Gb = ((Vb * fb)[..., None] * db).sum(1)
        c = -(Gf + 1.4 * rho0 * Gb) / (rho * rho)[:, None]
        s2 = (mj * f * f * r2).sum(1)
        div = (mj * f * dot(v[:, None] - v[j], d)).sum(1) + rho0 * dot(v, Gb)
        src = (rho0 - rho) - dt * rho0 / rho * div
        G = Gf + rho0 * Gb
        AA = dt * dt * rho0 / rho * (dot(c, G) - m / (rho * rho) * s2)
        live = AA.abs() > 1e-9
        rcp = torch.where(live, 1.0 / torch.where(live, AA, torch.ones_like(AA)),
                          torch.zeros_like(AA))
        p = torch.zeros_like(rho)
        for it in range(1, self.sc.iisph_max_iterations + 1):
            pr = p / (rho * rho)
            a = p[:, None] * c - ((mj * pr[j] * f)[..., None] * d).sum(1)
            Ap = dt * dt * rho0 / rho * (dot(a, G) - (mj * f * dot(a[j], d)).sum(1))
            p = (p + self.omega * (src - Ap) * rcp).clamp(min=0) * live
            aprde = float(((Ap - src) / rho0 * (p > 1e-9)).sum())
            if it >= self.sc.iisph_min_iterations and aprde / len(p) < self.sc.iisph_tolerance:
                break
        v = v + dt * a

        iv = self.sc.implicit_viscosity
        if iv in (1, 2):
            eye = torch.eye(3, device=v.device, dtype=v.dtype)
            kf = 10 * mu / rho[:, None] * mj / rho[j] / (r2 + hh)
            kb = 10 * mub / rho[:, None] * rho0 * Vb / rho[:, None] / (r2b + hh)
            g, gb = f[..., None] * d, fb[..., None] * db
            if iv == 2:
                M = -torch.einsum("nka,nkb->nab", (mj / rho[:, None] * f)[..., None] * d, d)
                L = _pinv(M)
                g, gb = g @ L.transpose(1, 2), gb @ L.transpose(1, 2)
            D = (torch.matmul((kf[..., None] * g).transpose(1, 2).contiguous(), d) +
                 torch.matmul((kb[..., None] * gb).transpose(1, 2).contiguous(), db))
            P = torch.linalg.inv(eye - dt * D)

            def product(w):
                o = ((kf * dot(w[:, None] - w[j], d))[..., None] * g).sum(1)
                o = o + ((kb * dot(w[:, None], db))[..., None] * gb).sum(1)
                return w - dt * o

            def precond(w):
                return (P * w[:, None, :]).sum(2)

            sol = _cg(product, precond, v, v, float(np.float32(self.sc.wkbb18_maximum_error)),
                      self.sc.wkbb18_maximum_iterations)
            a = (sol - v) / dt
            v = v + dt * a
        elif iv == 3:
            v = self._pt16(v, rho, j, d, W, f, mj, (Vb * Wb).sum(1), W0)
        self.x = self.x + dt * v
        self.v, self.a, self.rho, self.p = v, a, rho, p

    def _pt16(self, v, rho, j, d, W, f, mj, vb, W0):
        sc, m, rho0 = self.sc, self.m, self.rho0
        xi = float(np.float32(sc.pt16_strain_rate_viscosity))
        c = mj * W
        same = m * W0 + c.sum(1)
        prho = same + rho0 * vb
        dv = v[j] - v[:, None]
        vg = ((mj * f)[..., None, None] * dv[..., :, None] * d[..., None, :]).sum(1)
        vg = vg / rho[:, None, None]
        div = vg.diagonal(dim1=1, dim2=2).sum(1)
        R = (vg - vg.transpose(1, 2)) / 2
        Vm = (div / 3)[:, None, None] * torch.eye(3, device=v.device, dtype=v.dtype)
        S = (vg + vg.transpose(1, 2)) / 2 - Vm
        om = 2 * torch.stack([R[:, 2, 1], R[:, 0, 2], R[:, 1, 0]], 1)
        on = ((rho - rho0 >= 0) | (-div >= 0)).to(v.dtype)
        tvg = Vm * on[:, None, None] + xi * S
        diag0 = same - m * W0

        def solve(diag, rhs, guess, tol, max_k):
            cols = []
            for k in range(3):
                cols.append(_cg(lambda w: (diag - m * W0) * w - (c * w[j]).sum(1),
                                lambda w: w / diag0, rhs[:, k], guess[:, k],
                                float(np.float32(tol)), max_k))
            return torch.stack(cols, 1)

        rhs = xi * (c[..., None] * (om[:, None] - om[j])).sum(1)
        om = solve(same, rhs, om, sc.pt16_vorticity_maximum_error,
                   sc.pt16_vorticity_maximum_iterations)
        hw = 0.5 * om
        z = torch.zeros_like(hw[:, 0])
        tvg = tvg + torch.stack([z, -hw[:, 2], hw[:, 1], hw[:, 2], z, -hw[:, 0], -hw[:, 1],
                                 hw[:, 0], z], 1).reshape(-1, 3, 3)
        rhs = torch.zeros_like(v)
        for k in range(3):
            row = tvg[:, k]
            rhs[:, k] = (0.5 * c * ((row[:, None] + row[j]) * d).sum(2)).sum(1)
        return solve(prho, rhs, v, sc.pt16_velocity_maximum_error,
                     sc.pt16_velocity_maximum_iterations)

    def outputs(self, fields):
        named = {"position": self.x, "velocity": self.v, "acceleration": self.a,
                 "density": self.rho, "pressure": self.p}
        return {f: named[f].cpu() for f in fields}


def _pinv(M):
    """Pseudo-inverse of 3x3 matrices, singular values up to 3 eps of the
    largest counted as zero (eps of FP32); full-rank ones by their inverse."""
    eps = float(np.finfo(np.float32).eps)
    det = torch.linalg.det(M)
    fro = (M * M).sum((1, 2)).sqrt()
    full = det.abs() > 6 * eps * fro ** 3
    eye = torch.eye(3, device=M.device, dtype=M.dtype)
    out = torch.linalg.inv(torch.where(full[:, None, None], M, eye))
    rest = torch.nonzero(~full).flatten()
    if rest.numel():
        out[rest] = torch.from_numpy(np.linalg.pinv(M[rest].cpu().numpy(), rcond=3 * eps)).to(
            M.device)
    return out


def _exact_trace(sc, case):
    """The marched image: per step the least rounded-box distance over all
    occupied cells (edge 4 h), tightened by the particles' implicit function
    near the surface."""
    dev = torch.device("cuda")
    x = torch.from_numpy(sc.fluid_x.astype(np.float64)).to(dev)
    gd = 4 * float(np.float32(sc.smoothing_scale))
    half = gd / 2
    cell = (x / gd).floor().long()
    lo = cell.min(0).values - 2
    dim = (cell.max(0).values + 3 - lo).tolist()
    mul = torch.tensor([1, dim[0], dim[0] * dim[1]], device=dev)
    key, order = torch.sort(((cell - lo) * mul).sum(1), stable=True)
    xs = x[order]
    start = torch.searchsorted(key, torch.arange(dim[0] * dim[1] * dim[2] + 1, device=dev))
    occ = torch.unique(key)
    centre = torch.stack([occ % dim[0], occ // dim[0] % dim[1], occ // (dim[0] * dim[1])],
                         1).add(lo).double() * gd + half
    cam = _camera(case)

    def unit(a):
        return a / a.norm(dim=-1, keepdim=True)

    O = torch.tensor(list(cam.origin), device=dev, dtype=torch.float64)
    vv = unit(torch.tensor(list(cam.up), device=dev, dtype=torch.float64))
    pp = unit(torch.tensor(list(cam.principal), device=dev, dtype=torch.float64))
    hh = unit(torch.linalg.cross(vv, pp))
    wd, ht = case["width"], case["height"]
    ix = (torch.arange(wd, device=dev).double() - (wd - 1) / 2) / wd
    iy = (torch.arange(ht, device=dev).double() - (ht - 1) / 2) / wd
    ray = unit(O - (O + ix[None, :, None] * hh + iy[:, None, None] * vv -
                    cam.focal_length * pp)).reshape(-1, 3)
    top, phi0 = gd * 10000, 0.5 * 4 * ALPHA / half ** 3
    lip = -ALPHA * (12 * (1 / 3) ** 2 - 3 * (4 / 3) ** 2) / half ** 4
    n = ray.shape[0]
    t = torch.zeros(n, device=dev, dtype=torch.float64)
    normal = torch.zeros((n, 3), device=dev, dtype=torch.float64)
    live = torch.arange(n, device=dev)
    for _ in range(case["steps"]):
        if not live.numel():
            break
        rx = O + t[live, None] * ray[live]
        sdf = torch.empty(live.numel(), device=dev, dtype=torch.float64)
        for s in range(0, live.numel(), 1 << 14):
            q = (rx[s:s + (1 << 14), None] - centre).abs_().sub_(gd)
            mc = q.max(2).values.clamp_(max=0)
            sdf[s:s + (1 << 14)] = (q.clamp_(min=0).square_().sum(2).sqrt_().add_(mc) -
                                    gd).min(1).values
        near = torch.nonzero(sdf < gd).flatten()
        if near.numel():
            y = rx[near]
            base = (y / gd).floor().long() - lo
            phi = torch.full((near.numel(),), phi0, device=dev, dtype=torch.float64)
            grad = torch.zeros((near.numel(), 3), device=dev, dtype=torch.float64)
            count = torch.zeros(near.numel(), device=dev, dtype=torch.float64)
            for c in range(27):
                off = torch.tensor([c // 9 - 1, c // 3 % 3 - 1, c % 3 - 1], device=dev)
                at = base + off
                inside = ((at >= 0) & (at < torch.tensor(dim, device=dev))).all(1)
                lin = torch.where(inside, (at * mul).sum(1), torch.zeros_like(at[:, 0]))
                b, e = start[lin], torch.where(inside, start[lin + 1], start[lin])
                for u in range(int((e - b).max())):
                    k = torch.nonzero(b + u < e).flatten()
                    dv = y[k] - xs[b[k] + u]
                    r2 = (dv * dv).sum(1)
                    w, f = _kernel(r2, half, r2 < 4 * half * half)
                    hit = w > 0
                    phi[k] -= w * hit
                    grad[k] -= (f * hit)[:, None] * dv
                    count[k] += hit.double()
            some = count > 0
            s = lip * count.clamp(min=1)
            nrm = grad / s[:, None]
            normal[live[near]] = torch.where(some[:, None], nrm, normal[live[near]])
            sdf[near] = torch.maximum(sdf[near], torch.where(some, phi / s,
                                                             torch.full_like(phi, gd / 4)))
        stop = sdf < 1e-6
        t[live] = torch.where(stop, t[live], t[live] + sdf)
        live = live[~stop & (t[live] < top)]
    t[live] = top
    shade = -(ray * normal).sum(1) / normal.norm(dim=1).clamp(min=1e-300)
    img = torch.where(t == top, torch.zeros_like(t),
                      torch.where(t > top, torch.full_like(t, 0.3), shade))
    return {"image": img.reshape(ht, wd).cpu(), "parameter": t.reshape(ht, wd).cpu()}


def exact(case, seed):
    kind = case["kind"]
    scs = _scenes(case, seed)
    if kind == "trace":
        return _exact_trace(scs[0], case)
    fields = {"procedures": PROC_FIELDS, "step": STEP_FIELDS}.get(kind, ("position", "velocity"))
    outs = []
    for sc in scs:
        e = _Exact(sc)
        for _ in range(case["k"]):
            e.step()
        outs.append(e.outputs(fields))
        del e
    return outs
