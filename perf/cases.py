"""Performance cases of the forward time step and of the calls around it.

Every case is a piece of work that a program on ses3d_amd.api has the library
do: time steps of one simulation, of a batch, of many sources on one model,
one whole run from model arrays to seismograms, and the snapshot and adjoint
calls of a step. `prepare` builds what such a program holds before the call
(mesh, Earth model, sources, receivers and the wavefield of a run that is
under way), `run` is one pass through the public calls, `exact` the same
outputs from the equations in FP64, written with torch alone.

Fields and seismograms of an FP32 simulation are returned in FP32, as the raw
snapshot and SAC files hold them; FP64 simulations return FP64.

Case fields
  kind     loop      one step() call per time step and the velocity range, as
                     the Fortran host's time loop calls them
           steps     step(n), then the velocity snapshot
           run       simulation built, stepped to nt, seismograms read, closed
           batch     several independent simulations of uneven size in a Batch
           sources   several sources on one shared model in a Batch
           snapshot  adjoint / snapshot step: curl capture, one step, the
                     sensitivity sum and every field written to disk
  p, nx, ny, nz      GLL order and elements
  mode               precision mode (MODES)
  visco, words       visco-elastic model; memory words per mechanism
  aniso              anisotropic model (A, B, C)
  buffers            state blocks (0: the default)
  steps              steps of one pass
  receivers          receivers of three channels each
  members            simulations of a batch, sources of a shared model
  tune               s3d_autotune at set-up, as the benchmark and the Fortran
                     host (tile = -1) do
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ses3d-nt_amd"))

RADIUS = 6371000.0
LAT = 20.0                  # half width of the section in degrees at NREF elements
NREF = 96
TAPER, SLOPE = 2, 1.2
TAU_P = (1000.0, 70.0, 5.25)

# precision modes: keyword arguments of api.Simulation
MODES = {
    "fp64": dict(precision="fp64", kahan_v=False, kahan_sigma=0),
    "fp32": dict(precision="fp32", kahan_v=False, kahan_sigma=0),
    "fp32_v": dict(precision="fp32", kahan_v=True, kahan_sigma=0),
    "fp32_v_s": dict(precision="fp32", kahan_v=True, kahan_sigma=1),
    "fp32_v_s16": dict(precision="fp32", kahan_v=True, kahan_sigma=2),
    "fp32_static16": dict(precision="fp32", kahan_v=True, kahan_sigma=0, bf16_static=True),
}


def _case(name, kind, p, nx, ny, nz, mode, visco, steps, words=6, aniso=False, buffers=0, receivers=16,
          members=1, tune=False):
    c = dict(kind=kind, p=p, nx=nx, ny=ny, nz=nz, mode=mode, visco=visco, words=words, aniso=aniso,
             buffers=buffers, steps=steps, receivers=receivers, members=members, tune=tune)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # the smallest mesh (the smoke test's), one call per step as the
        # Fortran host's loop makes them: launches and call latency
        _case("loop_6x6x4_f64", "loop", 4, 6, 6, 4, "fp64", False, 20, receivers=4),
        # the homogeneous elastic 12x12x8 workload in FP64, the default
        # precision: a mesh that does not fill the GPU
        _case("steps_12x12x8_f64", "steps", 4, 12, 12, 8, "fp64", False, 256),
        # a small regional event from model arrays to seismograms
        _case("run_16x14x10_v", "run", 4, 16, 14, 10, "fp32_v", True, 320, receivers=8),
        # a middle-sized visco-elastic section in the benchmark's mode
        _case("steps_64x60x28_timed", "steps", 4, 64, 60, 28, "fp32_v_s16", True, 256, words=5, receivers=64),
        # the largest: the layered section in the benchmark's mode, autotuned
        # as the benchmark does, state far larger than any cache
        _case("steps_96x96x48_timed", "steps", 4, 96, 96, 48, "fp32_v_s16", True, 240, words=5, receivers=256,
              tune=True),
        # visco-elastic FP64, the reference's double-precision build
        _case("steps_48x48x24_f64", "steps", 4, 48, 48, 24, "fp64", True, 160, receivers=32),
        # order 6 in the mode of the uneven batch
        _case("steps_40x36x20_p6", "steps", 6, 40, 36, 20, "fp32_v", True, 192, receivers=32),
        # order 5, anisotropic elastic, FP32 stress compensation, odd sizes
        _case("steps_37x29x19_p5_aniso", "steps", 5, 37, 29, 19, "fp32_v_s", False, 320, aniso=True),
        # order 3, plain FP32 elastic, one state block, odd sizes
        _case("steps_61x53x31_p3", "steps", 3, 61, 53, 31, "fp32", False, 384, buffers=1),
        # independent regional simulations of orders 4 and 6 and uneven size
        _case("batch_12_uneven", "batch", 4, 24, 24, 12, "fp32_v", True, 128, receivers=32, members=12),
        # several sources on one model
        _case("sources_6_shared", "sources", 4, 40, 40, 20, "fp32_v_s16", True, 96, words=5, buffers=1,
              receivers=32, members=6),
        # snapshot and adjoint output of a step
        _case("snapshot_40x40x20", "snapshot", 4, 40, 40, 20, "fp32_v_s16", True, 1, receivers=16),
    ]


def draw(rng):
    kind = rng.choice(["loop", "steps", "steps", "steps", "steps", "run", "batch", "sources", "snapshot"])
    p = rng.choice([2, 3, 4, 4, 5, 6, 7])
    mode = rng.choice(sorted(MODES))
    if kind in ("batch", "sources") and mode == "fp32_static16":
        mode = "fp32_v"                      # batches do not take BF16 statics
    visco = rng.random() < 0.6
    top = {"loop": 2e5, "steps": 2e7, "run": 6e5, "batch": 1.5e6, "sources": 1.5e6, "snapshot": 4e6}[kind]
    low = {"loop": 5e3, "steps": 5e4, "run": 3e4, "batch": 1e5, "sources": 1e5, "snapshot": 1e5}[kind]
    nodes = math.exp(rng.uniform(math.log(low), math.log(top)))
    if mode == "fp64":
        nodes = max(low, nodes / 2)
    n = max(4.0, (nodes / (p + 1) ** 3 * 2.0) ** (1.0 / 3.0))
    nx = max(4, round(n * rng.uniform(0.8, 1.25)))
    ny = max(4, round(n * rng.uniform(0.8, 1.25)))
    nz = max(3, round(n / 2 * rng.uniform(0.8, 1.25)))
    real = nx * ny * nz * (p + 1) ** 3
    steps = {"loop": rng.randint(10, 40), "steps": rng.randint(100, 400), "run": rng.randint(100, 400),
             "batch": rng.randint(40, 160), "sources": rng.randint(40, 160), "snapshot": 1}[kind]
    if kind in ("steps", "batch", "sources"):
        steps = max(8, min(steps, int(6e9 / real / (4 if kind != "steps" else 1))))
    return _case(None, kind, p, nx, ny, nz, mode, visco, steps, words=rng.choice([5, 6]),
                 aniso=rng.random() < 0.2, buffers=rng.choice([0, 0, 1]), receivers=rng.randint(1, 64),
                 members=rng.randint(2, 8) if kind in ("batch", "sources") else 1)


# ---------------------------------------------------------------------------
# inputs, from the case and the seed alone
# ---------------------------------------------------------------------------

def _gll(p):
    """GLL points, weights and dl[i, j] = l_i'(x_j)."""
    c = np.zeros(p + 1)
    c[p] = 1.0
    leg = np.polynomial.legendre
    d1, d2 = leg.legder(c), leg.legder(c, 2)
    x = np.sort(leg.legroots(d1).real)
    for _ in range(3):
        x = x - leg.legval(x, d1) / leg.legval(x, d2)
    x = 0.5 * (x - x[::-1])
    x = np.concatenate([[-1.0], x, [1.0]])
    w = 2.0 / (p * (p + 1) * leg.legval(x, c) ** 2)
    dl = np.zeros((p + 1, p + 1))
    for i in range(p + 1):
        for j in range(p + 1):
            if i == j:
                dl[i, j] = sum(1.0 / (x[i] - x[k]) for k in range(p + 1) if k != i)
            else:
                num = np.prod([x[j] - x[k] for k in range(p + 1) if k not in (i, j)])
                dl[i, j] = num / np.prod([x[i] - x[k] for k in range(p + 1) if k != i])
    return x, w, dl


class _Mesh:
    """Section of one simulation: sizes, geometry, time step and time axis."""

    def __init__(self, p, nx, ny, nz, nt):
        self.p, self.nx, self.ny, self.nz, self.nt = p, nx, ny, nz, nt
        self.lat, self.lon = LAT * nx / NREF, LAT * ny / NREF
        self.depth = 43750.0 * nz * 32.0 / 48.0
        self.x, self.w, self.dl = _gll(p)
        kn = 0.5 * (1.0 + self.x)
        self.t0, self.t1 = math.radians(90.0 - self.lat), math.radians(90.0 + self.lat)
        self.p0, self.p1 = math.radians(-self.lon), math.radians(self.lon)
        self.d = ((self.t1 - self.t0) / nx, (self.p1 - self.p0) / ny, self.depth / nz)
        # node positions in elements along each axis: a node shared by two
        # elements has the same position in both
        self.s = [np.arange(n)[None, :] + kn[:, None] for n in (nx, ny, nz)]
        self.theta = self.t0 + self.s[0] * self.d[0]
        self.r = RADIUS - self.s[2] * self.d[2]
        vp = _layers(RADIUS - self.r)[0] * 1.04
        dx = np.diff(self.x).min() * 0.5
        q = max(np.max(vp / self.r) / (dx * self.d[0]),
                np.max(vp / self.r) / (dx * self.d[1] * math.cos(math.radians(self.lat))),
                np.max(vp) / (dx * self.d[2]))
        self.dt = 0.3 / q

    def grid(self):
        from ses3d_amd import synth
        return synth.Grid(self.nx, self.ny, self.nz, self.p, -self.lat, self.lat, -self.lon, self.lon,
                          RADIUS - self.depth, RADIUS, TAPER, SLOPE, self.dt, self.nt)


def _layers(depth):
    """vp, vs, rho (SI) and Q of a crust over a mantle with two jumps."""
    d = depth / 1000.0
    vp = np.where(d < 35, 5.8 + 0.02 * d, np.where(d < 410, 8.0 + 0.0024 * d, 9.2 + 0.002 * d))
    vs = vp / np.where(d < 35, 1.78, 1.83)
    rho = np.where(d < 35, 2.6 + 0.008 * d, np.where(d < 410, 3.3 + 0.0006 * d, 3.6 + 0.0007 * d))
    return 1000.0 * vp, 1000.0 * vs, 1000.0 * rho, np.where(d < 35, 300.0, 600.0)


def _axis(mesh, a, v):
    """(p+1, n) values along axis a (0 theta, 1 phi, 2 r) for a 6-D product."""
    shape = [1] * 6
    shape[2 - a], shape[5 - a] = v.shape
    return torch.from_numpy(np.ascontiguousarray(v)).reshape(shape)


def _waves(mesh, rng, longest):
    """A smooth separable field of unit size: one harmonic per axis."""
    f = []
    for a, n in enumerate((mesh.nx, mesh.ny, mesh.nz)):
        k = 2.0 * math.pi / rng.uniform(3.0, max(4.0, min(longest, n)))
        f.append(_axis(mesh, a, np.cos(k * mesh.s[a] + rng.uniform(0.0, 6.28))))
    return f[0] * f[1] * f[2]


def _model(mesh, case, seed):
    """Model parameters by name, 6-D (k, j, i, ez, ey, ex) torch FP64."""
    rng = random.Random(1000003 * seed + 17)
    vp, vs, rho, q = _layers(RADIUS - mesh.r)
    full = (mesh.p + 1,) * 3 + (mesh.nz, mesh.ny, mesh.nx)
    g = _waves(mesh, rng, 24.0).mul_(0.03).add_(1.0)
    g.mul_(g)
    out = {"rhoinv": _axis(mesh, 2, 1.0 / rho).expand(full).contiguous(),
           "mu": g * _axis(mesh, 2, rho * vs * vs)}
    out["lambda"] = _axis(mesh, 2, rho * vp * vp) - 2.0 * out["mu"]
    if case["visco"]:
        out["q"] = _axis(mesh, 2, q).expand(full).contiguous()
    if case["aniso"]:
        for name, of in (("a", "lambda"), ("b", "mu"), ("c", "lambda")):
            out[name] = 0.02 * _waves(mesh, rng, 24.0) * out[of]
    return out


def _velocity(mesh, seed):
    rng = random.Random(1000003 * seed + 29)
    return [_waves(mesh, rng, 12.0).mul_(rng.uniform(0.5, 1.0) * 1e-5) for _ in range(3)]


def _points(mesh, seed, receivers):
    """The source (latitude, longitude, depth, moment tensor, onset, width)
    and the receivers (latitude, longitude) of a simulation."""
    rng = random.Random(1000003 * seed + 41)
    m = [rng.gauss(0.0, 1.0) for _ in range(6)]
    norm = math.sqrt(sum(v * v for v in m))
    src = (rng.uniform(-0.3, 0.3) * mesh.lat, rng.uniform(-0.3, 0.3) * mesh.lon,
           rng.uniform(0.1, 0.4) * mesh.depth, [1e17 * v / norm for v in m], 25.0 * mesh.dt, 40.0 * mesh.dt)
    return src, [(rng.uniform(-0.5, 0.5) * mesh.lat, rng.uniform(-0.5, 0.5) * mesh.lon)
                 for _ in range(receivers)]


def _members(case):
    """(order, nx, ny, nz) of the simulations of a batch: uneven around the
    case's size, orders 4 and 6 as the uneven-batch workload draws them."""
    rng = random.Random(case["nx"] * 7919 + case["members"])
    out = []
    for q in range(case["members"]):
        out.append((rng.choice([4, 6]) if case["p"] in (4, 6) else case["p"],
                    max(4, round(case["nx"] * rng.uniform(0.4, 1.4))),
                    max(4, round(case["ny"] * rng.uniform(0.4, 1.4))),
                    max(3, round(case["nz"] * rng.uniform(0.6, 1.4)))))
    return out


def _nt(case):
    """Length of the time axis: a run ends with it; the others are under way
    and leave room for further passes."""
    if case["kind"] == "run":
        return case["steps"]
    return max(2000, min(200000, int(4e11 / (case["nx"] * case["ny"] * case["nz"] * (case["p"] + 1) ** 3
                                             * case["members"]))))


def _meshes(case):
    nt = _nt(case)
    if case["kind"] == "batch":
        return [_Mesh(p, nx, ny, nz, nt) for p, nx, ny, nz in _members(case)]
    return [_Mesh(case["p"], case["nx"], case["ny"], case["nz"], nt)] * case["members"]


# ---------------------------------------------------------------------------
# the user's program
# ---------------------------------------------------------------------------

def _create(case, mesh, model):
    from ses3d_amd import api
    sim = api.Simulation(mesh.grid(), state_buffers=case["buffers"],
                         memory_vars=case["words"] if case["visco"] else 0, **MODES[case["mode"]])
    for name, par in (("rhoinv", api.RHOINV), ("lambda", api.LAMBDA), ("mu", api.MU), ("q", api.Q),
                      ("a", api.A), ("b", api.B), ("c", api.C_)):
        if name in model:
            sim.set_model(par, model[name])
    sim.init()
    if case["tune"]:
        sim.autotune()
    return sim


def _stations(sim, mesh, points):
    from ses3d_amd import api
    (lat, lon, depth, m, onset, width), recs = points
    e, vm = sim.locate(lat, lon, depth)
    sim.add_source_mt(e, vm, np.outer(m, api.wavelet("RICKER", onset, width, mesh.dt, mesh.nt)))
    for la, lo in recs:
        e, vm = sim.locate(la, lo, 0.0)
        sim.add_receiver(e, vm, ("vx", "vy", "vz"))


def prepare(case, seed):
    from ses3d_amd import api
    meshes = _meshes(case)
    if case["kind"] == "run":
        m = _model(meshes[0], case, seed)
        return dict(case=case, mesh=meshes[0], model={k: v.numpy() for k, v in m.items()},
                    points=_points(meshes[0], seed, case["receivers"]))
    sims = []
    for q, mesh in enumerate(meshes):
        if case["kind"] == "sources" and q > 0:
            sim = api.Simulation.shared(sims[0])
        else:
            sim = _create(case, mesh, {k: v.numpy() for k, v in _model(mesh, case, seed + 101 * q).items()})
        if case["kind"] == "snapshot":
            sim.enable_displacement_gradient()
        _stations(sim, mesh, _points(mesh, seed + 101 * q, case["receivers"]))
        for f, v in zip((api.VX, api.VY, api.VZ), _velocity(mesh, seed + 101 * q)):
            sim.set(f, v.numpy())
        sims.append(sim)
    state = dict(case=case, sims=sims)
    if case["kind"] in ("batch", "sources"):
        state["batch"] = api.Batch(sims)
    if case["kind"] == "snapshot":
        state["forward"] = [v.numpy() for v in _velocity(meshes[0], seed + 7)]
    for sim in sims:
        sim.synchronize()
    return state


def _field(case, sim, f):
    v = sim.get(f)
    return v if case["mode"] == "fp64" else v.astype(np.float32)


def run(state):
    from ses3d_amd import api
    case = state["case"]
    if case["kind"] == "run":
        sim = _create(case, state["mesh"], state["model"])
        _stations(sim, state["mesh"], state["points"])
        sim.step(case["steps"])
        t = np.array([[sim.trace(r, c) for c in range(3)] for r in range(case["receivers"])])
        sim.close()
        return t if case["mode"] == "fp64" else t.astype(np.float32)
    if case["kind"] in ("batch", "sources"):
        state["batch"].step(case["steps"])
        return [[_field(case, s, f) for f in (api.VX, api.VY, api.VZ)] for s in state["sims"]]
    sim = state["sims"][0]
    if case["kind"] == "snapshot":
        sim.capture_curl_strain()
        sim.step(1)
        sim.grad_add(*state["forward"], -1)
        names = dict(vx=api.VX, vy=api.VY, vz=api.VZ, sxx=api.SXX, sxy=api.SXY, sxz=api.SXZ, syy=api.SYY,
                     syz=api.SYZ, szz=api.SZZ, exx=api.EXX, exy=api.EXY, exz=api.EXZ, eyy=api.EYY,
                     eyz=api.EYZ, ezz=api.EZZ, rx=api.ROT_VX, ry=api.ROT_VY, rz=api.ROT_VZ, g=api.GRAD_RHO)
        out = {n: _field(case, sim, f) for n, f in names.items()}
        out["range"] = sim.vrange() if case["mode"] == "fp64" else sim.vrange().astype(np.float32)
        e = sim.kinetic_energy()
        out["energy"] = e if case["mode"] == "fp64" else np.float32(e)
        return out
    if case["kind"] == "loop":
        for _ in range(case["steps"]):
            sim.step(1)
        r = sim.vrange_noalloc()
        return [r if case["mode"] == "fp64" else r.astype(np.float32)] + \
            [_field(case, sim, f) for f in (api.VX, api.VY, api.VZ)]
    sim.step(case["steps"])
    return [_field(case, sim, f) for f in (api.VX, api.VY, api.VZ)]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _step_work(case, p, nx, ny, nz, shared=1):
    """Bytes and operations of one step of one simulation: state, velocity
    and its compensation read and written, static fields read (once for all
    sources of a shared model), per element-local node."""
    nodes = nx * ny * nz * (p + 1) ** 3
    u = (nx * p + 1) * (ny * p + 1) * (nz * p + 1) / nodes
    m = MODES[case["mode"]]
    s = 8 if m["precision"] == "fp64" else 4
    kv = 4 if m["kahan_v"] else 0
    ks = {0: 0, 1: 4, 2: 2}[m["kahan_sigma"]]
    st = 2 if m.get("bf16_static") else s
    visco = 1 if case["visco"] else 0
    b = s * (12 + 6 * case["words"] * visco + 6 * u) + 6 * kv * u + 12 * ks
    b += st * (2 + visco + 3 * bool(case["aniso"]) + u) / shared
    f = 36 * (p + 1) + 95 + (125 if visco else 18) + (30 if m["kahan_sigma"] else 6) + 12 * u
    return nodes * b, nodes * f


def work(case):
    p, nx, ny, nz, steps = (case[k] for k in ("p", "nx", "ny", "nz", "steps"))
    sims = _members(case) if case["kind"] == "batch" else [(p, nx, ny, nz)] * case["members"]
    word = 8 if case["mode"] == "fp64" else 4
    shared = case["members"] if case["kind"] == "sources" else 1
    bytes_, flops = 0.0, 0.0
    for q in sims:
        b, f = _step_work(case, *q, shared=shared)
        nodes = q[1] * q[2] * q[3] * (q[0] + 1) ** 3
        bytes_ += steps * b
        flops += steps * f
        if case["kind"] == "run":
            # model arrays in, seismograms out
            bytes_ += 8.0 * nodes * (3 + bool(case["visco"]) + 3 * bool(case["aniso"]))
            bytes_ += 3.0 * word * case["receivers"] * steps
        elif case["kind"] == "snapshot":
            # three forward components in, 19 fields out, gradients updated
            bytes_ += nodes * (3 * 8.0 + 19.0 * word + 2 * 6 * 8.0)
            flops += nodes * (60 + 18.0 * (q[0] + 1))
        else:
            bytes_ += 3.0 * word * nodes
    return {"bytes": bytes_, "flops": flops}


# ---------------------------------------------------------------------------
# the same outputs from the equations, FP64
# ---------------------------------------------------------------------------

class _Plain:
    """One simulation in FP64: displacement-free velocity-stress elastic or
    visco-elastic (three relaxation mechanisms) spectral elements."""

    def __init__(self, case, mesh, model, velocity, points):
        dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.case, self.mesh, self.dev = case, mesh, dev
        P1 = self.P1 = mesh.p + 1
        on = lambda v: v.to(dev)  # noqa: E731
        self.lam, self.mu = on(model["lambda"]), on(model["mu"])
        self.abc = [on(model[k]) for k in "abc"] if "a" in model else None
        self.tau = None
        if "q" in model:
            # single-precision literals in the reference's formula
            self.tau = float(np.float32(6.0814)) * on(model["q"]) ** float(np.float32(-1.015))
        self.v = [on(f) for f in velocity]
        zero = torch.zeros_like(self.lam)
        self.s = [zero.clone() for _ in range(6)]          # xx xy xz yy yz zz
        self.m = [[zero.clone() for _ in range(6)] for _ in range(3)] if self.tau is not None else None
        ax = lambda a, f: on(_axis(mesh, a, f))  # noqa: E731
        sin = np.sin(mesh.theta)
        self.sin, self.cot = ax(0, sin), ax(0, np.cos(mesh.theta) / sin)
        self.r = ax(2, mesh.r)
        jac = self.jac = mesh.d[0] * mesh.d[1] * mesh.d[2] / 8.0
        wx, wy, wz = (ax(a, np.repeat(mesh.w[:, None], n, 1)) for a, n in enumerate((mesh.nx, mesh.ny, mesh.nz)))
        self.www = wx * wy * wz
        rho = 1.0 / on(model["rhoinv"])
        self.rho = rho
        mass = self.join(-(jac * self.r ** 2 * self.sin * rho * self.www))
        self.dtm = mesh.dt / mass
        D = torch.from_numpy(mesh.dl.T.copy()).to(dev)     # D[i, q] = l_q'(x_i)
        W = torch.from_numpy(mesh.dl * mesh.w[None, :]).to(dev)   # W[i, q] = l_i'(x_q) w_q
        self.D = [2.0 * D / h for h in mesh.d]
        self.W = W
        self.c = [wy * wz * self.r * (2.0 / mesh.d[0] * jac), wx * wz * self.r * (2.0 / mesh.d[1] * jac),
                  wx * wy * self.sin * (-2.0 / mesh.d[2] * jac)]
        self.damp = self.taper()
        self.source = self.locate(*points[0][:3])
        self.recs = [self.locate(a, b, 0.0) for a, b in points[1]]
        _, _, _, self.tensor, onset, width = points[0]
        t = np.arange(min(mesh.nt, 2 * case["steps"] + 2)) * mesh.dt - onset
        a2 = -(math.pi / width) ** 2
        self.stf = 2.0 * (0.5 + a2 * t * t) * np.exp(a2 * t * t)
        self.it = 0
        self.grad = None

    def along(self, A, f, a):
        """A applied to the GLL index of axis a."""
        P1, sh = self.P1, f.shape
        lead = P1 ** (2 - a)
        return torch.matmul(A, f.reshape(lead, P1, -1)).reshape(sh)

    def join(self, f):
        """Sum of the element copies of every shared node."""
        f = f.clone()
        for a in range(3):
            dim, el = 2 - a, 5 - a
            n = f.shape[el]
            if n < 2:
                continue
            hi = f.select(dim, self.P1 - 1).narrow(el - 1, 0, n - 1)
            lo = f.select(dim, 0).narrow(el - 1, 1, n - 1)
            t = hi + lo
            hi.copy_(t)
            lo.copy_(t)
        return f

    def taper(self):
        m = self.mesh
        prof = []
        for a, n in enumerate((m.nx, m.ny, m.nz)):
            s, t = m.s[a], np.zeros(m.s[a].shape)
            e = np.arange(n)[None, :] + np.zeros((self.P1, 1))
            if a < 2:
                t = np.where(e < TAPER, SLOPE * ((TAPER - s) / TAPER) ** 2, t)
            t = np.where(e >= n - TAPER, SLOPE * (((n - TAPER) - s) / TAPER) ** 2, t)
            prof.append(_axis(m, a, t).to(self.dev))
        p = prof[0] + prof[1] + prof[2]
        p2 = 2.0 * p / (1.0 + p / SLOPE)
        return -torch.expm1(-float(np.float32(0.1)) * p2 * p2)

    def locate(self, lat, lon, depth):
        m = self.mesh
        pos = [(math.radians(90.0 - lat) - m.t0) / m.d[0], (math.radians(lon) - m.p0) / m.d[1], depth / m.d[2]]
        el, l = [], []
        for q, n in zip(pos, (m.nx, m.ny, m.nz)):
            e = min(max(int(math.floor(q)), 0), n - 1)
            x = 2.0 * (q - e) - 1.0
            el.append(e)
            l.append(np.array([np.prod([(x - m.x[k]) / (m.x[i] - m.x[k]) for k in range(self.P1) if k != i])
                               for i in range(self.P1)]))
        vm = torch.from_numpy(l[2][:, None, None] * l[1][None, :, None] * l[0][None, None, :]).to(self.dev)
        return el, vm

    def strain(self):
        """Raw velocity gradient parts after the spherical terms."""
        x, y, z = self.v
        r, rs = self.r, self.r * self.sin
        d = lambda a, f: self.along(self.D[a], f, a)  # noqa: E731
        e = {}
        e["xx"] = (z + d(0, x)) / r
        e["yy"] = d(1, y) / rs + (z + x * self.cot) / r
        e["zz"] = -d(2, z)
        e["zx"], e["zy"] = -d(2, x), -d(2, y)
        e["xz"] = (d(0, z) - x) / r
        e["yz"] = -y / r + d(1, z) / rs
        e["xy"] = d(0, y) / r
        e["yx"] = -y * self.cot / r + d(1, x) / rs
        return e

    def step(self):
        mesh, dt = self.mesh, self.mesh.dt
        self.it += 1
        g = self.strain()
        e = [g["xx"], 0.5 * (g["xy"] + g["yx"]), 0.5 * (g["xz"] + g["zx"]), g["yy"],
             0.5 * (g["yz"] + g["zy"]), g["zz"]]
        self.curl = (e[4], e[2], e[1], g["zy"], g["zx"], g["yx"])
        if self.grad is not None:
            for a, b in zip(self.grad, e):
                a += dt * b
        tr = e[0] + e[3] + e[5]
        if self.tau is None:
            lam, mu = self.lam, self.mu
        else:
            lam, mu = self.lam - 2.0 / 3.0 * self.tau * self.mu, self.mu * (1.0 + self.tau)
        rate = [2.0 * mu * b for b in e]
        for c in (0, 3, 5):
            rate[c] = rate[c] + lam * tr
        if self.tau is not None:
            sm = [a + b + c for a, b, c in zip(*self.m)]
            mt = (sm[0] + sm[3] + sm[5]) / 3.0
            for c in range(6):
                rate[c] = rate[c] + 2.0 * self.mu * (sm[c] - mt if c in (0, 3, 5) else sm[c])
            for q in range(3):
                for c in range(6):
                    self.m[q][c] -= dt / TAU_P[q] * (self.m[q][c] + self.tau / 3.0 * e[c])
        if self.abc:
            A, B, C = self.abc
            rate[0] = rate[0] + C * e[5] + A * (e[0] + e[3])
            rate[3] = rate[3] + C * e[5] + A * (e[0] + e[3])
            rate[5] = rate[5] + C * (e[0] + e[3])
            rate[2] = rate[2] + 2.0 * B * e[2]
            rate[4] = rate[4] + 2.0 * B * e[4]
        for c in range(6):
            self.s[c] += dt * rate[c]
        s = list(self.s)
        if self.it > 1:
            (ex, ey, ez), vm = self.source
            rr = (self.r ** 2 * self.sin * self.www * self.jac)[:, :, :, ez, ey, ex]
            for c in range(6):
                s[c] = s[c].clone()
                s[c][:, :, :, ez, ey, ex] -= self.tensor[c] * self.stf[self.it - 2] * vm / rr
        rows = ((0, 1, 2), (1, 3, 4), (2, 4, 5))
        for c in range(3):
            f = self.c[0] * self.along(self.W, self.sin * s[rows[0][c]], 0)
            f = f + self.c[1] * self.along(self.W, s[rows[1][c]], 1)
            f = f + self.c[2] * self.along(self.W, self.r ** 2 * s[rows[2][c]], 2)
            v = self.v[c] + self.join(f) * self.dtm
            self.v[c] = v - v * self.damp
        for c in range(6):
            self.s[c] -= self.s[c] * self.damp

    def record(self):
        return [[float((vm * f[:, :, :, e[2], e[1], e[0]]).sum()) for f in self.v] for e, vm in self.recs]


def exact(case, seed):
    meshes = _meshes(case)
    if sum(m.nx * m.ny * m.nz * (m.p + 1) ** 3 for m in meshes) * case["steps"] > \
            (1.5e10 if torch.cuda.is_available() else 2e7):
        return None
    cpu = lambda f: f.cpu().numpy()  # noqa: E731
    sims, out = [], []
    for q, mesh in enumerate(meshes):
        of = seed if case["kind"] == "sources" else seed + 101 * q
        velocity = _velocity(mesh, seed + 101 * q)
        if case["kind"] == "run":
            velocity = [torch.zeros_like(f) for f in velocity]
        s = _Plain(case, mesh, _model(mesh, case, of), velocity, _points(mesh, seed + 101 * q, case["receivers"]))
        if case["kind"] == "snapshot":
            s.grad = [torch.zeros_like(s.lam) for _ in range(6)]
        trace = []
        for _ in range(case["steps"]):
            s.step()
            if case["kind"] == "run":
                trace.append(s.record())
        if case["kind"] == "run":
            return np.ascontiguousarray(np.array(trace).transpose(1, 2, 0))
        out.append([cpu(f) for f in s.v])
        sims.append(s)
    if case["kind"] in ("batch", "sources"):
        return out
    v = np.concatenate([f.reshape(-1) for f in out[0]])
    span = np.array([v.min(), v.max()])
    if case["kind"] == "loop":
        return [span] + out[0]
    if case["kind"] == "steps":
        return out[0]
    s = sims[0]
    x, y, z = s.v
    ev = s.curl
    rs = s.r * s.sin
    forward = [f.to(s.dev) for f in _velocity(meshes[0], seed + 7)]
    got = dict(zip(("vx", "vy", "vz"), out[0]))
    got.update(zip(("sxx", "sxy", "sxz", "syy", "syz", "szz"), (cpu(f) for f in s.s)))
    got.update(zip(("exx", "exy", "exz", "eyy", "eyz", "ezz"), (cpu(f) for f in s.grad)))
    got["rx"] = cpu(-y / s.r + ev[0] / rs + ev[3])
    got["ry"] = cpu(-ev[4] + (x - ev[1]) / s.r)
    got["rz"] = cpu((ev[2] + y * s.cot - ev[5] / s.sin) / s.r)
    got["g"] = cpu(-s.mesh.dt * (forward[0] * x + forward[1] * y + forward[2] * z) / s.jac)
    got["range"] = span
    got["energy"] = float(0.5 * s.jac * (s.rho * (x * x + y * y + z * z) * s.r ** 2 * s.sin * s.www).sum())
    return got
