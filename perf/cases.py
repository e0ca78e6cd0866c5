"""Performance cases: what users of this package have it do, through its public entry points.

A case is a dict of plain values.  ``kind`` says which program it stands for:

  run       one whole simulation of a small mesh from rest: reset, all NSTEP steps, seismograms and the last frame
  resume    the next ``steps`` steps of a long simulation that goes on from a snapshot, with its seismograms
  gradient  one misfit gradient of one shot: forward run with checkpoints, recomputation and reverse sweep
  shots     the same for a batch of shots of one mesh, advanced together
  adjoint   a SIMULATION_TYPE=1 run with stored edges, then the SIMULATION_TYPE=3 run and its kernels
  uneven    a batch of simulations of different sizes and physics as unions of similar NSTEP

``exact`` restates the discretisation (5 x 5 GLL elements, explicit Newmark, Stacey edges, standard linear solids) in
64-bit torch for the cases without a CPML layer and without fluid-solid coupling.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from specfem2d_amd import config
from specfem2d_amd.config import ExternalMesh, SimulationConfig, Source
from specfem2d_amd.driver import ShotBatch, Simulation, UnevenRuns

R37 = math.sqrt(3.0 / 7.0)
XI = [-1.0, -R37, 0.0, R37, 1.0]
W = [0.1, 49.0 / 90.0, 32.0 / 45.0, 49.0 / 90.0, 0.1]

LISTED = [
    # the plain elastic half-space of the tests and the oracle's calibration: 80 x 60 elements, until the waves reach
    # the sides; the smallest thing that is run in earnest, bound by launches and their latency
    dict(name="run_plain_80x60", kind="run", physics="elastic", edges="stacey", nx=80, nz=60, nstep=1000, nrec=20,
         random=False),
    # the mesh of the fluid's absolute-amplitude example: 44 x 44 elements, pressure receivers
    dict(name="run_fluid_44x44", kind="run", physics="fluid", edges="stacey", nx=44, nz=44, nstep=800, nrec=5,
         random=False),
    # a mesh read from files: deformed quadrilaterals in a mesher's blockwise order, neither chains nor rectangles
    dict(name="run_quads_90x50", kind="run", physics="quads", edges="stacey", nx=90, nz=50, nstep=600, nrec=12,
         random=True),
    # the sensitivity-kernel example (80 x 32 elements): forward run with stored edges, adjoint run, three kernels
    dict(name="adjoint_80x32", kind="adjoint", physics="elastic", edges="stacey", nx=80, nz=32, nstep=500, nrec=6,
         random=True),
    # a mesh of the multi-shot survey (600 x 300) in a long run: fields that fit the last-level cache
    dict(name="resume_elastic_600x300", kind="resume", physics="elastic", edges="stacey", nx=600, nz=300, steps=300,
         nrec=64),
    # viscoelastic attenuation at every point (3 solids), the element state dominates the traffic
    dict(name="resume_visco_600x300", kind="resume", physics="visco", edges="stacey", nx=600, nz=300, steps=150,
         nrec=64),
    # water layer over a random solid with a CPML frame 20 elements thick, a quarter of the benchmark's mesh
    dict(name="resume_coupled_cpml_1000x500", kind="resume", physics="coupled", edges="cpml", nx=1000, nz=500,
         steps=100, nrec=100),
    # the large forward run: 2000 x 1000 elements, 32 M points, far beyond every cache
    dict(name="resume_elastic_2000x1000", kind="resume", physics="elastic", edges="stacey", nx=2000, nz=1000,
         steps=40, nrec=100),
    # one shot of a waveform inversion, checkpoint every 50 steps
    dict(name="gradient_400x200", kind="gradient", physics="elastic", edges="stacey", nx=400, nz=200, nstep=300,
         chunk=50, nrec=100, shots=1),
    # eight shots of a survey in one batch, checkpoint every 14 steps (about the square root of NSTEP)
    dict(name="shots_8x300x150", kind="shots", physics="elastic", edges="stacey", nx=300, nz=150, nstep=200, chunk=14,
         nrec=75, shots=8),
    # a batch of unlike simulations (water and viscoelastic solids, CPML 10 elements thick) in a few unions
    dict(name="uneven_8", kind="uneven", physics="mixed", edges="cpml", count=8, nx=300, nz=160, nstep=400, layout=5),
]


def listed():
    return [dict(c) for c in LISTED]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["run", "run", "resume", "resume", "resume", "gradient", "shots", "adjoint", "uneven"])
    if kind == "run":
        physics = rng.choice(["elastic", "elastic", "fluid", "quads", "visco", "coupled"])
        edges = "stacey" if physics == "quads" else rng.choice(["stacey", "cpml"])
        nx, nz = _log(rng, 24, 130), _log(rng, 20, 90)
        return dict(kind=kind, physics=physics, edges=edges, nx=nx, nz=nz,  # ends while the waves are in the mesh
                    nstep=150 + rng.randint(2, 10) * min(nx, nz), nrec=rng.randint(1, 40), random=rng.random() < 0.7)
    if kind == "resume":
        physics = rng.choice(["elastic", "visco", "coupled"])
        nx = _log(rng, 130, 1300)
        nz = max(40, int(nx * rng.uniform(0.35, 0.7)))
        steps = max(10, min(300, int((5e7 if physics != "visco" else 2.5e7) / (nx * nz))))
        return dict(kind=kind, physics=physics, edges=rng.choice(["stacey", "cpml"]), nx=nx, nz=nz, steps=steps,
                    nrec=rng.randint(8, 150))
    if kind == "adjoint":
        return dict(kind=kind, physics="elastic", edges="stacey", nx=_log(rng, 20, 120), nz=_log(rng, 20, 60),
                    nstep=rng.randint(100, 500), nrec=rng.randint(1, 12), random=rng.random() < 0.7)
    if kind == "uneven":
        return dict(kind=kind, physics="mixed", edges="cpml", count=rng.randint(3, 8), nx=_log(rng, 80, 300),
                    nz=_log(rng, 60, 160), nstep=rng.randint(120, 400), layout=rng.randint(1, 10000))
    nx = _log(rng, 60, 400) if kind == "gradient" else _log(rng, 60, 260)
    nz = max(30, int(nx * rng.uniform(0.4, 0.6)))
    nstep = rng.randint(80, 300) if kind == "gradient" else rng.randint(60, 180)
    return dict(kind=kind, physics="elastic", edges="stacey", nx=nx, nz=nz, nstep=nstep,
                chunk=rng.randint(8, 60) if kind == "gradient" else rng.randint(8, 16), nrec=rng.randint(10, 100),
                shots=1 if kind == "gradient" else rng.randint(2, 8))


# ----------------------------------------------------------------------------------------------------------------
# inputs, from the seed alone

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _waves(rng, n, lmin, lmax):
    """n plane-wave products: amplitude, wave numbers and phases with wavelengths in [lmin, lmax]."""
    k = 2 * np.pi / np.exp(rng.uniform(np.log(lmin), np.log(lmax), (n, 2)))
    return rng.standard_normal(n) / math.sqrt(n), k, rng.uniform(0, 2 * np.pi, (n, 2))


def _lattice(case, h):
    """GLL coordinates of the lattice columns and rows (x from 0, z from -depth to 0)."""
    nx, nz = case["nx"], case["nz"]
    t = torch.tensor(XI[:4], dtype=torch.float64, device=_dev())

    def line(n, lo):
        x = (torch.arange(n, dtype=torch.float64, device=_dev())[:, None] + (t[None, :] + 1) / 2).reshape(-1)
        return lo + h * torch.cat([x, torch.full((1,), float(n), dtype=torch.float64, device=_dev())])
    return line(nx, 0.0), line(nz, -nz * h)


def _field(waves, x, z):
    """The wave products on the lattice, [rows, columns]."""
    a, k, p = waves
    out = torch.zeros(len(z), len(x), dtype=torch.float64, device=x.device)
    for q in range(len(a)):
        out += (a[q] * torch.sin(k[q, 1] * z + p[q, 1]))[:, None] * torch.sin(k[q, 0] * x + p[q, 0])[None, :]
    return out


def _elements(grid, nx, nz):
    """Lattice values as element points [nspec, 25], elements row by row, i fastest."""
    e = grid.unfold(0, 5, 4).unfold(1, 5, 4)  # [nz, nx, 5, 5]
    return e.reshape(nx * nz, 25)


def _quad_order(nx, nz):
    """Elements of an nx x nz grid in blocks 7 wide and 5 high: (ex, ez) of each, in order."""
    e = [(x, z) for bz in range(0, nz, 5) for bx in range(0, nx, 7) for z in range(bz, min(bz + 5, nz))
         for x in range(bx, min(bx + 7, nx))]
    return np.array(e)


def _quads(case, h, rng):
    """A deformed mesh: nodes of the grid moved by up to a fifth of an element inside, kept in place on the sides."""
    nx, nz = case["nx"], case["nz"]
    X, Z = np.meshgrid(np.arange(nx + 1) * h, np.arange(nz + 1) * h - nz * h)
    inside = np.zeros_like(X)
    inside[1:-1, 1:-1] = 0.2 * h
    co = np.stack([X + inside * rng.uniform(-1, 1, X.shape), Z + inside * rng.uniform(-1, 1, X.shape)], -1)
    o = _quad_order(nx, nz)
    n0 = o[:, 1] * (nx + 1) + o[:, 0]
    ab = [(e, c) for e, (x, z) in enumerate(o) for c, on in ((1, z == 0), (2, x == nx - 1), (4, x == 0)) if on]
    ab = np.array(ab, np.int32)
    none = np.zeros(0, np.int32)
    return ExternalMesh(knods=np.stack([n0, n0 + 1, n0 + nx + 2, n0 + nx + 1], 1).astype(np.int32),
                        coorg=co.reshape(-1, 2), material=np.ones(len(o), np.int32), free_elem=none, free_code=none,
                        abs_elem=ab[:, 0], abs_code=ab[:, 1])


def _config(case, seed):
    """The simulation of a case: mesh, model, sources and receivers."""
    rng = np.random.default_rng(seed)
    nx, nz = case["nx"], case["nz"]
    kind, physics = case["kind"], case["physics"]
    h = {"run": 50.0, "adjoint": 50.0, "resume": 10.0}.get(kind, 20.0)
    dt = {50.0: 1.0e-3, 20.0: 4.0e-4, 10.0: 2.0e-4}[h]
    nstep = case["nstep"] if "nstep" in case else 12000
    width, depth = nx * h, nz * h
    fluid_rows = nz if physics == "fluid" else max(1, nz // 10) if physics == "coupled" else 0
    inner = rng.uniform(0.08, 0.92, (case["nrec"], 2))
    rec = np.stack([inner[:, 0] * width, -inner[:, 1] * depth], 1)
    if kind in ("gradient", "shots"):  # a line of surface receivers
        rec = np.stack([np.linspace(h, width - h, case["nrec"]), np.zeros(case["nrec"])], 1)
    f0 = {50.0: 8.0, 20.0: 25.0, 10.0: 8.0}[h]
    # an inversion's source lies just below the receivers, the others' at a third to a half of the depth
    down = 3 * h if kind == "gradient" else depth
    src = [Source(x=float(rng.uniform(0.4, 0.6) * width), z=float(-rng.uniform(0.3, 0.5) * down), f0=f0,
                  factor=1.0e4 if physics == "fluid" else 1.0e10, anglesource=float(rng.uniform(0, 90)))]
    # model: fluid rows on top of a solid, both homogeneous or with smooth +-10 % variations of 15 to 100 elements
    vary = case.get("random", True)
    if vary:
        x, z = _lattice(case, h)
        pert = 0.1 * torch.tanh(_field(_waves(rng, 4, 15 * h, 100 * h), x, z))
        pert = _elements(pert, nx, nz).cpu().numpy()
        if physics == "quads":
            o = _quad_order(nx, nz)
            pert = pert[o[:, 1] * nx + o[:, 0]]
    else:
        pert = np.zeros((nx * nz, 25))
    fluid = (np.repeat(np.arange(nz), nx) >= nz - fluid_rows)[:, None]
    vals = []
    for water, rock in ((1020.0, 2500.0), (1500.0, 3000.0), (0.0, 1732.0)):
        v = (1.0 + pert) * rock
        if fluid_rows:
            v = np.where(fluid, water * (1.0 + (pert if physics == "fluid" else 0.0)), v)
        vals.append(v.reshape(-1))
    cfg = SimulationConfig(
        name=kind, nx=nx, nz=nz, xmin=0.0, xmax=width, interfaces=[-depth, 0.0], nz_layers=[nz], nstep=nstep, dt=dt,
        rho=vals[0], vp=vals[1], vs=vals[2], material_mode=1, stacey=case["edges"] == "stacey",
        pml=case["edges"] == "cpml", nelem_pml=min(20, max(3, min(nx, nz) // 12)), absorbtop=False, sources=src,
        receivers=rec)
    if physics == "fluid":
        cfg = cfg.replace(seismotype=4, use_trick=True)
    if physics == "visco":
        cfg = cfg.replace(attenuation=True, qkappa=float(rng.uniform(40, 100)), qmu=float(rng.uniform(30, 80)))
    if physics == "quads":
        cfg = cfg.replace(mesh=_quads(case, h, rng))
    return cfg, h, rng


def _snapshot(case, cfg, h, rng):
    """Smooth displacement and velocity on the lattice (two components each), and a fluid potential."""
    x, z = _lattice(case, h)
    om = 2 * np.pi * 6.0
    u = [1e-3 * _field(_waves(rng, 5, 8 * h, 60 * h), x, z) for _ in range(2)]
    v = [1e-3 * om * _field(_waves(rng, 5, 8 * h, 60 * h), x, z) for _ in range(2)]
    pot = None
    if case["physics"] == "coupled":
        floor = 4 * (case["nz"] - max(1, case["nz"] // 10))
        for f in u + v:
            f[floor + 1:] = 0.0
        pot = _field(_waves(rng, 5, 8 * h, 60 * h), x, z) * torch.sin(z / 100.0)[:, None]
        pot[:floor] = 0.0
    return u, v, pot


def _points(sim, grids):
    """Lattice grids as point arrays [nglob, len(grids)] in the numbering of the simulation."""
    ib = torch.from_numpy(sim.ibool().astype(np.int64) - 1).to(_dev())
    out = torch.zeros(sim.nglob, len(grids), device=_dev())
    for c, g in enumerate(grids):
        out[ib.reshape(-1), c] = _elements(g, sim.cfg.nx, sim.cfg.nz).reshape(-1).float()
    return out.cpu().numpy()


def _observed(case, cfg, rng):
    """Observed seismograms of each shot: one arrival per receiver, a few per cent off the background's time."""
    t = np.arange(cfg.nstep) * cfg.dt - 1.2 / 25.0
    out = []
    for s in _shots(case, cfg):
        dist = np.hypot(cfg.receivers[:, 0] - s[0].x, cfg.receivers[:, 1] - s[0].z)
        late = t[None, :] - (dist / 3000.0 * (1 + 0.05 * rng.uniform(-1, 1, dist.size)))[:, None]
        a = (np.pi * 25.0) ** 2 * late ** 2
        wave = (1 - 2 * a) * np.exp(-a) * 0.2
        out.append(np.stack([wave * g for g in rng.uniform(-1, 1, 2)], 1))
    return np.stack(out)


def _shots(case, cfg):
    return config.surface_shots(cfg, case["shots"], f0=25.0) if case["kind"] == "shots" else [cfg.sources]


def _adjoint_traces(case, cfg, rng):
    t = np.arange(cfg.nstep) * cfg.dt
    f = rng.uniform(2, 6, (case["nrec"], 2, 1))
    win = np.sin(np.pi * np.arange(cfg.nstep) / max(1, cfg.nstep - 1)) ** 2
    return (np.sin(2 * np.pi * f * t + rng.uniform(0, 6, f.shape)) * win * 1e6).astype(np.float32)


def _uneven_configs(case, seed):
    """Sizes, physics and NSTEP of the instances from the case's layout; their models and sources from the seed."""
    rng = np.random.default_rng(seed)
    out = []
    for c in config.uneven_batch_instances(
            n=case["count"], seed=case["layout"], nelem_pml=10, nrec=10, nstep_range=(case["nstep"] // 4, case["nstep"]),
            size_range=((max(30, case["nx"] // 5), case["nx"]), (max(30, case["nz"] // 4), case["nz"]))):
        x, z = _lattice(dict(nx=c.nx, nz=c.nz), 20.0)
        p = 1.0 + 0.05 * torch.tanh(_elements(_field(_waves(rng, 4, 300.0, 2000.0), x, z), c.nx, c.nz)).reshape(-1)
        p = p.cpu().numpy()
        s = c.sources[0]
        s = Source(x=s.x + float(rng.uniform(-20, 20)), z=s.z + float(rng.uniform(-20, 20)), f0=30.0, factor=s.factor)
        rec = np.array([[s.x, s.z]]) + rng.uniform(-1, 1, (10, 2)) * [[0.2 * c.nx * 20.0, 0.15 * c.nz * 20.0]]
        out.append(c.replace(rho=c.rho * p, vp=c.vp * p, vs=c.vs * p, sources=[s], receivers=rec))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "uneven":
        return dict(case=case, sim=UnevenRuns(_uneven_configs(case, seed), max_groups=3))
    cfg, h, rng = _config(case, seed)
    state = dict(case=case, cfg=cfg)
    if kind == "shots":
        state["sim"] = ShotBatch(cfg, _shots(case, cfg))
        state["obs"] = _observed(case, cfg, rng)
    elif kind == "gradient":
        state["sim"] = Simulation(cfg)
        state["obs"] = _observed(case, cfg, rng)[0]
    elif kind == "adjoint":
        state["sim"] = Simulation(cfg, save_forward=True)
        state["adj"] = _adjoint_traces(case, cfg, rng)
    else:
        state["sim"] = Simulation(cfg)
        if kind == "resume":
            u, v, pot = _snapshot(case, cfg, h, rng)
            state["frame"] = _points(state["sim"], u), _points(state["sim"], v)
            state["pot"] = None if pot is None else _points(state["sim"], [pot])
            _restart(state)
    return state


def _restart(state):
    sim = state["sim"]
    sim.set_fields(*state["frame"])
    if state["pot"] is not None:
        sim.set_acoustic_fields(state["pot"])


def run(state):
    case, sim = state["case"], state["sim"]
    kind = case["kind"]
    if kind == "run":
        sim.reset()
        seis, _ = sim.forward()
        last = sim.acoustic_fields() if case["physics"] == "fluid" else sim.fields()
        if case["physics"] == "coupled":
            last = last + sim.acoustic_fields()
        return dict(seis=seis, last=list(last))
    if kind == "resume":
        if sim.steps_done + case["steps"] > sim.cfg.nstep:  # the run is over: the next one from the snapshot
            sim.reset()
            _restart(state)
        return dict(seis=sim.forward(nstep=case["steps"])[0])
    if kind in ("gradient", "shots"):
        chi, seis = sim.gradient_forward(state["obs"], chunk=case["chunk"])
        return dict(chi=chi, seis=seis, grad=sim.gradient_backward())
    if kind == "adjoint":
        sim.reset()
        seis, _, store = sim.forward(save_stacey=True)
        back = Simulation(state["cfg"], simulation_type=3)
        adj, kernels = back.adjoint(state["adj"], store, sim.fields())
        back.close()
        return dict(seis=seis, adj=adj, kernels=kernels)
    return dict(seis=sim.forward()[0])


def work(case):
    """Per step: every point's displacement and velocity read and written and its inverse mass read, every element
    point's moduli read (viscoelastic: its 12 state values read and written), 16 bytes of geometry per element (400
    where it is deformed); the multiply-adds of the element operator.  A gradient steps forward twice and back once
    and reads what it recomputes; an adjoint run steps three fields."""
    if case["kind"] == "uneven":
        n, scale = case["count"] * case["nx"] * case["nz"] / 4, case["nstep"] * 0.6
        return dict(bytes=n * scale * (0.5 * (16 * 20 + 25 * 4) + 0.5 * (16 * 36 + 25 * 104)), flops=n * scale * 3000)
    n = case["nx"] * case["nz"]
    steps = case.get("steps", case.get("nstep"))
    solid = 16 * 36 + 25 * 8 + (400 if case["physics"] == "quads" else 16)
    fluid = 16 * 20 + 25 * 4 + 16
    b, f = solid, 3000
    if case["physics"] == "visco":
        b, f = b + 25 * 96, f + 1500
    if case["physics"] == "fluid":
        b, f = fluid, 1350
    if case["physics"] == "coupled":
        b, f = 0.9 * solid + 0.1 * fluid, 0.9 * 3000 + 0.1 * 1350
    if case["kind"] in ("gradient", "shots"):  # two forward passes, one writing d, v', r; the sweep reads them
        k = case["shots"]
        return dict(bytes=n * steps * (k * (16 * (2 * 36 + 24 + 24 + 36)) + 3 * 216), flops=n * steps * k * 12000)
    if case["kind"] == "adjoint":
        b, f = 3 * b + 25 * 24, 3 * f + 2500
    return dict(bytes=float(n) * steps * b, flops=float(n) * steps * f)


def tolerance(case):
    """32-bit sums in another order.  The last frame of a run holds the acceleration, M^-1 times a force whose terms
    cancel to about one part in a thousand: 1.4e-4 off the 64-bit run was seen there (displacement 3e-6), 1e-7 to 6e-7
    in seismograms, kernels and gradients."""
    if case["kind"] == "run":
        return {"rel": 1e-3, "max": 4e-2}
    return {"rel": 1e-5, "max": 1e-3}


# ----------------------------------------------------------------------------------------------------------------
# the same in 64 bits

def _hp():
    """h'_k(xi_i), [i, k]."""
    h = np.zeros((5, 5))
    for i in range(5):
        for k in range(5):
            h[i, k] = sum(np.prod([(XI[i] - XI[m]) / (XI[k] - XI[m]) for m in range(5) if m not in (k, q)])
                          / (XI[k] - XI[q]) for q in range(5) if q != k)
    return h


def _weights(t):
    return np.array([np.prod([(t - XI[m]) / (XI[k] - XI[m]) for m in range(5) if m != k]) for k in range(5)])


def _solids(q, f0, dt):
    """Recursive-convolution coefficients (A, B) of the three standard linear solids of quality factor q: least
    squares of 1/Q over f0 / 10 .. 10 f0."""
    fmin, fmax, n = f0 / 10, f0 * 10, 3
    p = np.array([2 * np.pi * fmin * (fmax / fmin) ** float(np.float32(k) / np.float32(n - 1)) for k in range(n)])
    m, r = np.zeros((n, n)), np.zeros(n)
    for k in range(2 * n - 1):
        w = 2 * np.pi * fmin * (fmax / fmin) ** float(np.float32(k) / np.float32(2 * n - 2))
        b = w * (p - w / q) / (p * p + w * w)
        r += b / q
        m += np.outer(b, b)
    y = np.linalg.solve(m, r)
    ts = 1 / p
    te = ts * (1 + n * y)
    phi = (1 - te / ts) / ts / np.sum(te / ts)
    a = np.exp(-0.5 * dt / ts)
    return a, phi * (1 - a) * ts


class _Sem:
    """One mesh, model, source set and receiver set; elements as [nspec, 5 (j), 5 (i)], points by lattice index."""

    def __init__(self, case, cfg, sources):
        d = _dev()
        t64 = dict(dtype=torch.float64, device=d)
        nx, nz = cfg.nx, cfg.nz
        self.n, self.dt, self.cfg, self.lx = nx * nz, cfg.dt, cfg, 4 * nx + 1
        self.npt = self.lx * (4 * nz + 1)
        if cfg.mesh is not None:
            ex, ez = (torch.from_numpy(v).to(d) for v in _quad_order(nx, nz).T.copy())
            nodes = torch.as_tensor(cfg.mesh.coorg[cfg.mesh.knods], **t64)  # [n, 4, 2]
        else:
            e = torch.arange(self.n, device=d)
            ex, ez = e % nx, e // nx
            h = (cfg.xmax - cfg.xmin) / nx
            x0, z0 = ex * h + cfg.xmin, ez * h + cfg.interfaces[0]
            nodes = torch.stack([torch.stack([x0 + a * h, z0 + b * h], -1) for a, b in ((0, 0), (1, 0), (1, 1), (0, 1))],
                                1).to(torch.float64)
        self.ex, self.ez, self.nodes = ex, ez, nodes
        j, i = torch.meshgrid(torch.arange(5, device=d), torch.arange(5, device=d), indexing="ij")
        self.ib = ((4 * ez[:, None, None] + j) * self.lx + 4 * ex[:, None, None] + i)  # [n, 5, 5]
        xi = torch.tensor(XI, **t64)
        ga, x_ = xi[:, None].expand(5, 5), xi[None, :].expand(5, 5)
        dxi = 0.25 * torch.stack([ga - 1, 1 - ga, ga + 1, -ga - 1])
        dga = 0.25 * torch.stack([x_ - 1, -x_ - 1, x_ + 1, 1 - x_])
        J = torch.stack([torch.tensordot(nodes, v, ([1], [0])) for v in (dxi, dga)], 1)  # [n, (xi, ga), (x, z), 5, 5]
        self.jac = J[:, 0, 0] * J[:, 1, 1] - J[:, 0, 1] * J[:, 1, 0]
        self.xix, self.xiz = J[:, 1, 1] / self.jac, -J[:, 1, 0] / self.jac
        self.gax, self.gaz = -J[:, 0, 1] / self.jac, J[:, 0, 0] / self.jac
        self.hp = torch.tensor(_hp(), **t64)
        self.w = torch.tensor(W, **t64)
        self.hpw = self.w[:, None] * self.hp  # w_k h'_i(xi_k), [k, i]
        self.rho, self.vp, self.vs = (torch.as_tensor(np.asarray(v, np.float64), **t64).reshape(-1, 5, 5)
                                      for v in (cfg.rho, cfg.vp, cfg.vs))
        self.mu = self.rho * self.vs ** 2
        self.kappa = self.rho * self.vp ** 2 - self.mu
        self.ww = self.w[:, None] * self.w[None, :]
        self.edges()
        it = np.arange(cfg.nstep)
        self.src, self.rec = [], []
        for s in sources:
            t = it * cfg.dt - 1.2 / s.f0
            a = (np.pi * s.f0) ** 2
            if cfg.use_trick:
                f = -(2 * a * (3 - 12 * a * t ** 2 + 4 * a * a * t ** 4)) * np.exp(-a * t * t)
            else:
                f = (1 - 2 * a * t * t) * np.exp(-a * t * t)
            e, hh = self.locate(s.x, s.z)
            ang = math.radians(s.anglesource)
            self.src.append((e, hh, (math.sin(ang), -math.cos(ang)), torch.tensor(-s.factor * f, **t64)))
        loc = [self.locate(x, z) for x, z in cfg.receivers]
        self.rib = torch.stack([self.ib[e] for e, _ in loc])
        self.rw = torch.stack([w for _, w in loc])

    def locate(self, x, z):
        c = self.nodes.mean(1)
        near = torch.argsort((c[:, 0] - x) ** 2 + (c[:, 1] - z) ** 2)[:9].tolist()
        best = None
        for e in near:
            n = self.nodes[e].cpu().numpy()
            a = b = 0.0
            for _ in range(12):
                sh = 0.25 * np.array([(a - 1) * (b - 1), -(a + 1) * (b - 1), (a + 1) * (b + 1), -(a - 1) * (b + 1)])
                da = 0.25 * np.array([b - 1, 1 - b, b + 1, -b - 1])
                db = 0.25 * np.array([a - 1, -a - 1, a + 1, 1 - a])
                m = np.stack([da @ n, db @ n], 1)
                da, db = np.linalg.solve(m, np.array([x, z]) - sh @ n)
                a, b = a + da, b + db
            if best is None or max(abs(a), abs(b)) < best[0]:
                best = (max(abs(a), abs(b)), e, a, b)
        _, e, a, b = best
        return e, torch.tensor(np.outer(_weights(b), _weights(a)), dtype=torch.float64, device=_dev())

    def edges(self):
        """Absorbing sides left, right, bottom: points, weights, and the traction's normal axis; a corner point
        belongs to the vertical side.  Then the masses with their half-step term."""
        nx = self.cfg.nx
        at = [(self.ex == 0, slice(None), 0, 0), (self.ex == nx - 1, slice(None), 4, 0),
              (self.ez == 0, 0, slice(None), 1)]
        self.sides = []
        dto2 = 0.5 * self.dt
        fluid = bool((self.vs == 0).all())
        m = torch.zeros(self.npt, 1 if fluid else 2, dtype=torch.float64, device=_dev())
        base = (self.ww * self.jac / (self.rho * self.vp ** 2) if fluid else self.ww * self.jac * self.rho).reshape(-1, 1)
        m.index_add_(0, self.ib.reshape(-1), base.expand(-1, m.shape[1]).contiguous())
        for on, jj, ii, axis in at:
            e = torch.nonzero(on)[:, 0]
            # length element: |d(x, z)/d(gamma or xi)|
            l = torch.hypot(self.xix[e], self.xiz[e]) if axis == 0 else torch.hypot(self.gax[e], self.gaz[e])
            l = (l * self.jac[e])[:, jj, ii] * self.w
            if axis == 1:
                l = l.clone()
                l[self.ex[e] == 0, 0] = 0.0
                l[self.ex[e] == nx - 1, 4] = 0.0
            p = self.ib[e][:, jj, ii].reshape(-1)
            rvp, rvs = (self.rho * self.vp)[e][:, jj, ii], (self.rho * self.vs)[e][:, jj, ii]
            if fluid:
                c = (l / rvp).reshape(-1, 1)
            else:
                c = torch.stack([rvp, rvs] if axis == 0 else [rvs, rvp], -1) * l[..., None]
                c = c.reshape(-1, 2)
            self.sides.append((p, c, e, jj, ii, l, axis))
            m.index_add_(0, p, c * dto2)
        m[m <= 0] = 1.0
        self.minv = 1.0 / m

    def grad(self, u):
        """xi and gamma derivatives of a field's element values [n, 5, 5]."""
        return u @ self.hp.T, torch.matmul(self.hp, u)

    def strain(self, d):
        ux, uz = d[:, 0][self.ib], d[:, 1][self.ib]
        (ax, bx), (az, bz) = self.grad(ux), self.grad(uz)
        return (ax * self.xix + bx * self.gax, ax * self.xiz + bx * self.gaz, az * self.xix + bz * self.gax,
                az * self.xiz + bz * self.gaz)

    def back(self, t1, t2):
        return self.w[:, None] * (t1 @ self.hpw) + self.w[None, :] * torch.matmul(self.hpw.T, t2)

    def force(self, d, visco=None):
        """-K d, with the standard linear solids' state in visco."""
        uxx, uxz, uzx, uzz = self.strain(d)
        lam, lp = self.kappa - self.mu, self.kappa + self.mu
        sxx, szz, sxz = lp * uxx + lam * uzz, lp * uzz + lam * uxx, self.mu * (uxz + uzx)
        if visco is not None:
            th, g = uxx + uzz, uxz + uzx
            if "old" not in visco:
                z = torch.zeros_like(th)
                visco["old"], visco["e"] = (z, z, z), [[z, z, z] for _ in range(3)]
            oxx, ozz, og = visco["old"]
            for k in range(3):
                (a1, b1), (a2, b2) = ((v[0][k], v[1][k]) for v in (visco["kappa"], visco["mu"]))
                e = visco["e"][k]
                e[0] = a1 * a1 * e[0] + b1 * (th + a1 * (oxx + ozz))
                e[1] = a2 * a2 * e[1] + b2 * (uxx - 0.5 * th + a2 * (oxx - 0.5 * (oxx + ozz)))
                e[2] = a2 * a2 * e[2] + b2 * (g + a2 * og)
                sxx = sxx + self.kappa * e[0] + 2 * self.mu * e[1]
                szz = szz + self.kappa * e[0] - 2 * self.mu * e[1]
                sxz = sxz + self.mu * e[2]
            visco["old"] = (uxx, uzz, g)
        J = self.jac
        out = torch.zeros_like(d)
        fx = self.back(J * (sxx * self.xix + sxz * self.xiz), J * (sxx * self.gax + sxz * self.gaz))
        fz = self.back(J * (sxz * self.xix + szz * self.xiz), J * (sxz * self.gax + szz * self.gaz))
        out.index_add_(0, self.ib.reshape(-1), -torch.stack([fx, fz], -1).reshape(-1, 2))
        return out

    def force_fluid(self, p):
        u = p[:, 0][self.ib]
        a, b = self.grad(u)
        gx, gz = a * self.xix + b * self.gax, a * self.xiz + b * self.gaz
        f = self.jac / self.rho
        r = self.back(f * (gx * self.xix + gz * self.xiz), f * (gx * self.gax + gz * self.gaz))
        out = torch.zeros_like(p)
        out.index_add_(0, self.ib.reshape(-1), -r.reshape(-1, 1))
        return out

    def absorb(self, v, out):
        for p, c, *_ in self.sides:
            out.index_add_(0, p, -c * v[p])

    def record(self, d):
        return torch.einsum("rjic,rji->rc", d[self.rib], self.rw)

    def steps(self, d, v, it0, n, visco=None, keep=None, adj=None):
        """n steps after it0 of the field (d, v); a = 0 before the first.  Returns seismograms [n, nrec, c]."""
        dt, fluid = self.dt, d.shape[1] == 1
        a = torch.zeros_like(d)
        top = slice((self.npt // self.lx - 1) * self.lx, self.npt)  # the fluid's free surface
        seis = []
        for it in range(it0, it0 + n):
            d = d + dt * v + 0.5 * dt * dt * a
            v = v + 0.5 * dt * a
            if fluid:
                d[top] = 0
                v[top] = 0
                r = self.force_fluid(d)
            else:
                r = self.force(d, visco)
            self.absorb(v, r)
            if adj is not None:
                w = self.rw[..., None] * adj[it][:, None, None, :]
                r.index_add_(0, self.rib.reshape(-1), w.reshape(-1, 2))
            else:
                for e, h, dirs, f in self.src:
                    s = (h / (self.rho * self.vp ** 2)[e])[..., None] if fluid else torch.stack([h * q for q in dirs], -1)
                    r.index_add_(0, self.ib[e].reshape(-1), s.reshape(-1, d.shape[1]) * f[it])
            if keep is not None:
                keep(d, v, r)
            a = r * self.minv
            v = v + 0.5 * dt * a
            if fluid:
                d[top], v[top], a[top] = 0, 0, 0
            seis.append(self.record(d))
        return torch.stack(seis), d, v, a

    def first_touch(self):
        """Lattice index of each point in the numbering by first touch in element order."""
        ib = self.ib.reshape(-1).cpu().numpy()
        u, at = np.unique(ib, return_index=True)
        return torch.from_numpy(u[np.argsort(at)]).to(_dev())


def _zeros(sem, c=2):
    return torch.zeros(sem.npt, c, dtype=torch.float64, device=_dev())


def _gradient(sem, obs):
    """chi = 1/2 dt sum |s - o|^2 of a run from rest and its gradient with respect to rho, vp, vs."""
    kept = []
    seis, *_ = sem.steps(_zeros(sem), _zeros(sem), 0, sem.cfg.nstep, keep=lambda *q: kept.append(q))
    dt = sem.dt
    res = seis - torch.as_tensor(obs, dtype=torch.float64, device=_dev()).permute(2, 0, 1)
    chi = 0.5 * dt * float((res ** 2).sum())
    D, V, A = _zeros(sem), _zeros(sem), _zeros(sem)
    gk, gm = torch.zeros_like(sem.kappa), torch.zeros_like(sem.mu)
    gmass = _zeros(sem)
    gvp, gvs = torch.zeros_like(sem.kappa), torch.zeros_like(sem.kappa)
    for n in range(sem.cfg.nstep - 1, -1, -1):
        d, v, r = kept.pop()
        w = sem.rw[..., None] * (dt * res[n])[:, None, None, :]
        D.index_add_(0, sem.rib.reshape(-1), w.reshape(-1, 2))
        A = A + 0.5 * dt * V
        b = A * sem.minv
        gmass -= b * r * sem.minv
        D = D + sem.force(b)
        sem.absorb(b, V)
        e, f = sem.strain(d), sem.strain(b)
        J = sem.ww * sem.jac
        gk -= J * (e[0] + e[3]) * (f[0] + f[3])
        gm -= J * (e[0] * f[0] + e[3] * f[3] - e[0] * f[3] - e[3] * f[0] + (e[1] + e[2]) * (f[1] + f[2]))
        for p, c, el, jj, ii, l, axis in sem.sides:
            q = -(v[p] * b[p]).reshape(len(el), 5, 2) * l[..., None]
            gvp[el, jj, ii] += q[..., axis]
            gvs[el, jj, ii] += q[..., 1 - axis]
        V, A = V + dt * D, 0.5 * dt * V + 0.5 * dt * dt * D
    gr = sem.ww * sem.jac * gmass.sum(1)[sem.ib]
    for p, c, el, jj, ii, l, axis in sem.sides:
        q = 0.5 * dt * gmass[p].reshape(len(el), 5, 2) * l[..., None]
        gvp[el, jj, ii] += q[..., axis]
        gvs[el, jj, ii] += q[..., 1 - axis]
    rho, vp, vs = sem.rho, sem.vp, sem.vs
    return chi, seis, dict(rho=gk * (vp ** 2 - vs ** 2) + gm * vs ** 2 + gr + gvp * vp + gvs * vs,
                           vp=2 * rho * vp * gk + rho * gvp, vs=2 * rho * vs * (gm - gk) + rho * gvs)


def exact(case, seed):
    kind, physics = case["kind"], case["physics"]
    if case["edges"] == "cpml" or physics == "coupled":
        return None
    cfg, h, rng = _config(case, seed)
    if kind in ("gradient", "shots"):
        obs = _observed(case, cfg, rng)
        chi, seis, grad = 0.0, [], {}
        for k, src in enumerate(_shots(case, cfg)):
            c, s, g = _gradient(_Sem(case, cfg, src), obs[k])
            chi += c
            seis.append(s.permute(1, 2, 0))
            grad = {q: grad.get(q, 0) + g[q].reshape(-1, 25) for q in g}
        seis = torch.stack(seis)
        return dict(chi=chi, seis=seis if kind == "shots" else seis[0], grad=grad)
    sem = _Sem(case, cfg, cfg.sources)
    visco = None
    if cfg.attenuation:
        visco = {q: _solids(v, cfg.sources[0].f0, cfg.dt) for q, v in (("kappa", cfg.qkappa), ("mu", cfg.qmu))}
    if kind == "resume":
        u, v, _ = _snapshot(case, cfg, h, rng)
        u, v = (torch.stack([g.float().double().reshape(-1) for g in f], -1) for f in (u, v))
        seis, *_ = sem.steps(u, v, 0, case["steps"], visco)
        return dict(seis=seis.permute(1, 2, 0))
    if kind == "adjoint":
        adj = torch.as_tensor(_adjoint_traces(case, cfg, rng), dtype=torch.float64, device=_dev()).permute(2, 0, 1)
        frames, other = [], []
        seis, *_ = sem.steps(_zeros(sem), _zeros(sem), 0, cfg.nstep, keep=lambda d, v, r: frames.append(d))
        # the adjoint field runs on the reversed traces; step it meets the forward field of step NSTEP - it + 1
        aseis, *_ = sem.steps(_zeros(sem), _zeros(sem), 0, cfg.nstep, adj=adj.flip(0),
                              keep=lambda d, v, r: other.append((d, r * sem.minv)))
        kr, km, kk = (torch.zeros_like(sem.mu) for _ in range(3))
        for (d, a), b in zip(other, reversed(frames)):
            e, f = sem.strain(d), sem.strain(b)
            both = (e[0] + e[3]) * (f[0] + f[3])
            kr += (a * b).sum(1)[sem.ib]
            km += e[0] * f[0] + e[3] * f[3] + 0.5 * (e[1] + e[2]) * (f[1] + f[2]) - both / 3.0
            kk += both
        return dict(seis=seis.permute(1, 2, 0), adj=aseis.permute(1, 2, 0),
                    kernels=dict(rho=(-sem.rho * cfg.dt * kr).reshape(-1, 25), mu=(-2 * sem.mu * cfg.dt * km).reshape(-1, 25),
                                 kappa=(-sem.kappa * cfg.dt * kk).reshape(-1, 25)))
    c = 1 if physics == "fluid" else 2
    seis, d, v, a = sem.steps(_zeros(sem, c), _zeros(sem, c), 0, cfg.nstep, visco)
    order = sem.first_touch()
    seis = seis.permute(1, 2, 0)
    if physics == "fluid":
        seis = torch.cat([-seis, torch.zeros_like(seis)], 1)
        return dict(seis=seis, last=[f[order, 0] for f in (d, v, a)])
    return dict(seis=seis, last=[f[order] for f in (d, v, a)])
