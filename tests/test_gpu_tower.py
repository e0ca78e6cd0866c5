"""The fused time step (towers of chains and the interface between them) against the unfused kernels and the oracle,
at the shapes where it can go wrong: towers of one chain and of a whole column, chain remainders (a mesh width that is
not a multiple of 12 elements), a single row of elements, the three geometry forms, one and several attenuation
coefficient sets, and every kind of interface point (Stacey edges, sources, receivers, CPML, fluid-solid edges)."""
import ctypes as C

import numpy as np
import pytest

from oracle.oracle import OracleSim
from specfem2d_amd import config
from specfem2d_amd.config import Source
from specfem2d_amd.driver import ShotBatch, Simulation, UnevenBatch

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


def make(form, nx, nz, nstep=160):
    if form.startswith("coupled"):
        src = [Source(x=nx * 47.0, z=-nz * 70.0, f0=8.0, factor=1.0e9)]
        rec = np.array([[nx * 30.0, -nz * 80.0], [nx * 80.0, -60.0], [nx * 55.0, -nz * 45.0]])
        cfg = config.layered_fluid_solid(nx, nz, max(1, nz // 4), 100.0, nstep, 2.0e-3, sources=src, receivers=rec)
        return cfg.replace(stacey=False, pml=True, nelem_pml=3) if form == "coupled_cpml" else cfg
    if form.startswith("fluid"):  # pressure: minus the potential, or (the second form) its second derivative
        cfg = config.pressure_source_acoustic_44x44(nstep).replace(
            nx=nx, nz=nz, nz_layers=[nz], xmin=0.0, xmax=nx * 100.0, interfaces=[-nz * 100.0, 0.0], dt=2.0e-3, absorbtop=False,
            sources=[Source(x=nx * 46.0, z=-nz * 42.0, f0=15.0, factor=1.0e4)],
            receivers=np.array([[nx * 16.0, -nz * 60.0], [nx * 62.0, -nz * 18.0]]))
        return cfg if form == "fluid" else cfg.replace(stacey=False, pml=True, nelem_pml=3, use_trick=False)
    cfg = config.small_test_mesh(nx=nx, nz=nz, nstep=nstep, gll=True, seed=3)
    if form in ("cpml", "visco_cpml"):
        cfg = cfg.replace(stacey=False, pml=True, nelem_pml=3)
    if form == "layers":  # rows of two heights: affine elements, not all alike; z sources stay inside
        cfg = cfg.replace(interfaces=[-nz * 100.0, -nz * 45.0, 0.0], nz_layers=[nz // 2, nz - nz // 2])
    if form in ("visco", "visco_cpml"):
        cfg = cfg.replace(attenuation=True, qkappa=60.0, qmu=40.0)
    if form == "visco_sets":  # two coefficient sets
        q = np.where(np.repeat(np.arange(nx * nz) % nx < nx // 2, 25), 40.0, 70.0)
        cfg = cfg.replace(attenuation=True, qkappa=q, qmu=0.7 * q)
    return cfg


def check_route(sim, fused):
    """The solid and the fluid of a handle, where it has them, step on towers or do not."""
    mp = C.byref(C.c_long(sim.mesh_pointer))
    if sim.nspec_acoustic < sim.nspec:
        assert sim.fused_step() == fused
    if sim.nspec_acoustic:
        assert bool(sim.gpu.sf2d_tower_fluid_ready(mp)) == fused


def run(cfg, pieces=None, fused=True):
    sim = Simulation(cfg)
    check_route(sim, fused)
    seis = np.concatenate([sim.forward(nstep=n)[0] for n in (pieces or [cfg.nstep])], axis=-1)
    out = [seis]
    if sim.nspec_acoustic < cfg.nx * sum(cfg.nz_layers):
        out += list(sim.fields())
    if sim.nspec_acoustic:
        out += list(sim.acoustic_fields())
    sim.close()
    return out


# displacement and seismograms: sums of the same 32-bit terms in another order, grown over 160 steps: below 1e-5, the
# bound of every comparison with the oracle here.  The velocity and, more so, the acceleration M^-1 K d hold short
# waves whose terms cancel: omega_max / omega, about 1e2 at these element sizes, once and twice.  The potential and its
# derivatives behave alike; a pressure that is the second derivative is 3e-6 off 64 bits in the 32-bit oracle itself: ten
# times that.
BOUNDS = [1e-5, 1e-5, 1e-4, 1e-3, 1e-5, 1e-4, 1e-3]


@pytest.mark.parametrize("form", ["stacey", "cpml", "coupled", "layers", "points", "visco", "visco_sets", "visco_cpml",
                                  "coupled_cpml", "fluid", "fluid_cpml"])
@pytest.mark.parametrize("nx,nz,chains", [(12, 12, 1), (25, 17, 3), (38, 13, 64), (13, 2, 64)])
def test_fused_step_matches_the_unfused_one(form, nx, nz, chains, monkeypatch):
    if nz < 12 and form not in ("stacey", "points", "visco", "visco_sets", "fluid"):
        pytest.skip("too flat for layers")
    if form == "points":
        monkeypatch.setenv("SF2D_NO_AFFINE", "1")
    cfg = make("stacey" if form == "points" else form, nx, nz)
    monkeypatch.setenv("SF2D_TOWER_CHAINS", str(chains))
    fused = run(cfg)
    monkeypatch.setenv("SF2D_NO_TOWERS", "1")
    plain = run(cfg, fused=False)
    bounds = [3e-5] + BOUNDS[1:] if cfg.seismotype == 4 and not cfg.use_trick else BOUNDS
    for a, b, tol in zip(fused, plain, bounds):
        assert np.linalg.norm(b) > 0 and rel(a, b) < tol
        # sums keep the order and the roundings of the launch per colour, but for points where several boundary terms meet
        # (the flattest mesh, ends of the sea floor) and, in solids, attenuation and CPML
        if nz >= 12 and form in ("stacey", "points", "layers", "fluid", "fluid_cpml"):
            assert np.array_equal(a, b)
    ref = OracleSim(cfg, "sp").forward()
    assert rel(fused[0], ref) < bounds[0]


@pytest.mark.parametrize("form", ["stacey", "cpml", "coupled", "visco", "coupled_cpml", "fluid", "fluid_cpml"])
def test_a_run_in_pieces_gives_the_bits_of_the_run_in_one(form):
    cfg = make(form, 27, 16)
    for a, b in zip(run(cfg), run(cfg, [1, 2, 57, cfg.nstep - 60])):
        assert np.array_equal(a, b)


def test_setting_the_same_model_again_keeps_the_run():
    """New materials on a prepared handle: the fused step reads them (and the two inverse masses) from then on."""
    cfg = make("stacey", 25, 17)
    sim = Simulation(cfg)
    want = sim.forward()[0]
    sim.set_model(1.1 * cfg.rho, cfg.vp, cfg.vs)
    sim.reset()
    other = sim.forward()[0]
    sim.set_model(cfg.rho, cfg.vp, cfg.vs)
    sim.reset()
    again = sim.forward()[0]
    sim.close()
    assert rel(again, want) < 1e-6 and rel(other, want) > 1e-2


@pytest.mark.parametrize("form", ["stacey", "points", "layers"])
@pytest.mark.parametrize("nx,nz,chains", [(12, 12, 1), (25, 17, 3), (13, 2, 64)])
@pytest.mark.parametrize("shots", [1, 3])
def test_fused_reverse_sweep_matches_the_unfused_one(form, nx, nz, chains, shots, monkeypatch):
    """Gradients of one run and of a shot batch, segments that do and do not divide the run: sums of the same 32-bit
    products in another order, below the bound of every comparison here.  160 steps: the waves are at the receivers then,
    and the 32-bit oracle's traces 1e-6 off the 64-bit ones (4e-5 of a precursor after 60)."""
    if form == "points":
        monkeypatch.setenv("SF2D_NO_AFFINE", "1")
    if nz < 12 and form == "layers":
        pytest.skip("too flat for layers")
    cfg = make("stacey" if form == "points" else form, nx, nz)
    src = cfg.sources[0]
    more = [[Source(x=src.x * f, z=src.z, f0=src.f0, factor=src.factor)] for f in (1.0, 1.3, 0.6)]
    out = []
    for towers in (True, False):
        monkeypatch.setenv("SF2D_TOWER_CHAINS", str(chains))
        if not towers:
            monkeypatch.setenv("SF2D_NO_TOWERS", "1")
        sim = Simulation(cfg) if shots == 1 else ShotBatch(cfg, more)
        obs = np.zeros((cfg.nrec, 2, cfg.nstep) if shots == 1 else (shots, cfg.nrec, 2, cfg.nstep))
        check_route(sim, towers)
        for chunk in (64, 160):
            chi, seis = sim.gradient_forward(obs, chunk=chunk)
            out.append([np.array([chi]), seis, *sim.gradient_backward().values()])
            assert sim.gpu.sf2d_grad_fused(C.byref(C.c_long(sim.mesh_pointer))) == towers
        if shots == 1:  # both sweeps leave the fields after the first segment
            out[-1] += list(sim.fields())
        sim.close()
    for fused, plain in zip(out[:2], out[2:]):
        for a, b, tol in zip(fused, plain, [1e-5] * 5 + BOUNDS[1:4]):
            assert np.linalg.norm(b) > 0 and rel(a, b) < tol


@pytest.mark.parametrize("form,nx,nz,chains,block", [
    *[(f, *s, 0) for f in ("stacey", "points") for s in ((12, 12, 1), (25, 17, 3), (13, 2, 64))], ("layers", 25, 17, 3, 0),
    ("stacey", 25, 17, 3, 7), ("layers", 12, 12, 1, 1), ("stacey", 12, 12, 1, 159)])
def test_fused_adjoint_run_matches_the_unfused_one(form, nx, nz, chains, block, monkeypatch):
    """A SAVE_FORWARD run (its Stacey terms) and the SIMULATION_TYPE 3 run with its kernels, the terms in one block of all
    160 steps and in blocks that do and do not divide them.  The reconstruction runs backwards in time on rounded fields:
    what a change of 1e-7 in the stored terms and the adjoint traces does to the unfused run is the measure, ten times that
    the bound."""
    if form == "points":
        monkeypatch.setenv("SF2D_NO_AFFINE", "1")
    if block:
        monkeypatch.setenv("SF2D_STACEY_STEPS", str(block))
    cfg = make("stacey" if form == "points" else form, nx, nz)
    rng = np.random.default_rng(1)
    monkeypatch.setenv("SF2D_TOWER_CHAINS", str(chains))

    def adjoint(traces, store, last, fused):
        back = Simulation(cfg, simulation_type=3)
        check_route(back, fused)
        out = back.adjoint(traces, store, last)
        back.close()
        return [out[0], *out[1].values()] if isinstance(out[1], dict) else [out[0], *out[1]]

    runs = []
    for towers in (True, False):
        if not towers:
            monkeypatch.setenv("SF2D_NO_TOWERS", "1")
        sim = Simulation(cfg, save_forward=True)
        check_route(sim, towers)
        parts = [sim.forward(nstep=n, save_stacey=True) for n in (70, cfg.nstep - 70)]
        seis = np.concatenate([p[0] for p in parts], axis=-1)
        store = np.concatenate([p[2] for p in parts])
        last = sim.fields()
        sim.close()
        runs.append((seis, store, last, adjoint(seis[..., ::-1], store, last, towers)))
    (seis, store, last, fused), (seis0, store0, last0, plain) = runs
    assert rel(seis, seis0) < 1e-5 and rel(store, store0) < 1e-4
    noise = lambda a: a * (1 + 1e-7 * rng.choice([-1.0, 1.0], np.shape(a)))
    moved = adjoint(noise(seis0[..., ::-1]), noise(store0).astype(np.float32), [noise(x).astype(np.float32) for x in last0],
                    False)
    for a, b, c in zip(fused, plain, moved):
        assert np.linalg.norm(b) > 0 and rel(a, b) < 10 * max(rel(c, b), 1e-6)


@pytest.mark.parametrize("form", ["stacey", "layers", "points", "visco", "visco_sets", "cpml"])
def test_offsets_that_count_from_the_tower(form, monkeypatch):
    """The kernels for element arrays beyond 4 GiB, on a small mesh: the bits of the others (affine kernels on both sides) in a
    run; atomics meet in gradients and adjoint runs, whose bounds are those of a run repeated."""
    monkeypatch.setenv("SF2D_NO_RECT", "1")
    monkeypatch.setenv("SF2D_TOWER_CHAINS", "3")
    if form == "points":
        monkeypatch.setenv("SF2D_NO_AFFINE", "1")
    cfg = make("stacey" if form == "points" else form, 25, 17)
    out = []
    for wide in (False, True):
        if wide:
            monkeypatch.setenv("SF2D_WIDE_OFFSETS", "1")
        exact, close = run(cfg), []
        if form in ("stacey", "layers", "points"):
            sim = Simulation(cfg)
            sim.gradient_forward(np.zeros((cfg.nrec, 2, cfg.nstep)), chunk=40)
            close += sim.gradient_backward().values()
            sim.close()
            sim = Simulation(cfg, save_forward=True)
            seis, _, store = sim.forward(save_stacey=True)
            back = Simulation(cfg, simulation_type=3)
            adj, kernels = back.adjoint(seis[..., ::-1], store, sim.fields())
            close += [adj, *kernels.values()]
            back.close()
            sim.close()
        out.append((exact, close))
    for a, b in zip(out[1][0], out[0][0]):
        assert np.linalg.norm(b) > 0 and np.array_equal(a, b)
    for a, b in zip(out[1][1], out[0][1]):
        assert np.linalg.norm(b) > 0 and rel(a, b) < 1e-5


def test_a_union_in_pieces_and_after_a_reset():
    """A union of a solid and two fluids, of which the fluids step on a stream of their own: forked from the handle's and
    joined again in each piece of a run.  A missing wait would leave whole samples out; the order of atomics is 5e-6."""
    cfgs = [make("visco_cpml", 25, 17).replace(dt=2.0e-3), make("fluid", 19, 14), make("fluid_cpml", 26, 12)]
    cfgs = [c.replace(seismotype=1, use_trick=True) for c in cfgs]
    u = UnevenBatch(cfgs)
    check_route(u, True)
    runs = []
    for pieces in ([160], [1, 2, 57, 100], [1] * 20 + [140], [160]):
        u.reset()
        seis = np.concatenate([Simulation.forward(u, nstep=n)[0] for n in pieces], axis=-1)
        runs.append([seis, *u.fields(), *u.acoustic_fields()])
    u.close()
    for other in runs[1:]:
        for a, b, tol in zip(other, runs[0], BOUNDS):
            assert np.linalg.norm(b) > 0 and rel(a, b) < min(tol, 5e-6)


def blocks(nx, nz, h=100.0):
    """A grid of deformed quadrilaterals whose elements are numbered in blocks 5 wide and 3 high."""
    o = np.array([(x, z) for bz in range(0, nz, 3) for bx in range(0, nx, 5) for z in range(bz, min(bz + 3, nz))
                  for x in range(bx, min(bx + 5, nx))])
    X, Z = np.meshgrid(np.arange(nx + 1) * h, np.arange(nz + 1) * h - nz * h)
    rng = np.random.default_rng(4)
    X[1:-1, 1:-1] += 0.15 * h * rng.uniform(-1, 1, (nz - 1, nx - 1))
    Z[1:-1, 1:-1] += 0.15 * h * rng.uniform(-1, 1, (nz - 1, nx - 1))
    n0 = o[:, 1] * (nx + 1) + o[:, 0]
    edges = np.array([(e, c) for e, (x, z) in enumerate(o) for c, on in ((1, z == 0), (2, x == nx - 1), (4, x == 0)) if on],
                     np.int32)
    none = np.zeros(0, np.int32)
    return config.ExternalMesh(knods=np.stack([n0, n0 + 1, n0 + nx + 2, n0 + nx + 1], 1).astype(np.int32),
                               coorg=np.stack([X, Z], -1).reshape(-1, 2), material=np.ones(len(o), np.int32),
                               free_elem=none, free_code=none, abs_elem=edges[:, 0], abs_code=edges[:, 1])


@pytest.mark.parametrize("nx,nz,rows", [(12, 6, 1), (17, 9, 1), (4, 5, 1), (3, 7, 0)])
@pytest.mark.parametrize("external", [False, True])
def test_elements_in_any_order_form_rows(nx, nz, rows, external):
    """Elements numbered in blocks, and rows narrower than a patch, step on chains where these have four elements on
    average, and on the general kernel otherwise."""
    if not external and nx >= 10:
        pytest.skip("consecutive rows are chains as they are")
    cfg = make("stacey", nx, nz)
    if external:
        cfg = cfg.replace(mesh=blocks(nx, nz))
    sim = Simulation(cfg)
    assert sim.chain_kernel() == bool(rows)
    check_route(sim, bool(rows))
    seis = sim.forward()[0]
    sim.close()
    assert rel(seis, OracleSim(cfg, "sp").forward()) < 1e-5
