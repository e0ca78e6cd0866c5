"""What a handle does where the card has little memory left (SF2D_SPARE_MEMORY says so): the ways that need less, with the
same results, and no allocation at the end of a long run."""
import ctypes as C

import numpy as np
import pytest

import test_gpu_tower as towers
from specfem2d_amd import config
from specfem2d_amd.config import Source
from specfem2d_amd.driver import ShotBatch, Simulation

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


def free_bytes():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def make(nx, nz, shots, nstep=160):
    cfg = config.small_test_mesh(nx=nx, nz=nz, nstep=nstep, gll=True, seed=3)
    src = cfg.sources[0]
    if shots == 1:
        return Simulation(cfg), np.zeros((cfg.nrec, 2, nstep))
    more = [[Source(x=src.x * f, z=src.z, f0=src.f0, factor=src.factor)] for f in (1.0, 1.3, 0.6)[:shots]]
    return ShotBatch(cfg, more), np.zeros((shots, cfg.nrec, 2, nstep))


def fused_sweep(sim):
    return sim.gpu.sf2d_grad_fused(C.byref(C.c_long(sim.mesh_pointer)))


def gradient(nx, nz, shots, chunk, spare, monkeypatch, nstep=160):
    """The gradient with its parts, how the sweep ran and what the reverse sweep took of the card's memory."""
    with monkeypatch.context() as m:
        sim, obs = make(nx, nz, shots, nstep)
        sim.gradient_forward(obs, chunk=chunk)
        if spare is not None:
            m.setenv("SF2D_SPARE_MEMORY", str(spare(sim)))
        before = free_bytes()
        grad, parts = sim.gradient_backward(parts=True)
        taken = before - free_bytes()
        fused = fused_sweep(sim)
        sim.close()
    return [*grad.values(), *parts.values()], fused, taken


@pytest.mark.parametrize("shots", [1, 3])
def test_gradient_on_a_full_card(shots, monkeypatch):
    """Nothing to spare: the reverse sweep without towers, and the result formed in the segment's slots from a model on the
    host.  A little: towers, with one field of R~ in place of a ring.  The sums are those of 32-bit products in another
    order, below the bound of every comparison here."""
    want, fused, _ = gradient(25, 17, shots, 40, None, monkeypatch)
    assert fused == 1
    for spare, towers in ((lambda sim: 0, 0), (lambda sim: 8 * 8 * sim.nglob * shots, 1)):
        got, fused, _ = gradient(25, 17, shots, 40, spare, monkeypatch)
        assert fused == towers
        for a, b in zip(got, want):
            assert np.linalg.norm(b) > 0 and rel(a, b) < 1e-5


@pytest.mark.parametrize("shots", [1, 3])
def test_reverse_sweep_takes_nothing_of_a_full_card(shots, monkeypatch):
    """Model and result of 200 x 100 elements would be 46 MB."""
    _, fused, taken = gradient(200, 100, shots, 10, lambda sim: 0, monkeypatch, nstep=30)
    assert fused == 0 and taken <= 0


@pytest.mark.parametrize("nx,nz", [(25, 17), (3, 2)])
@pytest.mark.parametrize("spare", [None, 0])
def test_gradient_formed_in_pieces(nx, nz, spare, monkeypatch):
    """Segments of one step hold the result of a part of the elements only, and on a mesh of a few none of it."""
    want, _, _ = gradient(nx, nz, 1, 64, None, monkeypatch)
    got, _, _ = gradient(nx, nz, 1, 1, None if spare is None else lambda sim: spare, monkeypatch)
    for a, b in zip(got, want):
        assert np.linalg.norm(b) > 0 and rel(a, b) < 1e-5


def fluid_ready(sim):
    return sim.gpu.sf2d_tower_fluid_ready(C.byref(C.c_long(sim.mesh_pointer)))


@pytest.mark.parametrize("form", ["stacey", "coupled_cpml", "fluid_cpml"])
def test_no_towers_on_a_full_card(form, monkeypatch):
    """A handle made with nothing to spare steps phase by phase, as with SF2D_NO_TOWERS: the same bits where no atomics meet."""
    cfg = towers.make(form, 25, 17)
    out = []
    for env in (("SF2D_SPARE_MEMORY", "0"), ("SF2D_NO_TOWERS", "1")):
        with monkeypatch.context() as m:
            m.setenv(*env)
            sim = Simulation(cfg)
            seis = sim.forward()[0]
            assert not fluid_ready(sim) and (form == "fluid_cpml" or not sim.fused_step())
            sim.close()
        out.append(seis)
    assert np.linalg.norm(out[1]) > 0 and rel(*out) < (1e-5 if form == "coupled_cpml" else 1e-12)


def test_states_before_towers(monkeypatch):
    """A gradient whose states need what the towers hold gives these up."""
    sim, obs = make(25, 17, 1)
    assert sim.fused_step()
    chi, seis = sim.gradient_forward(obs, chunk=40)
    want = sim.gradient_backward()
    sim.close()
    sim, obs = make(25, 17, 1)
    monkeypatch.setenv("SF2D_SPARE_MEMORY", "0")
    chi0, seis0 = sim.gradient_forward(obs, chunk=40)
    assert not sim.fused_step()
    got = sim.gradient_backward()
    sim.close()
    assert abs(chi0 - chi) < 1e-5 * chi and rel(seis0, seis) < 1e-5
    for k in want:
        assert rel(got[k], want[k]) < 1e-5


def test_adjoint_run_on_a_full_card(monkeypatch):
    """No room for the second field arrays: the run takes the entry points one by one, as with SF2D_NO_TOWERS."""
    cfg = towers.make("stacey", 25, 17)
    sim = Simulation(cfg, save_forward=True)
    seis, _, store = sim.forward(save_stacey=True)
    last = sim.fields()
    sim.close()

    def adjoint(env=None):
        with monkeypatch.context() as m:
            back = Simulation(cfg, simulation_type=3)
            assert back.fused_step()
            if env:
                m.setenv(*env)
            before = free_bytes()
            adj, kernels = back.adjoint(seis[..., ::-1], store, last)
            taken = before - free_bytes()
            back.close()
        return [adj, *(kernels.values() if isinstance(kernels, dict) else kernels)], taken

    fused, _ = adjoint()
    plain, taken = adjoint(("SF2D_SPARE_MEMORY", "0"))
    assert taken <= 0
    with monkeypatch.context() as m:
        m.setenv("SF2D_NO_TOWERS", "1")
        back = Simulation(cfg, simulation_type=3)
        adj, kernels = back.adjoint(seis[..., ::-1], store, last)
        back.close()
    ref = [adj, *(kernels.values() if isinstance(kernels, dict) else kernels)]
    for a, b, c in zip(plain, ref, fused):
        assert np.linalg.norm(b) > 0 and rel(a, b) <= max(1e-6, 10 * rel(c, b))
