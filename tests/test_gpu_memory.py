"""What a handle does where the card has little memory left (SF2D_SPARE_MEMORY says so): the ways that need less, with the
same results, and no allocation at the end of a long run."""
import ctypes as C

import numpy as np
import pytest

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
