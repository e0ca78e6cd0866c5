"""Autotuner for the launch shape of a time step: elements per chain patch and shots per wave.

The patch plan of a mesh (``sf2d_mesh_set_chain_elems``, elements per chain patch, 1..12) fixes how many elements one
wave of the fused step or of the chain kernel holds and how many waves there are; the shots per wave of a batch that
steps phase by phase (``sf2d_mesh_set_shots_per_wave``) trade element-data reuse against waves in flight.  Which is
fastest depends on the mesh size, the number of shots and the device, so it is measured: every candidate runs
a short forward (``steps`` time steps from rest) on the workload's own mesh, model and shots, and the fastest
device time wins.  The fused step takes one shot per wave and does not read the second knob: a chain length is timed once
there, for all its candidates, and the choice leaves the knob at 0, its default.  The height of the towers is the
library's own rule and is not tuned.

``tune(cfg, shots)`` returns the choice and the table; ``settings(choice)`` gives it as the ``chain_elems`` and
``shots_per_wave`` arguments of the handle it is for (``Simulation`` / ``ShotBatch``): per handle, nothing
process-wide.
"""
from __future__ import annotations

from typing import Dict, Iterable, List, Optional, Sequence

from .config import SimulationConfig
from .driver import ShotBatch, Simulation

CHAIN_ELEMS = (4, 6, 8, 10, 12)
SHOTS_PER_WAVE = (1, 2, 4, 8, 16)


def _forward_ms(sim, steps: int, batch: bool) -> float:
    if batch:
        _, ms = sim.forward(timing=True)
        return ms
    sim.reset()
    _, t = sim.forward(nstep=steps)
    return t["loop_ms"]


def tune(cfg: SimulationConfig, shots: Optional[Sequence[list]] = None, steps: int = 20,
         chain_elems: Iterable[int] = CHAIN_ELEMS, shots_per_wave: Iterable[int] = SHOTS_PER_WAVE) -> Dict:
    """Time a ``steps``-step forward for every (elements per chain patch, shots per wave) candidate on this
    workload (a ShotBatch of ``shots`` when given, else a single simulation) and return
    ``{"chain_elems", "shots_per_wave", "ms_per_step", "table"}``; ``table`` lists every candidate.  A batch on the fused
    step does not read the shots per wave: one time for all, and 0 as the choice."""
    small = cfg.replace(nstep=steps)
    batch = shots is not None
    groups: List[int] = sorted({min(g, len(shots)) for g in shots_per_wave}) if batch else [0]
    table, unread = [], {}
    for n in chain_elems:
        sim = ShotBatch(small, shots, chain_elems=n) if batch else Simulation(small, chain_elems=n)
        try:
            if not sim.chain_kernel():
                continue  # the mesh's patches are not chains: nothing to tune
            read = batch and (sim.shot_minor() or not sim.fused_step())
            unread[sim.chain_elems()] = not read
            for g in groups:
                if read or g == groups[0]:
                    if read:
                        sim.set_shots_per_wave(g)
                    _forward_ms(sim, steps, batch)  # warm-up
                    ms = _forward_ms(sim, steps, batch)
                table.append({"chain_elems": sim.chain_elems(), "shots_per_wave": g, "ms_per_step": ms / steps})
        finally:
            sim.close()
    if not table:
        return {"chain_elems": None, "shots_per_wave": None, "ms_per_step": None, "table": []}
    best = min(table, key=lambda r: r["ms_per_step"])
    if unread[best["chain_elems"]]:
        best = dict(best, shots_per_wave=0)
    return dict(best, table=table)


def settings(choice: Dict) -> Dict:
    """The tuned choice as constructor arguments of ``Simulation`` / ``ShotBatch`` (per handle: the library reads
    them when it builds that handle's plan and launch shape)."""
    return {"chain_elems": int(choice.get("chain_elems") or 0), "shots_per_wave": int(choice.get("shots_per_wave") or 0)}
