"""What the batch autotuner times (CPU, against a stub in place of the library
and of the clock): launches as deep as those of ``advance``."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import beamz_amd as bz
from beamz_amd import batch as bt


class _Event:
    def __init__(self, **kw):
        pass

    def record(self, *a):
        pass

    def elapsed_time(self, other):
        return 1.0


def _launch_steps(nsteps, T):
    """The steps of a call's launches (``run_batch2d``): ceil(nsteps / T)
    launches, one more where that changes the banks' parity."""
    n = -(-nsteps // T)
    n += (nsteps - n) % 2
    return [nsteps // n + (i < nsteps % n) for i in range(n)]


@pytest.mark.parametrize("steps", [None, 1, 2, 6, 50])
def test_autotune_times_launches_of_full_depth(monkeypatch, steps):
    calls = []
    monkeypatch.setattr(bt.native, "call_batch2d", lambda sims, step, attrs: calls.append(attrs.nsteps))
    monkeypatch.setattr(bt.torch.cuda, "current_stream", lambda: None)
    monkeypatch.setattr(bt.torch.cuda, "synchronize", lambda: None)
    monkeypatch.setattr(bt.torch.cuda, "Event", _Event)
    monkeypatch.setattr(bt, "_TUNED", {})
    batch = bt.BatchedSimulation2D([bz.Simulation(np.full((20, 30), 2.0), 20e-9, device=torch.device("cpu"))])
    best = bt.autotune(batch) if steps is None else bt.autotune(batch, steps=steps)
    assert best[0] in bt.TILE_ROWS and len(best[2]) == len(bt.TILE_ROWS)
    assert calls and min(calls) >= (steps or 1)
    for n in calls:
        for T in (8, 6):
            assert set(_launch_steps(n, T)) == {T}
