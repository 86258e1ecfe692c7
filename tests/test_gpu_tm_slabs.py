"""Several slabs of one timing on the same cells of a multi-step launch (the
first is held in registers, the others are added from memory), against the
per-phase schedule, bit for bit."""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest
import torch

from tests.test_gpu_parity import _require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [2, 3])
@pytest.mark.parametrize("grid", [(40, 70), (300, 520)])
def test_overlapping_slabs(grid, count):
    _require_gpu()
    import beamz_amd as bz
    from beamz_amd import runtime
    ny, nx = grid
    print(f"case tm_steps {grid} with {count} slabs per target and timing", flush=True)
    rng = np.random.default_rng(8)
    srcs = []
    for comp, timing in (("Ez", "pre_e"), ("Hx", "h"), ("Hy", "h"), ("Ez", "e")):
        unit = 1.0 if comp == "Ez" else 1 / 377
        srcs += [bz.CustomSource(comp, (5 + q, 30 - q), rng.normal(size=(20, 9 + q)) * unit,
                                 rng.normal(size=17 + 5 * q), timing) for q in range(count)]
    sim = bz.Simulation(rng.uniform(1.5, 12.0, grid), 25e-9, boundaries=[bz.PML(cells=6)], sources=srcs, steps=32)
    prog = sim.compile()
    assert prog.workspace_floats > 0
    fields = {c.lower(): rng.normal(size=prog.shapes[c]) * (1.0 if c[0] == "E" else 1 / 377)
              for c in prog.shapes}
    a, b = (runtime.advance(sim.initial_state(fields), p, 23)
            for p in (prog, dataclasses.replace(prog, workspace_floats=0)))
    torch.cuda.synchronize()
    for x, y in zip((a.hx, a.hy, a.ez, *a.psi_h, *a.psi_e), (b.hx, b.hy, b.ez, *b.psi_h, *b.psi_e)):
        assert torch.isfinite(y).all() and torch.equal(x, y)
