"""The 3D per-phase kernels against the FP64 oracle, at sizes around the ends of
a wave's 64 cells and of a 4-row block, where waves change between the plain,
x-edge and general bodies, with scalar and per-cell coefficients, CPML on all
and on some faces, metal faces, and grids too thin for any plain wave.

Tolerance: the FP32-against-FP64 bounds of the parity tests (``_close``).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import fdtd64 as o
from tests.test_gpu_pair import _h_sources, _sources
from tests.test_gpu_parity import _compare_state, _require_gpu, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lossy", [False, True], ids=["uniform", "lossy"])
@pytest.mark.parametrize("grid,cpml,faces,metal", [
    ((1, 1, 1), None, None, ("left", "top")),
    ((3, 5, 63), None, None, None),
    ((9, 8, 64), 2, None, None),
    ((10, 13, 65), 3, ("left", "right"), ("bottom", "back")),
    ((12, 7, 128), 3, None, ("front",)),
    ((9, 12, 129), 1, ("front", "back", "top"), None),
    ((11, 18, 200), 4, None, None),
    ((30, 3, 2), None, None, ("front", "back", "bottom", "top", "left", "right"))])
def test_phase_kernels_parity(grid, cpml, faces, metal, lossy):
    _require_gpu()
    print(f"case phase3d grid={grid} cpml={cpml} faces={faces} metal={metal} lossy={lossy}", flush=True)
    sigma = None
    if lossy:
        sigma = np.random.default_rng(7).uniform(0.0, 2e4, grid)
    steps = 12
    sim, prog, state, prob, ost = _setup(grid, seed=57, steps=steps, cpml_cells=cpml, faces=faces,
                                         metallic=metal, fused=False, sigma=sigma)
    state = sim.advance(state, steps)
    torch.cuda.synchronize()
    o.run(prob, ost, steps)
    _compare_state(prog, state, prob, ost)


@pytest.mark.parametrize("grid,kw", [((13, 17, 130), dict(cpml_cells=3)), ((9, 28, 64), {}),
                                     ((11, 14, 67), dict(metallic=("bottom", "left", "back")))])
def test_folded_sources_parity(grid, kw):
    """E- and H-timed slabs added by the phase kernels, two of them overlapping
    on one component and some on masked (metal) faces."""
    _require_gpu()
    print(f"case phase3d_sources grid={grid} {kw}", flush=True)
    steps = 9
    srcs = _sources(grid, steps) + _h_sources(grid, steps)
    first = srcs[1]
    srcs.append(o.Source("Ex", "e", (first.start[0] + 1, 0, 0), first.coeff, first.waveform))
    sim, prog, state, prob, ost = _setup(grid, seed=58, steps=steps, fused=False, sources=srcs, **kw)
    state = sim.advance(state, steps)
    torch.cuda.synchronize()
    o.run(prob, ost, steps)
    _compare_state(prog, state, prob, ost)


def test_launched_and_folded_sources_parity():
    """A grid where a source over most rows gets a launch of its own and small
    sources run inside the phase kernels, both on one phase."""
    _require_gpu()
    grid, steps = (96, 128, 136), 6
    print(f"case phase3d_sources grid={grid}", flush=True)
    srcs = _sources(grid, steps) + _h_sources(grid, steps)
    wave = srcs[0].waveform
    srcs += [o.Source("Ey", "e", (2, 3, 9), np.full((90, 120, 1), 0.05), wave),
             o.Source("Hx", "h", (1, 2, 30), np.full((92, 122, 2), 1e-4), wave),
             o.Source("Ex", "e", (50, 60, 70), np.full((2, 1, 3), 0.1), wave)]
    sim, prog, state, prob, ost = _setup(grid, seed=59, steps=steps, fused=False, sources=srcs, cpml_cells=4)
    state = sim.advance(state, steps)
    torch.cuda.synchronize()
    o.run(prob, ost, steps)
    _compare_state(prog, state, prob, ost)
