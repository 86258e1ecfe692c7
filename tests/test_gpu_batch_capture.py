"""Batch calls inside a caller's graph: after one warm-up call, a call of any
other step count can be captured (no allocation, no synchronous copy), and each
replay gives what the same call gives eagerly."""

from __future__ import annotations

import pytest
import torch

from tests.test_gpu_batch import _member, _require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsteps", [2, 10, 14])
def test_capture_after_a_call_of_another_step_count(nsteps):
    _require_gpu()
    from beamz_amd.batch import BatchedSimulation2D
    print(f"case batch captured nsteps={nsteps}", flush=True)
    # (grids of their own per step count: tile lists are kept per set of shapes)
    members = [_member((y + nsteps, 90), s, cpml_cells=6, metallic=None, steps=64)[0] for y, s in ((50, 3), (77, 4))]
    batch = BatchedSimulation2D(members, tile_rows=32)
    got, want = batch.initial_state(), batch.initial_state()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        for st in (got, want):
            batch.run_chunk(st, 16)
            st["step"].fill_(16)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        batch.run_chunk(got, nsteps)
        got["step"].add_(nsteps)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        batch.run_chunk(want, nsteps)
        want["step"].add_(nsteps)
        torch.cuda.synchronize()
        for a, b in zip(got["members"], want["members"]):
            for x, y in ((a.ez[0], b.ez[0]), (a.hx[0], b.hx[0]), (a.hy[0], b.hy[0])):
                assert float(y.abs().max()) > 0.0 and torch.equal(x, y)
