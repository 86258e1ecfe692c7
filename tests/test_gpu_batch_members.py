"""Members of a batch against the same simulations run alone, for both tile
heights, odd step totals and every split of a call into launches: bit for bit
with CPML; without, a lone program rounds the curl once where a member rounds it
twice."""

from __future__ import annotations

import pytest
import torch

from tests.test_gpu_batch import _member, _require_gpu

pytestmark = pytest.mark.gpu

CALLS = (1, 2, 7, 17, 9)


@pytest.mark.parametrize("T", ["3", "6", "8"])
@pytest.mark.parametrize("tile_rows", [16, 32])
def test_members_match_lone_runs(tile_rows, T, monkeypatch):
    _require_gpu()
    from beamz_amd.batch import BatchedSimulation2D
    monkeypatch.setenv("BZH_TM_T", T)
    print(f"case batch members tile_rows={tile_rows} T={T}", flush=True)
    faces = ("bottom", "top", "left", "right")
    specs = [((70, 133), 3, 8, None), ((90, 40), 7, 0, faces), ((21, 30), 9, 4, None),
             ((49, 97), 11, 5, ("left",)), ((33, 64), 13, 0, faces)]
    sims = [_member(g, s, cpml_cells=L, metallic=m, steps=sum(CALLS))[0] for g, s, L, m in specs]
    batch = BatchedSimulation2D(sims, tile_rows=tile_rows)
    state = batch.initial_state()
    for n in CALLS:
        batch.advance(state, n)
    for sim, (_, _, L, _), m in zip(sims, specs, state["members"]):
        lone = sim.advance(sim.initial_state(), sum(CALLS))
        torch.cuda.synchronize()
        for got, want in ((m.ez[0], lone.ez), (m.hx[0], lone.hx), (m.hy[0], lone.hy)):
            peak = float(want.abs().max())
            assert peak > 0.0
            if L:
                assert torch.equal(got, want)
            else:
                # one more rounding of the curl's terms (2^-24 each) per step,
                # of waves whose curl times its coefficient stays below 4 peaks
                assert float((got - want).abs().max()) <= sum(CALLS) * 4 * 2.0 ** -24 * peak
