"""The chunk rule of the pair launches: the depth the library picks for a grid
gives bit for bit the fields, CPML memories and DFT arenas of 48-plane chunks
(each update reads the same inputs whatever the cut), at plane counts around
one chunk's limits and at grids that fill the GPU less and more than once."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.test_gpu_parity import _require_gpu, _setup
from tests.test_gpu_pair import _monitors, _sources

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,cpml", [((2, 14, 70), None), ((5, 30, 66), None),
                                       ((47, 20, 61), 3), ((48, 20, 61), 3), ((49, 33, 130), 4),
                                       ((97, 60, 250), 6), ((20, 215, 250), 5)])
def test_chunk_rule_is_bitwise(grid, cpml, monkeypatch):
    _require_gpu()
    from beamz_amd import native
    steps = 8

    def run(kz):
        if kz:
            monkeypatch.setenv("BZH_PAIR_KZ", kz)
        else:
            monkeypatch.delenv("BZH_PAIR_KZ", raising=False)
        mons = _monitors(grid) if grid[0] > 4 else ()
        sim, prog, state, _, _ = _setup(grid, seed=91, steps=steps, cpml_cells=cpml,
                                        sources=_sources(grid, steps) if grid[0] > 4 else (),
                                        monitors=mons)
        state = sim.advance(state, steps)
        torch.cuda.synchronize()
        assert native.last_program_pairs() == 4
        return [t.cpu().numpy() for t in (*state.fields(), *state.psi_h, *state.psi_e,
                                          state.dft_re, state.dft_im)]

    print(f"case chunk_rule grid={grid} cpml={cpml}", flush=True)
    for got, want in zip(run(None), run("48")):
        assert np.array_equal(got, want)
