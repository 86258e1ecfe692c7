"""A program whose monitors list no frequency runs, and leaves the spectra
untouched (frequencies [M, 0] at the positional entry point)."""

from __future__ import annotations

from dataclasses import replace

import numpy as np
import pytest
import torch

from tests.test_gpu_parity import _require_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots", ["1", "32"])
@pytest.mark.parametrize("grid", [(30, 41), (14, 20, 26)])
def test_monitors_without_frequencies(grid, slots, monkeypatch):
    _require_gpu()
    import beamz_amd as bz
    from beamz_amd import runtime
    monkeypatch.setenv("BZH_DFT_SLOTS", slots)
    print(f"case dft without frequencies grid={grid} slots={slots}", flush=True)
    sim = bz.Simulation(np.full(grid, 2.0), 25e-9, steps=9, monitors=[bz.FluxMonitor("x", 9, np.array([2e14]))])
    prog = sim.compile()
    freqs, counts = prog.packed_monitors[2], prog.packed_monitors[4].clone()
    counts[:, 0] = 0
    packed = (*prog.packed_monitors[:2], freqs[:, :0].contiguous(), prog.packed_monitors[3], counts,
              *prog.packed_monitors[5:])
    rng = np.random.default_rng(2)
    fields = {c.lower(): rng.normal(size=prog.shapes[c]) * (1.0 if c[0] == "E" else 1 / 377)
              for c in prog.shapes}
    got = runtime.advance(sim.initial_state(fields), replace(prog, packed_monitors=packed), 9)
    want = runtime.advance(sim.initial_state(fields), prog, 9)
    torch.cuda.synchronize()
    for a, b in zip(got.fields(), want.fields()):
        assert torch.equal(a, b)
    assert not got.dft_re.any() and not got.dft_im.any() and not got.dft_w.any()
