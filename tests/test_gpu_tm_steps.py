"""Several TMxy steps per launch against the per-phase schedule, bit for bit:
every form the multi-step route accepts (CPML or PEC edges, lossy media,
sources of each timing that overlap faces and each other, monitors on both
normals with gates and windows) at sizes around its tiles and at step counts
around its launches.  The DFT differs only in how float64 partial sums are
grouped (1e-12)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.test_gpu_parity import _require_gpu

pytestmark = pytest.mark.gpu

DX = 25e-9


def _simulation(ny, nx, *, pml, lossy, edges=(), sources=True, monitors=True, seed=3):
    import beamz_amd as bz
    rng = np.random.default_rng(seed)
    dt = 0.9 * DX / (bz.LIGHT_SPEED * np.sqrt(2.0))
    eps = rng.uniform(1.5, 12.0, (ny, nx))
    sigma = rng.uniform(0.0, 2e4, (ny, nx)) if lossy else None
    bounds = [bz.PML(cells=pml)] if pml else []
    if edges:
        bounds.append(bz.PEC(edges=edges))
    wave = np.cos(0.7 * np.arange(30)) * 0.3
    srcs = []
    if sources:
        y, x = ny // 3, nx // 2
        srcs = [bz.CustomSource("Ez", (y, x), rng.normal(size=(min(3, ny - y), 1)), wave, "pre_e"),
                bz.CustomSource("Ez", (0, x), rng.normal(size=(ny + 1, 2)), wave[::-1].copy(), "e"),
                bz.CustomSource("Ez", (y, 0), rng.normal(size=(1, nx + 1)), wave, "e"),
                bz.CustomSource("Hy", (0, 0), rng.normal(size=(ny + 1, 1)) / 377, wave, "h"),
                bz.CustomSource("Hx", (y, 0), rng.normal(size=(1, nx + 1)) / 377, wave, "h")]
    mons = []
    if monitors:
        f = np.array([1.8e14, 2.0e14, 2.3e14])
        mons = [bz.FluxMonitor("x", max(1, nx // 2), f, ranges={"y": (0, ny)}),
                bz.FluxMonitor("y", max(1, ny // 2), f[:2], ranges={"x": (0, nx)}, interval=2,
                               window="hann", t_start=3.5 * dt, t_end=20.5 * dt)]
    sim = bz.Simulation(eps, DX, dt=dt, boundaries=bounds, sources=srcs, monitors=mons, steps=64,
                        conductivity=sigma)
    prog = sim.compile()
    fields = {c.lower(): rng.normal(size=prog.shapes[c]) * (1.0 if c[0] == "E" else 1 / 377)
              for c in prog.shapes}
    return sim, prog, fields


def _run(sim, prog, fields, steps, multi):
    import dataclasses
    from beamz_amd import runtime
    prog = prog if multi else dataclasses.replace(prog, workspace_floats=0)
    state = sim.initial_state(fields)
    for n in steps:
        state = runtime.advance(state, prog, n)
    torch.cuda.synchronize()
    return state


def _check(sim, prog, fields, steps):
    a = _run(sim, prog, fields, steps, True)
    b = _run(sim, prog, fields, steps, False)
    assert len(a.fields_b) == 1 and b.fields_b == ()
    for got, want in zip((a.hx, a.hy, a.ez, *a.psi_h, *a.psi_e), (b.hx, b.hy, b.ez, *b.psi_h, *b.psi_e)):
        assert torch.isfinite(want).all()
        assert torch.equal(got, want)
    for got, want in zip((a.dft_re, a.dft_im, a.dft_w), (b.dft_re, b.dft_im, b.dft_w)):
        got, want = got.cpu().numpy(), want.cpu().numpy()
        assert np.abs(got - want).max(initial=0.0) <= 1e-12 * max(np.abs(want).max(initial=0.0), 1e-30)


@pytest.mark.parametrize("ny,nx,pml", [(3, 2, 0), (21, 30, 4), (47, 48, 10), (48, 95, 0),
                                       (130, 49, 8), (97, 200, 12)])
@pytest.mark.parametrize("lossy", [False, True])
def test_multi_step_matches_phases(ny, nx, pml, lossy):
    _require_gpu()
    print(f"case tm_steps {ny}x{nx} pml={pml} lossy={lossy}", flush=True)
    _check(*_simulation(ny, nx, pml=pml, lossy=lossy), steps=(2, 3, 1, 9, 33))


@pytest.mark.parametrize("edges", [("left",), ("top", "right"), ("bottom", "left", "right")])
def test_multi_step_partial_metal(edges):
    _require_gpu()
    print(f"case tm_steps edges={edges}", flush=True)
    _check(*_simulation(60, 77, pml=6, lossy=False, edges=edges), steps=(16, 5))


@pytest.mark.parametrize("parts", [(False, False), (True, False), (False, True)])
def test_multi_step_layouts(parts):
    """Programs without sources, without monitors, with one of them."""
    _require_gpu()
    print(f"case tm_steps sources={parts[0]} monitors={parts[1]}", flush=True)
    _check(*_simulation(64, 100, pml=5, lossy=False, sources=parts[0], monitors=parts[1]),
           steps=(20, 7))


@pytest.mark.parametrize("T", ["2", "3", "6", "8"])
def test_multi_step_shapes(T, monkeypatch):
    _require_gpu()
    monkeypatch.setenv("BZH_TM_T", T)
    print(f"case tm_steps T={T}", flush=True)
    _check(*_simulation(150, 190, pml=9, lossy=False), steps=(26,))
    _check(*_simulation(300, 700, pml=9, lossy=False), steps=(19,))    # four rows per lane
