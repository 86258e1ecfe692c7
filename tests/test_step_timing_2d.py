"""The timing helper runs and names the kernels that a 2D program's calls run
(CPU, against a stub in place of the native call), and programs that the
multi-step launch does not take hold no workspace for it."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import beamz_amd as bz
from beamz_amd import native, runtime


def _simulation(*, nmon=1, nslab=1, edges="all", timing="e"):
    wave = np.ones(4)
    return bz.Simulation(
        np.full((40, 50), 2.0), 25e-9, boundaries=[bz.PML(edges=edges, cells=4)], steps=8,
        sources=[bz.CustomSource("Ez", (8, 8 + q), np.ones((3, 1)), wave, timing) for q in range(nslab)],
        monitors=[bz.FluxMonitor("x", 10 + q, np.array([2e14]), ranges={"y": (5, 30)}) for q in range(nmon)])


@pytest.mark.parametrize("kw,multi", [
    ({}, True), ({"nmon": 8, "nslab": 12}, True), ({"nmon": 0, "nslab": 0}, True), ({"nmon": 9}, False),
    ({"nslab": 13}, False), ({"edges": ("left", "right")}, False)])
def test_workspace_only_where_launches_take_several_steps(kw, multi):
    prog = _simulation(**kw).compile()
    assert (prog.workspace_floats > 0) == multi
    assert runtime.step_kernel_name(prog) == ("tm_steps" if multi else "h_phase_tm+e_phase_tm")


class _Event:
    def __init__(self, **kw):
        pass

    def record(self, *a):
        pass

    def elapsed_time(self, other):
        return 480.0


class _Stream:
    def __init__(self, *a):
        pass

    def __enter__(self):
        return self

    def __exit__(self, *a):
        return False


@pytest.mark.parametrize("nmon,steps,count", [(1, 48, 1), (9, 4, 0)])
def test_step_timing_runs_the_program_s_kernels(monkeypatch, nmon, steps, count):
    sim = _simulation(nmon=nmon)
    prog, calls = sim.compile(), []
    monkeypatch.setattr(native, "call_program", lambda args, attrs: calls.append((len(args), attrs.nsteps, args[-1])))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: _Stream())
    monkeypatch.setattr(torch.cuda, "stream", _Stream)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    monkeypatch.setattr(torch.cuda, "Event", _Event)
    bare = len(runtime._graph_io(prog, sim.initial_state()))
    ms = runtime.time_step_kernel(sim.initial_state(), prog, launches=5)
    assert {c[:2] for c in calls} == {(bare + count, steps)}
    assert ms == 480.0 / (5 * steps)
    if count:
        assert calls[0][2].numel() == prog.workspace_floats


@pytest.mark.gpu
@pytest.mark.parametrize("kw,floats", [({"nmon": 9}, None), ({"nslab": 13}, None), ({}, 64)])
def test_refused_forms_run_the_phases(kw, floats):
    """Too many monitors or slabs, or a workspace that is too small, offered to
    the library all the same: the per-phase schedule's results."""
    import dataclasses
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU")
    native.library()
    print(f"case 2D fallback {kw} floats={floats}", flush=True)
    sim = _simulation(**kw)
    prog = sim.compile()
    rng = np.random.default_rng(3)
    fields = {c.lower(): rng.normal(size=prog.shapes[c]) * (1.0 if c[0] == "E" else 1 / 377)
              for c in prog.shapes}
    states = []
    for n in (floats or 1 << 22, 0):
        states.append(runtime.advance(sim.initial_state(fields), dataclasses.replace(prog, workspace_floats=n), 11))
    torch.cuda.synchronize()
    for name in ("hx", "hy", "ez", "dft_re", "dft_im", "dft_w"):
        assert torch.equal(getattr(states[0], name), getattr(states[1], name))
    for a, b in zip((*states[0].psi_h, *states[0].psi_e), (*states[1].psi_h, *states[1].psi_e)):
        assert torch.equal(a, b)
