"""A 2D state's launch scratch belongs to that state: a state forked from it
with tensors of its own gets another scratch, and copies and saved states carry
none (CPU; the forked runs on two streams need the GPU)."""

from __future__ import annotations

import copy
import io

import numpy as np
import pytest
import torch

import beamz_amd as bz
from beamz_amd import native, runtime

TENSORS = ("hx", "hy", "ez", "dft_re", "dft_im", "dft_w", "t", "current_step")


def _simulation(ny=70, nx=90):
    dx = 25e-9
    wave = np.cos(0.7 * np.arange(40)) * 0.3
    return bz.Simulation(
        np.random.default_rng(4).uniform(1.5, 12.0, (ny, nx)), dx, boundaries=[bz.PML(cells=6)], steps=64,
        sources=[bz.CustomSource("Ez", (10, 20), np.full((30, 1), 0.1), wave, "pre_e")],
        monitors=[bz.FluxMonitor("x", nx // 2, np.array([2.0e14]), ranges={"y": (0, ny)})])


def _fork(state):
    return state._replace(psi_h=tuple(t.clone() for t in state.psi_h),
                          psi_e=tuple(t.clone() for t in state.psi_e),
                          **{k: getattr(state, k).clone() for k in TENSORS})


def test_scratch_follows_the_state():
    sim = _simulation()
    prog = sim.compile()
    state = runtime.with_workspace_2d(sim.initial_state(), prog)
    assert prog.workspace_floats > 0 and len(state.fields_b) == 1
    assert runtime.with_workspace_2d(state, prog).fields_b[0] is state.fields_b[0]
    moved = state._replace(current_step=state.current_step.clone())
    assert runtime.with_workspace_2d(moved, prog).fields_b[0] is state.fields_b[0]
    forked = runtime.with_workspace_2d(_fork(state), prog)
    assert forked.fields_b[0].data_ptr() != state.fields_b[0].data_ptr()
    assert runtime.with_workspace_2d(forked, prog).fields_b[0] is forked.fields_b[0]


def test_copies_and_saved_states_carry_no_scratch():
    sim = _simulation()
    state = runtime.with_workspace_2d(sim.initial_state(), sim.compile())
    assert copy.deepcopy(state).fields_b == ()
    held = io.BytesIO()
    torch.save(tuple(state), held)
    held.seek(0)
    loaded = type(state)(*torch.load(held, weights_only=True))
    assert loaded.fields_b == () and torch.equal(loaded.ez, state.ez)


@pytest.mark.gpu
def test_forks_on_two_streams_match_lone_runs():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU")
    native.library()
    print("case forked 2D states on two streams", flush=True)
    sim = _simulation(300, 420)
    prog = sim.compile()
    rng = np.random.default_rng(5)
    fields = {c.lower(): rng.normal(size=prog.shapes[c]) * (1.0 if c[0] == "E" else 1 / 377)
              for c in prog.shapes}
    first = sim.advance(sim.initial_state(fields), 16)
    other = _fork(first)
    other.ez.mul_(-0.5)
    want = [sim.advance(_fork(s)._replace(fields_b=()), 48, chunk=16) for s in (first, other)]
    torch.cuda.synchronize()
    states = [first, other]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for _ in range(3):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                states[i] = runtime.run_chunk(states[i], prog, 16)
                states[i].current_step.add_(16)
                states[i].t.add_(16 * prog.dt)
    torch.cuda.synchronize()
    assert states[0].fields_b[0].data_ptr() != states[1].fields_b[0].data_ptr()
    for got, ref in zip(states, want):
        for a, b in zip((got.hx, got.hy, got.ez, *got.psi_h, *got.psi_e),
                        (ref.hx, ref.hy, ref.ez, *ref.psi_h, *ref.psi_e)):
            assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("warm", [False, True])
def test_captured_calls_replay(warm):
    """A call in a caller's graph, with and without a warm-up on its stream."""
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a GPU")
    native.library()
    print(f"case captured 2D call warm={warm}", flush=True)
    sim = _simulation(150, 230)
    prog = sim.compile()
    rng = np.random.default_rng(6)
    fields = {c.lower(): rng.normal(size=prog.shapes[c]) * (1.0 if c[0] == "E" else 1 / 377)
              for c in prog.shapes}

    def chunk(state):
        state = runtime.run_chunk(state, prog, 9)
        state.current_step.add_(9)
        state.t.add_(9 * prog.dt)
        return state

    got, want = sim.initial_state(fields), sim.initial_state(fields)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    if warm:
        with torch.cuda.stream(stream):
            got = chunk(got)
        want = chunk(want)
        torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        held = chunk(got)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        want = chunk(want)
        torch.cuda.synchronize()
        for a, b in zip((held.hx, held.hy, held.ez, *held.psi_h, *held.psi_e),
                        (want.hx, want.hy, want.ez, *want.psi_h, *want.psi_e)):
            assert torch.equal(a, b)
        for a, b in ((held.dft_re, want.dft_re), (held.dft_im, want.dft_im), (held.dft_w, want.dft_w)):
            assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())
