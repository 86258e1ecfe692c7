"""Lower Yee phases and multi-step programs to the HIP library's positional
entry points.

This module mirrors ``beamz/simulation/cuda/runtime.py`` function for function:
``update_h``/``update_e`` (``runtime.py:184-280``, one phase through
``bzh_streamed``), ``run_steps`` (``:685-750``), ``run_source_group_steps``
(``:496-527``) and ``run_program_steps`` (``:621-682``) through
``bzh_program`` with the same positional layouts (``abi_layout.json``).  State
tensors are updated in place (the reference's ``input_output_aliases``) and
the same state object is returned.
"""

from __future__ import annotations

import ctypes
import weakref

import torch

from . import _abi as abi
from . import native
from .program import CompiledProgram, SimulationState, field_bank

# Slots without elements: described, not allocated (34 of a 2D call's
# arguments; as zero-size tensors they took 60 of its 175 us).
_EMPTY = native.Absent()
_EMPTY_GROUP = (native.Absent((0, 1, 1, 1)), native.Absent((0, 1)),
                native.Absent((0, 3), torch.int32))


def _metrics(prog, phase):
    """The (z, y, x) derivative metrics of one phase (``cuda/runtime.py:89-94``):
    none on isotropic uniform grids (metric_kind 0)."""
    table = prog.h_metrics if phase == abi.PHASE_H else prog.e_metrics
    if table:
        return tuple(table)
    return (_EMPTY, _EMPTY, _EMPTY)


def _materials(prog, phase):
    c = prog.coeffs
    p = "h" if phase == abi.PHASE_H else "e"
    return (c[f"{p}_decay_x"], c[f"{p}_decay_y"], c[f"{p}_decay_z"],
            c[f"{p}_source_x"], c[f"{p}_source_y"], c[f"{p}_source_z"])


def _psi_slots(psi):
    return (*psi, *(_EMPTY,) * (abi.CPML_TERM_COUNT - len(psi)))


def _cpml_payload(prog, state, phase):
    if phase == abi.PHASE_H:
        return (*_materials(prog, phase), prog.h_meta, *prog.h_term_arrays,
                *_psi_slots(state.psi_h))
    return (*_materials(prog, phase), prog.e_meta, *prog.e_term_arrays,
            *_psi_slots(state.psi_e))


def _graph_io(prog: CompiledProgram, state: SimulationState):
    """Positional inputs of the 24-input (Yee) or 74-input (CPML) graph
    (``runtime.py:284-381``)."""
    if prog.cpml_enabled:
        return (*state.fields(), *_cpml_payload(prog, state, abi.PHASE_H),
                *_cpml_payload(prog, state, abi.PHASE_E), *_metrics(prog, abi.PHASE_H),
                *_metrics(prog, abi.PHASE_E))
    return (*state.fields(), *_materials(prog, abi.PHASE_H), *_materials(prog, abi.PHASE_E),
            *_metrics(prog, abi.PHASE_H), *_metrics(prog, abi.PHASE_E))


def _source_group_arguments(prog):
    return tuple(t for g in prog.source_groups for t in (_EMPTY_GROUP if g is None else g))


def _program_attrs(prog, nsteps, layout, monitor_count=0):
    return native.ProgramAttrs(
        abi_version=abi.ABI_VERSION, flags=prog.flags, nsteps=int(nsteps), dt=prog.dt,
        resolution=prog.abi_resolution, boundary_code=prog.boundary_code,
        metric_kind=prog.metric_kind, program_layout=layout, cpml_enabled=int(prog.cpml_enabled),
        monitor_count=int(monitor_count), coincident_source_group_mask=prog.coincident_mask)


def _phase(prog, state, phase):
    if phase == abi.PHASE_H:
        targets, sources = (state.hx, state.hy, state.hz), (state.ex, state.ey, state.ez)
    else:
        targets, sources = (state.ex, state.ey, state.ez), (state.hx, state.hy, state.hz)
    args = [*targets, *sources, *_materials(prog, phase)]
    if prog.cpml_enabled:
        meta = prog.h_meta if phase == abi.PHASE_H else prog.e_meta
        arrays = prog.h_term_arrays if phase == abi.PHASE_H else prog.e_term_arrays
        psi = state.psi_h if phase == abi.PHASE_H else state.psi_e
        n = prog.nterms
        args += [meta, *arrays[:3 * n], *psi[:n]]
    args += list(_metrics(prog, phase))
    attrs = native.PhaseAttrs(
        abi_version=abi.ABI_VERSION, flags=prog.flags, phase=phase, nterms=prog.nterms,
        dt=prog.dt, resolution=prog.abi_resolution, boundary_code=prog.boundary_code,
        metric_kind=prog.metric_kind)
    native.call_streamed(args, attrs)
    return state


def update_h(state: SimulationState, prog: CompiledProgram) -> SimulationState:
    """Advance the magnetic fields and their CPML memory (``runtime.py:184-231``)."""
    return _phase(prog, state, abi.PHASE_H)


def update_e(state: SimulationState, prog: CompiledProgram) -> SimulationState:
    """Advance the electric fields and their CPML memory (``runtime.py:234-280``)."""
    return _phase(prog, state, abi.PHASE_E)


def uses_two_banks(prog) -> bool:
    """The fused two-bank step applies to 3D programs with at most
    ``MAX_H_SLABS`` H-timed source slabs when the fused flag is set
    (``abi.FLAG_FUSED_STEP``)."""
    from .program import MAX_H_SLABS, h_source_slabs
    return (prog.is_3d and bool(prog.flags & abi.FLAG_FUSED_STEP)
            and h_source_slabs(prog.source_groups) <= MAX_H_SLABS)


def with_workspace(state):
    """Allocate the second field bank on first use (the CPML bank is allocated
    with the state, in the same arena as the first)."""
    if state.fields_b:
        return state
    fields_b = field_bank([tuple(t.shape) for t in state.fields()], state.hx.dtype,
                          state.hx.device)
    psi_b = state.psi_b
    if len(psi_b) != len(state.psi_h) + len(state.psi_e):
        psi_b = tuple(torch.empty_like(t) for t in (*state.psi_h, *state.psi_e))
    return state._replace(fields_b=fields_b, psi_b=psi_b)


def _swap_banks(state, nsteps):
    """After an odd step count the result lives in the workspace bank
    (``runtime.py:393-440``): exchange the bank roles."""
    if nsteps % 2 == 0:
        return state
    f = state.fields_b
    nh = len(state.psi_h)
    return state._replace(hx=f[0], hy=f[1], hz=f[2], ex=f[3], ey=f[4], ez=f[5],
                          psi_h=tuple(state.psi_b[:nh]), psi_e=tuple(state.psi_b[nh:]),
                          fields_b=state.fields(), psi_b=(*state.psi_h, *state.psi_e))


def _temporal_io(prog, state):
    if prog.cpml_enabled:
        return (*_graph_io(prog, state), *state.fields_b, *state.psi_b)
    return (*_graph_io(prog, state), *state.fields_b)


class Workspace2D(tuple):
    """A 2D state's launch scratch in its second-bank slot: one tensor, used by
    the state that holds ``ez`` and on the stream it was allocated on.  A state
    forked with tensors of its own, or a call on another stream, gets another
    one, so that two forks on two streams never write the same scratch, and a
    dropped one is reused only behind the work that was queued on it.  Its
    contents do not outlive a call: copies and pickles leave it out.  A caller's
    graph refers to the scratch of the state that the captured call returned."""

    def __new__(cls, tensor, ez, stream):
        self = super().__new__(cls, (tensor,))
        self.ez = weakref.ref(ez)
        self.stream = stream
        return self

    def fits(self, ez, stream, floats):
        return self.ez() is ez and self.stream == stream and self[0].numel() >= floats

    def __reduce__(self):
        return torch.Size, ((),)  # an empty tuple that ``weights_only`` loading accepts


def _stream(prog):
    """The current stream's handle, read once per call (None: no GPU)."""
    return native.current_stream_handle() if prog.device.type == "cuda" else None


def with_workspace_2d(state, prog, handle=None):
    """The state with the 2D program's multi-step workspace in its second-bank
    slot (:class:`Workspace2D`), allocated where the state has none of its own
    for the current stream (``handle``, from :func:`_stream`)."""
    n = prog.workspace_floats
    if n == 0 or prog.is_3d:
        return state
    if handle is None:
        handle = _stream(prog)
    stream = (handle.value or 0) if handle is not None else 0
    held = state.fields_b
    if isinstance(held, Workspace2D) and held.fits(state.ez, stream, n):
        return state
    tensor = torch.empty(n, dtype=torch.float32, device=prog.device)
    return state._replace(fields_b=Workspace2D(tensor, state.ez, stream))


def _workspace_args(state, prog):
    return tuple(state.fields_b[:1]) if prog.workspace_floats and not prog.is_3d else ()


def run_steps(state, prog, nsteps):
    """Source-free, monitor-free steps (``runtime.py:685-750``).  Returns the
    state holding the result (the bank roles swap after an odd count)."""
    if uses_two_banks(prog):
        return run_source_group_steps(state, prog, nsteps)
    layout = abi.PROGRAM_LAYOUT_CPML_IN_PLACE if prog.cpml_enabled else abi.PROGRAM_LAYOUT_YEE_IN_PLACE
    stream = _stream(prog)
    state = with_workspace_2d(state, prog, stream)
    native.call_program((*_graph_io(prog, state), *_workspace_args(state, prog)),
                        _program_attrs(prog, nsteps, layout), stream)
    return state


def run_source_group_steps(state, prog, nsteps, *, noalloc=False):
    """Steps with the nine slab-source groups (``runtime.py:496-527``);
    ``noalloc`` as in :func:`run_program_steps`."""
    if uses_two_banks(prog):
        state = with_workspace(state)
        args = (*_temporal_io(prog, state), *_source_group_arguments(prog), state.current_step)
        native.call_program(args, _program_attrs(prog, nsteps, abi.PROGRAM_LAYOUT_SOURCE_TEMPORAL_CPML),
                            noalloc=noalloc)
        return _swap_banks(state, nsteps)
    stream = _stream(prog)
    state = state if noalloc else with_workspace_2d(state, prog, stream)
    args = (*_graph_io(prog, state), *_source_group_arguments(prog), state.current_step,
            *_workspace_args(state, prog))
    native.call_program(args, _program_attrs(prog, nsteps, abi.PROGRAM_LAYOUT_SOURCE_IN_PLACE),
                        stream, noalloc=noalloc)
    return state


def _monitor_tail(state, prog, noalloc):
    """The source groups, packed monitors, DFT arenas and clocks that follow
    the field arguments of a monitor layout."""
    if state.dft_re.dtype != torch.float64:
        raise ValueError("the HIP program accumulates DFT monitors in float64")
    tail = (*_source_group_arguments(prog), *prog.packed_monitors,
            state.dft_re, state.dft_im, state.dft_w, state.t, state.current_step)
    if prog.monitor_boxes is not None and not noalloc:
        tail = (*tail, prog.monitor_boxes)      # host hint: the cells the monitors read
    return tail


def run_program_steps(state, prog, nsteps, *, noalloc=False):
    """Steps with sources and packed DFT monitors (``runtime.py:621-682``).
    ``noalloc`` calls ``bzh_program_noalloc``, which allocates no device
    memory (the state must already hold its workspace banks)."""
    tail = _monitor_tail(state, prog, noalloc)
    if uses_two_banks(prog):
        state = with_workspace(state)
        native.call_program((*_temporal_io(prog, state), *tail),
                            _program_attrs(prog, nsteps, abi.PROGRAM_LAYOUT_MONITOR_TEMPORAL_CPML,
                                           monitor_count=len(prog.monitors)), noalloc=noalloc)
        return _swap_banks(state, nsteps)
    stream = _stream(prog)
    state = state if noalloc else with_workspace_2d(state, prog, stream)
    native.call_program((*_graph_io(prog, state), *tail, *_workspace_args(state, prog)),
                        _program_attrs(prog, nsteps, abi.PROGRAM_LAYOUT_MONITOR_IN_PLACE,
                                       monitor_count=len(prog.monitors)), stream, noalloc=noalloc)
    return state


def run_chunk(state, prog, nsteps):
    """Pick the layout the program needs (``execute.py:595-681``); returns the
    state that holds the result."""
    if prog.monitors:
        return run_program_steps(state, prog, nsteps)
    if any(g is not None for g in prog.source_groups):
        return run_source_group_steps(state, prog, nsteps)
    return run_steps(state, prog, nsteps)


def prepare_chunk(state, prog, nsteps):
    """The program call :func:`run_chunk` makes for ``nsteps`` steps of
    ``state``, as a :class:`native.PreparedProgram` (arguments marshalled
    once), for loops that step one state many times in short chunks.  Only
    the in-place layouts qualify, whose steps leave every tensor in its role;
    None for a program that steps through two banks."""
    if uses_two_banks(prog):
        return None
    state = with_workspace_2d(state, prog)
    ws = _workspace_args(state, prog)
    if prog.monitors:
        return native.PreparedProgram(
            (*_graph_io(prog, state), *_monitor_tail(state, prog, False), *ws),
            _program_attrs(prog, nsteps, abi.PROGRAM_LAYOUT_MONITOR_IN_PLACE,
                           monitor_count=len(prog.monitors)), scratch=ws)
    if any(g is not None for g in prog.source_groups):
        return native.PreparedProgram(
            (*_graph_io(prog, state), *_source_group_arguments(prog), state.current_step, *ws),
            _program_attrs(prog, nsteps, abi.PROGRAM_LAYOUT_SOURCE_IN_PLACE), scratch=ws)
    layout = abi.PROGRAM_LAYOUT_CPML_IN_PLACE if prog.cpml_enabled else abi.PROGRAM_LAYOUT_YEE_IN_PLACE
    return native.PreparedProgram((*_graph_io(prog, state), *ws),
                                  _program_attrs(prog, nsteps, layout), scratch=ws)


GRAPH_MAX_STEPS = 256  # execute.py:64


def advance(state, prog, nsteps, *, chunk=GRAPH_MAX_STEPS):
    """Advance ``nsteps`` in chunks of at most ``chunk`` steps; the clocks are
    recomputed from the run origin after every chunk (``execute.py:622-657``).
    Returns the state holding the result."""
    done = int(state.current_step.item()) if nsteps > 0 else 0
    remaining = int(nsteps)
    while remaining > 0:
        n = min(chunk, remaining)
        state = run_chunk(state, prog, n)
        done += n
        remaining -= n
        state.current_step.fill_(done)
        state.t.fill_(prog.t0 + done * prog.dt)
    return state


def step_kernel_name(prog, pairs=False):
    """The step kernels as rocprofv3 names them; ``pairs`` when the last
    program call ran two steps per launch."""
    if uses_two_banks(prog):
        # one pair launch runs the general and the core bodies
        return "pair_step" if pairs else "fused_interior+fused_edge"
    if prog.is_3d:
        return "phase_3d"
    return "tm_steps" if prog.workspace_floats else "h_phase_tm+e_phase_tm"


def time_step_kernel(state, prog, *, launches=20, stream=None):
    """Average device time of one bare field step (no sources or monitors),
    measured with events on ``stream``: four steps per call (two pair launches
    where the pair kernel runs) so the banks return to their starting roles, 48
    (launches of eight or six steps) where a 2D program runs several per launch."""
    stream = stream or torch.cuda.current_stream()
    with torch.cuda.stream(stream):
        layout_state = state
        steps = 4
        start = torch.cuda.Event(enable_timing=True)
        stop = torch.cuda.Event(enable_timing=True)
        if uses_two_banks(prog):
            layout_state = with_workspace(layout_state)
            args = (*_temporal_io(prog, layout_state), *_EMPTY_GROUP * abi.SOURCE_GROUP_COUNT,
                    layout_state.current_step)
            attrs = _program_attrs(prog, steps, abi.PROGRAM_LAYOUT_SOURCE_TEMPORAL_CPML)
            attrs.coincident_source_group_mask = 0
        else:
            layout = abi.PROGRAM_LAYOUT_CPML_IN_PLACE if prog.cpml_enabled else abi.PROGRAM_LAYOUT_YEE_IN_PLACE
            layout_state = with_workspace_2d(layout_state, prog)
            ws = _workspace_args(layout_state, prog)
            steps = 48 if ws else steps
            args = (*_graph_io(prog, layout_state), *ws)
            attrs = _program_attrs(prog, steps, layout)
        native.call_program(args, attrs)  # warm (captures the graph)
        start.record(stream)
        for _ in range(launches):
            native.call_program(args, attrs)
        stop.record(stream)
    torch.cuda.synchronize()
    return start.elapsed_time(stop) / (steps * launches)


# ---- descriptor-level entry points (cuda/src/launch.h:12-77) -----------------
# The same work as the positional calls above, described by the structs that
# the reference's BeamzLaunchStreamed / BeamzLaunchProgram take
# (update.cu:919-971, program.cu:339-354).

def _fill(slots, tensors):
    for i, t in enumerate(tensors):
        slots[i] = native.buffer(t)


def _phase_launch(prog, phase, targets, sources, psi, out_targets, out_psi):
    """A :class:`native.Launch` of one phase: inputs in the streamed order
    (targets, sources, materials, metadata, 18 term arrays, psi), outputs the
    written targets and psi."""
    ln = native.Launch()
    ln.abi_version = abi.ABI_VERSION
    ln.flags = prog.flags
    ln.phase = phase
    ln.nterms = prog.nterms
    ln.metric_kind = prog.metric_kind
    ln.dt = prog.dt
    ln.resolution = prog.abi_resolution
    ln.inv_resolution = 1.0 / prog.abi_resolution
    ln.metallic_edges = prog.boundary_code & 0xFF
    ln.uniform_cpml_thickness = prog.boundary_code >> 8
    ins = [*targets, *sources, *_materials(prog, phase)]
    if prog.cpml_enabled:
        meta = prog.h_meta if phase == abi.PHASE_H else prog.e_meta
        arrays = prog.h_term_arrays if phase == abi.PHASE_H else prog.e_term_arrays
        ins += [meta, *arrays[:18], *_psi_slots(psi)]
    _fill(ln.inputs, ins + [None] * (37 - len(ins)))
    _fill(ln.metrics, _metrics(prog, phase))
    outs = [*out_targets]
    if prog.cpml_enabled:
        outs += list(_psi_slots(out_psi))
    _fill(ln.outputs, outs + [None] * (9 - len(outs)))
    return ln


def launch_phase(state, prog, phase):
    """One phase in place through ``bzh_launch_phase``."""
    if phase == abi.PHASE_H:
        t, src, psi = (state.hx, state.hy, state.hz), (state.ex, state.ey, state.ez), state.psi_h
    else:
        t, src, psi = (state.ex, state.ey, state.ez), (state.hx, state.hy, state.hz), state.psi_e
    native.call_launch_phase(_phase_launch(prog, phase, t, src, psi, t, psi))
    return state


def launch_program(state, prog, nsteps):
    """``nsteps`` steps with sources and monitors through
    ``bzh_launch_program`` (two field banks where the fused step applies).
    Returns the state holding the result, as :func:`run_chunk` does."""
    two = uses_two_banks(prog)
    if two:
        state = with_workspace(state)
    nh = len(state.psi_h)
    a_h, a_e = (state.hx, state.hy, state.hz), (state.ex, state.ey, state.ez)
    fb = state.fields_b if two else state.fields()
    b_h, b_e = tuple(fb[0:3]), tuple(fb[3:6])
    pb_h = tuple(state.psi_b[:nh]) if two else state.psi_h
    pb_e = tuple(state.psi_b[nh:]) if two else state.psi_e
    pl = native.ProgramLaunch()
    pl.h_ab = _phase_launch(prog, abi.PHASE_H, a_h, a_e, state.psi_h, b_h, pb_h)
    pl.e_ab = _phase_launch(prog, abi.PHASE_E, a_e, b_h, state.psi_e, b_e, pb_e)
    pl.h_ba = _phase_launch(prog, abi.PHASE_H, b_h, b_e, pb_h, a_h, state.psi_h)
    pl.e_ba = _phase_launch(prog, abi.PHASE_E, b_e, a_h, pb_e, a_e, state.psi_e)
    groups = (native.SourceGroup * abi.SOURCE_GROUP_COUNT)()
    flat = _source_group_arguments(prog)
    for gi in range(abi.SOURCE_GROUP_COUNT):
        g = groups[gi]
        g.coefficients = native.buffer(flat[3 * gi])
        g.waveforms = native.buffer(flat[3 * gi + 1])
        g.starts = native.buffer(flat[3 * gi + 2])
        g.current_step = native.buffer(state.current_step)
        g.component = gi % 3
        g.timing = gi // 3
        g.coincident = (prog.coincident_mask >> gi) & 1
    pl.source_groups = groups
    pl.source_group_count = abi.SOURCE_GROUP_COUNT
    keep = [groups]
    if prog.monitors:
        if state.dft_re.dtype != torch.float64:
            raise ValueError("the HIP program accumulates DFT monitors in float64")
        m = native.DftGroup()
        names = ("indices", "weights", "frequencies", "component_masks", "counts", "codes", "windows")
        for name, t in zip(names, prog.packed_monitors):
            setattr(m, name, native.buffer(t))
        m.dft_re = native.buffer(state.dft_re)
        m.dft_im = native.buffer(state.dft_im)
        m.dft_weight = native.buffer(state.dft_w)
        m.time = native.buffer(state.t)
        m.current_step = native.buffer(state.current_step)
        m.monitor_count = len(prog.monitors)
        pl.monitors = ctypes.pointer(m)
        keep.append(m)
    pl.field_bank_count = 2 if two else 1
    pl.nsteps = int(nsteps)
    native.call_launch_program(pl)
    del keep
    return _swap_banks(state, nsteps) if two else state
