"""``bzh_adjoint2d_recompute`` refuses record slots outside the record, also
where the slot and the step count together exceed 32 bits.  (CPU: the arguments
are refused before anything is launched.)"""

from __future__ import annotations

from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest
import torch

import beamz_amd as bz
from beamz_amd import native, runtime


@pytest.mark.parametrize("slot,nsteps", [(0, 9), (8, 1), (-1, 2), (2 ** 31 - 1, 5), (2 ** 31 - 4, 4)])
def test_record_slots_out_of_range(slot, nsteps):
    cpu = torch.device("cpu")
    sim = bz.Simulation(np.full((20, 30), 2.0), 25e-9, boundaries=[bz.PEC()], steps=8, device=cpu)
    prog, state = sim.compile(), sim.initial_state()
    shapes = prog.shapes
    keep = {"a_ez": torch.zeros(shapes["Ez"]), "a_hx": torch.zeros(shapes["Hx"]), "a_hy": torch.zeros(shapes["Hy"]),
            "record": torch.zeros(8, 4, 5), "grad": torch.zeros(4, 5, dtype=torch.float64),
            "e_decay": prog.coeffs["e_decay_z"], "e_source": prog.coeffs["e_source_z"],
            "h_decay": prog.coeffs["h_decay_x"], "h_source": prog.coeffs["h_source_x"]}
    work = [torch.zeros(shapes[c]) for c in ("Ez", "Ez", "Hy", "Hx")]
    adj = native.Adjoint2d()
    for k, t in keep.items():
        setattr(adj, k, native.buffer(t))
    for t in range(4):
        adj.work[t] = native.buffer(work[t])
        adj.a_psi[t] = native.buffer(None)
    adj.cpml_table = adj.source_profile = adj.source_time = native.buffer(None)
    adj.metallic, adj.resolution = int(prog.boundary_code & 0xFF), float(prog.abi_resolution)
    for q, v in enumerate((5, 9, 6, 11)):
        adj.design[q] = v
    call = runtime.prepare_chunk(state, prog, 1)
    # (on a thread of its own: the library keeps the last error per thread)
    with ThreadPoolExecutor(1) as pool, pytest.raises(native.HipLaunchError, match="record slots out of range"):
        pool.submit(call.recompute, adj, nsteps, slot, 0).result()
