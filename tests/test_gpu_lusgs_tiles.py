"""LU-SGS sweeps of more tiles than the GPU has compute units: a work-group's
LDS fills its compute unit, so the last tiles start only after others have ended
and find the values handed to them long before.  Three steps (both sweeps fill
and empty the same places each time) against the oracle at the bound of the
other implicit tests."""
import dataclasses
import sys

import numpy as np
import pytest

from binding import Oracle
from festgpu import cases as C
from festgpu.native import GpuBlock

pytestmark = pytest.mark.gpu
INNER = (slice(None),) + (slice(3, -3),) * 3


@pytest.mark.parametrize("turb", ["none", "sst"])
def test_more_tiles_than_compute_units(turb):
    ni, nj, nk = 8, 137, 129  # 18 x 17 = 306 tiles of 8 x 8 columns
    if turb == "none":
        case, nodes, q = C.laminar_box(ni, nj, nk)
        case = dataclasses.replace(case, time_local=1, bc_id=(-8, -4, -5, -6, -6, -6), fix_p=(case.p_inf,) * 6)
    else:
        case, nodes, q = C.sst_bump(ni, nj, nk, recon="muscl", first=2e-3)
        case = dataclasses.replace(case, bc_id=case.bc_id[:4] + (-6, -6))
    case = dataclasses.replace(case, time_accuracy="implicit")
    print("tiles", ni, nj, nk, turb, flush=True)
    sys.stdout.flush()
    o = Oracle(case)
    o.set_nodes(nodes)
    if turb != "none":
        o.wall_dist()
    o.set_state(q)
    o.temp_refresh()
    g = GpuBlock(case)
    g.set_grid(nodes, wall_dist=turb != "none")
    g.upload_state(q)
    for it in (1, 2, 3):
        assert o.step(it) == 0
        g.get_next_solution(it)
    a, b = g.download("qp")[INNER], o.arr("qp")[INNER]
    for l in range(case.n_var):
        assert np.abs(a[l] - b[l]).max() <= 1e-12 * max(np.abs(b[l]).max(), case.vel_mag if l in (1, 2, 3) else 0.0), l
