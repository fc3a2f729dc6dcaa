"""The face sweeps at the extents where their special paths meet: directions
of three to six cells, where every face, all but one or none takes a boundary
rule, and rows around the 64-wide tiles.  Against the oracle at the bound of
the other residual tests (1e-12 of each array's largest value)."""
import dataclasses
import sys

import numpy as np
import pytest

from binding import Oracle
from festgpu import cases as C
from festgpu.native import GpuBlock

pytestmark = pytest.mark.gpu
TOL = 1e-12


def relerr(a, b):
    assert np.isfinite(a).all() and np.isfinite(b).all()
    s = np.abs(b).max()
    return np.abs(a - b).max() / s if s > 0 else np.abs(a).max()


def pair(case, nodes, q, wall):
    o = Oracle(case)
    o.set_nodes(nodes)
    if wall:
        o.wall_dist()
    o.set_state(q)
    o.temp_refresh()
    g = GpuBlock(case)
    g.set_grid(nodes, wall_dist=wall)
    g.upload_state(q)
    return g, o


@pytest.mark.parametrize("recon", ["muscl", "ppm", "weno", "weno_NM"])
@pytest.mark.parametrize("ni,nj,nk", [(3, 3, 3), (4, 5, 6), (63, 6, 4), (64, 4, 5), (65, 7, 3)])
def test_boundary_and_inner_faces(ni, nj, nk, recon):
    case, nodes, q = C.sst_bump(ni, nj, nk, first=0.02)
    case = dataclasses.replace(case, recon=recon, bc_id=(-3, -4, -5, -8, -6, -2))
    print("faces", ni, nj, nk, recon, flush=True)
    sys.stdout.flush()
    g, o = pair(case, nodes, q, True)
    assert o.residual(1) == 0
    g.residual(1)
    out = g.download("qp", "F", "G", "H", "residue")
    for n, on in (("qp", "qp"), ("F", "F"), ("G", "G"), ("H", "H"), ("residue", "res")):
        assert relerr(out[n], o.arr(on)) <= TOL, n
