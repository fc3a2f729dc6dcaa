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


@pytest.mark.parametrize("turb", ["none", "sst", "sa", "kkl"])
@pytest.mark.parametrize("ni,nj,nk", [(5, 70, 1), (4, 64, 1), (6, 7, 3), (5, 17, 4), (7, 9, 8), (3, 17, 9), (9, 8, 16)])
def test_implicit_sweep_tiles(ni, nj, nk, turb):
    """LU-SGS sweeps where their 64-column tiles (64 x 1, 16 x 4 or 8 x 8) are
    full, just exceeded or mostly empty: one tile, a chain along j, both
    directions.  Two steps, every one handing values over the tile edges."""
    if turb == "none":
        case, nodes, q = C.laminar_box(ni, nj, nk)
        case = dataclasses.replace(case, time_local=1, bc_id=(-8, -4, -5, -6, -6, -6), fix_p=(case.p_inf,) * 6)
        nodes = C.cartesian_nodes(case, warp=0.03)
    else:
        case, nodes, q = C.sst_bump(ni, nj, nk, turb=turb, recon="muscl", first=2e-3)
        case = dataclasses.replace(case, bc_id=case.bc_id[:4] + (-6, -6))
    case = dataclasses.replace(case, time_accuracy="implicit")
    print("tiles", ni, nj, nk, turb, flush=True)
    g, o = pair(case, nodes, q, turb != "none")
    for it in (1, 2):
        assert o.step(it) == 0
        g.get_next_solution(it)
    inner = (slice(None),) + (slice(3, -3),) * 3
    assert relerr(g.download("qp")[inner], o.arr("qp")[inner]) <= TOL


@pytest.mark.parametrize("bcs", [(-3, -4, -5, -8, -9, -9), (-8, -2, -8, -6, -5, -8), (-9, -9, -6, -5, -8, -4),
                                 (-1, -11, -9, -9, -6, -6), (-7, -4, -6, -8, -11, -5)])
@pytest.mark.parametrize("ni,nj,nk", [(3, 4, 5), (4, 3, 9), (5, 7, 3), (6, 4, 4)])
def test_ghost_launches(ni, nj, nk, bcs):
    """Every ghost cell, edge and corner after one residual: faces that share
    a launch and those that may not, directions of three cells (where a face
    reads the other's ghosts) and more.  Both inflow-fix classes."""
    case, nodes, q = C.sst_bump(ni, nj, nk, first=0.02)
    tp = 1.02 * case.p_inf * (1 + 0.2 * case.MInf ** 2) ** 3.5
    case = dataclasses.replace(case, bc_id=bcs, fix_tp=(tp,) * 6)
    print("ghosts", ni, nj, nk, bcs, flush=True)
    g, o = pair(case, nodes, q, True)
    for it in (1, 3):
        assert o.residual(it) == 0
        g.residual(it)
        a, b = g.download("qp"), o.arr("qp")
        for l in range(7):
            assert relerr(a[l], b[l]) <= TOL, (it, l)


@pytest.mark.parametrize("turb", ["none", "kkl"])
@pytest.mark.parametrize("ni,nj,nk", [(3, 3, 3), (5, 4, 7), (64, 4, 3), (33, 65, 3), (127, 63, 35)])
def test_norm_sums(ni, nj, nk, turb):
    """The residual norms from one cell a thread and a mostly empty wave to
    more cells than 1024 work-groups have threads (127 x 63 x 35), against
    extended-precision sums of the downloaded residue and face fluxes.  Any
    order of m additions of positive terms is within m 2^-53 of the exact sum
    (3e-11 here); the imbalance is held to that of its terms' magnitudes."""
    if turb == "none":
        case, nodes, q = C.laminar_box(ni, nj, nk)
    else:
        case, nodes, q = C.sst_bump(ni, nj, nk, turb=turb, recon="muscl", first=0.02)
    g = GpuBlock(case)
    g.set_grid(nodes, wall_dist=turb != "none")
    g.upload_state(q)
    g.residual(1)
    out = g.download("residue", "F", "G", "H")
    norms = g.resnorm()
    m = ni * nj * nk
    v, rho, p = case.vel_mag, case.rho_inf, case.p_inf
    scale = [rho * v] + 3 * [rho * v * v] + [0.5 * rho * v**3 + case.gm / (case.gm - 1) * p]
    for l, s in enumerate(scale):
        r = out["residue"][l].astype(np.longdouble)
        assert norms[1 + l] == pytest.approx(float(np.sqrt((r * r).sum())) / s, rel=m * 2.0**-53 + 1e-14, abs=0)
    F, G, H = (out[n][0].astype(np.longdouble) for n in "FGH")
    ends = [F[:, :, 0], -F[:, :, -1], G[:, 0, :], -G[:, -1, :], H[0], -H[-1]]
    exact = abs(float(sum(e.sum() for e in ends)))
    mag = float(sum(abs(e).sum() for e in ends))
    assert abs(norms[0] - exact) <= (m * 2.0**-53 + 1e-14) * mag


@pytest.mark.parametrize("turb", ["none", "sst", "sa"])
@pytest.mark.parametrize("ni,nj,nk", [(5, 4, 1), (64, 3, 3), (65, 5, 4), (3, 9, 1)])
def test_gradients_next_to_boundaries(ni, nj, nk, turb):
    """Gradients and mu_t of interior and first ghost cells where a direction
    has one cell (both its faces belong to it), three or more, and rows that
    end at and past a wave."""
    if turb == "none":
        case, nodes, q = C.laminar_box(ni, nj, nk)
        nodes = C.cartesian_nodes(case, warp=0.03)
        case = dataclasses.replace(case, bc_id=(-8, -4, -5, -5, -6, -6), fix_p=(case.p_inf,) * 6)
    else:
        case, nodes, q = C.sst_bump(ni, nj, nk, turb=turb, recon="muscl", first=0.02)
        case = dataclasses.replace(case, bc_id=case.bc_id[:4] + (-6, -6))
    print("gradients", ni, nj, nk, turb, flush=True)
    g, o = pair(case, nodes, q, turb != "none")
    assert o.residual(3) == 0
    g.residual(3)
    out = g.download("grads", "mut", "residue")
    for d, n in enumerate(("gx", "gy", "gz")):
        assert relerr(out["grads"][d], o.arr(n)) <= TOL, n
    if turb != "none":
        inner = (slice(2, -2),) * 3
        assert relerr(out["mut"][inner], o.arr("mut")[inner]) <= TOL
    assert relerr(out["residue"], o.arr("res")) <= TOL
