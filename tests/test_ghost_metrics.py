"""The ghost cells' gradients of blocks far longer along k (or j) than along i.

The gradient ghost rule reads the J and K face metrics at the I-face linear
offset (src/gradients.f90:523-595); in these blocks that offset passes the end
of the arrays, and the face's own metrics are taken.  The oracle against the
rule written out in numpy (a dozen roundings: 1e-13 of the largest value), the
engine against the oracle at the bound of the other residual tests, and the
viscous adjoint against central differences of the engine's own residual (the
bound of test_gpu_vjp.py)."""
import dataclasses
import sys

import numpy as np
import pytest

from binding import Oracle
from festgpu import cases as C

SHAPES = [(3, 20, 63), (5, 8, 63), (3, 48, 36), (4, 5, 120)]


def make(ni, nj, nk, turb):
    if turb == "none":
        case, nodes, q = C.laminar_box(ni, nj, nk)
        nodes = C.cartesian_nodes(case, warp=0.02)
        return dataclasses.replace(case, bc_id=(-8, -4, -5, -6, -6, -5), fix_p=(case.p_inf,) * 6), nodes, q
    case, nodes, q = C.sst_bump(ni, nj, nk, turb=turb, recon="muscl", first=0.02)
    return dataclasses.replace(case, bc_id=case.bc_id[:4] + (-6, -8)), nodes, q


def oracle(case, nodes, q):
    o = Oracle(case)
    o.set_nodes(nodes)
    if case.turb != "none":
        o.wall_dist()
    o.set_state(q)
    o.temp_refresh()
    assert o.residual(3) == 0
    return o


@pytest.mark.parametrize("ni,nj,nk", SHAPES)
def test_oracle_follows_the_rule(ni, nj, nk):
    case, nodes, q = make(ni, nj, nk, "none")
    o = oracle(case, nodes, q)
    qp, vol = o.arr("qp"), o.arr("vol")
    g = np.stack([o.arr(n) for n in ("gx", "gy", "gz")])
    I, J, K = case.imx, case.jmx, case.kmx
    past = 0
    for d, letter, n in ((1, "j", J), (2, "k", K)):
        metrics = [o.arr(letter + m) for m in ("A", "nx", "ny", "nz")]
        flat = [m.reshape(-1) for m in metrics]
        at = n - 1, n  # the interior and the ghost cell of the max face
        worst = top = 0.0
        for c in range(1, K if d == 1 else J):
            for i in range(1, I):
                f = (i, n, c) if d == 1 else (i, c, n)
                o_i = (f[0] + 2) + (I + 6) * ((f[1] + 2) + (J + 5) * (f[2] + 2))
                if o_i < flat[0].size:
                    A, *nrm = [m[o_i] for m in flat]
                else:
                    past += 1
                    A, *nrm = [m[f[2] + 2, f[1] + 2, f[0] + 2] for m in metrics]
                nrm = np.array(nrm)
                ci, cg = [(c + 2, x + 2, i + 2) if d == 1 else (x + 2, c + 2, i + 2) for x in at]
                gi, gg = [(c, x, i) if d == 1 else (x, c, i) for x in at]
                own = g[(slice(None), 0) + gi]
                want = -(qp[(1,) + ci] - qp[(1,) + cg]) * A * nrm / vol[ci] + own - own.dot(nrm) * nrm
                worst = max(worst, np.abs(g[(slice(None), 0) + gg] - want).max())
                top = max(top, np.abs(want).max())
        assert worst <= 1e-13 * top
    assert past > 0


@pytest.mark.gpu
@pytest.mark.parametrize("turb", ["none", "sst", "sa"])
@pytest.mark.parametrize("ni,nj,nk", SHAPES)
def test_engine_follows_the_oracle(ni, nj, nk, turb):
    from festgpu.native import GpuBlock
    case, nodes, q = make(ni, nj, nk, turb)
    print("ghost metrics", ni, nj, nk, turb, flush=True)
    sys.stdout.flush()
    o = oracle(case, nodes, q)
    g = GpuBlock(case)
    g.set_grid(nodes, wall_dist=turb != "none")
    g.upload_state(q)
    g.residual(3)
    out = g.download("grads", "residue")
    for a, n in ((out["grads"][0], "gx"), (out["grads"][1], "gy"), (out["grads"][2], "gz"), (out["residue"], "res")):
        b = o.arr(n)
        assert np.isfinite(a).all()
        assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max(), n


@pytest.mark.gpu
def test_viscous_adjoint():
    from festgpu.native import GpuBlock
    from test_gpu_vjp import TOL, check_columns, gpu_residual, say
    case, nodes, q = C.euler_bump(4, 5, 60, flux="van_leer", recon="none", bc_id=(-3, -4, -5, -6, -6, -5))
    case = dataclasses.replace(case, mu_ref=0.02, mu_sutherland=1, S_ref=0.4)
    say("vjp ghost metrics")
    g = GpuBlock(case)
    g.set_grid(nodes)
    _, worst = check_columns(g, case, q, lambda x: gpu_residual(g, x), 19, sample=400)
    say("  worst", worst)
    assert worst <= TOL
