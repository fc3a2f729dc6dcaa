"""Quotients by zero and by infinity: what the oracle computes and accepts, the
engine does as well.  Values at the bound of the other residual tests."""
import dataclasses

import numpy as np
import pytest

from binding import Oracle
from festgpu import cases as C
from festgpu.native import GpuBlock

pytestmark = pytest.mark.gpu
INNER = (slice(None),) + (slice(3, -3),) * 3


def pair(case, nodes, q):
    o = Oracle(case)
    o.set_nodes(nodes)
    o.set_state(q)
    o.temp_refresh()
    g = GpuBlock(case)
    g.set_grid(nodes)
    g.upload_state(q)
    return g, o


@pytest.mark.parametrize("nk", [1, 4])
def test_implicit_step_with_cfl_0(nk):
    """The LU-SGS diagonal volume / dt is infinite, the update zero."""
    case, nodes, q = C.euler_bump(9, 6, nk)
    case = dataclasses.replace(case, time_accuracy="implicit", CFL=0.0)
    g, o = pair(case, nodes, q)
    for it in (1, 2):
        assert o.step(it) == 0
        g.get_next_solution(it)
    a, b = g.download("qp")[INNER], o.arr("qp")[INNER]
    assert np.isfinite(a).all()
    assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()
    assert np.abs(a - q[INNER]).max() <= 1e-12 * np.abs(q[INNER]).max()


@pytest.mark.parametrize("flux", ["ldfss0", "van_leer"])
def test_infinite_density(flux):
    """A cell of infinite density has a sound speed of 0 and infinite fluxes,
    no NaN."""
    case, nodes, q = C.euler_bump(6, 5, 4, flux=flux, recon="none")
    q[0, 5, 5, 5] = np.inf
    g, o = pair(case, nodes, q)
    assert o.residual(1) == 0
    g.residual(1)
    for n in "FGH":
        a, b = g.download(n), o.arr(n)
        f = np.isfinite(b)
        assert not f.all()
        assert np.array_equal(a[~f], b[~f])
        assert np.abs(a[f] - b[f]).max() <= 1e-12 * np.abs(b[f]).max()
