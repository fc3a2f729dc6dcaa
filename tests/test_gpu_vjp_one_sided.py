"""The adjoint of a block whose direction has one periodic face only.

A periodic face's ghost cells copy the three layers next to the opposite
face, so the transpose of its rule adds to cells that the opposite face's
transpose adds to as well.  Every interior input of 10 x 9 x 8 grids, by
central differences of the GPU's own residual as in test_gpu_vjp.py (WENO5 +
van Leer, smooth at this state; its step and its bound of 1e-6 of each
variable's largest adjoint), and the same bits from every repetition."""
import numpy as np
import pytest

from festgpu import cases as C
from festgpu.native import GpuBlock
from test_gpu_vjp import TOL, check_columns, gpu_residual, say, weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bcs", [
    (-9, -2, -5, -6, -9, -9),   # periodic at imin, a flat copy at imax
    (-5, -9, -5, -6, -6, -6),   # a no-slip wall reads four layers from imin
    (-3, -4, -9, -6, -9, -9),   # j: a slip wall at jmax
    (-3, -4, -5, -6, -2, -9),   # k
])
def test_jacobian_columns_one_periodic_face(bcs):
    say("vjp one periodic face", bcs)
    case, nodes, q = C.euler_bump(10, 9, 8, flux="van_leer", recon="weno", bc_id=bcs)
    g = GpuBlock(case)
    g.set_grid(nodes)
    bar, worst = check_columns(g, case, q, lambda x: gpu_residual(g, x), 13)
    say("  worst", worst)
    assert worst <= TOL
    g.upload_state(q)
    for _ in range(20):
        assert np.array_equal(g.vjp(weights(case, 13)), bar)
