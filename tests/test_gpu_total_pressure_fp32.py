"""The total-pressure inlet's eddy viscosity in the FP32 mode.

The ghost cells of a -11 face take the SST mu_t and F1 that their own gradients
give; a block that keeps FP32 gradients only has to take those.  They depend on
the current state alone, whatever gradients were widened for a download before
(equal bits), and agree with an FP64 handle's to the FP32 gradients' error: a
velocity of |V| rounded to 2^-24 against differences of 0.5% of it, 1.2e-5 of a
gradient, times the few that a strain invariant sums: held to 1e-3."""
import dataclasses

import numpy as np
import pytest

from bc_cases import total_pressure_case
from festgpu.native import GpuBlock

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("turb", ["sst", "sst2003"])
@pytest.mark.parametrize("face", [0, 1])
def test_ghost_eddy_viscosity(face, turb):
    case, nodes, q = total_pressure_case(face, turb)
    # an omega at which the strain, not omega, sets mu_t next to the wall
    case = dataclasses.replace(case, fix_tw=(0.01 * case.tw_inf,) * 6)
    q[6] *= 0.01
    other = q.copy()
    other[1:4, 3:-3, 3:-3, 3:-3] *= 1 + 0.05 * np.random.default_rng(5).uniform(-1, 1, other[1:4, 3:-3, 3:-3, 3:-3].shape)

    def block(precision):
        g = GpuBlock(case, precision=precision)
        g.set_grid(nodes, wall_dist=True)
        return g

    def ghosts(g):
        g.upload_state(q)
        g.residual(1)
        i = 2 if face == 0 else case.imx + 2
        out = g.download("mut", "f1", "F")
        return out["mut"][3:-3, 3:-3, i], out["f1"][3:-3, 3:-3, i], out["F"]

    used = block(1)
    used.upload_state(other)
    used.residual(1)
    used.download("grads")
    mut, f1, F = ghosts(used)
    for a, b in zip((mut, f1, F), ghosts(block(1))):
        assert np.array_equal(a, b)
    mut64, f164, _ = ghosts(block(0))
    assert np.abs(mut64 - mut64.mean()).max() > 0.1 * mut64.max()
    assert np.abs(mut - mut64).max() <= 1e-3 * np.abs(mut64).max()
    assert np.abs(f1 - f164).max() <= 1e-3
