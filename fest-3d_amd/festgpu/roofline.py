"""Algorithmic HBM bytes of the hot kernels, per launch, for the roofline.

Each figure counts the bytes a kernel must move at least once per launch:
every array element it reads or writes, taken once (stencil neighbours come
from cache), FP64 throughout.  Face arrays are counted per face, cell arrays
per cell of the launch's index box.  The numbers follow the kernels in
fest-3d_amd/csrc:

  flux_i/j/k (k_sweeps run for one direction D, as timed runs do; one thread
  per face of direction D):
    read  q (n_var planes), the face's A,nx,ny,nz (4), both cell centres
          (3, one per cell), the cell gradients (3 x n_grad), mu (+ mu_t, F1
          with SST)
    write the face flux (n_var); the face sound speed at stage 1 (1, a
          quarter per launch over the four RK stages)
  flux (k_sweeps of all three directions in one launch, as steps run it):
    read  per cell q, the centre, the gradients, mu (+ mu_t, F1 with SST)
          once, per face A,nx,ny,nz
    write as above
  grad (k_grad<NG>, one thread per cell 0..imx x 0..jmx x 0..kmx):
    read  the n_grad gradient variables, volume, the i/j/k face metrics
          (3 x 4), rho and p when mu follows Sutherland, rho, dist and mu
          (when constant) with SST
    write 3 x n_grad gradients, mu (Sutherland), mu_t, F1 and the two SST
          source terms
  update (k_update, one thread per interior cell), averaged over the four
    RK4 stages:
    read  the three face fluxes (3 x n_var, one face per direction per
          cell), the RK base state (n_var), dt, volume, the R accumulator
          (stages 2-4), the SST source (2), F1 and omega (SST)
    write q (n_var), the R accumulator (stages 1-3), the residue (stage 4)
  lusgs_sweep (k_lusgs_march, the LU-SGS update of the 'implicit' step: one
    launch a sweep, two a step, which the engine's event timer brackets as
    one; priced per bracket, i.e. both sweeps over every interior cell), per
    interior cell and sweep, from the hyperplane-major storage, whose values
    are kept in pairs (p = ceil(n_var / 2)):
    read  the state, the right-hand side and, backward, the cell's own
          forward value (p pairs each), the diagonal (1 pair, SST 2), three
          faces x {A,nx,ny,nz, the viscous factors (2, turbulent 4), radius}
          in 4 or 5 pairs
    write the sweep value (p pairs)
  lusgs_diag (k_to_skew + k_lusgs_prep, once a step), per interior cell:
    the copy of q into hyperplane-major storage (read + write, 2 n_var); the
    prep's stencil reads (q and residue, six faces x 4 metrics counted once a
    face, volume, mu, mu_t, F1, centres, dt: 2 n_var + 12 + 8) and writes (two
    right-hand sides, three radii, three faces' viscous factors, diagonal:
    2 n_var + 3 + 6 or 12 + 1 or 3)
  lusgs_apply (k_lusgs_apply): read q and the sweep value, write q (3 n_var)
"""

W = 8  # bytes per FP64 value


def _ngrad(case):
    return 6 if case.sst_family else 4


def launch_items(case, group):
    """Number of faces or cells one timed launch of `group` processes (for
    the sweep, cell-sweeps of both sweeps of a step)."""
    I, J, K = case.imx, case.jmx, case.kmx
    if group == "lusgs_sweep":
        return 2 * (I - 1) * (J - 1) * (K - 1)
    return {
        "flux_i": I * (J - 1) * (K - 1),
        "flux_j": (I - 1) * J * (K - 1),
        "flux_k": (I - 1) * (J - 1) * K,
        "grad": (I + 1) * (J + 1) * (K + 1),
        "update": (I - 1) * (J - 1) * (K - 1),
        "lusgs_diag": (I - 1) * (J - 1) * (K - 1),
        "lusgs_apply": (I - 1) * (J - 1) * (K - 1),
    }.get(group)


def bytes_per_item(case, group):
    """Algorithmic bytes per face or cell of one launch of `group`."""
    nv, ng, sst = case.n_var, _ngrad(case), case.sst_family
    if group in ("flux_i", "flux_j", "flux_k"):
        reads = nv + 4 + 3 + 3 * ng + (3 if sst else 1)
        writes = nv + 0.25
        return W * (reads + writes)
    if group == "grad":
        reads = ng + 1 + 12
        if case.mu_sutherland:
            reads += 2
        if sst:
            reads += 1 + (0 if case.mu_sutherland else 2)  # dist (+ rho, mu)
        writes = 3 * ng + (1 if case.mu_sutherland else 0) + (4 if sst else 0)
        return W * (reads + writes)
    if group == "update":
        base = 3 * nv + nv + 2 + nv  # fluxes, RK base, dt + vol, q write
        if sst:
            base += 2 + 2  # source, F1 + omega
        acc = (nv + 2 * nv + 2 * nv + 2 * nv) / 4.0  # R: write; read+write x2; read + residue write
        return W * (base + acc)
    ndg = 3 if sst else 1
    pairs, nvis = (nv + 1) // 2, 2 if nv == 5 else 4
    if group == "lusgs_sweep":
        reads = 2.5 * pairs + (ndg + 1) // 2 + 3 * (3 + nvis // 2)
        return 2 * W * (reads + pairs)
    if group == "lusgs_diag":
        return W * (2 * nv + (2 * nv + 12 + 8) + (2 * nv + 3 + 3 * nvis + ndg))
    if group == "lusgs_apply":
        return W * 3 * nv
    return None


def bytes_per_launch(case, group):
    if group == "flux":
        # the three directions together: what a cell holds for all of them
        # read once, each face's metrics and flux once
        nv, sst = case.n_var, case.sst_family
        cells = (case.imx - 1) * (case.jmx - 1) * (case.kmx - 1)
        faces = sum(launch_items(case, "flux_" + d) for d in "ijk")
        return W * (cells * (nv + 3 + 3 * _ngrad(case) + (3 if sst else 1)) + faces * (4 + nv + 0.25))
    n, b = launch_items(case, group), bytes_per_item(case, group)
    if n is None or b is None:
        return None
    return n * b


# whole RK stage at the fused minimum: q read and write, the RK base, the R
# accumulator, three owned faces x {A,nx,ny,nz}, volume, time step, cell
# centres, stale temperature and wall distance (stage-averaged)
BYTES_PER_CELL_STAGE = {"sst": 406.0, "none": 326.0}
HBM_PEAK_GBPS = 8000.0
