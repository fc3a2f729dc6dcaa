"""The work that users of this engine have it do, as cases to measure: time
steps (explicit and implicit, FP64 and FP32 faces, single blocks and groups)
with the norms a run prints beside them, single residuals, and the adjoint.

A case is a dict of plain values: `kind` (the flow), the cell counts
ni, nj, nk (a group: blocks, lo, hi), flux, recon, turb, time ("residual" and
"adjoint" are the two single evaluations) and fp32 (face arithmetic).
"""
import dataclasses
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fest-3d_amd"))
from festgpu import cases as C  # noqa: E402
from festgpu.native import GpuBlock, GpuGroup  # noqa: E402

INNER = (slice(3, -3),) * 3


def _case(name, kind, ni, nj, nk, flux, recon, turb, time, fp32=False):
    c = {"kind": kind, "ni": ni, "nj": nj, "nk": nk, "flux": flux, "recon": recon, "turb": turb, "time": time,
         "fp32": fp32}
    return dict(c, name=name) if name else c


def _chain(name, blocks, lo, hi, fp32):
    c = {"kind": "chain", "blocks": blocks, "lo": lo, "hi": hi, "flux": "ausmUP", "recon": "muscl", "turb": "none",
         "time": "RK4", "fp32": fp32}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the reference's CPU-sized laminar box: the smallest runs, where
        # launches count; a global time step, as a time-accurate run takes
        _case("box_64x64x4", "box", 64, 64, 4, "ausmP", "muscl", "none", "RK4"),
        # a 2-D SST flat plate under LU-SGS, as the reference's shipped
        # flat-plate cases are (one cell in k)
        _case("plate2d_lusgs_96x48", "plate", 96, 48, 1, "ausm", "muscl", "sst", "implicit"),
        # an ordinary laminar box of odd extents, PPM
        _case("box_ppm_71x53x37", "box", 71, 53, 37, "van_leer", "ppm", "none", "RK4"),
        # an ordinary RANS block of odd extents
        _case("bump_97x61x45", "bump", 97, 61, 45, "slau", "weno", "sst", "RK4"),
        # Spalart-Allmaras, MUSCL, the TVD integrator
        _case("bump_sa_128x96x64", "bump", 128, 96, 64, "ausmP", "muscl", "sa", "TVDRK3"),
        # the headline: the RANS bump, WENO5 + SLAU, RK4
        _case("bump_256x128x128", "bump", 256, 128, 128, "slau", "weno", "sst", "RK4"),
        # the same block in the throughput mode (FP32 faces)
        _case("bump_f32_256x128x128", "bump", 256, 128, 128, "slau", "weno", "sst", "RK4", True),
        # the largest: a wall-resolved flat plate, PPM + LDFSS(0)
        _case("plate_384x192x128", "plate", 384, 192, 128, "ldfss0", "ppm", "sst", "RK4"),
        # the implicit integrator on a RANS block
        _case("bump_lusgs_128x96x64", "bump", 128, 96, 64, "slau", "weno", "sst", "implicit"),
        # uneven laminar blocks joined in a chain, one batched group step
        _chain("chain_24x16..48", 24, 16, 48, True),
        # one residual evaluation, and its adjoint, as a design loop calls them
        _case("euler_residual_96x64x48", "euler", 96, 64, 48, "slau", "muscl", "none", "residual"),
        _case("euler_adjoint_96x64x48", "euler", 96, 64, 48, "slau", "muscl", "none", "adjoint"),
    ]


def draw(rng):
    def extent(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    if rng.random() < 0.12:
        return _chain(None, rng.randint(6, 24), rng.choice((12, 16, 20)), rng.randint(28, 48), rng.random() < 0.5)
    kind = rng.choice(("box", "bump", "bump", "plate", "euler"))
    ni, nj, nk = extent(24, 320), extent(20, 160), extent(6, 128)
    fp32 = False
    if kind == "euler":
        # the adjoint's arguments are host arrays
        ni, nj, nk = min(ni, 128), min(nj, 96), min(nk, 64)
        return _case(None, kind, ni, nj, nk, rng.choice(("slau", "ausmP", "van_leer")),
                     rng.choice(("muscl", "weno", "ppm")), "none", rng.choice(("residual", "adjoint")))
    if kind == "box":
        turb, time = "none", rng.choice(("RK4", "RK4", "RK2", "implicit"))
        recon, flux = rng.choice(("muscl", "weno", "ppm")), rng.choice(("ausmP", "slau", "van_leer"))
    else:
        turb, time = rng.choice(("sst", "sst", "sst2003", "sa", "kkl")), rng.choice(("RK4", "RK4", "TVDRK3", "implicit"))
        recon, flux = rng.choice(("weno", "muscl", "ppm")), rng.choice(("slau", "ldfss0", "ausmP"))
        fp32 = turb == "sst" and time == "RK4" and rng.random() < 0.3
        if kind == "plate" and rng.random() < 0.3:
            ni, nj, nk, fp32 = min(ni, 128), min(nj, 64), 1, False
    return _case(None, kind, ni, nj, nk, flux, recon, turb, time, fp32)


# ---------------------------------------------------------------- inputs
def _noise(c, q, rng, amp):
    """Uniform noise on the interior cells (velocities scaled by |V_inf|)."""
    for l in range(c.n_var):
        r = amp * (2 * rng.random((c.kmx - 1, c.jmx - 1, c.imx - 1)) - 1)
        if l in (1, 2, 3):
            q[(l,) + INNER] += c.vel_mag * r
        else:
            q[(l,) + INNER] *= 1 + r
    return q


def _block_inputs(case, seed):
    """The configuration, grid nodes and initial state of a one-block case."""
    rng = np.random.default_rng(seed)
    kind, ni, nj, nk = case["kind"], case["ni"], case["nj"], case["nk"]
    make = {"box": C.laminar_box, "bump": C.sst_bump, "plate": C.flat_plate, "euler": C.euler_bump}[kind]
    kw = {"flux": case["flux"], "recon": case["recon"]}
    if kind in ("bump", "plate"):
        kw["turb"] = case["turb"]
    small, _, _ = make(4, 4, 4, **kw)  # the flow's settings; they do not depend on the extents
    time = case["time"] if case["time"] not in ("residual", "adjoint") else "RK4"
    c = dataclasses.replace(small, imx=ni + 1, jmx=nj + 1, kmx=nk + 1, time_accuracy=time, name=kind)
    q = C.freestream_state(c)
    if kind == "box":
        nodes = C.cartesian_nodes(c)
        # smooth 1% disturbances
        x = [(np.arange(n) + 0.5) for n in (nk, nj, ni)]
        for _ in range(8):
            at = rng.random(3) * (nk, nj, ni)
            g = [np.exp(-(x[a] - at[a]) ** 2 / 32.0) for a in range(3)]
            bump = g[0][:, None, None] * g[1][None, :, None] * g[2][None, None, :]
            for l, s in enumerate((c.rho_inf, c.vel_mag, c.vel_mag, c.vel_mag, c.p_inf)):
                q[(l,) + INNER] += 0.01 * s * (2 * rng.random() - 1) * bump
        if case["time"] == "implicit":
            c = dataclasses.replace(c, time_local=1)
    elif kind == "bump":
        nodes = C.bump_nodes(c, first=1e-5)
        _noise(c, q, rng, 0.005)
    elif kind == "euler":
        nodes = C.bump_nodes(c, first=0.02 if nj < 40 else 0.5 / nj, span=0.25)
        _noise(c, q, rng, 0.02)
    else:
        length, height, span = 2.0, 0.5, 0.25
        xs, zs = np.linspace(0.0, length, c.imx), np.linspace(0.0, span, c.kmx)
        ys = C.tanh_stretch(c.jmx, 5.5e-6 / height, 1.0) * height
        nodes = np.zeros(c.node_shape())
        nodes[0, 3:-3, 3:-3, 3:-3] = xs[None, None, :]
        nodes[1, 3:-3, 3:-3, 3:-3] = ys[None, :, None]
        nodes[2, 3:-3, 3:-3, 3:-3] = zs[:, None, None]
        xc, yc = 0.5 * (xs[1:] + xs[:-1]) + 0.05 * length, 0.5 * (ys[1:] + ys[:-1])
        delta = 0.37 * xc * (c.rho_inf * c.vel_mag * xc / c.mu_ref) ** -0.2
        q[(1,) + INNER] = c.u_inf * np.minimum(1.0, (yc[:, None] / delta[None, :]) ** (1.0 / 7.0))[None]
        _noise(c, q, rng, 0.01)
    return c, nodes, q, kind in ("bump", "plate")


class _OnDevice:
    """A resident array of a block as a tensor; holds the block alive."""

    def __init__(self, block, name, shape):
        ptr, _ = block.device_ptr(name)
        self.block = block
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f8", "data": (ptr, False), "version": 3,
                                         "strides": None}


def _view(block, name):
    return torch.as_tensor(_OnDevice(block, name, block.shape_of(name)), device="cuda")


def prepare(case, seed):
    if case["kind"] == "chain":
        # the layout of the blocks belongs to the case, the state to the seed
        blocks, links = C.chain_blocks(case["blocks"], case["lo"], case["hi"])
        rng = np.random.default_rng(seed)
        made = []
        for c, nodes, _ in blocks:
            g = GpuBlock(c, precision=int(case["fp32"]))
            g.set_grid(nodes)
            g.upload_state(_noise(c, C.freestream_state(c), rng, 0.01))
            made.append(g)
        group = GpuGroup(made, links)
        group.set_option("batched", 1)
        return {"what": "group", "group": group, "it": 1, "out": {"qp": [_view(g, "qp") for g in made]}}
    c, nodes, q, walls = _block_inputs(case, seed)
    g = GpuBlock(c, precision=int(case["fp32"]))
    g.set_grid(nodes, wall_dist=walls)
    g.upload_state(q)
    out = {"qp": _view(g, "qp")}
    if not case["fp32"]:
        out["residue"] = _view(g, "residue")
    state = {"what": case["time"], "block": g, "it": 1, "out": out}
    if case["time"] == "adjoint":
        state["w"] = np.random.default_rng(seed + 1).uniform(-1.0, 1.0, g.shape_of("residue"))
    elif case["time"] != "residual":
        state["what"] = "step"
    return state


def run(state):
    what = state["what"]
    if what == "group":
        state["group"].get_next_solution(state["it"])
        state["it"] += 1
        return state["out"]
    if what == "adjoint":
        return {"bar_qp": state["block"].vjp(state["w"])}
    if what == "residual":
        state["block"].residual(1)
        return state["out"]
    state["block"].get_next_solution(state["it"])
    state["it"] += 1
    if "residue" not in state["out"]:
        return state["out"]
    return dict(state["out"], norms=state["block"].resnorm())


def work(case):
    """Per residual evaluation and cell: the state in and out, the RK base,
    three owned faces (area and normal), volume, centre, time step and, with a
    turbulence model, the wall distance; the adjoint reads w and the state and
    writes the state's adjoint.  Operations are rounded counts of the
    reconstruction, the flux, the viscous terms and the closures."""
    if case["kind"] == "chain":
        blocks, _ = _extents(case)
        cells = sum(a * b * c for a, b, c in blocks)
    else:
        cells = case["ni"] * case["nj"] * case["nk"]
    nv = {"none": 5, "sa": 6}.get(case["turb"], 7)
    viscous = case["kind"] != "euler"
    faces = 2 if case.get("nk") == 1 else 3
    recon = {"muscl": 60, "ppm": 40, "weno": 150}[case["recon"]]
    flops = faces * (nv * recon + 130 + (30 * nv if viscous else 0)) + (60 * nv if viscous else 0) + 20 * nv
    values = 3 * nv + 12 + 1 + (3 if viscous else 0) + 1 + (1 if case["turb"] != "none" else 0)
    stages = {"RK4": 4, "RK2": 2, "TVDRK3": 3}.get(case["time"], 1)
    if case["time"] == "adjoint":
        return {"bytes": 8.0 * cells * (3 * nv + 12), "flops": 4.0 * cells * flops}
    if case["time"] == "implicit":
        values += 2 * 2 * nv  # the sweep values written and read by each sweep
        flops += 2 * 3 * 250
    return {"bytes": 8.0 * cells * stages * values, "flops": float(cells * stages * flops)}


def _extents(case):
    """The cell counts of a chain's blocks, as chain_blocks draws them."""
    u = C.splitmix_uniform(3, 3 + case["blocks"])
    span = case["hi"] - case["lo"]
    pick = [int(case["lo"] + min(span, int(v * (span + 1)))) for v in u]
    sizes = [pick[:3]]
    for b in range(1, case["blocks"]):
        e = list(sizes[-1])
        e[(b - 1) % 3] = pick[3 + b]
        sizes.append(e)
    return sizes, None


# ---------------------------------------------------- the values in 64 bits
def _gt(a, b):
    return torch.where(a > b, a, b)


def _lt(a, b):
    return torch.where(a < b, a, b)


def _sgn(x):
    return torch.copysign(torch.ones_like(x), x)


class _Plain:
    """The explicit step of one three-dimensional block (inviscid, laminar,
    SST) written with whole-array operations in float64.  Arrays are
    [variable,] k, j, i with two cells of offset (cell i at index i + 2)."""

    def __init__(self, c, nodes, walls):
        self.c, self.dev = c, "cuda" if torch.cuda.is_available() else "cpu"
        self.N = (c.imx, c.jmx, c.kmx)
        self.sst = c.turb == "sst"
        self.ng = 6 if self.sst else 4
        x = torch.tensor(nodes, device=self.dev)
        for d in range(3):
            n, dim = self.N[d], 3 - d
            for g in (2, 1, 0):
                x.select(dim, g).copy_(2 * x.select(dim, g + 1) - x.select(dim, g + 2))
            for g in (n + 3, n + 4, n + 5):
                x.select(dim, g).copy_(2 * x.select(dim, g - 1) - x.select(dim, g - 2))

        def at(di, dj, dk, along=None):
            """Nodes moved by (di, dj, dk), cut to the cells (along: to the faces of a direction)."""
            v = x
            for d, o in enumerate((di, dj, dk)):
                if d != along:
                    v = v.narrow(3 - d, o, v.shape[3 - d] - 1)
            return v

        self.A, self.n = [], []
        for d in range(3):
            p = {0: ((0, 1, 1), (0, 0, 1), (0, 1, 0)), 1: ((1, 0, 1), (1, 0, 0), (0, 0, 1)),
                 2: ((1, 1, 0), (0, 1, 0), (1, 0, 0))}[d]
            s = 0.5 * torch.linalg.cross(at(*p[0], along=d) - at(0, 0, 0, along=d), at(*p[1], along=d) - at(*p[2], along=d),
                                         dim=0)
            area = s.square().sum(0).sqrt()
            self.A.append(area)
            self.n.append(s / torch.where(area == 0, torch.ones_like(area), area))
        corner = [at(*o) for o in ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))]

        def tet(a, b, e, f):
            a, b, e, f = corner[a], corner[b], corner[e], corner[f]
            return -((f - a) * torch.linalg.cross(b - a, e - a, dim=0)).sum(0) / 6.0

        v1 = tet(0, 4, 7, 5) + tet(6, 7, 5, 2) + tet(7, 3, 0, 2) + tet(5, 0, 2, 7) + tet(0, 1, 5, 2)
        v2 = tet(1, 5, 4, 6) + tet(7, 4, 6, 3) + tet(4, 0, 1, 3) + tet(6, 1, 3, 4) + tet(1, 2, 6, 3)
        self.vol = torch.maximum(v1, v2)
        self.ctr = 0.125 * sum(corner)
        self.dist = torch.ones_like(self.vol)
        if walls:
            w = []
            for f in range(6):
                if c.bc_id[f] == -5:
                    real = x[:, 3:-3, 3:-3, 3:-3].select(3 - f // 2, -1 if f & 1 else 0)
                    w.append(real.reshape(3, -1))
            # the reference's surface-node file holds eleven digits
            w = torch.cat(w, 1).cpu().numpy()
            w = torch.tensor([[float("%.10E" % v) for v in row] for row in w], dtype=torch.float64, device=self.dev)
            p = x.reshape(3, -1)
            near = torch.empty(p.shape[1], dtype=torch.float64, device=self.dev)
            step = max(1, (1 << 28) // w.shape[1])
            for s in range(0, p.shape[1], step):
                q = p[:, s: s + step]
                near[s: s + step] = sum((q[a][:, None] - w[a][None, :]).square_() for a in range(3)).amin(1)
            x = near.sqrt_().reshape((1,) + x.shape[1:])
            self.dist = sum(at_[0] for at_ in (x[:, dk: x.shape[1] - 1 + dk, dj: x.shape[2] - 1 + dj, di: x.shape[3] - 1 + di]
                                               for di in (0, 1) for dj in (0, 1) for dk in (0, 1))) * 0.125
        self.mu = torch.full_like(self.vol, c.mu_ref)
        self.mut, self.f1 = torch.zeros_like(self.vol), torch.zeros_like(self.vol)

    # -- ghost cells
    def layer(self, v, f, L):
        """The plane of layer L (1 the first cell, 0 the first ghost) of face f, interior columns."""
        d = f >> 1
        s = v.select(v.dim() - 1 - d, (self.N[d] - L if f & 1 else L) + 2)
        return s[..., 3:-3, 3:-3]

    def bnormal(self, f, d):
        """The stored normal (of direction d's faces) at face f's first face plane."""
        dim = f >> 1
        return self.n[d].select(3 - dim, (self.N[dim] if f & 1 else 1) + 2)[:, 3:3 + self.span(f)[1], 3:3 + self.span(f)[0]]

    def span(self, f):
        """The interior columns of face f along its first and second tangent."""
        d = f >> 1
        return [(self.N[a] - 1) for a in range(3) if a != d]

    def ghosts(self, q, it):
        c = self.c
        a2, a3 = 1.0 + c.accur, 0.5 * c.accur
        a1 = a2 - a3

        def symm(l, f):
            for g in range(3):
                self.layer(q[l], f, -g).copy_((a2 * self.layer(q[l], f, g + 1) - a3 * self.layer(q[l], f, g + 2)) / a1)

        def anti(l, f):
            for g in range(3):
                self.layer(q[l], f, -g).copy_(-self.layer(q[l], f, g + 1))

        def flat(l, f):
            for g in range(3):
                self.layer(q[l], f, -g).copy_(self.layer(q[l], f, 1).clone())

        def fixed(l, f, v):
            for g in range(3):
                self.layer(q[l], f, -g).fill_(v)

        values = [c.fix_rho, c.fix_u, c.fix_v, c.fix_w, c.fix_p, c.fix_tk, c.fix_tw]
        turb = range(5, q.shape[0])
        for f in range(6):
            id_, d, hi, N = c.bc_id[f], f >> 1, f & 1, self.N[f >> 1]
            if id_ == -3:
                if it <= 2:
                    for l in [0, 1, 2, 3, *turb]:
                        fixed(l, f, values[l][f])
                flat(4, f)
            elif id_ == -4:
                for l in [0, 1, 2, 3, *turb]:
                    flat(l, f)
                if it <= 2:
                    fixed(4, f, c.fix_p[f])
            elif id_ == -5:
                symm(4, f)
                tw = c.fix_twall[f]
                if tw > 1.0:
                    for g in range(3):
                        at = self.layer(q[4], f, 1 + g) / (c.R_gas * self.layer(q[0], f, 1 + g))
                        self.layer(q[0], f, -g).copy_(self.layer(q[4], f, -g) / (c.R_gas * (2 * tw - at)))
                else:
                    symm(0, f)
                for l in (1, 2, 3):
                    anti(l, f)
                if self.sst:
                    anti(5, f)
                    r0, r1, p0, p1 = (self.layer(q[l], f, L) for l in (0, 4) for L in (0, 1))
                    t = 0.5 * (p0 / r0 + p1 / r1) / c.R_gas
                    mu = c.mu_ref * (t / c.T_ref) ** 1.5 * ((c.T_ref + c.S_ref) / (t + c.S_ref))
                    ww = 120 * mu / (0.5 * (r0 + r1) * 0.075 * (2 * self.layer(self.dist, f, 1)) ** 2)
                    for g in range(3):
                        self.layer(q[6], f, -g).copy_(ww - self.layer(q[6], f, g + 1))
            elif id_ == -6:
                for l in (0, 4):
                    symm(l, f)
                n, r = self.bnormal(f, d), self.bnormal(f, 0)
                for g in range(3):
                    u = [self.layer(q[l], f, g + 1).clone() for l in (1, 2, 3)]
                    dot = u[0] * n[0] + u[1] * n[1] + u[2] * n[2]
                    for l in range(3):
                        self.layer(q[1 + l], f, -g).copy_(u[l] - 2.0 * dot * r[l])
            elif id_ == -8:
                n = self.bnormal(f, d)
                n = n if hi else -n
                s = [self.layer(q[l], f, 1).clone() for l in range(5)]
                gm = c.gm
                cinf = math.sqrt(gm * c.p_inf / c.rho_inf)
                un = s[1] * n[0] + s[2] * n[1] + s[3] * n[2]
                uinf = c.u_inf * n[0] + c.v_inf * n[1] + c.w_inf * n[2]
                low, high = uinf - 2 * cinf / (gm - 1), un + 2 * (gm * s[4] / s[0]).sqrt() / (gm - 1)
                ub, cb = 0.5 * (high + low), 0.25 * (gm - 1) * (high - low)
                out = ub > 0
                new = [None] * 5
                for l, inf in ((1, c.u_inf), (2, c.v_inf), (3, c.w_inf)):
                    new[l] = torch.where(out, s[l] + (ub - un) * n[l - 1], inf + (ub - uinf) * n[l - 1])
                sen = torch.where(out, s[4] / s[0] ** gm, torch.full_like(ub, c.p_inf / c.rho_inf ** gm))
                new[0] = (cb * cb / (gm * sen)) ** (1.0 / (gm - 1))
                new[4] = new[0] * cb * cb / gm
                for l in range(5):
                    self.layer(q[l], f, 0).copy_(new[l])
                for l in turb:
                    flat(l, f) if bool(out[-1, -1]) else fixed(l, f, values[l][f])
                for L in (1, 2):  # the outer layers copy the first over the whole plane
                    at = (N + L if hi else -L) + 2
                    q.select(3 - d, at).copy_(q.select(3 - d, (N if hi else 0) + 2).clone())
            elif id_ == -9:
                for g in range(3):
                    to, src = (N + g, 1 + g) if hi else (-2 + g, N - 3 + g)
                    q.select(3 - d, to + 2).copy_(q.select(3 - d, src + 2).clone())
        I, J, K = (n + 2 for n in self.N)
        for j, jn in ((2, 3), (J, J - 1)):
            for k, kn in ((2, 3), (K, K - 1)):
                q[:, k, j].copy_(0.33 * (q[:, kn, jn] + q[:, kn, j] + q[:, k, jn]))
        for i, n in ((2, 3), (I, I - 1)):
            for j, jn in ((2, 3), (J, J - 1)):
                q[:, :, j, i].copy_(0.33 * (q[:, :, jn, n] + q[:, :, j, n] + q[:, :, jn, i]))
        for i, n in ((2, 3), (I, I - 1)):
            for j, jn in ((2, 3), (J, J - 1)):
                for k, kn in ((2, 3), (K, K - 1)):
                    q[:, k, j, i].copy_(0.33 * (q[:, k, j, n] + q[:, k, jn, i] + q[:, kn, j, i]))

    # -- face states
    def muscl(self, a, b, e, sw, edge):
        fd, bd = e - b, b - a
        eps = 0.0 if edge else 1e-14

        def psi(x, y):
            r = x / (y + eps * _sgn(y)) if eps else x / y
            mid = (2 + r) / 3.0 if edge else (2.0 / 3.0) * (r - 1.0) + 1.0
            lim = _lt(_lt(2 * r, mid), torch.full_like(r, 2.0))
            return 1 - (1 - torch.where(lim < 0, torch.zeros_like(lim), lim)) * sw

        p1, p2 = psi(fd, bd), psi(bd, fd)
        third = 1.0 / 3.0
        return (b + 0.25 * ((1 - third) * p1 * bd + (1 + third) * p2 * fd),
                b - 0.25 * ((1 + third) * p1 * bd + (1 - third) * p2 * fd))

    @staticmethod
    def weno(a, b, m, e, f):
        """The face value of cell m on the side of e, f."""
        b1 = 13.0 / 12.0 * (a - 2 * b + m) ** 2 + 0.25 * (a - 4 * b + 3 * m) ** 2
        b2 = 13.0 / 12.0 * (b - 2 * m + e) ** 2 + 0.25 * (b - e) ** 2
        b3 = 13.0 / 12.0 * (m - 2 * e + f) ** 2 + 0.25 * (3 * m - 4 * e + f) ** 2
        w1, w2, w3 = 0.1 / (1e-6 + b1) ** 2, 0.6 / (1e-6 + b2) ** 2, 0.3 / (1e-6 + b3) ** 2
        return (w1 * (2 * a - 7 * b + 11 * m) + w2 * (-b + 5 * m + 2 * e) + w3 * (2 * m + 5 * e - f)) / (6 * (w1 + w2 + w3))

    @staticmethod
    def ppm(q, lo, hi, limit):
        """The limited lower- and upper-face values of a cell."""
        if not limit:
            return lo, hi
        ext = (hi - q) * (q - lo) <= 0
        d, d6 = hi - lo, 6.0 * (q - 0.5 * (lo + hi))
        over, under = d * d6 > d * d, -d * d > d * d6
        return (torch.where(ext, q, torch.where(over, 3 * q - 2 * hi, lo)),
                torch.where(ext, q, torch.where(~over & under, 3 * q - 2 * lo, hi)))

    def faces(self, q, d):
        c, N, dim = self.c, self.N[d], 3 - d
        cut = [slice(None)] * 4
        for a in range(3):
            if a != d:
                cut[3 - a] = slice(3, -3)
        v = q[tuple(cut)]
        w = [v.narrow(dim, m, N) for m in range(6)]
        sw = torch.tensor([c.lim[d]] * 5 + [c.tlim[d]] * (q.shape[0] - 5), dtype=torch.float64, device=q.device)
        sw = sw.reshape(-1, 1, 1, 1)
        if c.recon == "muscl":
            L, R = self.muscl(w[1], w[2], w[3], sw, False)[0], self.muscl(w[2], w[3], w[4], sw, False)[1]
        elif c.recon == "weno":
            L, R = self.weno(*w[:5]), self.weno(w[5], w[4], w[3], w[2], w[1])
        else:
            f = [(7.0 * (w[m] + w[m - 1]) - (w[m + 1] + w[m - 2])) / 12.0 for m in (2, 3, 4)]
            L = self.ppm(w[2], f[0], f[1], c.lim[d] == 1)[1]
            R = self.ppm(w[3], f[1], f[2], c.lim[d] == 1)[0]
        L, R = L.clone(), R.clone()
        at = lambda n: [w[m].select(dim, n - 1) for m in range(6)]  # noqa: E731
        one = sw[..., 0]
        first, last = c.bc_id[2 * d], c.bc_id[2 * d + 1]
        edge = c.recon != "muscl"
        x, y, y2, x2 = at(1), at(N), at(N - 1), at(2)
        gmin, gmax = first in (-8, -9), last in (-8, -9)
        if edge:
            L.select(dim, 1).copy_(self.muscl(x2[1], x2[2], x2[3], one, True)[0])
            R.select(dim, N - 2).copy_(self.muscl(y2[2], y2[3], y2[4], one, True)[1])
        if gmax:
            L.select(dim, N - 1).copy_(y[3])
        elif edge:
            L.select(dim, N - 1).copy_(self.muscl(y[1], y[2], y[3], one, True)[0])
        if gmin:
            R.select(dim, 0).copy_(x[2])
        elif edge:
            R.select(dim, 0).copy_(self.muscl(x[2], x[3], x[4], one, True)[1])
        L.select(dim, 0).copy_(x[2] if gmin else 0.5 * (x[2] + x[3]))
        R.select(dim, N - 1).copy_(y[3] if gmax else 0.5 * (y[2] + y[3]))
        return L, R

    def flux(self, L, R, n, A, shut):
        c, gm = self.c, self.c.gm
        (rL, uL, vL, wL, pL), (rR, uR, vR, wR, pR) = L[:5], R[:5]
        hL = 0.5 * (uL * uL + vL * vL + wL * wL) + gm / (gm - 1) * pL / rL
        hR = 0.5 * (uR * uR + vR * vR + wR * wR) + gm / (gm - 1) * pR / rR
        nL, nR = uL * n[0] + vL * n[1] + wL * n[2], uR * n[0] + vR * n[1] + wR * n[2]
        sound = 0.5 * ((gm * pL / rL).sqrt() + (gm * pR / rR).sqrt())
        if c.flux in ("ausmP", "slau"):
            if c.flux == "ausmP":
                cs = (2 * (gm - 1) * 0.5 * (hL + hR) / (gm + 1)).sqrt()
                C_ = _lt(cs * cs / _gt(cs, nL.abs()), cs * cs / _gt(cs, nR.abs()))
            else:
                C_ = sound
            mL, mR = nL / C_, nR / C_
            aL, aR = (mL.abs() < 1).double(), (mR.abs() < 1).double()
            upL, upR = 0.5 * (1 + _sgn(mL)) * (1 - aL), 0.5 * (1 - _sgn(mR)) * (1 - aR)
            bL = upL + aL * 0.25 * (1 + mL) ** 2 * (2 - mL)
            bR = upR + aR * 0.25 * (1 - mR) ** 2 * (2 + mR)
            if c.flux == "ausmP":
                m = upL * mL + aL * (0.25 * (1 + mL) ** 2 + 0.125 * (mL * mL - 1) ** 2)
                m = m + upR * mR - aR * (0.25 * (1 - mR) ** 2 + 0.125 * (mR * mR - 1) ** 2)
                bL = bL + aL * 0.1875 * (mL * mL - 1) ** 2 * mL
                bR = bR - aR * 0.1875 * (mR * mR - 1) ** 2 * mR
                p, mass = bL * pL + bR * pR, torch.where(m > 0, m * C_ * rL, m * C_ * rR)
            else:
                vt = (0.5 * (uL * uL + vL * vL + wL * wL + uR * uR + vR * vR + wR * wR)).sqrt()
                xi = (1 - _lt(torch.ones_like(vt), vt / C_)) ** 2
                va = (rL * nL.abs() + rR * nR.abs()) / (rL + rR)
                zero, unit = torch.zeros_like(mL), torch.ones_like(mL)
                g = -_gt(_lt(mL, zero), -unit) * _lt(_gt(mR, zero), unit)
                p = 0.5 * ((pL + pR) + (bL - bR) * (pL - pR) + (1 - xi) * (bL + bR - 1) * (pL + pR))
                mass = 0.5 * (rL * (nL + (1 - g) * va + g * nL.abs()) + rR * (nR - (1 - g) * va - g * nR.abs()) -
                              xi * (pR - pL) / C_)
            mass = mass * shut
            fp, fm = 0.5 * (mass + mass.abs()), 0.5 * (mass - mass.abs())
            out = [fp + fm] + [fp * L[l] + fm * R[l] + p * n[l - 1] for l in (1, 2, 3)] + [fp * hL + fm * hR]
        else:
            mL, mR = nL / sound, nR / sound
            ap, am = 0.5 * (1 + _sgn(mL)), 0.5 * (1 - _sgn(mR))
            bl, br = -(mL.abs() < 1).double(), -(mR.abs() < 1).double()
            sL, sR = 0.25 * (1 + mL) ** 2, 0.25 * (1 - mR) ** 2
            cp, cm = ap * (1 + bl) * mL - bl * sL, am * (1 + br) * mR + br * sR
            dp, dm = ap * (1 + bl) - bl * sL * (2 - mL), am * (1 + br) - br * sR * (2 + mR)
            if c.flux == "ldfss0":
                ml = 0.25 * bl * br * ((0.5 * (mL * mL + mR * mR)).sqrt() - 1) ** 2
                cp = cp - ml * (1 - (pL - pR) / (2 * rL * sound ** 2))
                cm = cm + ml * (1 - (pL - pR) / (2 * rR * sound ** 2))
            fp, fm = rL * sound * cp * shut, rR * sound * cm * shut
            out = [fp + fm] + [fp * L[l] + dp * pL * n[l - 1] + fm * R[l] + dm * pR * n[l - 1] for l in (1, 2, 3)]
            out += [fp * hL + fm * hR]
        out += [fp * L[l] + fm * R[l] for l in range(5, L.shape[0])]
        return torch.stack(out) * A, sound

    # -- gradients, viscosities, viscous fluxes
    def cells(self, v, *shift):
        """Cells 0..N of each direction, moved by `shift` along (i, j, k)."""
        for d in range(3):
            v = v.narrow(v.dim() - 1 - d, 2 + shift[d], self.N[d] + 1)
        return v

    def facing(self, v, d, up):
        """The lower (up: upper) face of direction d of the cells 0..N."""
        return self.cells(v, *[int(up and a == d) for a in range(3)])

    def gradients(self, q, temp):
        c = self.c
        var = torch.cat([q[1:4], temp[None], q[5:7]]) if self.sst else torch.cat([q[1:4], temp[None]])
        mid, g = self.cells(var, 0, 0, 0), 0
        for up in (False, True):
            for d in range(3):
                s = [0, 0, 0]
                s[d] = 1 if up else -1
                an = self.facing(self.n[d], d, up) * self.facing(self.A[d], d, up)
                g = g + (1 if up else -1) * (self.cells(var, *s) + mid)[:, None] * an[None]
        g = g / (2 * self.cells(self.vol, 0, 0, 0))
        rho, p = self.cells(q[0], 0, 0, 0), self.cells(q[4], 0, 0, 0)
        mu = self.cells(self.mu, 0, 0, 0)
        if c.mu_sutherland:
            t = p / (rho * c.R_gas)
            mu.copy_(c.mu_ref * (t / c.T_ref) ** 1.5 * ((c.T_ref + c.S_ref) / (t + c.S_ref)))
        src = None
        if self.sst:
            k, w, dist = self.cells(q[5], 0, 0, 0), self.cells(q[6], 0, 0, 0), self.cells(self.dist, 0, 0, 0)
            bs, s2 = 0.09, 0.856
            v1, v2 = k.clamp(min=0).sqrt() / (bs * w * dist), 500 * (mu / rho) / (dist * dist * w)
            vort = ((g[2, 1] - g[1, 2]) ** 2 + (g[0, 2] - g[2, 0]) ** 2 + (g[1, 0] - g[0, 1]) ** 2).sqrt()
            F2 = torch.tanh(_gt(2 * v1, v2) ** 2)
            self.cells(self.mut, 0, 0, 0).copy_(rho * 0.31 * k / _gt(0.31 * w, vort * F2).clamp(min=1e-20))
            cd = (2 * rho * s2 * (g[4] * g[5]).sum(0) / w).clamp(min=1e-20)
            F1 = torch.tanh(_lt(_gt(v1, v2), 4 * rho * s2 * k / (cd * dist * dist)) ** 4)
            self.cells(self.f1, 0, 0, 0).copy_(F1)
            mut, vol = self.cells(self.mut, 0, 0, 0), self.cells(self.vol, 0, 0, 0)
            g1, g2 = 0.075 / bs - 0.5 * 0.41 ** 2 / math.sqrt(bs), 0.0828 / bs - s2 * 0.41 ** 2 / math.sqrt(bs)
            dk, dw = bs * rho * w * k, (0.075 * F1 + 0.0828 * (1 - F1)) * rho * w * w
            pk = _lt(mut * vort ** 2 - 2.0 / 3.0 * rho * k * (g[0, 0] + g[1, 1] + g[2, 2]), 20 * dk)
            pw = rho * (g1 * F1 + g2 * (1 - F1)) / mut * pk
            src = torch.stack([(pk - dk) * vol, (pw - dw + (1 - F1) * cd) * vol])[:, 1:-1, 1:-1, 1:-1]
        # ghost cells: the normal part from the face's two cells; J and K
        # metrics are taken at the I-face offset of the reference
        for f in range(6):
            d, hi, id_ = f >> 1, f & 1, c.bc_id[f]
            N = self.N[d]
            idx = [torch.arange(1, self.N[a], device=self.dev) for a in range(3)]
            idx[d] = torch.tensor([N if hi else 1], device=self.dev)
            i, j, k = idx[0][None, None, :] + 2, idx[1][None, :, None] + 2, idx[2][:, None, None] + 2
            off = (i + (c.imx + 6) * (j + (c.jmx + 5) * k)).squeeze(2 - d)
            nrm, A = self.n[d].reshape(3, -1)[:, off], self.A[d].reshape(-1)[off]
            coef = A * nrm / self.layer(self.vol, f, 1)
            dq = self.layer(var, f, 1) - self.layer(var, f, 0)
            cut = [slice(None), slice(None), slice(1, -1), slice(1, -1), slice(1, -1)]
            cut[4 - d] = N - 1 if hi else 1
            gi = g[tuple(cut)]
            o = (-1 if hi else 1) * dq[:, None] * coef[None]
            if id_ == -5 and 0 <= c.fix_twall[f] < 1:
                o[3] = -gi[3]
            cut[4 - d] = N if hi else 0
            g[tuple(cut)] = o + gi - (gi * nrm[None]).sum(1, keepdim=True) * nrm[None]
            if self.sst:
                self.layer(self.mut, f, 0).copy_((-1 if id_ == -5 else 1) * self.layer(self.mut, f, 1))
                self.layer(self.f1, f, 0).copy_(self.layer(self.f1, f, 1))
        return g, src

    def viscous(self, q, g, d, n, A):
        c, N, dim = self.c, self.N[d], 2 - d

        def pair(v):
            """A padded array at the cells below and above the faces."""
            for a in range(3):
                v = v.narrow(v.dim() - 1 - a, 2 if a == d else 3, self.N[a] + (1 if a == d else -1))
            m = v.shape[v.dim() - 1 - d] - 1
            return v.narrow(v.dim() - 1 - d, 0, m), v.narrow(v.dim() - 1 - d, 1, m)

        def mean(v):
            a, b = pair(v)
            return 0.5 * (a + b)

        lo, up = pair(self.ctr)
        dx = up - lo
        gc = g[(slice(None), slice(None)) + tuple(slice(None) if 2 - a == d else slice(1, -1) for a in range(3))]
        gc = 0.5 * (gc.narrow(dim + 2, 0, N) + gc.narrow(dim + 2, 1, N))
        temp = q[4] / (q[0] * c.R_gas)
        var = torch.cat([q[1:4], temp[None], q[5:7]]) if self.sst else torch.cat([q[1:4], temp[None]])
        lo, up = pair(var)
        gc = gc + ((up - lo - (gc * dx[None]).sum(1)) / dx.square().sum(0))[:, None] * dx[None]
        mu, mut = mean(self.mu), mean(self.mut)
        t = mu + mut
        grad, vel = gc[:3], mean(q[1:4])
        div = (grad[0, 0] + grad[1, 1] + grad[2, 2]) / 3.0
        tau = t * (grad + grad.transpose(0, 1))
        for a in range(3):
            tau[a, a] = tau[a, a] - 2 * t * div
        tn = (tau * n[None]).sum(1)
        heat = (mu / c.Pr + mut / c.tPr) * c.gm * c.R_gas / (c.gm - 1)
        out = [torch.zeros_like(mu), tn[0], tn[1], tn[2], (tn * vel).sum(0) + heat * (gc[3] * n).sum(0)]
        if self.sst:
            F1 = mean(self.f1)
            kk = -2.0 / 3.0 * mean(q[0]) * mean(q[5])
            for a in range(3):
                out[1 + a] = out[1 + a] + kk * n[a]
            kf = (mu + (0.85 * F1 + 1 - F1) * mut) * (gc[4] * n).sum(0)
            out[4] = out[4] + kf
            out += [kf, (mu + (0.5 * F1 + 0.856 * (1 - F1)) * mut) * (gc[5] * n).sum(0)]
        return torch.stack(out) * A

    def residual(self, q, temp, it):
        """The residue of the interior cells; fills q's ghost cells."""
        c = self.c
        self.ghosts(q, it)
        g = src = None
        if c.mu_ref != 0:
            g, src = self.gradients(q, temp)
        res, self.sound, self.mass = 0, [], 0
        for d in range(3):
            N = self.N[d]
            cut = tuple(slice(3, 3 + N) if 2 - a == d else slice(3, -3) for a in range(3))
            n, A = self.n[d][(slice(None),) + cut], self.A[d][cut]
            L, R = self.faces(q, d)
            shut = torch.ones_like(A)
            for at, id_ in ((0, c.bc_id[2 * d]), (N - 1, c.bc_id[2 * d + 1])):
                if id_ in (-5, -6, -7):
                    shut.select(2 - d, at).zero_()
            F, s = self.flux(L, R, n, A, shut)
            if g is not None:
                F = F - self.viscous(q, g, d, n, A)
            self.sound.append(s)
            res = res + F.narrow(3 - d, 1, N - 1) - F.narrow(3 - d, 0, N - 1)
            self.mass = self.mass + (F[0].select(2 - d, 0).sum() - F[0].select(2 - d, N - 1).sum())
        if src is not None:
            res = torch.cat([res[:5], res[5:] - src])
        return res

    def time_step(self, q):
        c, tot = self.c, 0
        vol = self.vol[INNER]
        visc = [0, 0]
        cells = [slice(3, -3)] * 3

        def moved(v, d, o):
            s = list(cells)
            s[2 - d] = slice(3 + o, v.shape[v.dim() - 1 - d] - 3 + o)
            return v[(Ellipsis, *s)]

        for d in range(3):
            for up in (0, 1):
                sf = [slice(3, 3 + self.N[2 - a] - 1) for a in range(3)]
                sf[2 - d] = slice(3 + up, 3 + up + self.N[d] - 1)
                n, A = self.n[d][(slice(None), *sf)], self.A[d][tuple(sf)]
                qq = moved(q, d, up)
                tot = tot + A * ((qq[1:4] * n).sum(0).abs() + self.sound[d].narrow(2 - d, up, self.N[d] - 1))
                if c.mu_ref != 0:
                    gap = ((moved(self.ctr, d, up - 1) - moved(self.ctr, d, up)) * n).sum(0).abs()
                    for a, m in enumerate((self.mu, self.mut)):
                        visc[a] = visc[a] + A * moved(m, d, up) / (qq[0] * gap)
        dt = c.CFL * vol / tot
        if c.mu_ref != 0:
            for a in range(2 if self.sst else 1):
                dt = c.CFL * vol * 2.0 / (c.gm * visc[a] / (c.tPr if a else c.Pr) + 2 * c.CFL * vol / dt)
        return dt if c.time_local else torch.full_like(dt, float(dt.min()))

    def step(self, q, it):
        """One RK4 step in place; returns the last residue."""
        c, gm = self.c, self.c.gm
        temp, base, acc, dt = q[4] / (c.R_gas * q[0]), q.clone(), 0, None
        b = base[(slice(None),) + INNER]
        u1 = b * b[:1]
        u1[0] = b[0]
        u1[4] = b[4] / (gm - 1) + 0.5 * (u1[1] ** 2 + u1[2] ** 2 + u1[3] ** 2) / b[0]
        for s, (tf, sf) in enumerate(((0.5, 1.0), (0.5, 2.0), (1.0, 2.0), (1.0 / 6.0, 1.0))):
            res = self.residual(q, temp, it)
            dt = self.time_step(q) if dt is None else dt
            r = res.clone()
            if self.sst:
                F1, w = self.f1[INNER], q[6][INNER]
                beta = 0.075 * F1 + 0.0828 * (1 - F1)
                r[5], r[6] = r[5] / (1 + beta * w * dt), r[6] / (1 + 2 * beta * w * dt)
            acc = acc + sf * r
            u = u1 - (acc if s == 3 else r) * tf * dt / self.vol[INNER]
            new = u / u[:1]
            new[0] = u[0]
            new[4] = (gm - 1) * (u[4] - 0.5 * (u[1] ** 2 + u[2] ** 2 + u[3] ** 2) / u[0])
            q[:5, 3:-3, 3:-3, 3:-3] = new[:5]
            for l in range(5, q.shape[0]):
                q[(l,) + INNER] = torch.where(new[l] >= 0, new[l], q[(l,) + INNER])
        return res

    def norms(self, res):
        c, v = self.c, self.c.vel_mag
        scale = [c.rho_inf * v] + [c.rho_inf * v * v] * 3
        scale += [0.5 * c.rho_inf * v ** 3 + c.gm / (c.gm - 1) * c.p_inf, c.rho_inf * v * c.tk_inf, c.rho_inf * v * c.tw_inf]
        return np.array([abs(float(self.mass))] + [float(r.square().sum().sqrt()) / s for r, s in zip(res, scale)])


def exact(case, seed):
    """The values of one pass.  None where there is no short whole-array form:
    groups (exchange maps), the implicit sweeps (a recurrence over the cells),
    2-D grids' own rules, the other turbulence models and integrators; and the
    adjoint of the reconstructions whose boundary cells divide by zero
    differences (automatic differentiation returns NaN there)."""
    if case["kind"] == "chain" or case["turb"] not in ("none", "sst") or case["nk"] == 1:
        return None
    if case["time"] not in ("RK4", "residual", "adjoint"):
        return None
    if case["time"] == "adjoint" and case["recon"] != "muscl":
        return None
    c, nodes, q, walls = _block_inputs(case, seed)
    p = _Plain(c, nodes, walls)
    q = torch.tensor(q, device=p.dev)
    if case["time"] == "adjoint":
        w = torch.tensor(np.random.default_rng(seed + 1).uniform(-1.0, 1.0, (5, c.kmx - 1, c.jmx - 1, c.imx - 1)),
                         device=p.dev)
        inner = q[(slice(None),) + INNER].clone().requires_grad_()
        full = torch.zeros_like(q) + q
        full[(slice(None),) + INNER] = inner
        res = p.residual(full, None, 1)
        bar = torch.zeros_like(q)
        bar[(slice(None),) + INNER] = torch.autograd.grad((res * w).sum(), inner)[0]
        return {"bar_qp": bar}
    with torch.no_grad():
        if case["time"] == "residual":
            res = p.residual(q, q[4] / (c.R_gas * q[0]), 1)
            return {"qp": q, "residue": res}
        res = p.step(q, 1)
        return {"qp": q} if case["fp32"] else {"qp": q, "residue": res, "norms": p.norms(res)}
