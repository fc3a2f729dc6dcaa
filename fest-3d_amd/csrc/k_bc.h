// k_bc.h -- ghost-cell boundary conditions (faces in the reference's order
// imin, imax, jmin, jmax, kmin, kmax, those that do not read each other's
// ghosts in one launch), then the edge/corner averages.
// src/boundary/bc_primitive.f90:55-227 and the routines it calls; every face
// kernel gives one thread a column of three ghost cells, which only reads its
// own column, so the passes keep the reference's sequential
// semantics.  The bodies and helpers are here,
// their per-block kernels in k_bc_kernels.h (one translation unit).
#pragma once
// ghost cells and geometry keep the reference's unfused operation order
#pragma clang fp contract(off)
#include "blk.h"

namespace fest {

// cell of layer L (L >= 1 interior counted from the face, L <= 0 ghost) at
// tangential position (a, bb) of a face
__device__ __forceinline__ long fcell(const Blk &b, int face, int L, int a, int bb) {
  switch (face) {
    case 0: return ci(b, L, a, bb);
    case 1: return ci(b, b.imx - L, a, bb);
    case 2: return ci(b, a, L, bb);
    case 3: return ci(b, a, b.jmx - L, bb);
    case 4: return ci(b, a, bb, L);
    default: return ci(b, a, bb, b.kmx - L);
  }
}
__host__ __device__ inline int face_na(const Blk &b, int face) { return face < 2 ? b.jmx : b.imx; }
__host__ __device__ inline int face_nb(const Blk &b, int face) { return face < 4 ? b.kmx : b.jmx; }

enum { CP_ANTI = 0, CP_FLAT = 1, CP_SYMM = 2 };

// boundary id and fixed values of one face, gathered with compile-time
// indices: indexing the by-value kernel argument with a run-time face would
// make the compiler copy the whole argument block to private memory
struct FaceBC {
  int id;
  double fix[FX_N];
};
__device__ __forceinline__ FaceBC face_params(const Blk &b, int face) {
  FaceBC p;
  p.id = b.bc[0];
#pragma unroll
  for (int l = 0; l < FX_N; ++l) p.fix[l] = b.fix[l][0];
#pragma unroll
  for (int f = 1; f < 6; ++f)
    if (face == f) {
      p.id = b.bc[f];
#pragma unroll
      for (int l = 0; l < FX_N; ++l) p.fix[l] = b.fix[l][f];
    }
  return p;
}

__device__ __forceinline__ bool two_eq(const Blk &b) { return b.ng >= 6; }

// unit normal of the boundary face at (a, bb); the metric planes are picked
// per case with constant member indices (a run-time index into the
// by-value argument's pointer arrays would put them in private memory)
__device__ __forceinline__ void bnormal(const Blk &b, int face, int a, int bb, double &nx, double &ny, double &nz) {
  long f;
  const double *px, *py, *pz;
  switch (face) {
    case 0: f = fi(b, 0, 1, a, bb); px = b.fx[0]; py = b.fy[0]; pz = b.fz[0]; break;
    case 1: f = fi(b, 0, b.imx, a, bb); px = b.fx[0]; py = b.fy[0]; pz = b.fz[0]; break;
    case 2: f = fi(b, 1, a, 1, bb); px = b.fx[1]; py = b.fy[1]; pz = b.fz[1]; break;
    case 3: f = fi(b, 1, a, b.jmx, bb); px = b.fx[1]; py = b.fy[1]; pz = b.fz[1]; break;
    case 4: f = fi(b, 2, a, bb, 1); px = b.fx[2]; py = b.fy[2]; pz = b.fz[2]; break;
    default: f = fi(b, 2, a, bb, b.kmx); px = b.fx[2]; py = b.fy[2]; pz = b.fz[2]; break;
  }
  nx = px[f]; ny = py[f]; nz = pz[f];
}

// far-field Riemann state of one column (src/boundary/bc_primitive.f90:645-1234)
// or, when total, the total-pressure inlet (bc_primitive.f90:1237-1776):
// the same Riemann-invariant velocity, then the pressure from the total
// pressure tp and the boundary Mach number and the density from the
// boundary speed of sound.  c is the first interior cell's rho, u, v, w, p
// and nrm the boundary face's stored unit normal (bnormal); returns Unb and,
// when full, the ghost layer 0 state g.  Written for a type T: double, or
// the dual numbers of the adjoint (k_dual.h)
template <typename T>
__device__ __forceinline__ T riemann_state(const Blk &b, int face, const T (&c)[5], const T (&nrm)[3], bool full,
                                           bool total, double tp, T (&g)[5]) {
  const double gm = b.gm;
  T nx = nrm[0], ny = nrm[1], nz = nrm[2];
  if ((face & 1) == 0) { nx = -nx; ny = -ny; nz = -nz; }
  T cexp = sqrt(gm * c[4] / c[0]);
  double cinf = sqrt(gm * b.p_inf / b.rho_inf);
  T Unexp = c[1] * nx + c[2] * ny + c[3] * nz;
  T Uninf = b.u_inf * nx + b.v_inf * ny + b.w_inf * nz;
  T Rinf = Uninf - 2 * cinf / (gm - 1.);
  T Rexp = Unexp + 2 * cexp / (gm - 1.);
  T Unb = 0.5 * (Rexp + Rinf);
  T Cb = 0.25 * (gm - 1.) * (Rexp - Rinf);
  if (!full) return Unb;
  if (Unb > 0.) {
    T vd = Unb - Unexp;
    g[1] = c[1] + vd * nx;
    g[2] = c[2] + vd * ny;
    g[3] = c[3] + vd * nz;
    if (!total) {
      T sen = c[4] / pow(c[0], gm);
      g[0] = pow(Cb * Cb / (gm * sen), 1. / (gm - 1.));
      g[4] = (g[0] * Cb * Cb / gm);
    }
  } else {
    T vd = Unb - Uninf;
    g[1] = b.u_inf + vd * nx;
    g[2] = b.v_inf + vd * ny;
    g[3] = b.w_inf + vd * nz;
    if (!total) {
      double sen = b.p_inf / pow(b.rho_inf, gm);
      g[0] = pow(Cb * Cb / (gm * sen), 1. / (gm - 1.));
      g[4] = (g[0] * Cb * Cb / gm);
    }
  }
  if (total) {
    T Mb = sqrt(g[1] * g[1] + g[2] * g[2] + g[3] * g[3]) / Cb;
    g[4] = tp / pow((1 + 0.5 * (gm - 1.) * Mb * Mb), gm / (gm - 1.));
    g[0] = gm * g[4] / (Cb * Cb);
  }
  return Unb;
}
// Unb of the far-field or total-pressure state at column (a, bb)
__device__ __forceinline__ double riemann_unb(const Blk &b, int face, int a, int bb) {
  const long c1 = fcell(b, face, 1, a, bb);
  double c[5], g[5], nrm[3];
#pragma unroll
  for (int l = 0; l < 5; ++l) c[l] = b.qp[(long)l * b.nc + c1];
  bnormal(b, face, a, bb, nrm[0], nrm[1], nrm[2]);
  return riemann_state(b, face, c, nrm, false, false, 0.0, g);
}

// How a variable's three ghost cells follow from its first four interior
// cells (src/boundary/copy_bc.f90:58-131, bc_primitive.f90:484-525), or not:
// left as they are
enum { BK_LEFT = -1, BK_ANTI = CP_ANTI, BK_FLAT = CP_FLAT, BK_SYMM = CP_SYMM, BK_FIX = 3 };
constexpr int BC_NV = 8;

// The rules of every variable of a face: the turbulence variables are k and
// omega (SST), k and kL (k-kL), nu-tilde (SA); lctm2015's intermittency takes
// a flat copy wherever they copy (bc_primitive.f90:302, 385, 437, 475, 555) and
// its own fixed value wherever they are fixed (:262, :343).  kl_tw: the
// subsonic inlet fixes k-kL's kL from the omega values
// (src/boundary/bc_primitive.f90:333-336), which k-kL never reads from the
// boundary file (read_bc.f90:98-108)
struct BcRules {
  int kind[BC_NV];
  double val[BC_NV];
};
__device__ __forceinline__ void turb_copy(const Blk &b, BcRules &r, int kind) {
  if (b.ng >= 5) r.kind[5] = kind;
  if (two_eq(b)) r.kind[6] = kind;
  if (b.lctm) r.kind[7] = BK_FLAT;
}
__device__ __forceinline__ void turb_fix(const Blk &b, const FaceBC &p, BcRules &r, bool kl_tw) {
  if (b.ng >= 5) r.kind[5] = BK_FIX;
  r.val[5] = two_eq(b) ? p.fix[FX_TK] : p.fix[FX_TV];
  if (two_eq(b)) r.kind[6] = BK_FIX;
  r.val[6] = (b.kkl && !kl_tw) ? p.fix[FX_TKL] : p.fix[FX_TW];
  if (b.lctm) r.kind[7] = BK_FIX;
  r.val[7] = p.fix[FX_TGM];
}

// One column of populate_ghost_primitive.  The grid spans the padded
// tangential plane (-2..na+2) x (-2..nb+2); most conditions act on the face
// interior 1..na-1 x 1..nb-1, the periodic and far-field plane copies on the
// whole plane.  A launch may hold several faces when none reads what another
// writes (see the caller).  All of a column's cells are read before any is
// written: a rule that reads and writes variable by variable waits for memory
// once per variable.  With the launches joined (bc_launches) and the edges in
// one, a stage's ghosts of the SST bump at 97x61x45 take 26 us, not 56, those
// of the laminar box at 64x64x4 28, not 49.
__device__ __forceinline__ void k_bc_face_b(const Blk &b, int face, int a, int bb, int current_iter) {
  const int na = face_na(b, face), nb = face_nb(b, face);
  if (a > na + 2 || bb > nb + 2) return;
  const FaceBC p = face_params(b, face);
  const int id = p.id;
  if (id >= 0 || id == -10) return;  // filled by the interface exchange
  const bool inner = a >= 1 && a <= na - 1 && bb >= 1 && bb <= nb - 1;
  const bool riemann = id == -8 || id == -11;
  double *const q = b.qp;
  const long nc = b.nc;
  if (id == -9) {  // single-block periodic: whole plane, three layers
    // the reference's array assignment reads its source layers whole
    // before writing; with one or two cells in the direction they overlap
    // the destination layers.  Layers g = 0..2 sit at d0 + g*st (ghosts)
    // and s0 + g*st (their sources) along the face normal's stride st.
    long d0, s0, st;
    switch (face) {
      case 0: d0 = ci(b, -2, a, bb); s0 = ci(b, b.imx - 3, a, bb); st = 1; break;
      case 1: d0 = ci(b, b.imx, a, bb); s0 = ci(b, 1, a, bb); st = 1; break;
      case 2: d0 = ci(b, a, -2, bb); s0 = ci(b, a, b.jmx - 3, bb); st = b.pi; break;
      case 3: d0 = ci(b, a, b.jmx, bb); s0 = ci(b, a, 1, bb); st = b.pi; break;
      case 4: d0 = ci(b, a, bb, -2); s0 = ci(b, a, bb, b.kmx - 3); st = (long)b.pi * b.pj; break;
      default: d0 = ci(b, a, bb, b.kmx); s0 = ci(b, a, bb, 1); st = (long)b.pi * b.pj; break;
    }
    double v[BC_NV][3];
#pragma unroll
    for (int l = 0; l < BC_NV; ++l)
      if (l < b.nv) {
#pragma unroll
        for (int g = 0; g < 3; ++g) v[l][g] = q[l * nc + s0 + g * st];
      }
#pragma unroll
    for (int l = 0; l < BC_NV; ++l)
      if (l < b.nv) {
#pragma unroll
        for (int g = 0; g < 3; ++g) q[l * nc + d0 + g * st] = v[l][g];
      }
    return;
  }
  if (!inner) {
    // the far field's outer layers copy the first over the whole plane
    if (!riemann) return;
    const long g0 = fcell(b, face, 0, a, bb), g1 = fcell(b, face, -1, a, bb), g2 = fcell(b, face, -2, a, bb);
    double v[BC_NV];
#pragma unroll
    for (int l = 0; l < BC_NV; ++l)
      if (l < b.nv) v[l] = q[l * nc + g0];
#pragma unroll
    for (int l = 0; l < BC_NV; ++l)
      if (l < b.nv) {
        q[l * nc + g1] = v[l];
        q[l * nc + g2] = v[l];
      }
    return;
  }
  // the rule of every variable
  BcRules r;
#pragma unroll
  for (int l = 0; l < BC_NV; ++l) {
    r.kind[l] = BK_LEFT;
    r.val[l] = l < 5 ? p.fix[l] : 0.0;
  }
  auto flow = [&](int k0, int k1, int k2, int k3, int k4) {
    r.kind[0] = k0; r.kind[1] = k1; r.kind[2] = k2; r.kind[3] = k3; r.kind[4] = k4;
  };
  const bool fix = current_iter <= 2;
  switch (id) {
    case -1:  // supersonic inlet
      if (!fix) return;
      flow(BK_FIX, BK_FIX, BK_FIX, BK_FIX, BK_FIX);
      turb_fix(b, p, r, false);
      break;
    case -2:  // supersonic outlet
    case -7:  // pole
      flow(BK_FLAT, BK_FLAT, BK_FLAT, BK_FLAT, BK_FLAT);
      turb_copy(b, r, BK_FLAT);
      break;
    case -3:  // subsonic inlet
      if (fix) {
        flow(BK_FIX, BK_FIX, BK_FIX, BK_FIX, BK_LEFT);
        turb_fix(b, p, r, true);
      }
      r.kind[4] = BK_FLAT;
      break;
    case -4:  // subsonic outlet
      flow(BK_FLAT, BK_FLAT, BK_FLAT, BK_FLAT, fix ? BK_FIX : BK_LEFT);
      turb_copy(b, r, BK_FLAT);
      break;
    case -5:  // no-slip wall; the density by the wall temperature, SST's omega below
      flow(BK_SYMM, BK_ANTI, BK_ANTI, BK_ANTI, BK_SYMM);
      turb_copy(b, r, BK_ANTI);
      if (two_eq(b) && !b.kkl) r.kind[6] = BK_LEFT;
      break;
    case -6:  // slip wall; the velocity below
      flow(BK_SYMM, BK_LEFT, BK_LEFT, BK_LEFT, BK_SYMM);
      turb_copy(b, r, BK_SYMM);
      break;
    case -8:   // far field
    case -11:  // total-pressure inlet
      // the whole-face turbulent copy/fix of the reference ends as set by
      // the last face cell in its loop order
      if (b.turb) {
        if (riemann_unb(b, face, na - 1, nb - 1) > 0.) turb_copy(b, r, BK_FLAT);
        else turb_fix(b, p, r, false);
      }
      break;
    default:
      return;
  }
  long cin[4], cgh[3];
#pragma unroll
  for (int m = 0; m < 4; ++m) cin[m] = fcell(b, face, m + 1, a, bb);
#pragma unroll
  for (int g = 0; g < 3; ++g) cgh[g] = fcell(b, face, -g, a, bb);
  double in[BC_NV][4], gh[BC_NV][3];
#pragma unroll
  for (int l = 0; l < BC_NV; ++l)
    if (l < b.nv) {
#pragma unroll
      for (int m = 0; m < 4; ++m) in[l][m] = q[l * nc + cin[m]];
    }
#pragma unroll
  for (int l = 0; l < BC_NV; ++l) {
    if (l >= b.nv) continue;
    const int k = r.kind[l];
    const double a1 = k == BK_SYMM ? b.c1 : 1., a2 = k == BK_SYMM ? b.c2 : k == BK_ANTI ? -1. : 1.,
                 a3 = k == BK_SYMM ? b.c3 : 0.;
#pragma unroll
    for (int g = 0; g < 3; ++g) {
      // ghost layer g takes interior layer g+1 (anti, symm) or layer 1 (flat)
      const double v1 = k == BK_FLAT ? in[l][0] : in[l][g], v2 = k == BK_FLAT ? in[l][1] : in[l][g + 1];
      const double w = a2 * v1 - a3 * v2;
      gh[l][g] = k == BK_FIX ? r.val[l] : a1 == 1. ? w : w / a1;
    }
  }
  unsigned done = 0;  // variables whose ghosts a special rule has filled
  if (id == -5) {
    // src/boundary/bc_primitive.f90:1778-1945
    const double Tw = p.fix[FX_TWALL], R = b.R, gm = b.gm;
    if (Tw < 0.0) {
      const double stag = (in[4][0] / (R * in[0][0])) * (1 + (0.5 * (gm - 1.) * gm * in[4][0] / in[0][0]));
#pragma unroll
      for (int g = 0; g < 3; ++g) gh[0][g] = gh[4][g] / (R * stag);
    } else if (Tw > 1.0) {
#pragma unroll
      for (int g = 0; g < 3; ++g) gh[0][g] = gh[4][g] / (R * (2 * Tw - (in[4][g] / (R * in[0][g]))));
    }
    if (two_eq(b) && !b.kkl) {
      // src/boundary/bc_primitive.f90:564-643 (Sutherland mu whatever mu_variation)
      const double T_face = 0.5 * ((gh[4][0] / gh[0][0]) + (in[4][0] / in[0][0])) / b.R;
      const double mu = b.mu_ref * pow(T_face / b.T_ref, 1.5) * ((b.T_ref + b.S_ref) / (T_face + b.S_ref));
      const double rm = 0.5 * (gh[0][0] + in[0][0]);
      const double d2 = 2 * b.dist[cin[0]];
#pragma unroll
      for (int g = 0; g < 3; ++g) gh[6][g] = 120 * mu / (rm * 0.075 * (d2 * d2)) - in[6][g];
      done |= 1u << 6;
    }
  } else if (id == -6) {
    // src/boundary/FT_bc.f90:36-106; j and k faces reflect with the I-face
    // normal stored at the same index, as the reference does
    double nx, ny, nz;
    bnormal(b, face, a, bb, nx, ny, nz);
    long f;
    switch (face) {
      case 0: f = fi(b, 0, 1, a, bb); break;
      case 1: f = fi(b, 0, b.imx, a, bb); break;
      case 2: f = fi(b, 0, a, 1, bb); break;
      case 3: f = fi(b, 0, a, b.jmx, bb); break;
      case 4: f = fi(b, 0, a, bb, 1); break;
      default: f = fi(b, 0, a, bb, b.kmx); break;
    }
    const double rx = b.fx[0][f], ry = b.fy[0][f], rz = b.fz[0][f];
#pragma unroll
    for (int g = 0; g < 3; ++g) {
      const double dot = in[1][g] * nx + in[2][g] * ny + in[3][g] * nz;
      gh[1][g] = in[1][g] - (2.0 * dot * rx);
      gh[2][g] = in[2][g] - (2.0 * dot * ry);
      gh[3][g] = in[3][g] - (2.0 * dot * rz);
    }
    done |= 0xe;
  } else if (riemann) {
    double c[5], g0[5], nrm[3];
#pragma unroll
    for (int l = 0; l < 5; ++l) c[l] = in[l][0];
    bnormal(b, face, a, bb, nrm[0], nrm[1], nrm[2]);
    riemann_state(b, face, c, nrm, true, id == -11, p.fix[FX_TP], g0);
#pragma unroll
    for (int l = 0; l < 5; ++l) gh[l][0] = gh[l][1] = gh[l][2] = g0[l];
    done |= 0x1f;
  }
#pragma unroll
  for (int l = 0; l < BC_NV; ++l)
    if (l < b.nv && (r.kind[l] != BK_LEFT || (done >> l & 1))) {
#pragma unroll
      for (int g = 0; g < 3; ++g) q[l * nc + cgh[g]] = gh[l][g];
    }
}
__device__ __forceinline__ void k_bc_face_b(const Blk &b, const Wg &wg, int current_iter) {
  k_bc_face_b(b, wg.z, (int)(wg.x * 64 + threadIdx.x) - 2, (int)(wg.y * 4 + threadIdx.y) - 2, current_iter);
}

// Edges and corners, src/boundary/bc_primitive.f90:209-224: the four lines
// along i, then the four along k, then the eight corners, each from the three
// cells next to it.  One launch takes all three: a line's end cells that a
// later one overwrites are left out, and what a later one reads of an earlier
// one (the k lines' and corners' neighbours on the other lines) is formed
// again from the cells below, which none of the three writes.
__host__ __device__ inline long edge_cells(const Blk &b) { return 4L * (b.imx + 5) + 4L * (b.kmx + 5) + 8; }
__device__ __forceinline__ void k_bc_edges_b(const Blk &b, const Wg &wg) {
  long t = (long)wg.x * blockDim.x + threadIdx.x;
  const int I = b.imx, J = b.jmx, K = b.kmx;
  const long n = edge_cells(b);
  if (t >= n * b.nv) return;
  const int l = (int)(t / n);
  t -= l * n;
  double *v = b.qp + (long)l * b.nc;
  auto Q = [&](int i, int j, int k) -> double & { return v[ci(b, i, j, k)]; };
  // the line along i at (j, k) of i, the line along k at (i, j) of k: jn, kn, in the interior neighbours
  auto line_i = [&](int i, int j, int k, int jn, int kn) { return 0.33 * (Q(i, jn, kn) + Q(i, j, kn) + Q(i, jn, k)); };
  auto line_k = [&](int i, int j, int k, int in, int jn) { return 0.33 * (Q(in, jn, k) + Q(in, j, k) + Q(i, jn, k)); };
  if (t < 4 * (I + 5)) {
    const int s = (int)(t / (I + 5)), i = (int)(t % (I + 5)) - 2;
    if (i == 0 || i == I) return;  // the lines along k have these
    const int j = s < 2 ? 0 : J, k = s & 1 ? K : 0;
    Q(i, j, k) = line_i(i, j, k, s < 2 ? 1 : J - 1, s & 1 ? K - 1 : 1);
    return;
  }
  t -= 4 * (I + 5);
  if (t < 4 * (K + 5)) {
    const int s = (int)(t / (K + 5)), k = (int)(t % (K + 5)) - 2;
    if (k == 0 || k == K) return;  // the corners
    const int i = s == 0 || s == 3 ? I : 0, j = s < 2 ? 0 : J;
    Q(i, j, k) = line_k(i, j, k, i ? I - 1 : 1, j ? J - 1 : 1);
    return;
  }
  t -= 4 * (K + 5);
  const int i = t & 1 ? I : 0, j = t & 2 ? J : 0, k = t & 4 ? K : 0;
  const int in = i ? I - 1 : 1, jn = j ? J - 1 : 1, kn = k ? K - 1 : 1;
  Q(i, j, k) = 0.33 * (line_i(in, j, k, jn, kn) + Q(i, jn, k) + line_k(i, j, kn, in, jn));
}

}  // namespace fest
