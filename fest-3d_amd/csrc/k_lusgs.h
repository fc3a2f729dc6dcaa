// k_lusgs.h -- the LU-SGS implicit update of the 'implicit' integrator
// (src/lusgs.f90:134-1196, laminar and SST variants; dispatch
// src/update.f90:215-218).
//
// The reference sweeps the cells in loop order: forward k, j, i ascending,
// backward i, j, k descending.  A cell's forward value needs only its i-, j-
// and k- neighbours' forward values, its backward value only the i+, j+, k+
// neighbours' backward values and its own forward value.  All cells of one
// hyperplane i + j + k = s therefore depend only on hyperplane s - 1 (s + 1
// backward).  Each sweep is one launch: a work-group owns a tile of (j, k)
// columns and walks the hyperplanes, so the loop order's dependences hold
// exactly (k_lusgs_march).
//
// delQstar and delQ share one array: a cell's backward value overwrites its
// own forward value, which nothing else reads afterwards.  The sweeps read
// only hyperplane-major copies (Sk), so qp is updated after the backward
// sweep.
#pragma once
// multiply-adds may fuse, as in the residual kernels
#pragma clang fp contract(fast)
#include "blk.h"

namespace fest {

struct LuFace {
  double A, nx, ny, nz, vol, mm, tm, F1;
};

// The viscous factors of a face, which no sweep value enters: with
// g = area / volume, c[0] = (mu + mu_t) g, c[1] = K_heat g / R, and for SST
// and k-kL c[2], c[3] = (mu + sigma mu_t) g of the two turbulence variables,
// for SA c[2] = mu g / sigma, c[3] = g / sigma.  k-kL: F1 stays 0 and sigma_w2
// is 1, so both sigmas are 1 (src/lusgs.f90:1671-1672).
template <int NV>
__device__ __forceinline__ void lu_visc(const Blk &b, const LuFace &f, double (&c)[4]) {
  const double g = f.A / f.vol;
  c[0] = (f.mm + f.tm) * g;
  c[1] = (f.mm * b.iPr + f.tm * b.itPr) * (b.cpR / b.R) * g;
  c[2] = c[3] = 0.0;
  if constexpr (NV == 7) {
    const double sk = 0.85 * f.F1 + 1.0 * (1.0 - f.F1), sw = 0.5 * f.F1 + b.sigma_w2 * (1.0 - f.F1);
    c[2] = (f.mm + sk * f.tm) * g;
    c[3] = (f.mm + sw * f.tm) * g;
  }
  if constexpr (NV == 6) {
    c[2] = f.mm * g / Sa::sigma;
    c[3] = g / Sa::sigma;
  }
}

// Flux / SAFlux / SSTFlux (src/lusgs.f90:490-609, 2104-2259, 1027-1196): the
// flux through a face (area A, outward normal n, viscous factors c) of the
// neighbour state ql moved by du (conservative), against the cell's own
// primitive state qr.  The reference takes every gradient as a difference d
// times n area / volume and builds the stress tensor from them; the normal
// stress those components add up to is mu g (d (n.n) + n (d.n) / 3), which is
// what is formed here: 24 operations in place of some 100 with 18 quotients.
// KKL: the k-kL model
template <int NV, bool KKL>
__device__ __forceinline__ void lu_flux(const Blk &b, const double (&ql)[NV], const double (&qr)[NV],
                                        const double (&du)[NV], double A, double nx, double ny, double nz,
                                        const double (&c)[4], double (&out)[NV]) {
  const double gm1 = b.gm - 1.0, ig1 = 1.0 / gm1;
  double U[NV], W[NV];
  U[0] = ql[0];
  U[1] = ql[0] * ql[1];
  U[2] = ql[0] * ql[2];
  U[3] = ql[0] * ql[3];
  U[4] = ql[4] * ig1 + (0.5 * ql[0] * (ql[1] * ql[1] + ql[2] * ql[2] + ql[3] * ql[3]));
#pragma unroll
  for (int l = 5; l < NV; ++l) U[l] = ql[0] * ql[l];
#pragma unroll
  for (int l = 0; l < NV; ++l) U[l] = U[l] + du[l];
  const double rU = qdiv(1.0, U[0]);
  W[0] = U[0];
#pragma unroll
  for (int l = 1; l < NV; ++l) W[l] = U[l] * rU;
  const double half = 0.5 * (U[1] * W[1] + U[2] * W[2] + U[3] * W[3]);  // rho u^2 / 2
  W[4] = gm1 * (U[4] - half);
  if constexpr (KKL) {
    // KKLFlux floors k and kL (src/lusgs.f90:1605-1606)
    W[5] = fmx(W[5], 1e-8);
    W[6] = fmx(W[6], 1e-8);
  } else if constexpr (NV == 7) {
    // a negative k or omega falls back to the neighbour's old value
    W[5] = W[5] < 0. ? ql[5] : W[5];
    W[6] = W[6] < 0. ? ql[6] : W[6];
  }
  if constexpr (NV == 6) W[5] = fmx(W[5], 1e-8);
  const double *P = qr;
  const double m = W[0] * ((W[1] * nx) + (W[2] * ny) + (W[3] * nz));
  const double d1 = P[1] - W[1], d2 = P[2] - W[2], d3 = P[3] - W[3];
  const double nn = nx * nx + ny * ny + nz * nz, dn = (d1 * nx + d2 * ny + d3 * nz) * (1.0 / 3.0);
  const double t1 = c[0] * (d1 * nn + dn * nx), t2 = c[0] * (d2 * nn + dn * ny), t3 = c[0] * (d3 * nn + dn * nz);
  const double dT = P[4] * qdiv(1.0, P[0]) - W[4] * rU;  // R times the temperature difference
  double Fx[NV];
  Fx[0] = m;
  Fx[1] = (W[1] * m) + (W[4] * nx) - t1;
  Fx[2] = (W[2] * m) + (W[4] * ny) - t2;
  Fx[3] = (W[3] * m) + (W[4] * nz) - t3;
  Fx[4] = (b.gm * ig1 * W[4] + half) * rU * m -
          (0.5 * (t1 * (W[1] + P[1]) + t2 * (W[2] + P[2]) + t3 * (W[3] + P[3])) + c[1] * dT * nn);
  if constexpr (NV == 7) {
    Fx[5] = W[5] * m + c[2] * (P[5] - W[5]) * nn;
    Fx[6] = W[6] * m + c[3] * (P[6] - W[6]) * nn;
  }
  // nu-tilde diffusion with 0.25 (rho_L + rho_R)(nu_L + nu_R), added
  if constexpr (NV == 6)
    Fx[5] = W[5] * m + (c[2] + 0.25 * (P[0] + W[0]) * (P[5] + W[5]) * c[3]) * (P[5] - W[5]) * nn;
#pragma unroll
  for (int l = 0; l < NV; ++l) out[l] = Fx[l] * A;
}

// face n (0..5 = i-, j-, k-, i+, j+, k+) of cell c0 = (i, j, k) with
// neighbour cn, from the natural-layout arrays: the Flist arrays of
// src/lusgs.f90:260-312
__device__ __forceinline__ LuFace lu_face(const Blk &b, int n, int i, int j, int k, long c0, long cn) {
  const int d = n % 3;
  const bool up = n >= 3;
  const long g = fi(b, d, i + (d == 0 && up), j + (d == 1 && up), k + (d == 2 && up));
  LuFace f;
  f.A = b.fA[d][g];
  f.nx = up ? b.fx[d][g] : -b.fx[d][g];
  f.ny = up ? b.fy[d][g] : -b.fy[d][g];
  f.nz = up ? b.fz[d][g] : -b.fz[d][g];
  f.vol = 0.5 * (b.vol[cn] + b.vol[c0]);
  // mu holds zeros for inviscid flow and mu_t for laminar flow, the dummy
  // arrays of src/lusgs.f90:115-130
  f.mm = 0.5 * (b.mu[cn] + b.mu[c0]);
  f.tm = 0.5 * (b.mut[cn] + b.mut[c0]);
  f.F1 = 0.5 * (b.f1[cn] + b.f1[c0]);
  return f;
}

// SpectralRadius (src/lusgs.f90:612-660) of face f times its area; c1 the
// neighbour's centre, c2 the cell's
template <int NV>
__device__ __forceinline__ double lu_radius(const Blk &b, const double (&ql)[NV], const double (&qr)[NV],
                                            const LuFace &f, double c1x, double c1y, double c1z, double c2x,
                                            double c2y, double c2z) {
  const double gm = b.gm;
  double Vn = 0.5 * (((ql[1] + qr[1]) * f.nx) + ((ql[2] + qr[2]) * f.ny) + ((ql[3] + qr[3]) * f.nz));
  Vn = fabs(Vn);
  const double a = 0.5 * (sqrt(gm * ql[4] / ql[0]) + sqrt(gm * qr[4] / qr[0]));
  const double rho = 0.5 * (ql[0] + qr[0]);
  const double dx = c1x - c2x, dy = c1y - c2y, dz = c1z - c2z;
  const double dist = sqrt(dx * dx + dy * dy + dz * dz);
  const double vis = gm * (f.mm / b.Pr + f.tm / b.tPr) / (rho * dist);
  return (Vn + a + vis) * f.A;
}

template <int NV>
__device__ __forceinline__ void lu_load(const Blk &b, long c, double (&q)[NV]) {
#pragma unroll
  for (int l = 0; l < NV; ++l) q[l] = b.qp[(long)l * b.nc + c];
}

// The SA diagonal (src/lusgs.f90:1882-1914, the same backward): D plus the
// linearised SA production and destruction, one value for all six
// equations; gi the cell's gradient index
__device__ __forceinline__ double sa_diagonal(const Blk &b, long c0, long gi, double rho, double q6, double vol,
                                              double D) {
  const double *gx = b.g[0], *gy = b.g[1], *gz = b.g[2];
  const long ngr = b.ngr;
  const double Omega = sqrt(sqd(gy[2 * ngr + gi] - gz[ngr + gi]) + sqd(gz[gi] - gx[2 * ngr + gi]) +
                            sqd(gx[ngr + gi] - gy[gi]));
  const double dist_i = b.dist[c0], dist_i_2 = dist_i * dist_i, k2 = Sa::kappa * Sa::kappa;
  const double nu = b.mu[c0] / rho;
  const double Ji = q6 / nu, Ji_2 = Ji * Ji, Ji_3 = Ji_2 * Ji;
  const double fv1 = Ji_3 / (Ji_3 + Sa::cv1_3);
  const double fv2 = 1.0 - Ji / (1.0 + (Ji * fv1));
  const double inv_k2_d2 = 1.0 / (k2 * dist_i_2);
  const double Shat = fmx(Omega + q6 * fv2 * inv_k2_d2, 1.0e-10);
  const double inv_Shat = 1.0 / Shat;
  const double jc = Ji_3 + Sa::cv1_3, jf = 1.0 + Ji * fv1;
  const double dfv1 = 3.0 * Ji_2 * Sa::cv1_3 / (nu * (jc * jc));
  const double dfv2 = -((1.0 / nu) - Ji_2 * dfv1) / (jf * jf);
  const double dShat = (fv2 + q6 * dfv2) * inv_k2_d2;
  D = D - Sa::cb1 * (q6 * dShat + Shat) * vol;
  const double r = fmn(q6 * inv_Shat * inv_k2_d2, 10.0);
  const double r5 = (((r * r) * r) * r) * r;
  const double g = r + Sa::cw2 * ((r5 * r) - r);
  const double g_6 = ((((g * g) * g) * g) * g) * g;
  const double glim = pow((1.0 + Sa::cw3_6) / (g_6 + Sa::cw3_6), 1.0 / 6.0);
  const double fw = g * glim;
  const double dr = (Shat - q6 * dShat) * inv_Shat * inv_Shat * inv_k2_d2;
  const double dg = dr * (1.0 + Sa::cw2 * (6.0 * r5 - 1.0));
  const double dfw = dg * glim * (1.0 - g_6 / (g_6 + Sa::cw3_6));
  return D + Sa::cw1 * (dfw * q6 + 2 * fw) * q6 / dist_i_2 * vol;
}

// Hyperplane-major ("skewed") storage of everything the sweeps read.  Cell
// (i, j, k), 0 <= i <= imx, 0 <= j <= jmx, 0 <= k <= kmx, lies on hyperplane
// s = i + j + k at position r = k sk_j + j + 7.  Components are kept in pairs,
// eight positions form a group, and a group's pairs lie together: component
// 2 p + e is at (((s sk_g + r / 8) NP + p) 8 + r % 8) 2 + e.  A tile of columns
// j = 8 m + 1 .. 8 m + 8 (sk_j is a multiple of 8) so reads whole lines that
// no other tile reads, 16 bytes a lane, at immediate offsets from one address
// per cell.  The i-, j- and k- neighbours of a cell sit on hyperplane s - 1 at
// r, r - 1 and r - sk_j.
template <int NV>
struct Sk {
  static constexpr int NVP = (NV + 1) / 2;         // pairs of a state
  static constexpr int NVIS = NV == 5 ? 2 : 4;     // viscous factors of a face that are kept
  static constexpr int Q = 0;                      // state (cells 0..n+1)
  static constexpr int RF = NVP;                   // right-hand sides of the forward and the backward sweep
  static constexpr int RB = 2 * NVP;               //   (interior; k_lusgs_prep)
  static constexpr int DQ = 3 * NVP;               // delQstar / delQ (interior)
  static constexpr int DG = 4 * NVP;               // diagonal (interior; SST: 3 values)
  static constexpr int FACE = DG + (NV == 7 ? 2 : 1);
  static constexpr int NF = 3 + NVIS / 2;          // lower face d at FACE + NF d (cells 1..n+1): A, nx, ny, nz,
                                                   //   the viscous factors, radius x area
  static constexpr int NP = FACE + 3 * NF;
};
__host__ __device__ inline int sk_npair(int nv) {
  return nv == 5 ? (int)Sk<5>::NP : nv == 6 ? (int)Sk<6>::NP : (int)Sk<7>::NP;
}

// pair 0 of position r on hyperplane s; pair p is 8 p further
__device__ __forceinline__ double2 *sk_at(const Blk &b, int NP, int s, int r) {
  return (double2 *)b.sk + ((long)s * b.sk_g + (r >> 3)) * NP * 8 + (r & 7);
}
__device__ __forceinline__ int sk_pos(const Blk &b, int j, int k) { return k * b.sk_j + j + 7; }

// Copies n natural-layout planes into skewed pairs p0.. for the cells
// lo <= i, j, k <= imx-1+hi (layout 0: padded cell arrays, 2 + d: face arrays
// of direction d, the lower face of each cell).  32 x 32 (i, j) tiles of one k
// go through LDS: rows are read whole, and each diagonal i + j = const of the
// tile, a run of consecutive positions on one hyperplane, is written whole.
struct SkewIn {
  const double *p[8];
  int n, p0, layout, lo, hi;
};
__global__ void __launch_bounds__(256) k_to_skew(Blk b, SkewIn a) {
  __shared__ double tile[2][32][33];
  const int NP = sk_npair(b.nv);
  const int ilo = a.lo, ihi = b.imx - 1 + a.hi, jhi = b.jmx - 1 + a.hi;
  const int ntx = (ihi - ilo + 32) / 32;
  const int i0 = ilo + ((int)blockIdx.x % ntx) * 32, j0 = ilo + ((int)blockIdx.x / ntx) * 32;
  const int k = ilo + (int)blockIdx.y;
  const int tid = threadIdx.x;
  for (int c = 0; c < a.n; c += 2) {
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int ii = tid & 31, jj = (tid >> 5) + 8 * m, i = i0 + ii, j = j0 + jj;
      if (i <= ihi && j <= jhi) {
        const long o = a.layout == 0 ? ci(b, i, j, k) : fi(b, a.layout - 2, i, j, k);
        tile[0][jj][ii] = a.p[c][o];
        tile[1][jj][ii] = c + 1 < a.n ? a.p[c + 1][o] : 0.0;
      }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      // position e of the tile in diagonal order: diagonals 0..31 first,
      // then 32..62 as the mirror image of 30..0
      const int e = tid + 256 * m, em = e < 528 ? e : 1023 - e;
      int sg = (int)((sqrtf((float)(8 * em + 1)) - 1.0f) * 0.5f);
      // exact whatever sqrtf rounds to: sg (sg + 1) / 2 <= em < (sg + 1) (sg + 2) / 2
      if ((sg + 1) * (sg + 2) / 2 <= em) ++sg;
      if (sg * (sg + 1) / 2 > em) --sg;
      const int pos = em - sg * (sg + 1) / 2;
      int jj = pos, ii = sg - pos;
      if (e >= 528) { jj = 31 - jj; ii = 31 - ii; }
      const int i = i0 + ii, j = j0 + jj;
      if (i <= ihi && j <= jhi)
        sk_at(b, NP, i + j + k, sk_pos(b, j, k))[8 * (a.p0 + c / 2)] = make_double2(tile[0][jj][ii], tile[1][jj][ii]);
    }
    __syncthreads();
  }
}

// Everything of a cell the sweeps use that does not depend on them, written
// into hyperplane-major storage: the radius x area of the lower faces
// (src/lusgs.f90:612-660; a face's radius is the same seen from either of
// its cells -- the normal flips sign, every other operand pairs up
// commutatively -- so the backward sweep reads a cell's upper faces from the
// neighbours) and their viscous factors; the "Old" fluxes of the neighbours'
// unmoved states (src/lusgs.f90:314-319, 424-429), summed over the lower faces
// into the forward right-hand side -R + 0.5 sum and over the upper ones into
// the backward 0.5 sum; and the diagonal vol/dt + 0.5 sum of the six radii
// (src/lusgs.f90:329-345).  16 x 16 (i, j) tiles of one k over the cells
// 1..n+1 read the stencil whole; each value goes through LDS and out along
// the tile's diagonals, runs of consecutive positions of one hyperplane.
// Values of cells outside the interior are never read.
template <int NV, bool KKL>
__global__ void __launch_bounds__(256) k_lusgs_prep(Blk b) {
  using C = Sk<NV>;
  __shared__ double tile[2 * C::NVP][16][17];
  const int ntx = (b.imx + 15) / 16;
  const int i0 = 1 + ((int)blockIdx.x % ntx) * 16, j0 = 1 + ((int)blockIdx.x / ntx) * 16;
  const int k = 1 + (int)blockIdx.y;
  const int tid = threadIdx.x;
  const int ii = tid & 15, jj = tid >> 4;
  const int i = min(i0 + ii, b.imx), j = min(j0 + jj, b.jmx);  // clamped lanes compute, never write
  const bool inner = i <= b.imx - 1 && j <= b.jmx - 1 && k <= b.kmx - 1;
  // where the tile's diagonal order puts this thread on the way out
  int oi, oj;
  {
    const int e = tid, em = e < 136 ? e : 255 - e;
    int sg = (int)((sqrtf((float)(8 * em + 1)) - 1.0f) * 0.5f);
    if ((sg + 1) * (sg + 2) / 2 <= em) ++sg;
    if (sg * (sg + 1) / 2 > em) --sg;
    oj = em - sg * (sg + 1) / 2;
    oi = sg - oj;
    if (e >= 136) {
      oj = 15 - oj;
      oi = 15 - oi;
    }
  }
  const bool out_ok = i0 + oi <= b.imx && j0 + oj <= b.jmx;
  double2 *const out_base = sk_at(b, C::NP, i0 + oi + j0 + oj + k, sk_pos(b, j0 + oj, k));
  // the staged values' first np pairs to pairs p.. of the cell
  auto flush = [&](int np, int p) {
    __syncthreads();
    if (out_ok)
      for (int m = 0; m < np; ++m) out_base[8 * (p + m)] = make_double2(tile[2 * m][oj][oi], tile[2 * m + 1][oj][oi]);
    __syncthreads();
  };
  const long c0 = ci(b, i, j, k);
  double Q0[NV], Qn[NV], zero[NV], Old[NV], L[6], sum[2][NV];
  lu_load<NV>(b, c0, Q0);
#pragma unroll
  for (int l = 0; l < NV; ++l) zero[l] = sum[0][l] = sum[1][l] = 0.0;
#pragma unroll
  for (int up = 0; up < 2; ++up) {
#pragma unroll 1
    for (int d = 0; d < 3; ++d) {
      const long cn = up ? c0 + cstride(b, d) : c0 - cstride(b, d);
      lu_load<NV>(b, cn, Qn);
      const LuFace f = lu_face(b, 3 * up + d, i, j, k, c0, cn);
      L[3 * up + d] = lu_radius<NV>(b, Qn, Q0, f, b.cx[cn], b.cy[cn], b.cz[cn], b.cx[c0], b.cy[c0], b.cz[c0]);
      double vis[4];
      lu_visc<NV>(b, f, vis);
      lu_flux<NV, KKL>(b, Qn, Q0, zero, f.A, f.nx, f.ny, f.nz, vis, Old);
#pragma unroll
      for (int l = 0; l < NV; ++l) sum[up][l] += Old[l];
      if (!up) {
#pragma unroll
        for (int l = 0; l < C::NVIS; ++l) tile[l][jj][ii] = vis[l];
        tile[C::NVIS][jj][ii] = L[d];
        tile[C::NVIS + 1][jj][ii] = 0.0;
        flush(C::NVIS / 2 + 1, C::FACE + C::NF * d + 2);
      }
    }
  }
#pragma unroll
  for (int up = 0; up < 2; ++up) {
#pragma unroll
    for (int l = 0; l < 2 * C::NVP; ++l)
      tile[l][jj][ii] = l >= NV ? 0.0 : up ? 0.5 * sum[1][l < NV ? l : 0]
                        : 0.5 * sum[0][l < NV ? l : 0] - (inner ? b.res[(long)l * b.nres + ri(b, i, j, k)] : 0.0);
    flush(C::NVP, up ? C::RB : C::RF);
  }
  double dg = 0.0, d5 = 0.0, d6 = 0.0;
  if (inner) {
    const double sumL = L[0] + L[1] + L[2] + L[3] + L[4] + L[5];
    const double vol = b.vol[c0];
    dg = (vol / b.dt[ri(b, i, j, k)]) + 0.5 * sumL;
    if constexpr (NV == 6) dg = sa_diagonal(b, c0, gri(b, i, j, k), Q0[0], Q0[5], vol, dg);
    if constexpr (NV == 7) {
      if constexpr (KKL) {
        // the k-kL source terms (src/lusgs.f90:1359-1361)
        const double mu = b.mu[c0], d2 = b.dist[c0] * b.dist[c0];
        d5 = dg + (2.5 * (pow(0.09, 0.75)) * Q0[0] * (pow(Q0[5], 1.5)) * vol / Q0[6]);
        d5 = d5 + (2 * mu * vol / d2);
        d6 = dg + (6 * mu * vol / d2);
      } else {
        const double F1 = b.f1[c0], w = Q0[6];
        const double beta = F1 * 0.075 + (1.0 - F1) * 0.0828;
        d5 = (dg + (0.09 * w) * vol);
        d6 = (dg + 2.0 * beta * w * vol);
      }
    }
  }
  tile[0][jj][ii] = dg;
  tile[1][jj][ii] = d5;
  tile[2][jj][ii] = d6;
  tile[3][jj][ii] = 0.0;
  flush(NV == 7 ? 2 : 1, C::DG);
}

// One sweep, forward (BACK = 0, delQstar) or backward (BACK = 1, delQ), in one
// launch.  A work-group owns a tile of lu_tj x lu_tk = 64 (j, k) columns and
// walks the hyperplanes s = i + j + k that cross it, its four waves side by
// side on the CU's four SIMDs.  The first has a lane per column: the fluxes
// through the cell's three lower (backward: upper) faces of the neighbours'
// states moved by their sweep values (the "New" fluxes of src/lusgs.f90:
// 308-310, 418-420), minus the radius terms, the right-hand side and the
// quotient by the diagonal.  The second moves the sweep values: to memory, and
// between the tiles.  The other two bring everything else a hyperplane needs
// into LDS two hyperplanes ahead (16 bytes a lane straight to LDS), so that no
// memory latency is left in the first wave; loads it issued itself, into
// registers, were drained once a hyperplane (2.3 us each in place of 1.5, 128x96x64 SST).
//
// The neighbours' values of the hyperplane before are in LDS (two alternating
// buffers, one barrier a hyperplane).  Across a tile boundary they come from
// the work-group next to it through xj / xk.  Each slot there carries one
// value from one writer to one reader: the reader waits for it to differ from
// LU_EMPTY and puts LU_EMPTY back, so the value is its own signal and neither
// side orders memory or waits for the other's stores.  Loads and stores of
// slots are device-scope atomics, which the XCDs' L2 caches do not hold back.
// (LU_EMPTY is a NaN that no operation makes of others.)
//
// Every wait ends: work-groups take their tile from a counter in the order in
// which they start, and a tile waits only for tiles before it in that order
// (lower j and k tiles forward, higher ones backward), which have started and
// wait for nothing after them.  Should the wait end without a value all the
// same, the sweep raises ERR_SWEEP and runs out on zeros.
//
// What bounds it: the serial chain of hyperplanes.  A launch per hyperplane
// took 7.2 us each at 128x96x64 (SST, 572 launches: 4.2 ms a step) and 5.2 us
// at 96x48x1 (1.5 ms).  Here a hyperplane costs the first wave's arithmetic
// (some 450 instructions), an LDS exchange and a barrier, and a work-group
// runs behind its neighbours by the hand-over's latency once, not once per
// hyperplane: 0.89 and 0.30 ms a step, 1.0 us a hyperplane in one tile, 1.5
// with the hand-overs.
constexpr unsigned long long LU_EMPTY = 0xfff8dead0000beefull;
constexpr int LU_COLUMNS = 64, LU_SLOT = 8, LU_SPINS = (1 << 23) - 1;
// sweep values in LDS: the columns', the halos' along j and k, a zero for the
// values outside the block and a place for those of no cell
constexpr int LU_HALO_J = LU_COLUMNS, LU_HALO_K = LU_HALO_J + 8, LU_ZERO = LU_HALO_K + 8, LU_NOWHERE = LU_ZERO + 1,
              LU_VALUES = LU_NOWHERE + 1;

__global__ void k_lusgs_empty(double *x, long n) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) ((unsigned long long *)x)[t] = LU_EMPTY;
}

// The barrier of a hyperplane: LDS is made visible, memory is not waited for.
__device__ __forceinline__ void lu_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
// waits until at most N of the wave's vector memory operations are under way
template <int N>
__device__ __forceinline__ void lu_wait_loads() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4) << 14 | 7 << 4 | 15 << 8);
  asm volatile("" ::: "memory");
}

template <int NV, int BACK, bool KKL>
__global__ void __launch_bounds__(4 * LU_COLUMNS) k_lusgs_march(Blk b) {
  using C = Sk<NV>;
  constexpr int ND = NV == 7 ? 3 : 1, NDP = NV == 7 ? 2 : 1;
  // pairs staged per hyperplane: the cell's state, its j and k neighbours',
  // the three faces, the right-hand side, the diagonal and, backward, the
  // forward value
  constexpr int L_J = C::NVP, L_K = 2 * C::NVP, L_F = 3 * C::NVP, L_R = L_F + 3 * C::NF, L_D = L_R + C::NVP,
                L_W = L_D + NDP, NL = L_W + (BACK ? C::NVP : 0);
  __shared__ double2 stage[3][NL][LU_COLUMNS];
  __shared__ double dq[2][NV][LU_VALUES];
  __shared__ int my_tile;
  const int ni = b.imx - 1, nj = b.jmx - 1, nk = b.kmx - 1;
  const int ltj = __builtin_ctz(b.lu_tj), tj = b.lu_tj, tk = b.lu_tk;
  const int ntj = (nj + tj - 1) >> ltj, ntk = (nk + tk - 1) / tk;
  const int tid = (int)threadIdx.x, lane = tid & (LU_COLUMNS - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / LU_COLUMNS);
  if (tid == 0) {
    const int n = (int)(atomicAdd(b.ticket, 1ull) % (unsigned long long)(ntj * ntk));
    my_tile = BACK ? ntj * ntk - 1 - n : n;
  }
  for (int e = tid; e < 2 * NV * LU_VALUES; e += 4 * LU_COLUMNS) (&dq[0][0][0])[e] = 0.0;
  __syncthreads();
  const int tile = __builtin_amdgcn_readfirstlane(my_tile);
  const int bj = tile % ntj, bk = tile / ntj, j0 = bj * tj + 1, k0 = bk * tk + 1;
  const int lo = j0 + k0 + 1, hi = min(nj, j0 + tj - 1) + min(nk, k0 + tk - 1) + ni;
  const int sg = BACK ? -1 : 1, first = BACK ? hi : lo, n = hi - lo + 1;
  const long plane = (long)b.sk_g * C::NP * 8;
  auto off = [&](int p) { return (long)(p >> 3) * C::NP * 8 + (p & 7); };
  // column c of the tile
  auto col_j = [&](int c) { return j0 + (c & (tj - 1)); };
  auto col_k = [&](int c) { return k0 + (c >> ltj); };
  const double2 *const base = (const double2 *)b.sk;
  const int jj = lane & (tj - 1), kk = lane >> ltj, j = j0 + jj, k = k0 + kk;
  const bool inside = j <= nj && k <= nk;
  // a lane outside the block reads column (1, 1)
  const int r = inside ? sk_pos(b, j, k) : sk_pos(b, 1, 1);
  const long o_own = off(r);
  if (wave >= 2) {
    // ---- the loading waves, taking the pairs in turn.  Every lane loads on
    // every hyperplane, cell or not: the storage holds all of them.
    constexpr int N0 = (NL + 1) / 2, N1 = NL / 2;  // pairs of each wave
    const long nb_plane = BACK ? plane : -plane;
    const long o_j = off(BACK ? r + 1 : r - 1) + nb_plane, o_k = off(BACK ? r + b.sk_j : r - b.sk_j) + nb_plane;
    // the lower faces of the cell forward, of the neighbours backward
    const long o_f[3] = {BACK ? o_own + plane : o_own, BACK ? o_j : o_own, BACK ? o_k : o_own};
    auto load = [&](int m) {
      const double2 *const S = base + (long)(first + sg * min(m, n - 1)) * plane;
      double2(*const to)[LU_COLUMNS] = stage[m % 3];
#pragma unroll
      for (int p = 0; p < NL; ++p) {
        if ((p & 1) != (wave & 1)) continue;
        const double2 *from;
        if (p < L_J) from = S + o_own + 8 * (C::Q + p);
        else if (p < L_K) from = S + o_j + 8 * (C::Q + p - L_J);
        else if (p < L_F) from = S + o_k + 8 * (C::Q + p - L_K);
        else if (p < L_R) from = S + o_f[(p - L_F) / C::NF] + 8 * (C::FACE + p - L_F);
        else if (p < L_D) from = S + o_own + 8 * ((BACK ? C::RB : C::RF) + p - L_R);
        else if (p < L_W) from = S + o_own + 8 * (C::DG + p - L_D);
        else from = S + o_own + 8 * (C::DQ + p - L_W);
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)from,
                                         (__attribute__((address_space(3))) void *)&to[p][0], 16, 0, 0);
      }
    };
    auto ready = [&]() {  // all but the newest hyperplane's loads have arrived
      if (wave & 1) lu_wait_loads<N1>();
      else lu_wait_loads<N0>();
    };
    load(0);
    load(1);
    ready();
    __builtin_amdgcn_s_barrier();
    for (int m = 0; m < n; ++m) {
      asm volatile("" ::: "memory");
      load(m + 2);
      ready();
      __builtin_amdgcn_s_barrier();
    }
    lu_wait_loads<0>();
    return;
  }
  if (wave == 0) {
    // ---- the computing wave
    int from[3] = {lane, BACK ? lane + 1 : lane - 1, BACK ? lane + tj : lane - tj};
    if (jj == (BACK ? tj - 1 : 0)) from[1] = LU_HALO_J + kk;
    if (kk == (BACK ? tk - 1 : 0)) from[2] = LU_HALO_K + (jj & 7);
    if (j == (BACK ? nj : 1)) from[1] = LU_ZERO;
    if (k == (BACK ? nk : 1)) from[2] = LU_ZERO;
    if (!inside) from[0] = from[1] = from[2] = LU_ZERO;
    auto get = [&](double *to, const double2(*p)[LU_COLUMNS], int np) {
#pragma unroll
      for (int m = 0; m < np; ++m) {
        const double2 v = p[m][lane];
        to[2 * m] = v.x;
        to[2 * m + 1] = v.y;
      }
    };
    // the i neighbour's state is the cell's own on the hyperplane before
    double nbi[2 * C::NVP], own[2 * C::NVP];
    {
      const double2 *const S = base + (long)(first - sg) * plane + o_own + 8 * C::Q;
#pragma unroll
      for (int m = 0; m < C::NVP; ++m) {
        const double2 v = S[8 * m];
        nbi[2 * m] = v.x;
        nbi[2 * m + 1] = v.y;
      }
    }
    lu_barrier();
    for (int m = 0; m < n; ++m) {
      const int s = first + sg * m, i = s - j - k;
      const double2(*const st)[LU_COLUMNS] = stage[m % 3];
      double sum[NV];
      get(own, st, C::NVP);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        double nb[2 * C::NVP], fc[2 * C::NF], ql[NV], qr[NV], dn[NV], New[NV];
        if (d > 0) get(nb, st + (d == 1 ? L_J : L_K), C::NVP);
        get(fc, st + L_F + d * C::NF, C::NF);
#pragma unroll
        for (int l = 0; l < NV; ++l) {
          ql[l] = d > 0 ? nb[l] : nbi[l];
          qr[l] = own[l];
          dn[l] = dq[(s + 1) & 1][l][from[d]];
        }
        double vis[4] = {fc[4], fc[5], 0.0, 0.0};
        if constexpr (C::NVIS == 4) {
          vis[2] = fc[6];
          vis[3] = fc[7];
        }
        // outward normal of this cell: the lower face's own normal flipped forward
        const double o = BACK ? 1.0 : -1.0;
        lu_flux<NV, KKL>(b, ql, qr, dn, fc[0], o * fc[1], o * fc[2], o * fc[3], vis, New);
#pragma unroll
        for (int l = 0; l < NV; ++l) {
          const double t = New[l] - fc[2 * C::NF - 2] * dn[l];
          sum[l] = d == 0 ? t : sum[l] + t;
        }
      }
      double rhs[2 * C::NVP], fwd[2 * C::NVP], dg[2 * NDP];
      get(rhs, st + L_R, C::NVP);
      get(dg, st + L_D, NDP);
      if constexpr (BACK) get(fwd, st + L_W, C::NVP);
      const int to = inside && i >= 1 && i <= ni ? lane : LU_NOWHERE;
#pragma unroll
      for (int l = 0; l < NV; ++l) {
        const double t = qdiv(rhs[l] - 0.5 * sum[l], dg[ND == 3 && l >= 5 ? l - 4 : 0]);
        dq[s & 1][l][to] = BACK ? fwd[l] + t : t;
      }
#pragma unroll
      for (int l = 0; l < NV; ++l) nbi[l] = own[l];
      lu_barrier();
    }
    return;
  }
  // ---- the second wave.  Hand-overs: lanes 4 e .. 4 e + 3 take two values
  // each of edge column e: 0..7 along the tile's j boundary, 8..15 its k
  // boundary (which only a tile of 8 x 8 columns has)
  const int e = (lane >> 2) & 7, sub = lane & 3;
  const bool kdir = lane >= 32;
  const bool exists = kdir ? e < tj : e < tk;
  const int near_ = BACK ? (kdir ? tk : tj) - 1 : 0, far_ = BACK ? 0 : (kdir ? tk : tj) - 1;
  // the columns that read across the boundary and that are read
  const int cin = kdir ? near_ * tj + e : e * tj + near_, cout = kdir ? far_ * tj + e : e * tj + far_;
  const int nt = kdir ? ntk : ntj, me = kdir ? bk : bj;
  const int jin = col_j(cin), kin = col_k(cin), jout = col_j(cout), kout = col_k(cout);
  const bool has_in = exists && (BACK ? me < nt - 1 : me > 0) && jin <= nj && kin <= nk;
  const bool has_out = exists && (BACK ? me > 0 : me < nt - 1) && jout <= nj && kout <= nk;
  auto slot = [&](int bound, int j, int k) {
    return (unsigned long long *)(kdir ? b.xk + ((long)bound * nj + (j - 1)) * ni * LU_SLOT
                                       : b.xj + ((long)bound * nk + (k - 1)) * ni * LU_SLOT);
  };
  unsigned long long *const xin = has_in ? slot(BACK ? me : me - 1, jin, kin) : nullptr;
  unsigned long long *const xout = has_out ? slot(BACK ? me - 1 : me, jout, kout) : nullptr;
  const long o_dq = o_own + 8 * C::DQ;
  bool given_up = false;
  // hyperplane s's values from the neighbouring tiles, for the cells of the next one
  auto take = [&](int s) {
    const int i = s + sg - jin - kin;
    if (!xin || i < 1 || i > ni) return;
    unsigned long long *const p = xin + (long)(i - 1) * LU_SLOT + 2 * sub;
    const bool two = 2 * sub + 1 < NV;
    if (2 * sub >= NV) return;
    unsigned long long x0, x1;
    for (int t = 0;; ++t) {
      x0 = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      x1 = two ? __hip_atomic_load(p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
      if ((x0 != LU_EMPTY && x1 != LU_EMPTY) || given_up) break;
      if (t >= LU_SPINS) atomicOr(b.err, ERR_SWEEP);
      if ((t & 1023) == 1023 && (__hip_atomic_load(b.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & ERR_SWEEP))
        given_up = true;
    }
    const int h = (kdir ? LU_HALO_K : LU_HALO_J) + e;
    dq[s & 1][2 * sub][h] = given_up ? 0.0 : __longlong_as_double((long long)x0);
    __hip_atomic_store(p, LU_EMPTY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (two) {
      dq[s & 1][2 * sub + 1][h] = given_up ? 0.0 : __longlong_as_double((long long)x1);
      __hip_atomic_store(p + 1, LU_EMPTY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  };
  // hyperplane s's values of this tile to the neighbouring tiles and to memory
  auto give = [&](int s) {
    const int io = s - jout - kout;
    if (xout && io >= 1 && io <= ni) {
      unsigned long long *const p = xout + (long)(io - 1) * LU_SLOT + 2 * sub;
      if (2 * sub < NV)
        __hip_atomic_store(p, (unsigned long long)__double_as_longlong(dq[s & 1][2 * sub][cout]), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      if (2 * sub + 1 < NV)
        __hip_atomic_store(p + 1, (unsigned long long)__double_as_longlong(dq[s & 1][2 * sub + 1][cout]),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const int i = s - j - k;
    if (inside && i >= 1 && i <= ni) {
      double2 *const W = (double2 *)b.sk + (long)s * plane + o_dq;
#pragma unroll
      for (int m = 0; m < C::NVP; ++m)
        W[8 * m] = make_double2(dq[s & 1][2 * m][lane], 2 * m + 1 < NV ? dq[s & 1][2 * m + 1 < NV ? 2 * m + 1 : 0][lane] : 0.0);
    }
  };
  take(first - sg);
  lu_barrier();
  for (int m = 0; m < n; ++m) {
    const int s = first + sg * m;
    if (m > 0) give(s - sg);
    if (m + 1 < n) take(s);
    lu_barrier();
  }
  give(first + sg * (n - 1));
}

// qp += delQ in conservative variables (src/lusgs.f90:456-486, 996-1022)
template <int NV>
__global__ void __launch_bounds__(256) k_lusgs_apply(Blk b) {
  using C = Sk<NV>;
  int i, j;
  if (!flat_ij(b.imx - 1, b.jmx - 1, i, j, (int)blockIdx.x)) return;
  i += 1;
  j += 1;
  const int k = blockIdx.y + 1;
  const long c = ci(b, i, j, k), nc = b.nc;
  const double2 *const at = sk_at(b, C::NP, i + j + k, sk_pos(b, j, k)) + 8 * C::DQ;
  double dq[2 * C::NVP];
#pragma unroll
  for (int m = 0; m < C::NVP; ++m) {
    const double2 v = at[8 * m];
    dq[2 * m] = v.x;
    dq[2 * m + 1] = v.y;
  }
  const double gm = b.gm;
  double q[NV], U[NV];
  lu_load<NV>(b, c, q);
  U[0] = q[0];
  U[1] = q[0] * q[1];
  U[2] = q[0] * q[2];
  U[3] = q[0] * q[3];
  U[4] = (q[4] / (gm - 1.0)) + (0.5 * q[0] * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]));
  if constexpr (NV == 7) {
    U[5] = q[0] * q[5];
    U[6] = q[0] * q[6];
  }
  if constexpr (NV == 6) U[5] = q[0] * q[5];
#pragma unroll
  for (int l = 0; l < NV; ++l) U[l] = U[l] + dq[l];
  b.qp[c] = U[0];
  b.qp[nc + c] = U[1] / U[0];
  b.qp[2 * nc + c] = U[2] / U[0];
  b.qp[3 * nc + c] = U[3] / U[0];
  b.qp[4 * nc + c] = (gm - 1.0) * (U[4] - (0.5 * (U[1] * U[1] + U[2] * U[2] + U[3] * U[3]) / U[0]));
  if constexpr (NV == 7) {
    if (b.kkl) {  // src/lusgs.f90:1502-1505
      b.qp[5 * nc + c] = fmx(U[5] / U[0], 1.e-8);
      b.qp[6 * nc + c] = fmx(U[6] / U[0], 1.e-8);
    } else {
      if (U[5] > 0) b.qp[5 * nc + c] = U[5] / U[0];
      if (U[6] > 0) b.qp[6 * nc + c] = U[6] / U[0];
    }
  }
  if constexpr (NV == 6) b.qp[5 * nc + c] = fmx(U[5] / U[0], 1.e-8);  // src/lusgs.f90:2096-2097
}

}  // namespace fest
