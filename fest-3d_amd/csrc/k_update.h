// k_update.h -- residue (flux divergence, src/face/flux/convective/
// scheme.f90:111-141), SST source (src/source.f90:158-270), the
// conservative RK stage update (src/update.f90:367-485), the local/global
// time step (src/time.f90:122-531) and the residual norms
// (src/resnorm.f90:171-225).
#pragma once
// the residual kernels let multiply-adds fuse into FMA: results differ from
// the unfused reference order by rounding only, far inside the 1e-12 parity
// bound, and the FP64 instruction count, which bounds these kernels, drops
#pragma clang fp contract(fast)
#include "blk.h"

namespace fest {

// Temp = p/(R rho) on the whole padded array (src/update.f90:170) and the RK
// base U_store = qp (src/update.f90:178)
__device__ __forceinline__ void k_step_begin_b(const Blk &b, const Wg &wg, int store_u) {
  long t = (long)wg.x * blockDim.x + threadIdx.x;
  if (t >= b.nc) return;
  double rho = b.qp[t];
  b.temp[t] = b.qp[4 * b.nc + t] / (b.R * rho);
  if (store_u)
    for (int l = 0; l < b.nv; ++l) b.ust[(long)l * b.nc + t] = b.qp[(long)l * b.nc + t];
}
__global__ void k_step_begin(Blk b, int store_u) {
  k_step_begin_b(b, FEST_WG_HW, store_u);
}

// q = a U_store + c q over the whole padded primitive array, the TVD-RK
// blends of src/update.f90:204,206,213
__global__ void k_blend(Blk b, double a, double c) {
  long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= b.nc * b.nv) return;
  b.qp[t] = a * b.ust[t] + c * b.qp[t];
}

__device__ __forceinline__ double sspd(const Blk &b, int d, long o) { return b.csnd[d][o]; }

// local time step of one cell (src/time.f90:122-246, 366-531)
// Memory bound.  The face metrics, speeds and velocities are asked for at once,
// the centres with them, and the viscous limit's six quotients serve mu and
// mu_t alike (one each, times two, in turn before): 256 x 128 x 128 256 -> 234
// us (1.35 GB, 5.8 TB/s), 24 blocks of 1.1 M cells 75 -> 55, 128 x 96 x 64 49 -> 42.
__device__ __forceinline__ void k_dt_b(const Blk &b, const Wg &wg) {
  int i, j;
  bool active = flat_ij(b.imx - 1, b.jmx - 1, i, j, (int)wg.x);
  i += 1;
  j += 1;
  const int k = wg.y + 1;
  active = active && k <= b.kmx - 1;
  double dtv = 1e300;
  if (active) {
    const long nc = b.nc;
    const double *qp = b.qp;
    const long c = ci(b, i, j, k), st[3] = {1, b.pi, (long)b.pi * b.pj};
    // faces 0..2 the cell's lower ones along i, j, k, 3..5 its upper ones with
    // the neighbour's velocity, as the reference takes them
    double n[6][4], cs[6], V[4][3];
    const long f[6] = {fi(b, 0, i, j, k),     fi(b, 1, i, j, k),     fi(b, 2, i, j, k),
                       fi(b, 0, i + 1, j, k), fi(b, 1, i, j + 1, k), fi(b, 2, i, j, k + 1)};
    const long o[6] = {fli(b, 0, i, j, k),     fli(b, 1, i, j, k),     fli(b, 2, i, j, k),
                       fli(b, 0, i + 1, j, k), fli(b, 1, i, j + 1, k), fli(b, 2, i, j, k + 1)};
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      V[0][l] = qp[(l + 1) * nc + c];
#pragma unroll
      for (int d = 0; d < 3; ++d) V[d + 1][l] = qp[(l + 1) * nc + c + st[d]];
    }
#pragma unroll
    for (int s = 0; s < 6; ++s) {
      const int d = s % 3;
      n[s][0] = b.fx[d][f[s]]; n[s][1] = b.fy[d][f[s]]; n[s][2] = b.fz[d][f[s]]; n[s][3] = b.fA[d][f[s]];
      cs[s] = sspd(b, d, o[s]);
    }
    const double vol = b.vol[c];
    __builtin_amdgcn_sched_barrier(0);
    // the viscous part's inputs: the neighbours' centres, then the densities
    // and viscosities
    const bool visc = b.mu_ref != 0.0;
    double x[7][3], rho[4], mu[4], mt[4];
    if (visc) {
      const double *cc[3] = {b.cx, b.cy, b.cz};
#pragma unroll
      for (int l = 0; l < 3; ++l) {
        x[6][l] = cc[l][c];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          x[d][l] = cc[l][c - st[d]];
          x[d + 3][l] = cc[l][c + st[d]];
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    double lsum = 0.0;
#pragma unroll
    for (int s = 0; s < 6; ++s) {
      const double *v = V[s < 3 ? 0 : s - 2];
      lsum = lsum + n[s][3] * (fabs((v[0] * n[s][0]) + (v[1] * n[s][1]) + (v[2] * n[s][2])) + cs[s]);
    }
    dtv = 1. / lsum;
    dtv = dtv * vol * b.CFLv;
    if (visc) {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const long cm = m ? c + st[m - 1] : c;
        rho[m] = qp[cm];
        mu[m] = b.mu[cm];
        mt[m] = b.turb ? b.mut[cm] : 0.0;
      }
      __builtin_amdgcn_sched_barrier(0);
      // A / (rho |centre distance . n|) of each face, for mu and mu_t alike
      double w[6];
#pragma unroll
      for (int s = 0; s < 6; ++s) {
        const double *u = s < 3 ? x[s] : x[6], *v = s < 3 ? x[6] : x[s];
        w[s] = n[s][3] / (rho[s < 3 ? 0 : s - 2] *
                          fabs(((u[0] - v[0]) * n[s][0]) + ((u[1] - v[1]) * n[s][1]) + ((u[2] - v[2]) * n[s][2])));
      }
      for (int pass = 0; pass < 2; ++pass) {
        if (pass == 1 && !b.turb) break;
        const double *m = pass == 0 ? mu : mt;
        double ls = ((w[0] + w[1]) + w[2]) * m[0] + w[3] * m[1] + w[4] * m[2] + w[5] * m[3];
        ls = b.gm * ls / (pass == 0 ? b.Pr : b.tPr);
        ls = 2. / (ls + (2. * b.CFLv * vol / dtv));
        dtv = b.CFLv * (ls * vol);
      }
    }
    b.dt[ri(b, i, j, k)] = dtv;
  }
  if (!b.time_local) {
    // block minimum for the global step (src/time.f90:248-289)
    __shared__ double smin[256];
    int tid = threadIdx.x;
    smin[tid] = dtv;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
      if (tid < st) smin[tid] = fmn(smin[tid], smin[tid + st]);
      __syncthreads();
    }
    if (tid == 0) {
      long blk = wg.x + (long)wg.nx * wg.y;
      b.red[blk] = smin[0];
    }
  }
}
__global__ void __launch_bounds__(256) k_dt(Blk b) {
  k_dt_b(b, FEST_WG_HW);
}

// global step: minimum of the block minima, broadcast into delta_t
__global__ void k_dt_min(Blk b, long nblk) {
  __shared__ double s[256];
  double m = 1e300;
  for (long t = threadIdx.x; t < nblk; t += blockDim.x) m = fmn(m, b.red[t]);
  s[threadIdx.x] = m;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (threadIdx.x < st) s[threadIdx.x] = fmn(s[threadIdx.x], s[threadIdx.x + st]);
    __syncthreads();
  }
  if (threadIdx.x == 0) b.dtmin[0] = s[0];
}
__global__ void k_dt_fill(Blk b, int use_fixed) {
  long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= b.nres) return;
  b.dt[t] = use_fixed ? b.global_dt : b.dtmin[0];
}

enum { UPD_FIRST = 1, UPD_LAST = 2, UPD_WRITE_RES = 4, UPD_APPLY = 8, UPD_STORE = 16 };

// the SA point-implicit destruction factor of the update (src/update.f90:
// 405-420): xi takes the conservative nu-tilde times the current density
__device__ __forceinline__ double sa_implicit(const Blk &b, long c, long gi, double u1_0, double u1_5, double dt) {
  const double *gx = b.g[0], *gy = b.g[1], *gz = b.g[2];
  const long ngr = b.ngr;
  double vort = sqrt(sqd(gy[2 * ngr + gi] - gz[ngr + gi]) + sqd(gz[gi] - gx[2 * ngr + gi]) +
                     sqd(gx[ngr + gi] - gy[gi]));
  double dist = b.dist[c];
  double kd = Sa::kappa * dist, kd2 = kd * kd;
  double xi = u1_5 * b.qp[c] / b.mu[c];
  double x3 = (xi * xi) * xi;
  double fv1 = x3 / (x3 + Sa::cv1_3);
  double fv2 = 1.0 - xi / (1 + xi * fv1);
  double scap = vort + u1_5 * fv2 / kd2;
  double rsa = fmn(u1_5 / (scap * kd2), 10.0);
  double r6 = ((((rsa * rsa) * rsa) * rsa) * rsa) * rsa;
  double g = rsa + Sa::cw2 * (r6 - rsa);
  double g6 = ((((g * g) * g) * g) * g) * g;
  double fw = g * pow((1.0 + Sa::cw3_6) / (g6 + Sa::cw3_6), 1.0 / 6.0);
  return 1. + ((-1.0 * u1_0 * Sa::cb1 * scap) + (2.0 * u1_0 * Sa::cw1 * fw * u1_5 / (dist * dist))) * dt;
}

// residue + SST/SA source, then (UPD_APPLY) the conservative update of the cell.
// Bound by memory: 1.79 GB (a stage's average) at 256 x 128 x 128 (SST) in 345
// us, 5.2 TB/s.  The stage's base state, R accumulator, source, volume and time
// step are asked for ahead of the fluxes and those two variables ahead of their
// sums, all of it with the variable count known at compile time; one variable
// after another, each flux when its difference came up, took 355 us there, 7.9
// us (now 4.7) at 64 x 64 x 4 and 64 us (now 43) over 24 blocks of 1.1 M cells.
// What the turbulence models' implicit factors read follows the sums.
template <int NV>
__device__ __forceinline__ void k_update_b(const Blk &b, const Wg &wg, double TF, double SF, int flags) {
  int i, j;
  if (!flat_ij(b.imx - 1, b.jmx - 1, i, j, plane_block(wg, b.xcd_remap))) return;
  i += 1;
  j += 1;
  const int k = wg.y + 1;
  if (k > b.kmx - 1) return;
  constexpr int nv = NV;
  const long nc = b.nc;
  long c = ci(b, i, j, k);
  long r = ri(b, i, j, k);
  long F0 = fli(b, 0, i, j, k), G0 = fli(b, 1, i, j, k), H0 = fli(b, 2, i, j, k);
  long sG = b.nfi[1], sH = (long)b.nfi[2] * b.nfj[2];
  const bool apply = flags & UPD_APPLY, more = apply && (flags & UPD_STORE) && !(flags & UPD_FIRST);
  const double *Qu = (flags & UPD_STORE) ? b.ust : b.qp;
  double R[NV], q0[NV], r0[NV], src[3] = {0.0, 0.0, 0.0};
  double dt = 0.0, vol = 0.0;
  if (apply) {
    dt = b.dt[r];
    vol = b.vol[c];
#pragma unroll
    for (int l = 0; l < nv; ++l) q0[l] = Qu[(long)l * nc + c];
  }
  if (more)
#pragma unroll
    for (int l = 0; l < nv; ++l) r0[l] = b.rst[(long)l * b.nres + r];
  if (nv >= 6) src[0] = b.src[r];
  if (nv >= 7) src[1] = b.src[b.nres + r];
  if (nv == 8) src[2] = b.src[2 * b.nres + r];
  // FP32 mode: the face fluxes are stored in FP32, the sums taken in FP64
  auto sums = [&](auto z) {
    using S = decltype(z);
    constexpr int AHEAD = 2;
    S w[AHEAD + 1][6];
    auto load = [&](int l, S (&f)[6]) {
      const S *F = (const S *)b.flux[0] + (long)l * b.nfl[0], *G = (const S *)b.flux[1] + (long)l * b.nfl[1],
              *H = (const S *)b.flux[2] + (long)l * b.nfl[2];
      f[0] = F[F0]; f[1] = F[F0 + 1];
      f[2] = G[G0]; f[3] = G[G0 + sG];
      f[4] = H[H0]; f[5] = H[H0 + sH];
    };
#pragma unroll
    for (int l = 0; l < AHEAD; ++l) load(l, w[l]);
#pragma unroll
    for (int l = 0; l < nv; ++l) {
      if (l + AHEAD < nv) load(l + AHEAD, w[(l + AHEAD) % (AHEAD + 1)]);
      __builtin_amdgcn_sched_barrier(0);
      const S(&f)[6] = w[l % (AHEAD + 1)];
      R[l] = ((double)f[1] - (double)f[0]) + ((double)f[3] - (double)f[2]) + ((double)f[5] - (double)f[4]);
    }
  };
  if (b.fp32) sums(0.0f);
  else sums(0.0);
  if constexpr (nv >= 7) {
    // SST source (src/source.f90:158-270), computed with the gradients
    R[5] = R[5] - src[0];
    R[6] = R[6] - src[1];
  }
  if constexpr (nv == 8) R[7] = R[7] - src[2];  // src/source.f90:454-456
  if constexpr (nv == 6) R[5] = R[5] - src[0];  // SA source (src/source.f90:835-983)
  if (flags & UPD_WRITE_RES)
#pragma unroll
    for (int l = 0; l < nv; ++l) b.res[(long)l * b.nres + r] = R[l];
  if (!apply) return;
  // src/update.f90:367-485
  const double gm = b.gm;
  double u1[NV], u2[NV];
  u1[0] = q0[0];
#pragma unroll
  for (int l = 1; l < nv; ++l) u1[l] = q0[l] * u1[0];
  u1[4] = (u1[4] / (gm - 1.) + 0.5 * (u1[1] * u1[1] + u1[2] * u1[2] + u1[3] * u1[3])) / u1[0] + 0.0;
  if constexpr (nv == 6) R[5] = R[5] / sa_implicit(b, c, gri(b, i, j, k), u1[0], u1[5], dt);
  if constexpr (nv >= 7) {
  if (b.kkl) {
    // k-kL point-implicit destruction, sqrt(rho) in the k factor
    // (src/update.f90:399-404)
    const double mu = b.mu[c], dist = b.dist[c];
    const double eta = u1[0] * dist * (sqrt(0.3 * u1[5]) / (20 * mu));
    const double fphi = (1 + 4.7 * eta) / (1 + ((eta * eta) * eta) * eta);
    const double d2 = sqd(dist);
    R[5] = R[5] / (1. + ((2.5 * ((pow(0.09, 0.75)) * sqrt(u1[0]) * (pow(u1[5], 1.5)) / fmx(u1[6], 1.e-20)) +
                          (2 * mu / d2)) * dt));
    R[6] = R[6] / (1. + (6 * mu * fphi / d2) * dt);
  } else {
    double F1 = b.f1[c];
    double beta = 0.075 * F1 + (1. - F1) * 0.0828;
    double w7 = b.qp[6 * nc + c];
    R[5] = R[5] / (1 + (beta * w7 * dt));
    R[6] = R[6] / (1 + (2 * beta * w7 * dt));
  }
  }
  if (flags & UPD_STORE) {
#pragma unroll
    for (int l = 0; l < nv; ++l) {
      double rn = more ? r0[l] + SF * R[l] : 0.0 + SF * R[l];
      if (flags & UPD_LAST) R[l] = rn;
      else b.rst[(long)l * b.nres + r] = rn;
    }
  }
  double fac = TF * dt / vol;
#pragma unroll
  for (int l = 0; l < nv; ++l) u2[l] = u1[l] - R[l] * fac;
#pragma unroll
  for (int l = 1; l < nv; ++l) u2[l] = u2[l] / u2[0];
  u2[4] = (gm - 1.) * u2[0] * (u2[4] - (0.5 * (u2[1] * u2[1] + u2[2] * u2[2] + u2[3] * u2[3])) - 0.0);
  bool bad = (u2[0] < 0.) || (u2[4] < 0.);
#pragma unroll
  for (int l = 0; l < nv; ++l) bad |= isnan(u2[l]);
  if (bad) {
    atomicOr(b.err, ERR_NONPHYS);
    return;
  }
  // variables 1-5 and the two turbulence variables; lctm2015's
  // intermittency is not written back (src/update.f90:456-484)
#pragma unroll
  for (int l = 0; l < 5; ++l) b.qp[(long)l * nc + c] = u2[l];
  if constexpr (nv >= 7) {
    if (u2[5] >= 0.) b.qp[5 * nc + c] = u2[5];
    if (u2[6] >= 0.) b.qp[6 * nc + c] = u2[6];
  }
  if constexpr (nv == 6) b.qp[5 * nc + c] = fmx(u2[5], 1.e-12);
}
template <int NV>
__global__ void __launch_bounds__(256) k_update(Blk b, double TF, double SF, int flags) {
  k_update_b<NV>(b, FEST_WG_HW, TF, SF, flags);
}

// NORM_ACC sums of a norm: the mass imbalance and up to 8 variables.
constexpr int NORM_ACC = 9;

// the sums of acc over a 256-thread work-group, in s[0 .. NORM_ACC): the
// waves take the sums in turn, 4 values a lane out of LDS and then across the
// lanes, one barrier each side of it
__device__ __forceinline__ void norm_sums(const double *acc, double (*s)[256], double *sum) {
#pragma unroll
  for (int l = 0; l < NORM_ACC; ++l) s[l][threadIdx.x] = acc[l];
  __syncthreads();
  const int lane = threadIdx.x & 63;
  for (int l = threadIdx.x >> 6; l < NORM_ACC; l += 4) {
    double v = (s[l][lane] + s[l][lane + 128]) + (s[l][lane + 64] + s[l][lane + 192]);
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o);
    if (lane == 0) sum[l] = v;
  }
  __syncthreads();
}

// per-block sums of residue^2 and of the boundary mass fluxes.  The residue
// is taken flat, so that every lane of every wave has a cell whatever the row
// length, its n_var loads in flight together: 64 x 64 x 4 x 5 15 -> 6 us,
// 256 x 128 x 128 x 7 90 -> 70 us (3.3 TB/s) against rows taken in turn, with
// the mass fluxes tested for at every cell and an 8-barrier tree.
__global__ void __launch_bounds__(256) k_norm_partial(Blk b, double *red) {
  __shared__ double s[NORM_ACC][256];
  __shared__ double sum[NORM_ACC];
  const int nv = b.nv;
  double acc[NORM_ACC] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  const int ni = b.imx - 1, nj = b.jmx - 1, nk = b.kmx - 1;
  const long step = (long)gridDim.x * 256, t0 = (long)blockIdx.x * 256 + threadIdx.x;
  for (long t = t0; t < b.nres; t += step) {
#pragma unroll
    for (int l = 0; l < NORM_ACC - 1; ++l)
      if (l < nv) {
        const double v = b.res[(long)l * b.nres + t];
        acc[1 + l] += v * v;
      }
  }
  // the mass fluxes of the boundary faces (FP32 in the FP32 mode), each
  // direction's first face plus and its last face minus
  auto fl = [&](int d, long o) -> double {
    return b.fp32 ? (double)((const float *)b.flux[d])[o] : b.flux[d][o];
  };
  for (long t = t0; t < (long)nj * nk; t += step) {
    const int j = (int)(t % nj) + 1, k = (int)(t / nj) + 1;
    acc[0] += fl(0, fli(b, 0, 1, j, k)) - fl(0, fli(b, 0, b.imx, j, k));
  }
  for (long t = t0; t < (long)ni * nk; t += step) {
    const int i = (int)(t % ni) + 1, k = (int)(t / ni) + 1;
    acc[0] += fl(1, fli(b, 1, i, 1, k)) - fl(1, fli(b, 1, i, b.jmx, k));
  }
  for (long t = t0; t < (long)ni * nj; t += step) {
    const int i = (int)(t % ni) + 1, j = (int)(t / ni) + 1;
    acc[0] += fl(2, fli(b, 2, i, j, 1)) - fl(2, fli(b, 2, i, j, b.kmx));
  }
  norm_sums(acc, s, sum);
  if (threadIdx.x < NORM_ACC) red[(long)blockIdx.x * NORM_ACC + threadIdx.x] = sum[threadIdx.x];
}

// final norms, src/resnorm.f90:128-225: 256 threads sum the block
// partials in a fixed order (strided, then as norm_sums).  out receives the
// n_var+1 norms and, with shares, from out[NORM_SHARE] the block's unassembled
// share.  With err, the block's error word goes to out[NORM_SLOTS], so that a
// host that reads out needs no second transfer.
__global__ void __launch_bounds__(256) k_norm_final(Blk b, int nblk, const double *red, double *out, int shares,
                                                    const unsigned *err) {
  __shared__ double s[NORM_ACC][256];
  __shared__ double sum[NORM_ACC];
  double part[NORM_ACC] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int t = threadIdx.x; t < nblk; t += blockDim.x)
#pragma unroll
    for (int l = 0; l < NORM_ACC; ++l) part[l] += red[(long)t * NORM_ACC + l];
  norm_sums(part, s, sum);
  if (err && threadIdx.x == NORM_ACC) out[NORM_SLOTS] = (double)*err;
  const int l = threadIdx.x;
  if (l > b.nv) return;
  const double v = b.vel_mag;
  // lctm2015's intermittency: resnorm.f90:128-168 leaves Res_scale(8)
  // unset, so the reference's value is undefined; scaled here like the
  // other turbulence variables
  const double scale = l == 0 ? 1.
                       : l == 1 ? b.rho_inf * v
                       : l <= 4 ? b.rho_inf * v * v
                       : l == 5 ? (0.5 * b.rho_inf * (v * v * v) + ((b.gm / (b.gm - 1.)) * b.p_inf))
                       : l == 6 ? b.rho_inf * v * (b.ng == 5 ? b.tv_inf : b.tk_inf)  // nu-tilde for SA (resnorm.f90:158)
                       : l == 7 ? b.rho_inf * v * (b.kkl ? b.tkl_inf : b.tw_inf)     // kL for k-kL (resnorm.f90:153)
                                : b.rho_inf * v * b.tgm_inf;
  // the norm, and the block's share before the cross-block assembly
  // (src/resnorm.f90:171-225): the signed mass imbalance and sum(R_l^2)/scale_l^2
  const double share = l == 0 ? sum[0] / scale : sum[l] / (scale * scale);
  out[l] = l == 0 ? fabs(share) : sqrt(share);
  if (shares) out[NORM_SHARE + l] = share;
}

// the blocks' error words into host memory, one lane a block
__global__ void k_report(const unsigned *const *err, int n, unsigned *out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) out[t] = *err[t];
}
__global__ void k_report_one(const unsigned *err, unsigned *out) { *out = *err; }

}  // namespace fest
