// flux_launch.hip -- launchers of the face sweeps for FEST_NV variables
// (compiled once for each of 5, 6, 7 and 8; declared in flux_launch.h),
// specialised on the reconstruction and the precision.
#include <hip/hip_runtime.h>

#include "flux_launch.h"
#include "k_flux.h"
#include "k_flux_walk.h"

namespace fest {
namespace {

constexpr int NV = FEST_NV;

template <bool FLAT, typename T>
void launch_recon(const Blk &b, const Sweeps &s, int only, int count, hipStream_t st, int store_csnd) {
  const dim3 g((unsigned)count), t(256);
  switch (b.recon) {
    case 0: hipLaunchKernelGGL((k_sweeps<NV, 0, FLAT, T>), g, t, 0, st, b, s, only, store_csnd); break;
    case 1: hipLaunchKernelGGL((k_sweeps<NV, 1, FLAT, T>), g, t, 0, st, b, s, only, store_csnd); break;
    case 2: hipLaunchKernelGGL((k_sweeps<NV, 2, FLAT, T>), g, t, 0, st, b, s, only, store_csnd); break;
    case 3: hipLaunchKernelGGL((k_sweeps<NV, 3, FLAT, T>), g, t, 0, st, b, s, only, store_csnd); break;
    default: hipLaunchKernelGGL((k_sweeps<NV, 4, FLAT, T>), g, t, 0, st, b, s, only, store_csnd); break;
  }
}
// the k faces of a 2-D grid (one cell in k) carry no convective flux
template <typename T>
void launch_flat(const Blk &b, const Sweeps &s, int only, int count, hipStream_t st, int store_csnd) {
  if (b.kmx == 2) launch_recon<true, T>(b, s, only, count, st, store_csnd);
  else launch_recon<false, T>(b, s, only, count, st, store_csnd);
}
template <typename T>
void batched_recon(int recon, hipStream_t st, const Blk *blks, const WorkItem *items, int n, unsigned grid,
                   int store_csnd) {
  const dim3 g(grid), t(256);
  switch (recon) {
    case 0: hipLaunchKernelGGL((km_sweeps<NV, 0, T>), g, t, 0, st, blks, items, n, store_csnd); break;
    case 1: hipLaunchKernelGGL((km_sweeps<NV, 1, T>), g, t, 0, st, blks, items, n, store_csnd); break;
    case 2: hipLaunchKernelGGL((km_sweeps<NV, 2, T>), g, t, 0, st, blks, items, n, store_csnd); break;
    case 3: hipLaunchKernelGGL((km_sweeps<NV, 3, T>), g, t, 0, st, blks, items, n, store_csnd); break;
    default: hipLaunchKernelGGL((km_sweeps<NV, 4, T>), g, t, 0, st, blks, items, n, store_csnd); break;
  }
}

}  // namespace

// FP64 face arithmetic, or FP32 when the handle was created with
// FEST_PREC_FP32_FLUX (lctm2015, 8 variables, runs in FP64 only)
template <>
void launch_sweeps<NV>(const Blk &b, const Sweeps &s, int only, int count, hipStream_t st, int store_csnd) {
  if constexpr (NV != 8) {
    if (b.fp32) {
      launch_flat<float>(b, s, only, count, st, store_csnd);
      return;
    }
  }
  launch_flat<double>(b, s, only, count, st, store_csnd);
}

#if FEST_NV == 5 || FEST_NV == 7
template <>
void launch_sweeps_batched<NV>(const Blk &b0, hipStream_t st, const Blk *blks, const WorkItem *items, int n,
                               unsigned grid, int store_csnd) {
  if (b0.fp32) batched_recon<float>(b0.recon, st, blks, items, n, grid, store_csnd);
  else batched_recon<double>(b0.recon, st, blks, items, n, grid, store_csnd);
}
#endif

}  // namespace fest
