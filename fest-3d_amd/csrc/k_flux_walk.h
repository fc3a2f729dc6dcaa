// k_flux_walk.h -- the face sweeps of a batched group step: one launch over
// the work list of all blocks' tiles in all directions, running k_flux_b on
// each tile.
#pragma once
#include "k_flux.h"
#include "k_walk.h"

namespace fest {

// an item's z: its direction and, from bit 8, the block's tile width
template <int NV, int RECON, typename T>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
km_sweeps(const Blk *__restrict__ blks, const WorkItem *__restrict__ items, int n, int store_csnd) {
  FEST_WALK((k_sweeps_b<NV, RECON, false, T>(b, it.z & 255, wg, it.z >> 8, store_csnd)))
}

}  // namespace fest
