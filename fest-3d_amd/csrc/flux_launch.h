// flux_launch.h -- launchers of the face-sweep kernels (k_sweeps, km_sweeps),
// compiled in translation units of their own, one per variable count
// (flux_launch.hip): the sweeps' many specialisations (variables x
// reconstruction x precision) then build beside the rest of the library.
#pragma once
#include <hip/hip_runtime.h>

#include "blk.h"

namespace fest {

struct WorkItem;

// the face sweeps of one block of NV variables (k_sweeps), count work-groups:
// all three (only -1) or one
template <int NV>
void launch_sweeps(const Blk &b, const struct Sweeps &s, int only, int count, hipStream_t st, int store_csnd);

// the face sweeps over the work list of a batched group step of blocks of NV
// (5 or 7) variables (n items, `grid` work-groups); b0 is any block of the
// group (they share one kernel variant)
template <int NV>
void launch_sweeps_batched(const Blk &b0, hipStream_t st, const Blk *blks, const WorkItem *items, int n,
                           unsigned grid, int store_csnd);

}  // namespace fest
