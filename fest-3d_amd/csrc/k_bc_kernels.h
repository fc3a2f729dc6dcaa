// k_bc_kernels.h -- the per-block kernels of the ghost-cell passes, whose
// bodies are in k_bc.h.  Not templates: one translation unit includes this.
#pragma once
#include "k_bc.h"

namespace fest {

// faces first .. first + gridDim.z - 1
__global__ void __launch_bounds__(256) k_bc_face(Blk b, int first, int current_iter) {
  const Wg wg{(int)blockIdx.x, (int)blockIdx.y, first + (int)blockIdx.z, 0};
  k_bc_face_b(b, wg, current_iter);
}
__global__ void __launch_bounds__(256) k_bc_edges(Blk b) {
  k_bc_edges_b(b, FEST_WG_HW);
}

}  // namespace fest
