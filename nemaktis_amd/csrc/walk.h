// Line solvers on the slab material (walk_kernels.hip), FP64.
#pragma once

#include "device_common.h"
#include "kernels.h"

namespace nmk {

// Slab material of a launch: per slot walk_points(Mx, My) points of five
// 16-byte values, the line axis slow -- nat for lines along y, tr for lines
// along x (WalkRing)
struct WalkMaterial {
    const c64 *nat, *tr;
};

// launch shape of one axis: chunks of a line, lines per block (16, 8, 4 or 2)
struct WalkShape {
    LinePlan lp;
    int W;
};

// LDS distance of two lines of the block's transposed result
__host__ __device__ inline int walk_line_pitch(int M) { return M + (M >> 3) + 1; }

// see k_walk; per_slot: propagations per wavelength slot
void launch_walk(int axis, int neumann, const c64 *src, c64 *dst, const c64 *accin, c64 *acc, bool flip,
                 const WalkMaterial &wm, const Geo &g, const SlotParams *sp, const PropParams *pp, int nprops,
                 int per_slot, const WalkShape &sh, hipStream_t st);

}  // namespace nmk
