// Line solvers on the slab material (walk_kernels.hip), FP64.
#pragma once

#include "device_common.h"
#include "kernels.h"

namespace nmk {

// Factors of the mu*R stencils (R = (D S^-1 + S^-1 D)/4 + i W, mu = i dZ/2) at one wavelength: (dZ/8) times 1/dX^2,
// 1/dY^2 and 1/(4 dX dY), and dZ/2 times 1/(8 dX), 1/(8 dY).  A table of all wavelengths belongs to the solvers' buffers
// (divided by each block of the launches instead: 64^2 x 20 1.112 -> 1.134 ms, 161^2 x 161 16.9 -> 17.1).
struct WalkSteps {
    double rx2, ry2, rxy, gx, gy;
};

// Slab material of a launch: per slot walk_points(Mx, My) points of five
// 16-byte values, the line axis slow -- nat for lines along y, tr for lines
// along x (WalkRing); the stencils' factors of every wavelength
struct WalkMaterial {
    const c64 *nat, *tr;
    const WalkSteps *steps;
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
                 const WalkMaterial &wm, const Geo &g, const PropParams *pp, int nprops, int per_slot,
                 const WalkShape &sh, hipStream_t st);

}  // namespace nmk
