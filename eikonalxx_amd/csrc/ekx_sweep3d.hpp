// ekx_sweep3d.hpp -- what the 3D sweep kernels share.
#pragma once
#include "ekx_device.hpp"

namespace ekx
{

// The Cartesian update of a problem's grid: non-uniform, or uniform with or
// without the roots' range tests (cartesian_uniform3d).
enum Grid3D { kNonUniform, kUniform, kUniformScaled };

// First node of each permuted axis that a sweep updates: 1 for refinement
// sweeps (getLoopLimits, solverUtilities3d.hpp:944-1052), the source octant
// for initialization sweeps (:1075-1184).
struct Octant
{
    int jx0, jy0, jz0;
};

__device__ __forceinline__ Octant sweep_octant(const Problem3D &p, int sweep,
                                               int initialize)
{
    Octant o{1, 1, 1};
    if (initialize)
    {
        int negX = sweep & 1, negY = (sweep >> 1) & 1, negZ = (sweep >> 2) & 1;
        o.jx0 = negX ? max(p.nx - 2 - p.srcCellX, 1) : max(1, p.srcCellX);
        o.jy0 = negY ? max(p.ny - 2 - p.srcCellY, 1) : max(1, p.srcCellY);
        o.jz0 = negZ ? max(p.nz - 2 - p.srcCellZ, 1) : max(1, p.srcCellZ);
    }
    return o;
}

} // namespace ekx
