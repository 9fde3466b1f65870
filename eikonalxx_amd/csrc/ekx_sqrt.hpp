// ekx_sqrt.hpp -- the FP64 square root of the local updates.
#pragma once
#include <hip/hip_runtime.h>

namespace ekx
{

// Correctly rounded square root of a double in [2^-767, DBL_MAX]: the
// reciprocal-square-root estimate refined by one Goldschmidt step and two
// corrections with exact FMA residuals (d = a - g*g).  This is the sequence
// the compiler emits for sqrt(double) on gfx950 minus its range handling:
// below 2^-767 it scales the argument by 2^256 (so that the residuals stay
// normal) and it returns zero and infinity unchanged, which costs 8 of its
// 18 instructions.  The callers pass positive determinants of travel-time
// differences, so the unscaled form serves every lane except for arguments
// under 2^-767 (zero included), which take the full sqrt.
__device__ __forceinline__ double sqrt_normal_range(double a)
{
    const double y = __builtin_amdgcn_rsq(a);
    double g = a*y;
    double h = y*0.5;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    double d = fma(-g, g, a);
    h = fma(h, r, h);
    g = fma(d, h, g);
    d = fma(-g, g, a);
    return fma(d, h, g);
}

} // namespace ekx
