// ekx_local3d.hpp -- the 3D local (per-node) update on the device.
//
// This is the arithmetic of finiteDifference in
// include/private/solverUtilities3d.hpp (uniform :258-558, non-uniform
// :562-824) and computeAnalyticalTravelTime (:138-208).  Every expression
// keeps the reference's operation order: the library is compiled with
// -ffp-contract=off, so in double precision the result is the same value
// the reference produces, bit for bit, given correctly rounded sqrt and
// division.
//
// Neighbour naming follows the reference (in the sweep's own frame, where
// the wave travels towards +x, +y, +z):
//   t1 = T(x-1,y,z)  t2 = T(x-1,y-1,z)  t3 = T(x,y-1,z)  t4 = T(x,y,z-1)
//   t5 = T(x-1,y,z-1) t6 = T(x-1,y-1,z-1) t7 = T(x,y-1,z-1)
//   s0 = cell(x-1,y-1,z-1), s1 = (x,y-1,z-1), s2 = (x,y,z-1),
//   s3 = (x-1,y,z-1), s4 = (x-1,y-1,z), s5 = (x,y-1,z), s7 = (x-1,y,z)
// (cells indexed by their lower corner, clamped to the model).
#pragma once
#include "ekx_device.hpp"
#include "ekx_sqrt.hpp"

namespace ekx
{

template <typename R> struct Math;
template <> struct Math<double>
{
    static __device__ __forceinline__ double min(double a, double b)
    { return fmin(a, b); }
    static __device__ __forceinline__ double max(double a, double b)
    { return fmax(a, b); }
    static __device__ __forceinline__ double fma(double a, double b, double c)
    { return ::fma(a, b, c); }
    static __device__ __forceinline__ double sqrt(double a)
    {
        double r = sqrt_normal_range(a);
        const bool normal = a >= 0x1p-767;
        // a wave-uniform branch, so that the full sqrt is not evaluated
        // alongside (lanes outside the range are overwritten here)
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(!normal) != 0, 0))
        {
            r = normal ? r : ::sqrt(a);
        }
        return r;
    }
    // of an argument known to lie in sqrt_normal_range's range
    static __device__ __forceinline__ double sqrt_in_range(double a)
    { return sqrt_normal_range(a); }
    // the same, or of zero: the root of the clamped argument, 2^-500, minus
    // itself (which changes no root of an argument in the range)
    static __device__ __forceinline__ double sqrt_or_zero(double a)
    { return sqrt_normal_range(fmax(a, 0x1p-1000)) - 0x1p-500; }
};
template <> struct Math<float>
{
    static __device__ __forceinline__ float min(float a, float b)
    { return fminf(a, b); }
    static __device__ __forceinline__ float max(float a, float b)
    { return fmaxf(a, b); }
    static __device__ __forceinline__ float fma(float a, float b, float c)
    { return ::fmaf(a, b, c); }
    // One-ulp hardware square root: the FP32 modes are validated against
    // the FP64 solve at 1e-5 relative, far above this rounding.
    static __device__ __forceinline__ float sqrt(float a)
    { return __builtin_amdgcn_sqrtf(a); }
    static __device__ __forceinline__ float sqrt_in_range(float a)
    { return sqrt(a); }
    static __device__ __forceinline__ float sqrt_or_zero(float a)
    { return sqrt(a); }
};

struct Sweep3D
{
    int signX, signY, signZ;        // getSweepFiniteDifferenceSigns
    int ixShift, iyShift, izShift;
};

// Sweep k (0..7): bit0 x decreasing, bit1 y decreasing, bit2 z decreasing
// (enums.hpp:66-76, solverUtilities3d.hpp:843-925).
__device__ __forceinline__ Sweep3D make_sweep3d(int sweep)
{
    Sweep3D s;
    int negX = sweep & 1, negY = (sweep >> 1) & 1, negZ = (sweep >> 2) & 1;
    s.signX = negX ? -1 : 1;
    s.signY = negY ? -1 : 1;
    s.signZ = negZ ? -1 : 1;
    s.ixShift = negX ? 1 : -1;
    s.iyShift = negY ? 1 : -1;
    s.izShift = negZ ? 1 : -1;
    return s;
}

// computeAnalyticalTravelTime (solverUtilities3d.hpp:138-156).
__device__ __forceinline__ double analytic_time3d(
    int ix, int iy, int iz, double dx, double dy, double dz,
    double xs, double ys, double zs, double slow)
{
    double x = ix*dx;
    double y = iy*dy;
    double z = iz*dz;
    double deltaX = x - xs;
    double deltaY = y - ys;
    double deltaZ = z - zs;
    double distance = ::sqrt(deltaX*deltaX + deltaY*deltaY + deltaZ*deltaZ);
    return slow*distance;
}

// computeAnalyticalTravelTime with derivatives (:180-208).
__device__ __forceinline__ void analytic_time_deriv3d(
    int ix, int iy, int iz, double dx, double dy, double dz,
    double xs, double ys, double zs, double slow,
    double &t, double &dtdx, double &dtdy, double &dtdz)
{
    double x = ix*dx;
    double y = iy*dy;
    double z = iz*dz;
    double deltaX = x - xs;
    double deltaY = y - ys;
    double deltaZ = z - zs;
    double distance = ::sqrt(deltaX*deltaX + deltaY*deltaY + deltaZ*deltaZ);
    t = slow*distance;
    dtdx = 0;
    dtdy = 0;
    dtdz = 0;
    if (distance > 0)
    {
        dtdx = (slow*deltaX)/distance;
        dtdy = (slow*deltaY)/distance;
        dtdz = (slow*deltaZ)/distance;
    }
}

__device__ __forceinline__ bool in_factored_box(const Problem3D &p, int ix,
                                                int iy, int iz)
{
    return !(abs(p.srcCellX - ix) > p.radius ||
             abs(p.srcCellY - iy) > p.radius ||
             abs(p.srcCellZ - iz) > p.radius);
}

// Cartesian branch, uniform grid (:281-371) in arithmetic R, from the cells'
// h s (h min(a, b) = min(h a, h b): rounding is monotone).  hs03: the
// minimum of hs0 and hs3; hs47 returns that of hs4 and hs7, which is the
// next plane's hs03.
//
// The candidates' minimum is kept in one running value instead of the
// reference's per-candidate HUGE defaults and final minimum: the same
// minimum over the valid candidates, except when no 2D or 3D candidate is
// valid and t1d exceeds HUGE, where the reference returns HUGE.  Neither
// is then below the node's own value (never above HUGE), so the update
// keeps the node and the field is the same.
//
// The instruction count bounds the sweeps, so: a pair's two causality tests
// are one (max <= min + hs: the other holds by itself), and the products by
// 2 and 1/2, which are exact, are fused into the sum after them (one
// rounding, the reference's).  SCALED: every hs at least 2^-300, so a
// positive 2D determinant 2 hs hs - c c is hs hs-sized or, where its terms
// cancel, a multiple of their last place, and its root needs no range test.
template <typename R, bool SCALED>
__device__ __forceinline__ R cartesian_uniform3d(
    R hs0, R hs1, R hs2, R hs3, R hs4, R hs5, R hs7, R hs03, R &hs47,
    R t1, R t2, R t3, R t4, R t5, R t6, R t7)
{
    using M = Math<R>;
    auto root = [](R a)
    {
        return SCALED ? M::sqrt_in_range(a) : M::sqrt(a);
    };
    hs47 = M::min(hs4, hs7);
    const R hs01 = M::min(hs0, hs1);
    const R hs04 = M::min(hs0, hs4);
    R t1d1 = t1 + M::min(hs03, hs47);
    R t1d2 = t3 + M::min(hs04, M::min(hs1, hs5));
    R t1d3 = t4 + M::min(hs01, M::min(hs2, hs3));
    R best = M::min(M::min(t1d1, t1d2), t1d3);
    const R max14 = M::max(t1, t4);
    R dtCrossXZ = t1 - t4;
    R detXZ = M::fma(2, hs03*hs03, -(dtCrossXZ*dtCrossXZ));
    if ((detXZ > 0) & (max14 <= M::min(t1, t4) + hs03))
    {
        best = M::min(best, t5 + root(detXZ));
    }
    R dtCrossYZ = t3 - t4;
    R detYZ = M::fma(2, hs01*hs01, -(dtCrossYZ*dtCrossYZ));
    if ((detYZ > 0) & (M::max(t3, t4) <= M::min(t3, t4) + hs01))
    {
        best = M::min(best, t7 + root(detYZ));
    }
    R dtCrossXY = t1 - t3;
    R detXY = M::fma(2, hs04*hs04, -(dtCrossXY*dtCrossXY));
    if ((detXY > 0) & (M::max(t1, t3) <= M::min(t1, t3) + hs04))
    {
        best = M::min(best, t2 + root(detXY));
    }
    // min(t1d, t2d) > max(t1, t4, t3) of the reference
    if (best > M::max(max14, t3))
    {
        const R third = (R) 0.33333333333333333333333;
        const R half = (R) 0.5;
        R Tx = M::fma(half, -t4 + t5 - t3 + t2, t1) - t7 + t6;
        R Ty = M::fma(half, -t4 + t7 - t1 + t2, t3) - t5 + t6;
        R Tz = M::fma(half, -t1 + t5 - t3 + t7, t4) - t2 + t6;
        R det = 27*hs0*hs0
              - (Tx - Ty)*(Tx - Ty)
              - (Tx - Tz)*(Tx - Tz)
              - (Ty - Tz)*(Ty - Tz);
        if (det >= 0)
        {
            best = M::min(best, third*((Tx + Ty + Tz) + M::sqrt(det)));
        }
    }
    return best;
}

// v where valid, else a number above HUGE (HUGE's next high word): one
// select instead of two, the low word does not matter.
__device__ __forceinline__ double valid_or_huge(double v, bool valid)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t hi = valid ? (uint32_t) (u >> 32) : 0x4202A060u;
    return __builtin_bit_cast(double,
                              ((uint64_t) hi << 32) | (uint32_t) u);
}
__device__ __forceinline__ float valid_or_huge(float v, bool valid)
{
    return valid ? v : 2*(float) kHuge;
}

// cartesian_uniform3d<R, true> without branches: every candidate is
// evaluated, and an invalid one is replaced by a number above HUGE.  For
// waves that have a SIMD nearly to themselves, where each branch is a wait
// (one 257 x 257 x 193 grid by diagonals: 49.4 ms with branches, 46.4
// without); where the launches fill the chip the branches skip work (64
// sources on 385 x 385 x 193: 615 and 648 ms, 62 on 206 x 173 x 44: 30 and
// 32 ms).
template <typename R>
__device__ __forceinline__ R cartesian_uniform3d_flat(
    R hs0, R hs1, R hs2, R hs3, R hs4, R hs5, R hs7, R hs03, R &hs47,
    R t1, R t2, R t3, R t4, R t5, R t6, R t7)
{
    using M = Math<R>;
    hs47 = M::min(hs4, hs7);
    const R hs01 = M::min(hs0, hs1);
    const R hs04 = M::min(hs0, hs4);
    R t1d1 = t1 + M::min(hs03, hs47);
    R t1d2 = t3 + M::min(hs04, M::min(hs1, hs5));
    R t1d3 = t4 + M::min(hs01, M::min(hs2, hs3));
    R best = M::min(M::min(t1d1, t1d2), t1d3);
    const R max14 = M::max(t1, t4);
    R dtCrossXZ = t1 - t4;
    R detXZ = M::fma(2, hs03*hs03, -(dtCrossXZ*dtCrossXZ));
    R dtCrossYZ = t3 - t4;
    R detYZ = M::fma(2, hs01*hs01, -(dtCrossYZ*dtCrossYZ));
    R dtCrossXY = t1 - t3;
    R detXY = M::fma(2, hs04*hs04, -(dtCrossXY*dtCrossXY));
    const bool cXZ = (detXZ > 0) & (max14 <= M::min(t1, t4) + hs03);
    const bool cYZ = (detYZ > 0) & (M::max(t3, t4) <= M::min(t3, t4) + hs01);
    const bool cXY = (detXY > 0) & (M::max(t1, t3) <= M::min(t1, t3) + hs04);
    best = M::min(best, valid_or_huge(t5 + M::sqrt_in_range(detXZ), cXZ));
    best = M::min(best, valid_or_huge(t7 + M::sqrt_in_range(detYZ), cYZ));
    best = M::min(best, valid_or_huge(t2 + M::sqrt_in_range(detXY), cXY));
    const R third = (R) 0.33333333333333333333333;
    const R half = (R) 0.5;
    R Tx = M::fma(half, -t4 + t5 - t3 + t2, t1) - t7 + t6;
    R Ty = M::fma(half, -t4 + t7 - t1 + t2, t3) - t5 + t6;
    R Tz = M::fma(half, -t1 + t5 - t3 + t7, t4) - t2 + t6;
    R det = 27*hs0*hs0
          - (Tx - Ty)*(Tx - Ty)
          - (Tx - Tz)*(Tx - Tz)
          - (Ty - Tz)*(Ty - Tz);
    const bool c3 = (best > M::max(max14, t3)) & (det >= 0);
    return M::min(best, valid_or_huge(third*((Tx + Ty + Tz) +
                                             M::sqrt_or_zero(det)), c3));
}

// Factored (spherical) branch, uniform grid (:281-294, :372-553); always
// evaluated in double.
__device__ __forceinline__ double factored_uniform3d(
    const Problem3D &p, const Sweep3D &sw, int ix, int iy, int iz,
    double s0, double s1, double s2, double s3, double s4, double s5,
    double s7, double t1, double t2, double t3, double t4, double t5,
    double t6, double t7)
{
    const double huge = kHuge;
    const double h = p.dx;
    const double sourceSlowness = p.srcSlowness;
    double minS0S3 = fmin(s0, s3);
    double minS0S1 = fmin(s0, s1);
    double minS0S4 = fmin(s0, s4);
    double t1d1 = t1 + h*fmin(minS0S3, fmin(s4, s7));
    double t1d2 = t3 + h*fmin(minS0S4, fmin(s1, s5));
    double t1d3 = t4 + h*fmin(minS0S1, fmin(s2, s3));
    double t1d = fmin(fmin(t1d1, t1d2), t1d3);
    double hs03 = h*minS0S3;
    double hs01 = h*minS0S1;
    double hs04 = h*minS0S4;
    const double xs = p.srcOffX, ys = p.srcOffY, zs = p.srcOffZ;
    double t0, dt0dx, dt0dy, dt0dz;
    analytic_time_deriv3d(ix, iy, iz, h, h, h, xs, ys, zs, s0,
                          t0, dt0dx, dt0dy, dt0dz);
    double tau1 = t1 - analytic_time3d(ix + sw.ixShift, iy, iz,
                                       h, h, h, xs, ys, zs, s0);
    double tau2 = t2 - analytic_time3d(ix + sw.ixShift, iy + sw.iyShift, iz,
                                       h, h, h, xs, ys, zs, s0);
    double tau3 = t3 - analytic_time3d(ix, iy + sw.iyShift, iz,
                                       h, h, h, xs, ys, zs, s0);
    double tau4 = t4 - analytic_time3d(ix, iy, iz + sw.izShift,
                                       h, h, h, xs, ys, zs, s0);
    double tau5 = t5 - analytic_time3d(ix + sw.ixShift, iy, iz + sw.izShift,
                                       h, h, h, xs, ys, zs, s0);
    double tau6 = t6 - analytic_time3d(ix + sw.ixShift, iy + sw.iyShift,
                                       iz + sw.izShift,
                                       h, h, h, xs, ys, zs, s0);
    double tau7 = t7 - analytic_time3d(ix, iy + sw.iyShift, iz + sw.izShift,
                                       h, h, h, xs, ys, zs, s0);
    dt0dx = sw.signX*dt0dx;
    dt0dy = sw.signY*dt0dy;
    dt0dz = sw.signZ*dt0dz;
    double dTauTxXZ = tau1 - tau4 + tau5;
    double dTauTzXZ = tau4 - tau1 + tau5;
    const double half = 0.5;
    double hi = 1/h;
    double h2inv = 1/(h*h);
    double a = h2inv;
    double b = (2*hi)*(dt0dx + dt0dz)
             - (2*h2inv)*tau5;
    double c = (half*h2inv)*(dTauTxXZ*dTauTxXZ + dTauTzXZ*dTauTzXZ)
             - (2*hi)*(dt0dx*dTauTxXZ + dt0dz*dTauTzXZ)
             + 2*(sourceSlowness*sourceSlowness - s0*s0 + dt0dy*dt0dy);
    double detXZ = b*b - 4*a*c;
    double tau = 0;
    double t2d1 = huge;
    if (detXZ > 0 && t4 <= t1 + hs03 && t1 <= t4 + hs03)
    {
        tau = (-b + ::sqrt(detXZ))/(2*a);
        t2d1 = t0 + tau;
        if (t2d1 < t1 || t2d1 < t4) { t2d1 = huge; }
    }
    double t2d = t2d1;
    double dTauTyYZ = tau3 - tau4 + tau7;
    double dTauTzYZ = tau4 - tau3 + tau7;
    b = (2*hi)*(dt0dy + dt0dz)
      - (2*h2inv)*tau7;
    c = (half*h2inv)*(dTauTyYZ*dTauTyYZ + dTauTzYZ*dTauTzYZ)
      - (2*hi)*(dt0dy*dTauTyYZ + dt0dz*dTauTzYZ)
      + 2*(sourceSlowness*sourceSlowness - s0*s0 + dt0dx*dt0dx);
    double detYZ = b*b - 4*a*c;
    double t2d2 = huge;
    if (detYZ >= 0 && t3 <= t4 + hs01 && t4 <= t3 + hs01)
    {
        tau = (-b + ::sqrt(detYZ))/(2*a);
        t2d2 = t0 + tau;
        if (t2d2 < t3 || t2d2 < t4) { t2d2 = huge; }
    }
    t2d = fmin(t2d, t2d2);
    double dTauTxXY = tau1 - tau3 + tau2;
    double dTauTyXY = tau3 - tau1 + tau2;
    b = (2*hi)*(dt0dx + dt0dy)
      - (2*h2inv)*tau2;
    c = (half*h2inv)*(dTauTxXY*dTauTxXY + dTauTyXY*dTauTyXY)
      - (2*hi)*(dt0dx*dTauTxXY + dt0dy*dTauTyXY)
      + 2*(sourceSlowness*sourceSlowness - s0*s0 + dt0dz*dt0dz);
    double detXY = b*b - 4*a*c;
    double t2d3 = huge;
    if (detXY >= 0 && t3 <= t1 + hs04 && t1 <= t3 + hs04)
    {
        tau = (-b + ::sqrt(detXY))/(2*a);
        t2d3 = t0 + tau;
        if (t2d3 < t1 || t2d3 < t3) { t2d3 = huge; }
    }
    t2d = fmin(t2d, t2d3);
    double t3d = huge;
    if (fmin(t1d, t2d) > fmax(fmax(t1, t4), t3))
    {
        double taux = tau1 + half*(-tau4 + tau5 - tau3 + tau2) - tau7 + tau6;
        double tauy = tau3 + half*(-tau4 + tau7 - tau1 + tau2) - tau5 + tau6;
        double tauz = tau4 + half*(-tau1 + tau5 - tau3 + tau7) - tau2 + tau6;
        a = 3*h2inv;
        b =-2*h2inv*(taux + tauy + tauz)
          + (6*hi)*(dt0dx + dt0dy + dt0dz);
        c = h2inv*(taux*taux + tauy*tauy + tauz*tauz)
          - (6*hi)*(dt0dx*taux + dt0dy*tauy + dt0dz*tauz)
          + 9*(sourceSlowness*sourceSlowness - s0*s0);
        double det = b*b - 4*a*c;
        if (det >= 0)
        {
            t3d = t0 + (-b + ::sqrt(det))/(2*a);
        }
        if (t3d < t1 || t3d < t3 || t3d < t4) { t3d = huge; }
    }
    return fmin(t1d, fmin(t2d, t3d));
}

// Cartesian branch, non-uniform grid (:591-680) in arithmetic R, with the
// running minimum of cartesian_uniform3d.
template <typename R>
__device__ __forceinline__ R cartesian_nonuniform3d(
    const Problem3D &p, R s0, R s1, R s2, R s3, R s4, R s5, R s7,
    R t1, R t2, R t3, R t4, R t5, R t6, R t7)
{
    using M = Math<R>;
    const R dx = (R) p.dx, dy = (R) p.dy, dz = (R) p.dz;
    const NonUniform3D &nu = p.nu;
    const R dx2Inv = (R) nu.dx2Inv, dy2Inv = (R) nu.dy2Inv;
    const R dz2Inv = (R) nu.dz2Inv;
    const R dx_dz = (R) nu.dx_dz, dz_dx = (R) nu.dz_dx;
    const R dy_dz = (R) nu.dy_dz, dz_dy = (R) nu.dz_dy;
    const R dx_dy = (R) nu.dx_dy, dy_dx = (R) nu.dy_dx;
    const R dx2_p_dz2_inv = (R) nu.dx2_p_dz2_inv;
    const R dy2_p_dz2_inv = (R) nu.dy2_p_dz2_inv;
    const R dx2_p_dy2_inv = (R) nu.dx2_p_dy2_inv;
    R minS0S3 = M::min(s0, s3);
    R minS0S1 = M::min(s0, s1);
    R minS0S4 = M::min(s0, s4);
    R t1d1 = t1 + dx*M::min(minS0S3, M::min(s4, s7));
    R t1d2 = t3 + dy*M::min(minS0S4, M::min(s1, s5));
    R t1d3 = t4 + dz*M::min(minS0S1, M::min(s2, s3));
    R best = M::min(M::min(t1d1, t1d2), t1d3);
    R dtCrossXZ = t1 - t4;
    R detXZ = (dx*dx + dz*dz)*(minS0S3*minS0S3) - dtCrossXZ*dtCrossXZ;
    if (detXZ > 0 && t1 < t4 + dz*minS0S3 && t4 < t1 + dx*minS0S3)
    {
        R TxXZ = t1 - t4 + t5;
        R TzXZ = t4 - t1 + t5;
        R t2d1 = (TxXZ*dz_dx + TzXZ*dx_dz) + 2*M::sqrt(detXZ);
        best = M::min(best, ((dx*dz)*dx2_p_dz2_inv)*t2d1);
    }
    R dtCrossYZ = t3 - t4;
    R detYZ = (dy*dy + dz*dz)*(minS0S1*minS0S1) - dtCrossYZ*dtCrossYZ;
    if (detYZ > 0 && t3 < t4 + dz*minS0S1 && t4 < t3 + dy*minS0S1)
    {
        R TyYZ = t3 - t4 + t7;
        R TzYZ = t4 - t3 + t7;
        R t2d2 = (TyYZ*dz_dy + TzYZ*dy_dz) + 2*M::sqrt(detYZ);
        best = M::min(best, ((dy*dz)*dy2_p_dz2_inv)*t2d2);
    }
    R dtCrossXY = t1 - t3;
    R detXY = (dx*dx + dy*dy)*(minS0S4*minS0S4) - dtCrossXY*dtCrossXY;
    if (detXY > 0 && t3 < t1 + dx*minS0S4 && t1 < t3 + dy*minS0S4)
    {
        R TxXY = t1 - t3 + t2;
        R TyXY = t3 - t1 + t2;
        R t2d3 = (TxXY*dy_dx + TyXY*dx_dy) + 2*M::sqrt(detXY);
        best = M::min(best, ((dx*dy)*dx2_p_dy2_inv)*t2d3);
    }
    // min(t1d, t2d) > max(t1, t4, t3) of the reference
    if (best > M::max(M::max(t1, t4), t3))
    {
        const R half = (R) 0.5;
        R Tx = t1 + half*(-t4 + t5 - t3 + t2) - t7 + t6;
        R Ty = t3 + half*(-t4 + t7 - t1 + t2) - t5 + t6;
        R Tz = t4 + half*(-t1 + t5 - t3 + t7) - t2 + t6;
        R det = 9*(s0*s0)*(dx2Inv + dy2Inv + dz2Inv)
              - ((Tx - Tz)*(Tx - Tz))*(dx2Inv*dz2Inv)
              - ((Ty - Tz)*(Ty - Tz))*(dy2Inv*dz2Inv)
              - ((Tx - Ty)*(Tx - Ty))*(dx2Inv*dy2Inv);
        if (det >= 0)
        {
            best = M::min(best, (Tx*dx2Inv + Ty*dy2Inv + Tz*dz2Inv +
                                 M::sqrt(det))/(dx2Inv + dy2Inv + dz2Inv));
        }
    }
    return best;
}

// Factored branch, non-uniform grid (:591-599, :681-821), in double.
__device__ __forceinline__ double factored_nonuniform3d(
    const Problem3D &p, const Sweep3D &sw, int ix, int iy, int iz,
    double s0, double s1, double s2, double s3, double s4, double s5,
    double s7, double t1, double t2, double t3, double t4, double t5,
    double t6, double t7)
{
    const double huge = kHuge;
    const double dx = p.dx, dy = p.dy, dz = p.dz;
    const double sourceSlowness = p.srcSlowness;
    const NonUniform3D &nu = p.nu;
    const double dxInv = nu.dxInv, dyInv = nu.dyInv, dzInv = nu.dzInv;
    const double dx2Inv = nu.dx2Inv, dy2Inv = nu.dy2Inv, dz2Inv = nu.dz2Inv;
    double minS0S3 = fmin(s0, s3);
    double minS0S1 = fmin(s0, s1);
    double minS0S4 = fmin(s0, s4);
    double t1d1 = t1 + dx*fmin(minS0S3, fmin(s4, s7));
    double t1d2 = t3 + dy*fmin(minS0S4, fmin(s1, s5));
    double t1d3 = t4 + dz*fmin(minS0S1, fmin(s2, s3));
    double t1d = fmin(fmin(t1d1, t1d2), t1d3);
    const double xs = p.srcOffX, ys = p.srcOffY, zs = p.srcOffZ;
    double t0, dt0dx, dt0dy, dt0dz;
    analytic_time_deriv3d(ix, iy, iz, dx, dy, dz, xs, ys, zs, s0,
                          t0, dt0dx, dt0dy, dt0dz);
    double tau1 = t1 - analytic_time3d(ix + sw.ixShift, iy, iz,
                                       dx, dy, dz, xs, ys, zs, s0);
    double tau2 = t2 - analytic_time3d(ix + sw.ixShift, iy + sw.iyShift, iz,
                                       dx, dy, dz, xs, ys, zs, s0);
    double tau3 = t3 - analytic_time3d(ix, iy + sw.iyShift, iz,
                                       dx, dy, dz, xs, ys, zs, s0);
    double tau4 = t4 - analytic_time3d(ix, iy, iz + sw.izShift,
                                       dx, dy, dz, xs, ys, zs, s0);
    double tau5 = t5 - analytic_time3d(ix + sw.ixShift, iy, iz + sw.izShift,
                                       dx, dy, dz, xs, ys, zs, s0);
    double tau6 = t6 - analytic_time3d(ix + sw.ixShift, iy + sw.iyShift,
                                       iz + sw.izShift,
                                       dx, dy, dz, xs, ys, zs, s0);
    double tau7 = t7 - analytic_time3d(ix, iy + sw.iyShift, iz + sw.izShift,
                                       dx, dy, dz, xs, ys, zs, s0);
    dt0dx = sw.signX*dt0dx;
    dt0dy = sw.signY*dt0dy;
    dt0dz = sw.signZ*dt0dz;
    double dTauTxXZ = tau1 - tau4 + tau5;
    double dTauTzXZ = tau4 - tau1 + tau5;
    double a = dx2Inv + dz2Inv;
    double b = 4*(dxInv*dt0dx + dzInv*dt0dz)
             - 2*(dTauTxXZ*dx2Inv + dTauTzXZ*dz2Inv);
    double c = (dTauTxXZ*dTauTxXZ)*dx2Inv + (dTauTzXZ*dTauTzXZ)*dz2Inv
             - 4*((dt0dx*dTauTxXZ)*dxInv + (dt0dz*dTauTzXZ)*dzInv)
             + 4*(sourceSlowness*sourceSlowness - s0*s0 + dt0dy*dt0dy);
    double detXZ = b*b - 4*a*c;
    double t2d1 = huge;
    if (detXZ > 0 && t1 < t4 + dz*minS0S3 && t4 < t1 + dx*minS0S3)
    {
        t2d1 = t0 + (-b + ::sqrt(detXZ))/(2*a);
        if (t2d1 < t1 || t2d1 < t4) { t2d1 = huge; }
    }
    double t2d = t2d1;
    double dTauTyYZ = tau3 - tau4 + tau7;
    double dTauTzYZ = tau4 - tau3 + tau7;
    a = dy2Inv + dz2Inv;
    b = 4*(dyInv*dt0dy + dzInv*dt0dz)
      - 2*(dTauTyYZ*dy2Inv + dTauTzYZ*dz2Inv);
    c = (dTauTyYZ*dTauTyYZ)*dy2Inv + (dTauTzYZ*dTauTzYZ)*dz2Inv
      - 4*((dt0dy*dTauTyYZ)*dyInv + (dt0dz*dTauTzYZ)*dzInv)
      + 4*(sourceSlowness*sourceSlowness - s0*s0 + dt0dx*dt0dx);
    double detYZ = b*b - 4*a*c;
    double t2d2 = huge;
    if (detYZ > 0 && t3 < t4 + dz*minS0S1 && t4 < t3 + dy*minS0S1)
    {
        t2d2 = t0 + (-b + ::sqrt(detYZ))/(2*a);
        if (t2d2 < t3 || t2d2 < t4) { t2d2 = huge; }
    }
    t2d = fmin(t2d, t2d2);
    double dTauTxXY = tau1 - tau3 + tau2;
    double dTauTyXY = tau3 - tau1 + tau2;
    a = dx2Inv + dy2Inv;
    b = 4*(dxInv*dt0dx + dyInv*dt0dy)
      - 2*(dTauTxXY*dx2Inv + dTauTyXY*dy2Inv);
    c = (dTauTxXY*dTauTxXY)*dx2Inv + (dTauTyXY*dTauTyXY)*dy2Inv
      - 4*((dt0dx*dTauTxXY)*dxInv + (dt0dy*dTauTyXY)*dyInv)
      + 4*(sourceSlowness*sourceSlowness - s0*s0 + dt0dz*dt0dz);
    double detXY = b*b - 4*a*c;
    double t2d3 = huge;
    if (detXY > 0 && t3 < t1 + dx*minS0S4 && t1 < t3 + dy*minS0S4)
    {
        t2d3 = t0 + (-b + ::sqrt(detXY))/(2*a);
        if (t2d3 < t1 || t2d3 < t3) { t2d3 = huge; }
    }
    t2d = fmin(t2d, t2d3);
    double t3d = huge;
    if (fmin(t1d, t2d) > fmax(fmax(t1, t4), t3))
    {
        const double half = 0.5;
        double taux = tau1 + half*(-tau4 + tau5 - tau3 + tau2) - tau7 + tau6;
        double tauy = tau3 + half*(-tau4 + tau7 - tau1 + tau2) - tau5 + tau6;
        double tauz = tau4 + half*(-tau1 + tau5 - tau3 + tau7) - tau2 + tau6;
        a = dx2Inv + dy2Inv + dz2Inv;
        b =-2*(taux*dx2Inv + tauy*dy2Inv + tauz*dz2Inv)
          + 6*(dxInv*dt0dx + dyInv*dt0dy + dzInv*dt0dz);
        c = (taux*taux)*dx2Inv + (tauy*tauy)*dy2Inv + (tauz*tauz)*dz2Inv
          - 6*(dt0dx*taux*dxInv + dt0dy*tauy*dyInv + dt0dz*tauz*dzInv)
          + 9*(sourceSlowness*sourceSlowness - s0*s0);
        double det = b*b - 4*a*c;
        if (det >= 0)
        {
            t3d = t0 + (-b + ::sqrt(det))/(2*a);
        }
        if (t3d < t1 || t3d < t3 || t3d < t4) { t3d = huge; }
    }
    return fmin(t1d, fmin(t2d, t3d));
}

// The grid constants of the branch-free updates, by value (in registers
// across a step loop).
template <typename R>
struct FlowGrid
{
    R dx, dy, dz, dx2Inv, dy2Inv, dz2Inv;
    R dx_dz, dz_dx, dy_dz, dz_dy, dx_dy, dy_dx;
    R dx2_p_dz2_inv, dy2_p_dz2_inv, dx2_p_dy2_inv;
};

template <typename R>
__device__ __forceinline__ FlowGrid<R> flow_grid(const Problem3D &p)
{
    const NonUniform3D &nu = p.nu;
    return FlowGrid<R>{
        (R) p.dx, (R) p.dy, (R) p.dz, (R) nu.dx2Inv, (R) nu.dy2Inv,
        (R) nu.dz2Inv, (R) nu.dx_dz, (R) nu.dz_dx, (R) nu.dy_dz,
        (R) nu.dz_dy, (R) nu.dx_dy, (R) nu.dy_dx, (R) nu.dx2_p_dz2_inv,
        (R) nu.dy2_p_dz2_inv, (R) nu.dx2_p_dy2_inv};
}

// cartesian_nonuniform3d without branches, for models whose h s are in
// range (as cartesian_uniform3d_flat).
template <typename R>
__device__ __forceinline__ R cartesian_nonuniform3d_flat(
    const FlowGrid<R> &g, R s0, R s1, R s2, R s3, R s4, R s5, R s7,
    R t1, R t2, R t3, R t4, R t5, R t6, R t7)
{
    using M = Math<R>;
    const R dx = g.dx, dy = g.dy, dz = g.dz;
    R minS0S3 = M::min(s0, s3);
    R minS0S1 = M::min(s0, s1);
    R minS0S4 = M::min(s0, s4);
    R t1d1 = t1 + dx*M::min(minS0S3, M::min(s4, s7));
    R t1d2 = t3 + dy*M::min(minS0S4, M::min(s1, s5));
    R t1d3 = t4 + dz*M::min(minS0S1, M::min(s2, s3));
    R best = M::min(M::min(t1d1, t1d2), t1d3);
    // the candidate of the plane of axes u (neighbour tu) and v (tv), corner
    // tc: same expressions as the branching form
    auto plane = [](R tu, R tv, R tc, R s, R du, R dv, R du_dv, R dv_du,
                    R inv)
    {
        R dtCross = tu - tv;
        R det = (du*du + dv*dv)*(s*s) - dtCross*dtCross;
        const bool c = (det > 0) & (tu < tv + dv*s) & (tv < tu + du*s);
        R Tu = tu - tv + tc;
        R Tv = tv - tu + tc;
        R t = (Tu*dv_du + Tv*du_dv) + 2*M::sqrt_in_range(det);
        return valid_or_huge(((du*dv)*inv)*t, c);
    };
    best = M::min(best, plane(t1, t4, t5, minS0S3, dx, dz, g.dx_dz, g.dz_dx,
                              g.dx2_p_dz2_inv));
    best = M::min(best, plane(t3, t4, t7, minS0S1, dy, dz, g.dy_dz, g.dz_dy,
                              g.dy2_p_dz2_inv));
    best = M::min(best, plane(t1, t3, t2, minS0S4, dx, dy, g.dx_dy, g.dy_dx,
                              g.dx2_p_dy2_inv));
    const R half = (R) 0.5;
    R Tx = M::fma(half, -t4 + t5 - t3 + t2, t1) - t7 + t6;
    R Ty = M::fma(half, -t4 + t7 - t1 + t2, t3) - t5 + t6;
    R Tz = M::fma(half, -t1 + t5 - t3 + t7, t4) - t2 + t6;
    const R sumInv = g.dx2Inv + g.dy2Inv + g.dz2Inv;
    R det = 9*(s0*s0)*sumInv
          - ((Tx - Tz)*(Tx - Tz))*(g.dx2Inv*g.dz2Inv)
          - ((Ty - Tz)*(Ty - Tz))*(g.dy2Inv*g.dz2Inv)
          - ((Tx - Ty)*(Tx - Ty))*(g.dx2Inv*g.dy2Inv);
    const bool c3 = (best > M::max(M::max(t1, t4), t3)) & (det >= 0);
    R t = (Tx*g.dx2Inv + Ty*g.dy2Inv + Tz*g.dz2Inv + M::sqrt_or_zero(det))/
          sumInv;
    return M::min(best, valid_or_huge(t, c3));
}

// The source and the grid constants of the branch-free factored updates, by
// value; on a uniform grid opaque too, so that no step loads them again and
// waits (33 x 29 x 25: 1.55 -> 1.53 ms; the 13 values of the other grids are
// more than the scalar registers hold).
struct FactoredGrid
{
    double dx, dy, dz, x, y, z, slowness2;
    double dxInv, dyInv, dzInv, dx2Inv, dy2Inv, dz2Inv;
};

template <bool UNIFORM>
__device__ __forceinline__ FactoredGrid factored_grid(const Problem3D &p)
{
    auto opaque = [](double v)
    {
        if (!UNIFORM) { return v; }
        uint64_t u = __builtin_bit_cast(uint64_t, v);
        uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t) u);
        uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t) (u >> 32));
        __asm__ __volatile__("" : "+s"(lo), "+s"(hi));
        return __builtin_bit_cast(double, ((uint64_t) hi << 32) | lo);
    };
    const NonUniform3D &nu = p.nu;
    FactoredGrid g;
    g.dx = g.dy = g.dz = opaque(p.dx);
    g.dxInv = g.dyInv = g.dzInv = opaque(nu.dxInv);
    g.dx2Inv = g.dy2Inv = g.dz2Inv = opaque(nu.dx2Inv);
    g.x = opaque(p.srcOffX);
    g.y = opaque(p.srcOffY);
    g.z = opaque(p.srcOffZ);
    g.slowness2 = opaque(p.srcSlowness*p.srcSlowness);
    if (!UNIFORM)
    {
        g.dy = opaque(p.dy);
        g.dz = opaque(p.dz);
        g.dyInv = opaque(nu.dyInv);
        g.dzInv = opaque(nu.dzInv);
        g.dy2Inv = opaque(nu.dy2Inv);
        g.dz2Inv = opaque(nu.dz2Inv);
    }
    return g;
}

// What the branch-free factored update keeps from step to step: the
// distances from the source to the node and its three neighbours in the
// plane (x-1, (x-1, y-1), y-1), which are the next plane's neighbours in z.
struct FactoredDistances
{
    double d0, d1, d2, d3;
};

// The distances at a node (natural indices).
__device__ __forceinline__ FactoredDistances factored_distances(
    const FactoredGrid &k, const Sweep3D &sw, int ix, int iy, int iz)
{
    const double x = ix*k.dx - k.x;
    const double x1 = (ix + sw.ixShift)*k.dx - k.x;
    const double y = iy*k.dy - k.y;
    const double y1 = (iy + sw.iyShift)*k.dy - k.y;
    const double z = iz*k.dz - k.z;
    const double xx = x*x, xx1 = x1*x1, yy = y*y, yy1 = y1*y1, zz = z*z;
    const double a0 = xx + yy + zz, a1 = xx1 + yy + zz;
    const double a2 = xx1 + yy1 + zz, a3 = xx + yy1 + zz;
    FactoredDistances d{sqrt_normal_range(a0), sqrt_normal_range(a1),
                        sqrt_normal_range(a2), sqrt_normal_range(a3)};
    const bool normal = fmin(fmin(a0, a1), fmin(a2, a3)) >= 0x1p-767;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!normal) != 0, 0))
    {
        d = FactoredDistances{::sqrt(a0), ::sqrt(a1), ::sqrt(a2),
                              ::sqrt(a3)};
    }
    return d;
}

// The roots of the determinants of a node's valid candidates (1 for the
// others): one test for arguments under sqrt_normal_range's range.
struct FactoredRoots
{
    double xz, yz, xy, xyz;
};

__device__ __forceinline__ double valid_or_one(double v, bool valid)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t hi = valid ? (uint32_t) (u >> 32) : 0x3FF00000u;
    return __builtin_bit_cast(double,
                              ((uint64_t) hi << 32) | (uint32_t) u);
}

__device__ __forceinline__ FactoredRoots factored_roots(double xz, double yz,
                                                        double xy, double xyz)
{
    FactoredRoots r{sqrt_normal_range(xz), sqrt_normal_range(yz),
                    sqrt_normal_range(xy), sqrt_normal_range(xyz)};
    const bool normal = fmin(fmin(xz, yz), fmin(xy, xyz)) >= 0x1p-767;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!normal) != 0, 0))
    {
        r = FactoredRoots{::sqrt(xz), ::sqrt(yz), ::sqrt(xy), ::sqrt(xyz)};
    }
    return r;
}

// The factored update without branches, from the distances at the node's
// plane (d) and at the plane before (e): same values as factored_uniform3d
// (the causality test of a pair, the exact products by 2 and 1/2 and h s as
// in cartesian_uniform3d; an invalid candidate is above HUGE).  For the flow
// kernel, whose lone waves wait at each branch and pay for each instruction:
// half of a node's eight distances are those of the plane before, and the
// quotients that depend on the grid alone come with the problem.  8 x 8 x 33
// with radius 3, 8 sweeps: 497 us with the branching form and its eight
// distances, 383 now (about 200 without a box).
__device__ __forceinline__ double factored_uniform3d_flat(
    const FactoredGrid &k, const Sweep3D &sw, const FactoredDistances &d,
    const FactoredDistances &e, int ix, int iy, int iz, double s0, double hs0,
    double hs1, double hs2, double hs3, double hs4, double hs5, double hs7,
    double t1, double t2, double t3, double t4, double t5, double t6,
    double t7)
{
    const double h = k.dx, hInv = k.dxInv, h2Inv = k.dx2Inv;
    const double hs03 = fmin(hs0, hs3), hs01 = fmin(hs0, hs1);
    const double hs04 = fmin(hs0, hs4);
    const double t1d =
        fmin(fmin(t1 + fmin(hs03, fmin(hs4, hs7)),
                  t3 + fmin(hs04, fmin(hs1, hs5))),
             t4 + fmin(hs01, fmin(hs2, hs3)));
    const double t0 = s0*d.d0;
    const bool off = d.d0 > 0;
    auto slope = [&](int i, double source, int sign)
    {
        const double q = (s0*(sign*(i*h - source)))/d.d0;
        return off ? q : 0.0;
    };
    const double gx = slope(ix, k.x, sw.signX);
    const double gy = slope(iy, k.y, sw.signY);
    const double gz = slope(iz, k.z, sw.signZ);
    const double tau1 = t1 - s0*d.d1, tau2 = t2 - s0*d.d2;
    const double tau3 = t3 - s0*d.d3, tau4 = t4 - s0*e.d0;
    const double tau5 = t5 - s0*e.d1, tau6 = t6 - s0*e.d2;
    const double tau7 = t7 - s0*e.d3;
    const double excess = k.slowness2 - s0*s0;
    const double h2Half = 0.5*h2Inv, hTwice = 2*hInv, h2Twice = 2*h2Inv;
    double b[3], det[3];
    // the pair (u, v), its corner's tau and the third axis' slope
    auto pair = [&](int m, double tauU, double tauV, double tauC, double gu,
                    double gv, double gw)
    {
        const double Tu = tauU - tauV + tauC, Tv = tauV - tauU + tauC;
        b[m] = hTwice*(gu + gv) - h2Twice*tauC;
        const double c = fma(2.0, excess + gw*gw,
                             h2Half*(Tu*Tu + Tv*Tv) -
                                 hTwice*(gu*Tu + gv*Tv));
        det[m] = b[m]*b[m] - (4*h2Inv)*c;
    };
    pair(0, tau1, tau4, tau5, gx, gz, gy);
    pair(1, tau3, tau4, tau7, gy, gz, gx);
    pair(2, tau1, tau3, tau2, gx, gy, gz);
    const double taux = fma(0.5, -tau4 + tau5 - tau3 + tau2, tau1) - tau7 +
                        tau6;
    const double tauy = fma(0.5, -tau4 + tau7 - tau1 + tau2, tau3) - tau5 +
                        tau6;
    const double tauz = fma(0.5, -tau1 + tau5 - tau3 + tau7, tau4) - tau2 +
                        tau6;
    const double a3 = 3*h2Inv, h6 = 6*hInv;
    const double b3 = -2*h2Inv*(taux + tauy + tauz) + h6*(gx + gy + gz);
    const double c3 = h2Inv*(taux*taux + tauy*tauy + tauz*tauz) -
                      h6*(gx*taux + gy*tauy + gz*tauz) + 9*excess;
    const double det3 = b3*b3 - (4*a3)*c3;
    const double max14 = fmax(t1, t4), max34 = fmax(t3, t4);
    const double max13 = fmax(t1, t3);
    const bool cXZ = (det[0] > 0) & (max14 <= fmin(t1, t4) + hs03);
    const bool cYZ = (det[1] >= 0) & (max34 <= fmin(t3, t4) + hs01);
    const bool cXY = (det[2] >= 0) & (max13 <= fmin(t1, t3) + hs04);
    const bool cXYZ = det3 >= 0;
    const FactoredRoots r = factored_roots(
        valid_or_one(det[0], cXZ), valid_or_one(det[1], cYZ),
        valid_or_one(det[2], cXY), valid_or_one(det3, cXYZ));
    auto candidate = [&](bool c, double bm, double root, double a2,
                         double upwind)
    {
        const double t = t0 + (-bm + root)/a2;
        return valid_or_huge(t, c & (t >= upwind));
    };
    double t2d = candidate(cXZ, b[0], r.xz, h2Twice, max14);
    t2d = fmin(t2d, candidate(cYZ, b[1], r.yz, h2Twice, max34));
    t2d = fmin(t2d, candidate(cXY, b[2], r.xy, h2Twice, max13));
    const double best = fmin(t1d, t2d), max134 = fmax(max14, t3);
    return fmin(best, candidate(cXYZ & (best > max134), b3, r.xyz, 2*a3,
                                max134));
}

// The same for factored_nonuniform3d.
__device__ __forceinline__ double factored_nonuniform3d_flat(
    const FactoredGrid &k, const Sweep3D &sw, const FactoredDistances &d,
    const FactoredDistances &e, int ix, int iy, int iz, double s0, double s1,
    double s2, double s3, double s4, double s5, double s7, double t1,
    double t2, double t3, double t4, double t5, double t6, double t7)
{
    const double dx = k.dx, dy = k.dy, dz = k.dz;
    const double dxInv = k.dxInv, dyInv = k.dyInv, dzInv = k.dzInv;
    const double dx2Inv = k.dx2Inv, dy2Inv = k.dy2Inv, dz2Inv = k.dz2Inv;
    const double s03 = fmin(s0, s3), s01 = fmin(s0, s1), s04 = fmin(s0, s4);
    const double t1d = fmin(fmin(t1 + dx*fmin(s03, fmin(s4, s7)),
                                 t3 + dy*fmin(s04, fmin(s1, s5))),
                            t4 + dz*fmin(s01, fmin(s2, s3)));
    const double t0 = s0*d.d0;
    const bool off = d.d0 > 0;
    auto slope = [&](int i, double h, double source, int sign)
    {
        const double q = (s0*(sign*(i*h - source)))/d.d0;
        return off ? q : 0.0;
    };
    const double gx = slope(ix, dx, k.x, sw.signX);
    const double gy = slope(iy, dy, k.y, sw.signY);
    const double gz = slope(iz, dz, k.z, sw.signZ);
    const double tau1 = t1 - s0*d.d1, tau2 = t2 - s0*d.d2;
    const double tau3 = t3 - s0*d.d3, tau4 = t4 - s0*e.d0;
    const double tau5 = t5 - s0*e.d1, tau6 = t6 - s0*e.d2;
    const double tau7 = t7 - s0*e.d3;
    const double excess = k.slowness2 - s0*s0;
    double b[3], det[3];
    auto pair = [&](int m, double tauU, double tauV, double tauC, double gu,
                    double gv, double gw, double uInv, double vInv,
                    double u2Inv, double v2Inv)
    {
        const double Tu = tauU - tauV + tauC, Tv = tauV - tauU + tauC;
        b[m] = 4*(uInv*gu + vInv*gv) - 2*(Tu*u2Inv + Tv*v2Inv);
        const double c = fma(4.0, excess + gw*gw,
                             (Tu*Tu)*u2Inv + (Tv*Tv)*v2Inv -
                                 4*((gu*Tu)*uInv + (gv*Tv)*vInv));
        det[m] = b[m]*b[m] - 4*(u2Inv + v2Inv)*c;
    };
    pair(0, tau1, tau4, tau5, gx, gz, gy, dxInv, dzInv, dx2Inv, dz2Inv);
    pair(1, tau3, tau4, tau7, gy, gz, gx, dyInv, dzInv, dy2Inv, dz2Inv);
    pair(2, tau1, tau3, tau2, gx, gy, gz, dxInv, dyInv, dx2Inv, dy2Inv);
    const double taux = fma(0.5, -tau4 + tau5 - tau3 + tau2, tau1) - tau7 +
                        tau6;
    const double tauy = fma(0.5, -tau4 + tau7 - tau1 + tau2, tau3) - tau5 +
                        tau6;
    const double tauz = fma(0.5, -tau1 + tau5 - tau3 + tau7, tau4) - tau2 +
                        tau6;
    const double a3 = dx2Inv + dy2Inv + dz2Inv;
    const double b3 = -2*(taux*dx2Inv + tauy*dy2Inv + tauz*dz2Inv) +
                      6*(dxInv*gx + dyInv*gy + dzInv*gz);
    const double c3 = (taux*taux)*dx2Inv + (tauy*tauy)*dy2Inv +
                      (tauz*tauz)*dz2Inv -
                      6*(gx*taux*dxInv + gy*tauy*dyInv + gz*tauz*dzInv) +
                      9*excess;
    const double det3 = b3*b3 - 4*a3*c3;
    const bool cXZ = (det[0] > 0) & (t1 < t4 + dz*s03) & (t4 < t1 + dx*s03);
    const bool cYZ = (det[1] > 0) & (t3 < t4 + dz*s01) & (t4 < t3 + dy*s01);
    const bool cXY = (det[2] > 0) & (t3 < t1 + dx*s04) & (t1 < t3 + dy*s04);
    const bool cXYZ = det3 >= 0;
    const FactoredRoots r = factored_roots(
        valid_or_one(det[0], cXZ), valid_or_one(det[1], cYZ),
        valid_or_one(det[2], cXY), valid_or_one(det3, cXYZ));
    auto candidate = [&](bool c, double bm, double root, double a,
                         double upwind)
    {
        const double t = t0 + (-bm + root)/(2*a);
        return valid_or_huge(t, c & (t >= upwind));
    };
    const double max14 = fmax(t1, t4);
    double t2d = candidate(cXZ, b[0], r.xz, dx2Inv + dz2Inv, max14);
    t2d = fmin(t2d, candidate(cYZ, b[1], r.yz, dy2Inv + dz2Inv,
                              fmax(t3, t4)));
    t2d = fmin(t2d, candidate(cXY, b[2], r.xy, dx2Inv + dy2Inv,
                              fmax(t1, t3)));
    const double best = fmin(t1d, t2d), max134 = fmax(max14, t3);
    return fmin(best, candidate(cXYZ & (best > max134), b3, r.xyz, a3,
                                max134));
}

// The factored update as a call, for kernels in which it is rare.
static __device__ __noinline__ double factored3d(
    const Problem3D &p, const Sweep3D &sw, int ix, int iy, int iz, double s0,
    double s1, double s2, double s3, double s4, double s5, double s7,
    double t1, double t2, double t3, double t4, double t5, double t6,
    double t7)
{
    return p.uniform
        ? factored_uniform3d(p, sw, ix, iy, iz, s0, s1, s2, s3, s4, s5, s7,
                             t1, t2, t3, t4, t5, t6, t7)
        : factored_nonuniform3d(p, sw, ix, iy, iz, s0, s1, s2, s3, s4, s5,
                                s7, t1, t2, t3, t4, t5, t6, t7);
}

// The complete local update: the factored branch inside the
// (2 radius + 1)^3 box around the source cell, Cartesian outside
// (:296-298).  ix, iy, iz are natural grid indices.
template <typename R>
__device__ __forceinline__ R local_update3d(
    const Problem3D &p, const Sweep3D &sw, int ix, int iy, int iz,
    R s0, R s1, R s2, R s3, R s4, R s5, R s7,
    R t1, R t2, R t3, R t4, R t5, R t6, R t7)
{
    if (!in_factored_box(p, ix, iy, iz))
    {
        if (p.uniform)
        {
            const R h = (R) p.dx;
            R hs47;
            return cartesian_uniform3d<R, false>(
                h*s0, h*s1, h*s2, h*s3, h*s4, h*s5, h*s7,
                Math<R>::min(h*s0, h*s3), hs47, t1, t2, t3, t4, t5, t6, t7);
        }
        return cartesian_nonuniform3d<R>(p, s0, s1, s2, s3, s4, s5, s7,
                                         t1, t2, t3, t4, t5, t6, t7);
    }
    return (R) factored3d(p, sw, ix, iy, iz, s0, s1, s2, s3, s4, s5, s7, t1,
                          t2, t3, t4, t5, t6, t7);
}

} // namespace ekx
