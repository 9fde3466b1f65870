// ekx_kernels2d.hip -- the 2D fast-sweeping solver on the device (gfx950).
//
// The schedule is Solver2D::solve with the fast-sweeping method
// (src/solver2d.cpp:462-565): source initialisation, the four
// initialization sweeps, then nSweeps x four refinement sweeps.  Each sweep
// runs in anti-diagonal order (levels jx + jz = L in the sweep's permuted
// frame, solverUtilities2d.hpp:1065-1147); a node reads only neighbours on
// earlier levels, so the result equals the serial loop of
// Solver2DSweep::updateFSM (include/private/solver2d.hpp:203-327).
//
// One workgroup owns one problem for the whole solve, so one launch covers
// it: the band kernel (64 rows per wave) up to 1024 rows, the level kernel
// (global memory, a block barrier per level) for taller and wider grids.
#include "ekx_kernels.hpp"
#include "ekx_sqrt.hpp"

#include <algorithm>
#include <type_traits>

namespace ekx
{

// Distance of node (ix, iz) from the source.
__device__ __forceinline__ double distance2d(int ix, int iz, double dx,
                                             double dz, double xs, double zs)
{
    double x = ix*dx;
    double z = iz*dz;
    double deltaX = x - xs;
    double deltaZ = z - zs;
    return ::hypot(deltaX, deltaZ);
}

// computeAnalyticalTravelTime 2D (solverUtilities2d.hpp:159-174).
__device__ __forceinline__ double analytic_time2d(int ix, int iz, double dx,
                                                  double dz, double xs,
                                                  double zs, double slow)
{
    return slow*distance2d(ix, iz, dx, dz, xs, zs);
}

// (solverUtilities2d.hpp:192-215), given the distance r
__device__ __forceinline__ void analytic_time_deriv2d(
    int ix, int iz, double dx, double dz, double xs, double zs, double slow,
    double r, double &t, double &dtdx, double &dtdz)
{
    double x = ix*dx;
    double z = iz*dz;
    double deltaX = x - xs;
    double deltaZ = z - zs;
    t = slow*r;
    dtdx = 0;
    dtdz = 0;
    if (r > 0)
    {
        dtdx = (slow*deltaX)/r;
        dtdz = (slow*deltaZ)/r;
    }
}

constexpr double kSqrt1_2 = 0.70710678118654752440;

// v where valid, else HUGE or (SCALED: no time is above HUGE) a number above
// it, HUGE's next high word: one select instead of two, the low word does
// not matter.
template <bool SCALED>
__device__ __forceinline__ double valid_or_huge(double v, bool valid)
{
    if (!SCALED) { return valid ? v : kHuge; }
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t hi = valid ? (uint32_t) (u >> 32) : 0x4202A060u;
    return __builtin_bit_cast(double,
                              ((uint64_t) hi << 32) | (uint32_t) u);
}

// The Cartesian part of finiteDifference, uniform grid
// (solverUtilities2d.hpp:345-400).  Branch-free: every candidate is
// evaluated and the invalid ones are replaced by a number above HUGE, so
// the three square roots of a node run side by side; along a front nearly
// every wave has lanes that need each of them.  deta and detb of the
// reference are positive whenever their other conditions hold (0 <= dT <=
// h s0 / sqrt 2), so their own tests are left out; 2 (hs0 hs0) is exact, so
// the fused form of detc rounds once like the reference's subtraction.
//
// SCALED (models in range, Route2D): 2^-700 <= hs0 hs0 in every cell, so every valid
// determinant is in the range of sqrt_normal_range: deta and detb are at
// least about half of hs0 hs0, and a positive detc = 2 q - c c is q-sized
// or, where the terms cancel, a multiple of their last place, 2^-53 q.
template <bool SCALED>
__device__ __forceinline__ double cartesian2d_uniform(
    double h, double s0, double s1, double s3, double t1, double t2,
    double t3)
{
    double best = fmin(t1 + h*fmin(s0, s3), t3 + h*fmin(s0, s1));
    const double hs0 = h*s0;
    const double q = hs0*hs0;
    const double dTx = t3 - t2;
    const double dTz = t1 - t2;
    const double hs = h*(kSqrt1_2*s0);
    const double deta = q - dTz*dTz;
    const double detb = q - dTx*dTx;
    const double dtCross = t1 - t3;
    const double detc = fma(2.0, q, -(dtCross*dtCross));
    const bool ca = dTz >= 0 && dTz <= hs;
    const bool cb = dTx >= 0 && dTx <= hs;
    const bool cc = dTx >= 0 && dTz >= 0 && detc > 0 && t3 <= t1 + hs0 &&
                    t1 <= t3 + hs0;
    double ra, rb, rc;
    if constexpr (SCALED)
    {
        ra = sqrt_normal_range(deta);
        rb = sqrt_normal_range(detb);
        rc = sqrt_normal_range(detc);
    }
    else
    {
        ra = ::sqrt(ca ? deta : q);
        rb = ::sqrt(cb ? detb : q);
        rc = ::sqrt(cc ? detc : q);
    }
    best = fmin(best, valid_or_huge<SCALED>(t1 + h*ra, ca));
    best = fmin(best, valid_or_huge<SCALED>(t3 + h*rb, cb));
    return fmin(best, valid_or_huge<SCALED>(t2 + rc, cc));
}

// The spacings and ratios of the Cartesian updates.
struct Grid2D
{
    double dx, dz, dx_dz, dz_dx, cosTheta, sinTheta;
};

__device__ __forceinline__ Grid2D grid2d(const Problem2D &p)
{
    return Grid2D{p.dx, p.dz, p.dx_dz, p.dz_dx, p.cosTheta, p.sinTheta};
}

// The same, non-uniform grid (solverUtilities2d.hpp:474-560).
template <bool SCALED>
__device__ __forceinline__ double cartesian2d_nonuniform(
    const Grid2D &p, double s0, double s1, double s3, double t1, double t2,
    double t3)
{
    const double dx = p.dx, dz = p.dz;
    const double dx_dz = p.dx_dz, dz_dx = p.dz_dx;
    const double cosTheta = p.cosTheta, sinTheta = p.sinTheta;
    double best = fmin(t1 + dx*fmin(s0, s3), t3 + dz*fmin(s0, s1));
    const double dTx = t3 - t2;
    const double dTz = t1 - t2;
    const double sx = cosTheta*s0;
    const double sz = sinTheta*s0;
    const double hxs0 = dx*s0;
    const double hzs0 = dz*s0;
    const double deta = hzs0*hzs0 - dTz*dTz;
    const double detb = hxs0*hxs0 - dTx*dTx;
    const double tildeTx = t1 - t3 + t2;
    const double tildeTz = t3 - t1 + t2;
    const double dtCross = t1 - t3;
    const double detc = hxs0*hxs0 + hzs0*hzs0 - dtCross*dtCross;
    const bool ca = dTz >= 0 && deta >= 0 && dTz <= dz*sz;
    const bool cb = dTx >= 0 && detb >= 0 && dTx <= dx*sx;
    const bool cc = dTx >= 0 && dTz >= 0 && detc > 0 && t1 < t3 + hzs0 &&
                    t3 < t1 + hxs0;
    double ra, rb, rc;
    if constexpr (SCALED)
    {
        // With very unequal spacings a valid deta or detb can cancel to
        // zero; the root then taken, 2^-500, adds nothing to t1 or t3,
        // which are at least dT, about h s0 there.
        ra = sqrt_normal_range(fmax(deta, 0x1p-1000));
        rb = sqrt_normal_range(fmax(detb, 0x1p-1000));
        rc = sqrt_normal_range(detc);
    }
    else
    {
        ra = ::sqrt(ca ? deta : 1.0);
        rb = ::sqrt(cb ? detb : 1.0);
        rc = ::sqrt(cc ? detc : 1.0);
    }
    best = fmin(best, valid_or_huge<SCALED>(t1 + dx_dz*ra, ca));
    best = fmin(best, valid_or_huge<SCALED>(t3 + dz_dx*rb, cb));
    double tc = tildeTx*dz_dx + tildeTz*dx_dz + 2*rc;
    tc = (cosTheta*sinTheta)*tc;
    // a negative candidate is dropped (t0Update3 < 0 of the reference)
    return fmin(best, valid_or_huge<SCALED>(tc, cc && !(tc < 0)));
}

// A sweep's directions (bit 0: x decreasing, bit 1: z decreasing) and the
// first node of each permuted axis that it updates: 1, or the source
// quadrant in an initialisation sweep (getLoopLimits,
// solverUtilities2d.hpp:1004-1053).
struct Sweep2D
{
    int negX, negZ, signX, signZ, izShift, jx0, jz0;
};

__device__ __forceinline__ Sweep2D make_sweep2d(const Problem2D &p, int sweep,
                                                int initialize)
{
    Sweep2D s;
    s.negX = sweep & 1;
    s.negZ = (sweep >> 1) & 1;
    s.signX = s.negX ? -1 : 1;
    s.signZ = s.negZ ? -1 : 1;
    s.izShift = s.negZ ? 1 : -1;
    s.jx0 = 1;
    s.jz0 = 1;
    if (initialize)
    {
        s.jx0 = s.negX ? max(p.nx - 2 - p.srcCellX, 1) : max(p.srcCellX, 1);
        s.jz0 = s.negZ ? max(p.nz - 2 - p.srcCellZ, 1) : max(p.srcCellZ, 1);
    }
    return s;
}

// What the factored update and the source cell need, by value: the band
// kernel keeps it in scalar registers (through the descriptor, every step
// would load it again).
struct Source2D
{
    double dx, dz;              // dz: dx on a uniform grid
    double xs, zs, slowness;
    double dxinv, dzinv, hx2inv, hz2inv, twoOverH, twoOverH2, halfOverH2;
    int cellX, cellZ, radius;
    bool uniform;
};

__device__ __forceinline__ Source2D source2d(const Problem2D &p)
{
    return Source2D{p.dx, p.uniform ? p.dx : p.dz, p.srcOffX, p.srcOffZ,
                    p.srcSlowness, p.dxinv, p.dzinv, p.hx2inv, p.hz2inv,
                    p.twoOverH, p.twoOverH2, p.halfOverH2, p.srcCellX,
                    p.srcCellZ, p.radius, p.uniform != 0};
}

// Distance of node (ix, iz) from the source.
__device__ __forceinline__ double distance2d(const Source2D &s, int ix, int iz)
{
    return distance2d(ix, iz, s.dx, s.dz, s.xs, s.zs);
}

// finiteDifference near the source: the analytic time factored out, uniform
// grid (solverUtilities2d.hpp:400-472) and non-uniform (:560-614).  r0..r3:
// the distances from the source of the node and of its neighbours 1, 2
// and 3; the
// quotients of the spacings come from the descriptor.
__device__ __forceinline__ double factored2d(
    const Source2D &p, const Sweep2D &w, int ix, int iz, double s0,
    double s1, double s3, double t1, double t2, double t3, double r0,
    double r1, double r2, double r3)
{
    const double huge = kHuge;
    const double dx = p.dx, dz = p.dz;
    const double sourceSlowness = p.slowness;
    double t0x = t1 + dx*fmin(s0, s3);
    double t0z = t3 + dz*fmin(s0, s1);
    double t0Update1 = fmin(t0x, t0z);
    double dTx = t3 - t2;
    double dTz = t1 - t2;
    double hxs0 = dx*s0;
    double hzs0 = dz*s0;
    double t0Update3 = huge;
    if (dTx >= 0 && dTz >= 0 && t1 < t3 + hzs0 && t3 < t1 + hxs0)
    {
        double dt0dx, dt0dz, t0;
        analytic_time_deriv2d(ix, iz, dx, dz, p.xs, p.zs,
                              sourceSlowness, r0, t0, dt0dx, dt0dz);
        double tau1 = t1 - sourceSlowness*r1;
        double tau2 = t2 - sourceSlowness*r2;
        double tau3 = t3 - sourceSlowness*r3;
        dt0dx = w.signX*dt0dx;
        dt0dz = w.signZ*dt0dz;
        double tauX = tau1 - tau3 + tau2;
        double tauZ = tau3 - tau1 + tau2;
        const double two = 2, four = 4;
        double a, b, c;
        if (p.uniform)
        {
            a = p.hx2inv;
            b = p.twoOverH*(dt0dx + dt0dz) - p.twoOverH2*tau2;
            c = p.halfOverH2*(tauX*tauX + tauZ*tauZ)
              - p.twoOverH*(dt0dx*tauX + dt0dz*tauZ)
              + two*(sourceSlowness*sourceSlowness - s0*s0);
        }
        else
        {
            a = p.hx2inv + p.hz2inv;
            b = four*(p.dxinv*dt0dx + p.dzinv*dt0dz)
              - two*(tauX*p.hx2inv + tauZ*p.hz2inv);
            c = (tauX*tauX)*p.hx2inv + (tauZ*tauZ)*p.hz2inv
              - four*((dt0dx*tauX)*p.dxinv + (dt0dz*tauZ)*p.dzinv)
              + four*(sourceSlowness*sourceSlowness - s0*s0);
        }
        double det = b*b - four*a*c;
        if (det >= 0)
        {
            double tau = (-b + ::sqrt(det))/(two*a);
            t0Update3 = t0 + tau;
        }
        if (t0Update3 < t1 || t0Update3 < t3) { t0Update3 = huge; }
    }
    return fmin(t0Update1, t0Update3);
}

__device__ __forceinline__ bool in_factored_box2d(const Source2D &p, int ix,
                                                  int iz)
{
    return !(abs(p.cellX - ix) > p.radius || abs(p.cellZ - iz) > p.radius);
}

// ---------------------------------------------------------------------------
// Band kernel: one workgroup solves one problem.  The grid's rows are cut
// into bands of 64 (grid rows 64 m .. 64 m + 63), one wave each, for the
// whole solve.  In the sweep's permuted frame lane i owns row i of its band
// and at step t works on column t - i: its x neighbour is its own previous
// value, its z neighbour the value that lane i - 1 computed one step
// earlier, one cross-lane move (wave_shr) away.  A band's last row goes to
// the next band through a ring in LDS; the next band runs kLag2d groups of
// kGroup2d steps behind, and one block barrier per group is all the
// synchronisation there is.  The lags are constant, so every wave derives
// its start in each sweep from the sizes alone, and a sweep that keeps the
// z direction follows the one before it without a gap.
//
// What bounds it: the chain of nx + nz dependent node updates per sweep, on
// waves that have a SIMD to themselves (up to 4 bands): such a wave issues
// one instruction every 4 cycles, scalar ones included, so a step costs its
// instruction count, not its latency.  Hence the group kinds below (what a
// group cannot meet costs it nothing), fixed strides (immediate offsets
// instead of address arithmetic) and stores without a mask.
//
// Times between sweeps: step records of 64 values, in the step and lane
// order of the sweep that reads them, so that every access of the step loop
// is coalesced.  The x direction reverses with every sweep, so a sweep
// always writes its records backwards, into the other of two buffers; a
// lane outside the grid writes a padding element (its column is outside
// the reader's grid too).  The last sweep writes the natural-order field.
//
// 201 x 201, 2 iterations: LDS-level kernel 2.81 ms, this kernel 1.24 ms;
// 701 x 523, 3 iterations: 31.4 ms (memory-only levels) and 9.4 ms.
// ---------------------------------------------------------------------------
constexpr int kBand2d = 64;
constexpr int kGroup2d = 8;
// groups between a band and the next: the first column of the band's last
// row is done at step 63, i.e. within group 8
constexpr int kLag2d = kBand2d/kGroup2d + 1;
// columns of a band's last row kept for the next band: written up to 16
// ahead of the reader
constexpr int kRing2d = 64;

// Doubles in device memory: through generic pointers the accesses would be
// FLAT ones, which the waits for LDS also wait for.
using GlobalDouble = __attribute__((address_space(1))) double;

// lane i's value of lane i - 1; lane 0 takes `first`
__device__ __forceinline__ double from_previous_lane(double v, double first)
{
    constexpr int kWaveShr1 = 0x138;
    const uint64_t a = __builtin_bit_cast(uint64_t, v);
    const uint64_t f = __builtin_bit_cast(uint64_t, first);
    const uint32_t lo = (uint32_t) __builtin_amdgcn_update_dpp(
        (int) (uint32_t) f, (int) (uint32_t) a, kWaveShr1, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t) __builtin_amdgcn_update_dpp(
        (int) (f >> 32), (int) (a >> 32), kWaveShr1, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((uint64_t) hi << 32) | lo);
}

// LDS accesses done, then the barrier: values exchanged between waves are
// in LDS, global accesses stay in flight.  The compiler treats both
// builtins as touching no memory, so empty asm statements keep the accesses
// on their side.
__device__ __forceinline__ void group_barrier()
{
    __asm__ __volatile__("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
    __asm__ __volatile__("" ::: "memory");
}

// What a group of steps can meet.  kFull: every lane is on a column that
// the sweep updates, none in the factored box.  kIdle: no lane updates
// anything.  kAny: lanes enter or leave the columns.  kRare: kAny in the
// solve's first sweep (old times HUGE and the source cell's corners) or its
// last one (writes the field), or with lanes in the factored box.
enum Group2D { kFull, kIdle, kAny, kRare };

// A band's wave within one sweep; AHEAD: steps that a record is loaded
// ahead.
template <int AHEAD>
struct Band2D
{
    Source2D src;
    Sweep2D w;
    Grid2D grid;
    int lane, iz, nx;
    bool row;               // the lane's row is in the grid
    uint32_t liveSpan;      // columns it updates (from jx0)
    double floor;           // kFull: above HUGE in lanes that update nothing
    bool first, last;       // the solve's first or last sweep
    int boxLo, boxHi;       // steps with lanes in the box
    int t;                  // first step of the next AHEAD
    const GlobalDouble *old, *cells;    // records AHEAD steps ahead
    GlobalDouble *out;
    // From AHEAD steps to the next.  Lanes whose whole 128 byte line has no
    // row stay in their first records, which costs nothing and takes their
    // values out of a traffic that bounds batches (256 problems of 201 x 201,
    // 55 lanes of the last band without a row: 1.87 ms, 1.76 so; 4096: 29.4
    // and 28.0; lines written in part are slower than whole ones: 1024
    // problems of 120 x 60 1.04 ms, 1.13 with their four lanes left out too).
    // Not in the instances of more than 8 bands, where one lane in 9 at most
    // has no row and the two registers are spilled.
    static constexpr bool kStays = AHEAD == kGroup2d;
    uint32_t steps[2];
    __device__ __forceinline__ uint32_t record_step() const
    { return kStays ? steps[0] : (uint32_t) (AHEAD*kBand2d); }
    __device__ __forceinline__ uint32_t cell_step() const
    { return kStays ? steps[1] : (uint32_t) (AHEAD*kCellRecord2d); }
    double cur, s1Prev, t3Prev, hand;
    // in the box's steps: distances from the source of the lane's previous
    // node and of that node's z neighbour
    double r0, r3;
    double T0[AHEAD], SA[AHEAD], SB[AHEAD];

    // the records of steps t .. t + AHEAD - 1, which old and cells point at
    __device__ __forceinline__ void load()
    {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
        {
            T0[u] = old[u*kBand2d];
            SA[u] = cells[u*kCellRecord2d];
            SB[u] = cells[u*kCellRecord2d + 1];
        }
        old += record_step();
        cells += cell_step();
    }
    // the first sweep's old time of the lane's node in column ix
    __device__ __forceinline__ double start_time(int ix) const
    {
        const int ox = ix - src.cellX, oz = iz - src.cellZ;
        double v = kHuge;
        if (ox >= 0 && ox <= 1 && oz >= 0 && oz <= 1)
        {
            v = analytic_time2d(ix, iz, grid.dx, grid.dz, src.xs, src.zs,
                                src.slowness);
        }
        return v;
    }
    template <bool UNIFORM, bool SCALED>
    __device__ __forceinline__ double cartesian(double s0, double s1,
                                                double s3, double t1,
                                                double t2, double t3) const
    {
        if constexpr (UNIFORM)
        {
            return cartesian2d_uniform<SCALED>(grid.dx, s0, s1, s3, t1,
                                               t2, t3);
        }
        else
        {
            return cartesian2d_nonuniform<SCALED>(grid, s0, s1, s3, t1,
                                                  t2, t3);
        }
    }
};

// AHEAD steps.  ri: the previous band's last row (column t + u + 1 in
// ri[u]); hp: where lane 63 leaves this band's.
template <bool UNIFORM, bool SCALED, Group2D KIND, int AHEAD>
__device__ __forceinline__ void band_steps(Band2D<AHEAD> &b, const double *ri,
                                           double *hp)
{
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
    {
        const double t3 = from_previous_lane(b.cur, b.hand);
        b.hand = ri[u];
        const double t1 = b.cur, t2 = b.t3Prev;
        const double s0 = b.s1Prev, s1 = b.SA[u], s3 = b.SB[u];
        double t0 = b.T0[u];
        // the record AHEAD steps on, into the freed registers
        b.T0[u] = b.old[u*kBand2d];
        b.SA[u] = b.cells[u*kCellRecord2d];
        b.SB[u] = b.cells[u*kCellRecord2d + 1];
        b.t3Prev = t3;
        b.s1Prev = s1;
        const int jx = b.t + u - b.lane;
        const int ix = b.w.negX ? b.nx - 1 - jx : jx;
        if constexpr (KIND == kIdle) { b.cur = t0; }
        else
        {
            double v = b.template cartesian<UNIFORM, SCALED>(s0, s1, s3, t1,
                                                             t2, t3);
            if constexpr (KIND == kFull)
            {
                b.cur = fmin(fmax(v, b.floor), t0);
            }
            else
            {
                const bool live = (uint32_t) (jx - b.w.jx0) < b.liveSpan;
                if constexpr (KIND == kRare)
                {
                    if (b.first) { t0 = b.start_time(ix); }
                    if (b.t + u >= b.boxLo - 1 && b.t + u <= b.boxHi)
                    {
                        // the node's x neighbour is the lane's previous
                        // node
                        const double r1 = b.r0, r2 = b.r3;
                        b.r0 = distance2d(b.src, ix, b.iz);
                        b.r3 = distance2d(b.src, ix, b.iz + b.w.izShift);
                        if (live && in_factored_box2d(b.src, ix, b.iz))
                        {
                            v = factored2d(b.src, b.w, ix, b.iz, s0, s1, s3,
                                           t1, t2, t3, b.r0, r1, r2, b.r3);
                        }
                    }
                }
                b.cur = live && v < t0 ? v : t0;
            }
        }
        hp[u] = b.cur;
        if (KIND == kRare && b.last)
        {
            if (b.row && (uint32_t) jx < (uint32_t) b.nx)
            {
                b.out[ix] = b.cur;
            }
        }
        else { b.out[-u*kBand2d] = b.cur; }
    }
    b.t += AHEAD;
    b.old += b.record_step();
    b.cells += b.cell_step();
    if (!(KIND == kRare && b.last)) { b.out -= b.record_step(); }
}

// One sweep of one band.  old: record of step 0 (this lane's value); cells:
// the sweep's cell records; out: this lane's result of step 0, the next
// steps' each one record before it (last: the start of the lane's row in
// the field).
template <bool UNIFORM, bool SCALED, int AHEAD>
__device__ __forceinline__ void band_sweep(
    const Problem2D &p, const Sweep2D &w, int band, int height, int lane,
    int groups, bool first, bool last, const GlobalDouble *old, const GlobalDouble *cells,
    GlobalDouble *out, const double *ringIn, double *ringOut, double *sink)
{
    const int nx = p.nx, nz = p.nz;
    const int iz = kBand2d*band + (w.negZ ? height - 1 - lane : lane);
    const int jz = w.negZ ? nz - 1 - iz : iz;
    const bool row = lane < height && iz < nz;
    const bool rowLive = row && jz >= w.jz0;
    const bool anyRow = __builtin_amdgcn_ballot_w64(rowLive) != 0;
    const int line = kBand2d*band +
                     (w.negZ ? height - 1 - (lane | 15) : lane & ~15);
    const bool stream = (lane & ~15) < height && line < nz;
    // the constants of the step loop in registers (the barriers' memory
    // clobbers would reload them)
    Band2D<AHEAD> b{source2d(p), w, grid2d(p), lane, iz, nx, row,
                    rowLive ? (uint32_t) (nx - w.jx0) : 0u,
                    rowLive ? -kHuge : 4*kHuge, first, last, 1, 0, 0, old,
                    cells + lane, out,
                    {stream ? AHEAD*kBand2d : 0u,
                     stream ? AHEAD*kCellRecord2d : 0u}, 0, 0, 0, 0, 0, 0, {}, {},
                    {}};
    // Runs of groups of one kind: [0, idleEnd) idle, [fullLo, fullHi) full,
    // [boxLo, boxEnd) with lanes in the box or on the step before it.
    // (the step before the first live one is not idle: it leaves the box's
    // distances)
    const int idleEnd = anyRow ? min((w.jx0 - 1)/kGroup2d, groups) : groups;
    const int fullLo = (w.jx0 + height - 2)/kGroup2d + 1;
    const int fullHi = nx/kGroup2d;
    int boxGroup = groups, boxEnd = groups;
    const int zLo = max(p.srcCellZ - p.radius, 0);
    const int zHi = min(p.srcCellZ + p.radius, nz - 1);
    if (p.radius >= 0 && zHi >= kBand2d*band && zLo < kBand2d*(band + 1))
    {
        const int xLo = max(p.srcCellX - p.radius, 0);
        const int xHi = min(p.srcCellX + p.radius, nx - 1);
        // the lanes of the box's rows in this band
        const int iLo = max(zLo - kBand2d*band, 0);
        const int iHi = min(zHi - kBand2d*band, height - 1);
        b.boxLo = (w.negX ? nx - 1 - xHi : xLo) +
                  (w.negZ ? height - 1 - iHi : iLo);
        b.boxHi = (w.negX ? nx - 1 - xLo : xHi) +
                  (w.negZ ? height - 1 - iLo : iHi);
        boxGroup = max(b.boxLo - 1, 0)/kGroup2d;
        boxEnd = b.boxHi/kGroup2d + 1;
    }
    b.load();
    // groups [g, end) of one kind; step(ri, hp) runs AHEAD steps.
    // ri: the previous band's last row at the columns after the step's
    // (column c in slot c - 1, so that the writer's eight are contiguous),
    // read one step ahead; hp: lane 63 writes column t - 63 (from the group
    // that holds column 0 on), the other lanes into a sink.
    auto run = [&](int g, int end, auto &&step)
    {
        for (; g < end; ++g)
        {
            const int t = g*kGroup2d;
            b.hand = ringIn[(t - 1) & (kRing2d - 1)];
            const double *ri = ringIn + (t & (kRing2d - 1));
            double *hp = lane == kBand2d - 1 && g >= kLag2d - 2
                             ? ringOut + (t & (kRing2d - 1)) : sink;
#pragma unroll 1
            for (int part = 0; part < kGroup2d; part += AHEAD)
            {
                step(ri + part, hp + part);
            }
            group_barrier();
        }
    };
    for (int g = 0; g < groups;)
    {
        int end = groups;
        if (g < idleEnd) { end = min(end, idleEnd); }
        if (g < fullLo) { end = min(end, fullLo); }
        if (g < fullHi) { end = min(end, fullHi); }
        if (g < boxGroup) { end = min(end, boxGroup); }
        if (g < boxEnd) { end = min(end, boxEnd); }
        if (first || last || (g >= idleEnd && g >= boxGroup && g < boxEnd))
        {
            run(g, end, [&](const double *ri, double *hp)
                { band_steps<UNIFORM, SCALED, kRare>(b, ri, hp); });
        }
        else if (g < idleEnd)
        {
            run(g, end, [&](const double *ri, double *hp)
                { band_steps<UNIFORM, SCALED, kIdle>(b, ri, hp); });
        }
        else if (g >= fullLo && g < fullHi)
        {
            run(g, end, [&](const double *ri, double *hp)
                { band_steps<UNIFORM, SCALED, kFull>(b, ri, hp); });
        }
        else
        {
            run(g, end, [&](const double *ri, double *hp)
                { band_steps<UNIFORM, SCALED, kAny>(b, ri, hp); });
        }
        g = end;
    }
}

template <int WAVES, int AHEAD, bool SCALED>
__global__ void __launch_bounds__(kBand2d*WAVES)
solve2d_bands_kernel(const Problem2D *__restrict__ problems,
                     double *__restrict__ T, double *work,
                     const double *__restrict__ cells)
{
    // (a group's last read-ahead takes the value after the ring)
    __shared__ double ring[WAVES][kRing2d + 1];
    __shared__ double sinks[WAVES][kBand2d + kGroup2d];
    const Problem2D &p = problems[blockIdx.x];
    if (p.route != (SCALED ? kBands2d : kBandsAnyRange2d)) { return; }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int nx = p.nx, nz = p.nz;
    const int nb = bands2d(nz);
    // a wave without a band leaves: barriers count the running waves
    if (wave >= nb) { return; }
    // the two buffers of the band's records, at step 0
    const int64_t perBand = (int64_t) band_records2d(nx)*kBand2d;
    GlobalDouble *rec[2];
    rec[0] = (GlobalDouble *) work + p.wOffset + wave*perBand +
             kBandPad2d*kBand2d;
    rec[1] = rec[0] + nb*perBand;
    const GlobalDouble *bandCells = (const GlobalDouble *) cells +
        p.cOffset + (int64_t) wave*cell_steps2d(nx)*kCellRecord2d;
    double *sink = &sinks[wave][lane];
    const int nSweeps = 4*(1 + p.nSweeps);
    // the last lane with rows ends the band's steps: a band alone is as high
    // as the grid (10 x 10, 12 sweeps: 0.31 ms with all 64 lanes, 0.14)
    const int height = nb == 1 ? nz : kBand2d;
    const int groups = (nx + height - 1 + kGroup2d - 1)/kGroup2d;
    int now = 0, base = 0;
    for (int k = 0; k < nSweeps; ++k)
    {
        const int sweep = k & 3;
        const bool last = k == nSweeps - 1;
        const Sweep2D w = make_sweep2d(p, sweep, k < 4);
        const bool nextNegZ = (k + 1) & 2;
        // z reverses with every second sweep: the band that was last is
        // first, and the others wait for it
        if (k > 0) { base += groups + ((k & 1) ? 0 : kLag2d*(nb - 1)); }
        const int pos = w.negZ ? nb - 1 - wave : wave;
        for (; now < base + kLag2d*pos; ++now) { group_barrier(); }
        const GlobalDouble *old = ((k & 1) ? rec[1] : rec[0]) + lane;
        // the result of step t, column jx = t - lane: the next sweep's
        // lane i' of the same row at its step (nx - 1 - jx) + i'
        // (a lane without a row writes a slot of its own)
        const int i = nextNegZ == (bool) w.negZ || lane >= height
                          ? lane : height - 1 - lane;
        GlobalDouble *out = ((k & 1) ? rec[0] : rec[1]) +
                            (int64_t) (nx - 1 + lane + i)*kBand2d + i;
        if (last)
        {
            const int izl = kBand2d*wave +
                            (w.negZ ? height - 1 - lane : lane);
            out = (GlobalDouble *) T + p.tOffset + (int64_t) izl*nx;
        }
        const int upstream = w.negZ ? min(wave + 1, nb - 1)
                                    : max(wave - 1, 0);
        const GlobalDouble *sc = bandCells +
            (int64_t) sweep*nb*cell_steps2d(nx)*kCellRecord2d;
        if (p.uniform)
        {
            band_sweep<true, SCALED, AHEAD>(p, w, wave, height, lane, groups,
                                            k == 0, last, old, sc, out,
                                            ring[upstream], ring[wave], sink);
        }
        else
        {
            band_sweep<false, SCALED, AHEAD>(p, w, wave, height, lane, groups,
                                             k == 0, last, old, sc, out,
                                             ring[upstream], ring[wave],
                                             sink);
        }
        now += groups;
        // the next sweep reads this one's records, by other lanes of the
        // wave: the stores first
        __asm__ __volatile__("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0);
        __asm__ __volatile__("" ::: "memory");
    }
}

// The skewed cell records of one model for the four sweeps: value i of
// step t of a band is the cell at permuted column t - i, permuted row
// (the node row of lane i) - 1, clamped to the model: lane i's own cell
// row (its cells 0 and 1) in value i, and in value i + 1 the row beyond
// (its cell 3: column t - i - 1, row + 1).
__global__ void __launch_bounds__(256)
skew_cells2d_kernel(int nx, int nz, const double *__restrict__ s,
                    double *__restrict__ out)
{
    // grid (x): the values of a band's steps; (y): bands of the four sweeps
    const int ncx = nx - 1, ncz = nz - 1;
    const int nb = bands2d(nz), values = cell_steps2d(nx)*kCellRecord2d;
    const int e = blockIdx.x*blockDim.x + threadIdx.x;
    if (e >= values) { return; }
    const int sweep = (int) blockIdx.y/nb, band = (int) blockIdx.y - sweep*nb;
    const int t = e/kCellRecord2d, i = e - t*kCellRecord2d;
    const bool negX = sweep & 1, negZ = sweep & 2;
    // permuted row of lane 0 of the band (a band alone: as high as the grid)
    const int jzBase = nb == 1 ? 0
                       : negZ ? nz - kBand2d*(band + 1) : kBand2d*band;
    const int pcx = min(max(t - i, 0), ncx - 1);
    const int pcz = min(max(jzBase + i - 1, 0), ncz - 1);
    const int cx = negX ? ncx - 1 - pcx : pcx;
    const int cz = negZ ? ncz - 1 - pcz : pcz;
    out[(int64_t) blockIdx.y*values + e] = s[(int64_t) cz*ncx + cx];
}

// ---------------------------------------------------------------------------
// Level kernel, for grids that the band kernel does not take: one sweep of
// one problem in anti-diagonal order (levels jx + jz), levels separated by
// block barriers, global memory only.
// ---------------------------------------------------------------------------
__device__ void sweep2d_block(const Problem2D &p, int sweep, int initialize,
                              double *__restrict__ T,
                              const double *__restrict__ S)
{
    const int nx = p.nx, nz = p.nz, ncx = nx - 1, ncz = nz - 1;
    const Sweep2D w = make_sweep2d(p, sweep, initialize);
    const Source2D src = source2d(p);
    const int lastLevel = (nx - 1) + (nz - 1);
    for (int level = w.jx0 + w.jz0; level <= lastLevel; ++level)
    {
        const int kLo = max(w.jz0, level - (nx - 1));
        const int kHi = min(nz - 1, level - w.jx0);
        for (int jz = kLo + (int) threadIdx.x; jz <= kHi; jz += blockDim.x)
        {
            const int jx = level - jz;
            const int ix = w.negX ? nx - 1 - jx : jx;
            const int iz = w.negZ ? nz - 1 - jz : jz;
            const int ixU = w.negX ? ix + 1 : ix - 1;
            const int izU = w.negZ ? iz + 1 : iz - 1;
            // gridToSurroundingSlowness (solverUtilities2d.hpp:1279-1370)
            // in the permuted frame: home (jx-1, jz-1), offsets clamped.
            const int pcxH = jx - 1, pcxO = min(jx, ncx - 1);
            const int pczH = jz - 1, pczO = min(jz, ncz - 1);
            const int cxH = w.negX ? ncx - 1 - pcxH : pcxH;
            const int cxO = w.negX ? ncx - 1 - pcxO : pcxO;
            const int czH = w.negZ ? ncz - 1 - pczH : pczH;
            const int czO = w.negZ ? ncz - 1 - pczO : pczO;
            const double s0 = S[czH*ncx + cxH];
            const double s1 = S[czH*ncx + cxO];
            const double s3 = S[czO*ncx + cxH];
            const int i0 = iz*nx + ix;
            const double t0 = T[i0];
            const double t1 = T[iz*nx + ixU];
            const double t2 = T[izU*nx + ixU];
            const double t3 = T[izU*nx + ix];
            double tUpd;
            if (in_factored_box2d(src, ix, iz))
            {
                tUpd = factored2d(src, w, ix, iz, s0, s1, s3, t1, t2, t3,
                                  distance2d(src, ix, iz),
                                  distance2d(src, ixU, iz),
                                  distance2d(src, ixU, izU),
                                  distance2d(src, ix, izU));
            }
            else if (p.uniform)
            {
                tUpd = cartesian2d_uniform<false>(p.dx, s0, s1, s3, t1, t2, t3);
            }
            else
            {
                tUpd = cartesian2d_nonuniform<false>(grid2d(p), s0, s1, s3,
                                                     t1, t2, t3);
            }
            if (tUpd < t0) { T[i0] = tUpd; }
        }
        __syncthreads();
    }
}

__global__ void __launch_bounds__(1024)
solve2d_kernel(const Problem2D *__restrict__ problems, double *__restrict__ T,
               const double *__restrict__ S)
{
    const Problem2D &p = problems[blockIdx.x];
    if (p.route != kLevels2d) { return; }
    double *Tp = T + p.tOffset;
    const double *Sp = S + p.sOffset;
    const int n = p.nx*p.nz;
    // Solver2DImpl::initializeTravelTimes (src/solver2d.cpp:61-105)
    for (int i = threadIdx.x; i < n; i += blockDim.x)
    {
        int iz = i/p.nx, ix = i - iz*p.nx;
        int ox = ix - p.srcCellX, oz = iz - p.srcCellZ;
        double v = kHuge;
        if (ox >= 0 && ox <= 1 && oz >= 0 && oz <= 1)
        {
            v = analytic_time2d(ix, iz, p.dx, p.dz, p.srcOffX, p.srcOffZ,
                                p.srcSlowness);
        }
        Tp[i] = v;
    }
    __syncthreads();
    for (int sweep = 0; sweep < 4; ++sweep)
    {
        sweep2d_block(p, sweep, 1, Tp, Sp);
    }
    for (int k = 0; k < p.nSweeps; ++k)
    {
        for (int sweep = 0; sweep < 4; ++sweep)
        {
            sweep2d_block(p, sweep, 0, Tp, Sp);
        }
    }
}

// Solver2DImpl::interpolateTravelTimes (src/solver2d.cpp:106-167) with
// bilinear (src/ray/bilinear.hpp).  Station (x, z) offsets and cells are
// computed on the host exactly as Station2D does.
__global__ void __launch_bounds__(256)
stations2d_kernel(const Problem2D *__restrict__ problem, int n,
                  const double *__restrict__ xOff,
                  const double *__restrict__ zOff,
                  const int *__restrict__ cellX, const int *__restrict__ cellZ,
                  const double *__restrict__ T, double *__restrict__ out)
{
    const int i = blockIdx.x*blockDim.x + threadIdx.x;
    if (i >= n) { return; }
    const Problem2D &p = *problem;
    const double *Tp = T + p.tOffset;
    const double dx = p.dx, dz = p.dz;
    const double dxi = 1./dx;
    const double dzi = 1./dz;
    const double xi = xOff[i], zi = zOff[i];
    const int cx = cellX[i], cz = cellZ[i];
    if (cx == p.srcCellX && cz == p.srcCellZ)
    {
        out[i] = ::hypot(xi - p.srcOffX, zi - p.srcOffZ)*p.srcSlowness;
        return;
    }
    const int i00 = cz*p.nx + cx;
    const int i10 = i00 + 1;
    const int i01 = i00 + p.nx;
    const int i11 = i01 + 1;
    const double x1 = cx*dx;
    const double x2 = (cx + 1)*dx;
    const double z1 = cz*dz;
    const double z2 = (cz + 1)*dz;
    const double f00 = Tp[i00], f01 = Tp[i01], f10 = Tp[i10], f11 = Tp[i11];
    double x2mx = x2 - xi;
    double xmx1 = xi - x1;
    double fxz1 = dxi*(x2mx*f00 + xmx1*f10);
    double fxz2 = dxi*(x2mx*f01 + xmx1*f11);
    double z2mz = z2 - zi;
    double zmz1 = zi - z1;
    out[i] = dzi*(z2mz*fxz1 + zmz1*fxz2);
}

__global__ void __launch_bounds__(256)
nodal_to_cell2d(int nx, int nz, const double *__restrict__ v, int ordering,
                double *__restrict__ slow)
{
    const int ncx = nx - 1, ncz = nz - 1;
    for (int i = blockIdx.x*blockDim.x + threadIdx.x; i < ncx*ncz;
         i += gridDim.x*blockDim.x)
    {
        int iz = i/ncx, ix = i - iz*ncx;
        int idx1, idx2, idx3, idx4;
        if (ordering == 0)
        {
            idx1 = iz*(ncx + 1) + ix;
            idx2 = idx1 + 1;
            idx3 = idx1 + (ncx + 1);
            idx4 = idx3 + 1;
        }
        else
        {
            idx1 = ix*(ncz + 1) + iz;
            idx2 = idx1 + 1;
            idx3 = idx1 + (ncz + 1);
            idx4 = idx3 + 1;
        }
        double sum1 = v[idx1] + v[idx2];
        double sum2 = v[idx3] + v[idx4];
        slow[i] = 4.0/(sum1 + sum2);
    }
}

// Workgroups that a CU should hold, 0: as many as fit.  Half of the sweeps
// write lane i's value two records from lane i - 1's, so lines leave L2 partly
// written, and where the records of the resident problems spill from the 256
// MB Infinity Cache each costs memory traffic (4096 problems of 201 x 201 with
// two a CU, 424 MB: 61 GB written for 27 GB of records).  So no bound up to 128
// MB in all, else what keeps 230 MB, up to a wave a SIMD or two workgroups
// (three of two bands up to 128 MB).  ms with 1, 2, 3, 4 and 8 a CU, and the MB
// of one on every CU:
//   4096 of 201 x 201  212 MB  28.0 31.8
//   4096 of 120 x 180  129     14.5 15.2
//   4096 of 40 x 250   103     12.5 10.1
//   4096 of 60 x 200    98     13.7 13.1
//   4096 of 120 x 128   94     12.2  8.5 10.5 11.7
//   4096 of 300 x 60    87     17.8  9.6  9.8 10.8 13.3
//   4096 of 80 x 100    59     10.3  6.7  7.3  8.7
//   4096 of 40 x 100    41      8.4  5.2  4.7  5.8
//   8192 of 51 x 41     19     13.9  7.5  6.1  6.1  8.8
//   4096 of 5 x 100     27      6.6  4.0  3.2  3.4
//   1024 of 5 x 100 (109 MB in all)      1.66 1.06 1.00 0.72
//   2048 of 20 x 40 (106 MB in all)      2.18 1.18 1.01 0.86 0.77
static int64_t band_workgroups_per_cu(const Plan2D &plan)
{
    constexpr int64_t kCUs = 256, kMB = (int64_t) 1 << 20;
    const int64_t n = plan.problems[kBands2d] +
                      plan.problems[kBandsAnyRange2d];
    if (plan.recordBytes <= 128*kMB) { return 0; }
    const int64_t each = plan.recordBytes/n*kCUs;
    const int64_t waves = 4*n/plan.bands;       // of one a SIMD
    if (waves == 2 && 3*each <= 128*kMB) { return 3; }
    return std::max<int64_t>(1, std::min(std::max<int64_t>(2, waves),
                                         230*kMB/each));
}

// LDS that a band workgroup asks for beyond its own, so that a CU holds no
// more of them.
static size_t band_residency_lds(const Plan2D &plan, size_t own)
{
    constexpr size_t kLdsPerCU = 160*1024;
    const size_t groups = (size_t) band_workgroups_per_cu(plan);
    if (groups == 0) { return 0; }
    // (a margin of 2 KB for the allocation's granules)
    const size_t share = kLdsPerCU/groups/1024*1024 - 2048;
    return share > own ? share - own : 0;
}

template <int WAVES, int AHEAD, bool SCALED>
static void launch_bands2d(const Problem2D *dProblems, int nProblems,
                           const Plan2D &plan, double *T, double *work,
                           const double *cells, hipStream_t stream)
{
    constexpr size_t kOwn =
        WAVES*(kRing2d + 1 + kBand2d + kGroup2d)*sizeof(double);
    hipLaunchKernelGGL((solve2d_bands_kernel<WAVES, AHEAD, SCALED>),
                       dim3((unsigned) nProblems),
                       dim3(kBand2d*bands2d(plan.maxNz)),
                       band_residency_lds(plan, kOwn), stream, dProblems, T,
                       work, cells);
}

// Registers per wave set the read-ahead: 8 steps (223 registers) while
// at most 2 waves share a SIMD, 4 steps (168) for 3 waves, 2 for 4 waves
// (128).  201 x 41, one band: 266 ns a step with 4 steps, 239 with 8.
template <bool SCALED>
static void launch_bands2d(const Problem2D *dProblems, int nProblems,
                           const Plan2D &plan, double *T, double *work,
                           const double *cells, hipStream_t stream)
{
    const int nb = bands2d(plan.maxNz);
    if (nb <= 8)
    {
        launch_bands2d<8, 8, SCALED>(dProblems, nProblems, plan, T, work,
                                     cells, stream);
    }
    else if (nb <= 12)
    {
        launch_bands2d<12, 4, SCALED>(dProblems, nProblems, plan, T, work,
                                      cells, stream);
    }
    else
    {
        launch_bands2d<kMaxBands2d, 2, SCALED>(dProblems, nProblems, plan, T,
                                               work, cells, stream);
    }
}

hipError_t launch_solve2d(const Problem2D *dProblems, int nProblems,
                          const Plan2D &plan, double *T, const double *S,
                          double *work, const double *cells,
                          hipStream_t stream)
{
    if (plan.problems[kLevels2d] > 0)
    {
        hipLaunchKernelGGL(solve2d_kernel, dim3((unsigned) nProblems),
                           dim3(256), 0, stream, dProblems, T, S);
    }
    if (plan.problems[kBands2d] > 0)
    {
        launch_bands2d<true>(dProblems, nProblems, plan, T, work, cells,
                             stream);
    }
    if (plan.problems[kBandsAnyRange2d] > 0)
    {
        launch_bands2d<false>(dProblems, nProblems, plan, T, work, cells,
                              stream);
    }
    return hipGetLastError();
}

// (one launch, 10 us less than reading the slowness back and uploading)
__global__ void __launch_bounds__(64)
store_problem2d_kernel(Problem2D p, const double *__restrict__ cell,
                       Problem2D *__restrict__ dst)
{
    if (threadIdx.x != 0) { return; }
    p.srcSlowness = *cell;
    *dst = p;
}

hipError_t launch_store_problem2d(const Problem2D &p, const double *cell,
                                  Problem2D *dst, hipStream_t stream)
{
    hipLaunchKernelGGL(store_problem2d_kernel, dim3(1), dim3(64), 0, stream,
                       p, cell, dst);
    return hipGetLastError();
}

hipError_t launch_skew_cells2d(int nx, int nz, const double *s, double *out,
                               hipStream_t stream)
{
    const int values = cell_steps2d(nx)*kCellRecord2d;
    hipLaunchKernelGGL(skew_cells2d_kernel,
                       dim3((unsigned) ((values + 255)/256),
                            (unsigned) (4*bands2d(nz))),
                       dim3(256), 0, stream, nx, nz, s, out);
    return hipGetLastError();
}

hipError_t launch_stations2d(const Problem2D *dProblem, int n,
                             const double *xOff, const double *zOff,
                             const int *cellX, const int *cellZ,
                             const double *T, double *out, hipStream_t stream)
{
    if (n <= 0) { return hipSuccess; }
    hipLaunchKernelGGL(stations2d_kernel, dim3((unsigned) ((n + 255)/256)),
                       dim3(256), 0, stream, dProblem, n, xOff, zOff, cellX,
                       cellZ, T, out);
    return hipGetLastError();
}

hipError_t launch_nodal_to_cell2d(int nx, int nz, const double *v,
                                  int ordering, double *slow,
                                  hipStream_t stream)
{
    int nCell = (nx - 1)*(nz - 1);
    unsigned g = (unsigned) ((nCell + 255)/256);
    if (g > 4096) { g = 4096; }
    hipLaunchKernelGGL(nodal_to_cell2d, dim3(g), dim3(256), 0, stream, nx, nz,
                       v, ordering, slow);
    return hipGetLastError();
}

} // namespace ekx
