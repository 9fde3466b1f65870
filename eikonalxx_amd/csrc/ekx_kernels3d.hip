// ekx_kernels3d.hip -- HIP kernels of the 3D fast-sweeping solver (gfx950).
//
// Sweep k (0..7) visits nodes in the order of Solver3DSweep<k>::updateFSM
// (include/private/solver3d.hpp:150-326).  In the sweep's permuted frame
// (solverUtilities3d.hpp:1197-1257) every sweep runs towards +x, +y, +z and
// a node reads only its 7 upwind neighbours, which lie on earlier
// hyperplanes jx+jy+jz.  Any schedule that finishes those neighbours first
// therefore reproduces the serial loop exactly; both kernels below are such
// schedules.
#include "ekx_kernels.hpp"
#include "ekx_local3d.hpp"
#include "ekx_storage.hpp"
#include "ekx_sweep3d.hpp"

namespace ekx
{

// Columns (8 x 8 tiles, indexed in the sweep's visiting order) that
// overlap the factored-eikonal box |i - iSrc| <= radius
// (solverUtilities3d.hpp:296-298), in units of columns (x, y) and z-chunks
// of `chunk` planes of the permuted frame.  Empty (lo > hi) when the radius
// is negative.
struct BoxColumns
{
    int bxLo, bxHi, byLo, byHi, bzLo, bzHi;
};

__device__ __forceinline__ BoxColumns box_columns(const Problem3D &p,
                                                  int sweep, int chunk)
{
    BoxColumns c{1, 0, 1, 0, 1, 0};
    if (p.radius < 0) { return c; }
    const int negX = sweep & 1, negY = (sweep >> 1) & 1;
    const int negZ = (sweep >> 2) & 1;
    int xLo = max(p.srcCellX - p.radius, 0);
    int xHi = min(p.srcCellX + p.radius, p.nx - 1);
    int yLo = max(p.srcCellY - p.radius, 0);
    int yHi = min(p.srcCellY + p.radius, p.ny - 1);
    int zLo = max(p.srcCellZ - p.radius, 0);
    int zHi = min(p.srcCellZ + p.radius, p.nz - 1);
    if (xLo > xHi || yLo > yHi || zLo > zHi) { return c; }
    // tiles are aligned to the grid's own axes: tile t holds nodes
    // 8 t .. 8 t + 7 in every sweep, and a sweep that reverses an axis
    // visits its tiles in reverse order
    const int mxLo = xLo/kColumnTile, mxHi = xHi/kColumnTile;
    const int myLo = yLo/kColumnTile, myHi = yHi/kColumnTile;
    c.bxLo = negX ? p.nTX - 1 - mxHi : mxLo;
    c.bxHi = negX ? p.nTX - 1 - mxLo : mxHi;
    c.byLo = negY ? p.nTY - 1 - myHi : myLo;
    c.byHi = negY ? p.nTY - 1 - myLo : myHi;
    int jzLo = negZ ? p.nz - 1 - zHi : zLo, jzHi = negZ ? p.nz - 1 - zLo : zHi;
    c.bzLo = jzLo/chunk;
    c.bzHi = jzHi/chunk;
    return c;
}

// ---------------------------------------------------------------------------
// Source initialisation (Solver3DImpl::initializeTravelTimes,
// src/solver3d.cpp:21-84): HUGE everywhere (one streaming fill over the
// fields of all problems, which lie back to back, tile padding and edge
// records included), then the analytic time at the 8 corners of each
// problem's source cell.
// ---------------------------------------------------------------------------
template <typename TS>
__global__ void __launch_bounds__(256)
init_travel_times3d(TS *__restrict__ T, int64_t n)
{
    // 16-byte stores over the aligned body, element stores for the tail
    constexpr int kPer = 16/sizeof(TS);
    union Pack
    {
        TS v[kPer];
        uint4 u;
    } pack;
#pragma unroll
    for (int k = 0; k < kPer; ++k) { pack.v[k] = Store<TS>::kHugeCode; }
    const int64_t nVec = n/kPer;
    uint4 *V = reinterpret_cast<uint4 *>(T);
    const int64_t stride = (int64_t) gridDim.x*blockDim.x;
    const int64_t first = (int64_t) blockIdx.x*blockDim.x + threadIdx.x;
    for (int64_t i = first; i < nVec; i += stride)
    {
        V[i] = pack.u;
    }
    for (int64_t i = nVec*kPer + first; i < n; i += stride)
    {
        T[i] = Store<TS>::kHugeCode;
    }
}

// Then the 8 corners of each problem's source cell (thread 8 k + c:
// problem k, corner c), in the field's layout.
template <typename TS>
__global__ void __launch_bounds__(64)
init_source_corners3d(const Problem3D *__restrict__ problems, int nProblems,
                      TS *__restrict__ T)
{
    const int t = blockIdx.x*blockDim.x + threadIdx.x;
    if (t >= 8*nProblems) { return; }
    const Problem3D &p = problems[t >> 3];
    const int c = t & 7;
    const int ix = p.srcCellX + (c & 1);
    const int iy = p.srcCellY + ((c >> 1) & 1);
    const int iz = p.srcCellZ + (c >> 2);
    if (ix >= p.nx || iy >= p.ny || iz >= p.nz) { return; }
    T[p.tOffset + node_index(p, ix, iy, iz)] = Store<TS>::code(
        (typename Store<TS>::R) analytic_time3d(
            ix, iy, iz, p.dx, p.dy, p.dz, p.srcOffX, p.srcOffY, p.srcOffZ,
            p.srcSlowness), p);
}

// ---------------------------------------------------------------------------
// Hyperplane kernel: all nodes of one level L = jx+jy+jz of one sweep (the
// level-set method of src/graph3d.cpp:119-221, with the node set computed
// in closed form instead of stored lists).  Threads enumerate (jz, jy)
// pairs; jx follows from the level.  Reads and writes global memory
// directly.
// ---------------------------------------------------------------------------
template <typename TS>
__global__ void __launch_bounds__(256)
sweep_hyperplane3d(const Problem3D *__restrict__ problems, int problem,
                   int sweep, int initialize, int level, int kLo, int nPairs,
                   TS *__restrict__ T, const TS *__restrict__ S,
                   unsigned int *__restrict__ change)
{
    const int pid = blockIdx.x*blockDim.x + threadIdx.x;
    if (pid >= nPairs) { return; }
    const Problem3D &p = problems[problem];
    const Octant o = sweep_octant(p, sweep, initialize);
    const int nyRange = p.ny - o.jy0;
    const int jz = kLo + pid/nyRange;
    const int jy = o.jy0 + pid%nyRange;
    const int jx = level - jy - jz;
    if (jx < o.jx0 || jx > p.nx - 1 || jz > p.nz - 1) { return; }
    const int negX = sweep & 1, negY = (sweep >> 1) & 1, negZ = (sweep >> 2) & 1;
    const int nx = p.nx, ny = p.ny, nz = p.nz;
    const int ncx = nx - 1, ncy = ny - 1, ncz = nz - 1;
    // natural indices of the node and of its upwind neighbour per axis
    const int ix = negX ? nx - 1 - jx : jx;
    const int iy = negY ? ny - 1 - jy : jy;
    const int iz = negZ ? nz - 1 - jz : jz;
    const int ixU = negX ? ix + 1 : ix - 1;
    const int iyU = negY ? iy + 1 : iy - 1;
    const int izU = negZ ? iz + 1 : iz - 1;
    // cells: permuted index j-1 (home) and min(j, nCell-1) (offset)
    auto cellx = [&](int pc) { return negX ? ncx - 1 - pc : pc; };
    auto celly = [&](int pc) { return negY ? ncy - 1 - pc : pc; };
    auto cellz = [&](int pc) { return negZ ? ncz - 1 - pc : pc; };
    const int cxH = cellx(jx - 1), cxO = cellx(min(jx, ncx - 1));
    const int cyH = celly(jy - 1), cyO = celly(min(jy, ncy - 1));
    const int czH = cellz(jz - 1), czO = cellz(min(jz, ncz - 1));
    using St = Store<TS>;
    using R = typename St::R;
    const TS *Sp = S + p.sOffset;
    auto sAt = [&](int cx, int cy, int cz)
    {
        return St::slowness(Sp[((int64_t) cz*ncy + cy)*ncx + cx], p);
    };
    TS *Tp = T + p.tOffset;
    auto tIdx = [&](int x, int y, int z)
    {
        return ((int64_t) z*ny + y)*nx + x;
    };
    const R s0 = sAt(cxH, cyH, czH);
    const R s1 = sAt(cxO, cyH, czH);
    const R s2 = sAt(cxO, cyO, czH);
    const R s3 = sAt(cxH, cyO, czH);
    const R s4 = sAt(cxH, cyH, czO);
    const R s5 = sAt(cxO, cyH, czO);
    const R s7 = sAt(cxH, cyO, czO);
    const int64_t i0 = tIdx(ix, iy, iz);
    const TS own = Tp[i0];
    const R t1 = St::time(Tp[tIdx(ixU, iy, iz)], p);
    const R t2 = St::time(Tp[tIdx(ixU, iyU, iz)], p);
    const R t3 = St::time(Tp[tIdx(ix, iyU, iz)], p);
    const R t4 = St::time(Tp[tIdx(ix, iy, izU)], p);
    const R t5 = St::time(Tp[tIdx(ixU, iy, izU)], p);
    const R t6 = St::time(Tp[tIdx(ixU, iyU, izU)], p);
    const R t7 = St::time(Tp[tIdx(ix, iyU, izU)], p);
    const Sweep3D sw = make_sweep3d(sweep);
    const R tUpd = local_update3d<R>(p, sw, ix, iy, iz, s0, s1, s2, s3, s4,
                                     s5, s7, t1, t2, t3, t4, t5, t6, t7);
    const TS c = St::code(tUpd, p);
    if (c < own)
    {
        Tp[i0] = c;
        if (change != nullptr)
        {
            // largest decrease of the sweep (positive floats order as
            // their bit patterns)
            const float drop = (float) (St::time(own, p) -
                                        St::finite_time(c, p));
            atomicMax(change, __float_as_uint(drop));
        }
    }
}

// ---------------------------------------------------------------------------
// Column kernel.  One 64-lane wave owns an 8 x 8 (x, y) tile of one problem
// and marches through z.  In the sweep's permuted frame lane (a, b) works on
// plane q = step - (a + b) (relative to the first plane of the sweep), so at
// every step the lanes hold nodes on one hyperplane and a lane's x- and
// y-neighbours on the same plane were finished one or two steps earlier by
// the neighbouring lanes.  Travel-time planes are staged in a 15-slot LDS
// ring of 9 x 9 values (the tile plus the upwind halo row and column, which
// the previous column diagonal has already finished; slots padded against
// LDS bank conflicts), slowness in a 4-record ring; the z-neighbours stay
// in registers.  Planes are prefetched DL steps ahead and written back once the
// last lane has finished them.  The waves of a block are independent: there
// is no block barrier.
//
// Memory (tiled layout): the tile's plane records are one contiguous run,
// read and written 64 values at a time; the halo comes from the edge
// records that the upwind columns wrote in this sweep (their last x column
// and y row), and the column writes its own edge records with each plane.
// Where the upwind column did not run in this sweep (it lies outside an
// initialisation sweep's octant) the halo is read from the tile records
// directly: those nodes keep their values through the sweep.  Slowness
// comes from the tile's bricks, records of 9 x 9 cells skewed to the lanes'
// planes, so that a 4-record LDS ring serves every lane.
//
// Launch: one launch per column diagonal bx + by (+ bz) = d, bx and by
// counting tiles in the sweep's visiting order.  Columns on one diagonal
// never read or write each other's nodes or edge records; their halos
// belong to the diagonals before.
//
// Instances: FACTORED = false runs the Cartesian operators, and with MERGED
// also the columns that overlap the factored box around the source (with
// the full local update): on single grids and small batches, where a
// second launch per diagonal costs more than the registers of the factored
// branch, and in the work-queue form.  FACTORED = true runs the full local
// update on exactly the box columns (at most boxPerDiag per problem and
// diagonal), with items derived from the problem's source instead of the
// item list, beside the bulk instances without MERGED, which keep the
// register count of the Cartesian update.
// ---------------------------------------------------------------------------
// Keeps the compiler from moving memory accesses across this point.  The
// column kernel's lanes exchange values through LDS within one wave, whose
// DS instructions execute in issue order, so program order is all the
// exchange needs: no wait for the LDS counter (a wave-scope fence made the
// compiler wait for every outstanding LDS access before the next store).
__device__ __forceinline__ void lds_order()
{
    __asm__ __volatile__("" ::: "memory");
}

// Travel-time accesses of a column.  COHERENT (work-queue launches, where
// chunks of one launch on different XCDs exchange planes): agent-scope
// relaxed atomics, i.e. loads and stores that bypass the XCD-local caches
// the other XCDs do not see.
template <bool COHERENT, typename TS>
__device__ __forceinline__ TS load_time(const TS *p)
{
    if constexpr (COHERENT)
    {
        using U = typename std::conditional<sizeof(TS) == 8, uint64_t,
                                            uint32_t>::type;
        const U u = __hip_atomic_load(const_cast<U *>(
                                          reinterpret_cast<const U *>(p)),
                                      __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
        return __builtin_bit_cast(TS, u);
    }
    else
    {
        return *p;
    }
}

template <bool COHERENT, typename TS>
__device__ __forceinline__ void store_time(TS *p, TS v)
{
    if constexpr (COHERENT)
    {
        using U = typename std::conditional<sizeof(TS) == 8, uint64_t,
                                            uint32_t>::type;
        __hip_atomic_store(reinterpret_cast<U *>(p),
                           __builtin_bit_cast(U, v), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    else
    {
        *p = v;
    }
}

// A run of nValues elements of type TS from base (a column's tile, edge or
// slowness records): loads and stores at a per-lane byte offset plus a
// wave-uniform one.  BUFFER: through a buffer resource, the uniform offset
// in a scalar register, so that advancing it is scalar work; else through
// a flat pointer (the instances whose scalar registers are already taken,
// where the resources would spill).
template <typename TS, bool BUFFER>
struct ColumnRun
{
    // raw buffer data format of gfx9 (32-bit elements, no swizzle)
    static constexpr int kBufferFlags = 0x00020000;
    const char *base;
    __amdgpu_buffer_rsrc_t rsrc;
    // base and nValues are wave-uniform; read from the first lane so that
    // the resource lives in scalar registers
    __device__ ColumnRun(const void *b, int64_t nValues)
        : base((const char *) b)
    {
        if constexpr (BUFFER)
        {
            rsrc = __builtin_amdgcn_make_buffer_rsrc(
                uniform_pointer(b), (short) 0,
                __builtin_amdgcn_readfirstlane(
                    (int) (nValues*(int64_t) sizeof(TS))),
                kBufferFlags);
        }
    }
    static __device__ __forceinline__ void *uniform_pointer(const void *p)
    {
        const uint64_t a = (uint64_t) p;
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t) a);
        const uint32_t hi = __builtin_amdgcn_readfirstlane(
            (uint32_t) (a >> 32));
        return (void *) (((uint64_t) hi << 32) | lo);
    }
    __device__ __forceinline__ TS load(uint32_t laneOff, int32_t off) const
    {
        if constexpr (!BUFFER)
        {
            return *(const TS *) (base + off + laneOff);
        }
        else if constexpr (sizeof(TS) == 8)
        {
            return __builtin_bit_cast(
                TS, __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int) laneOff,
                                                         off, 0));
        }
        else
        {
            return __builtin_bit_cast(
                TS, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int) laneOff,
                                                         off, 0));
        }
    }
    __device__ __forceinline__ void store(uint32_t laneOff, int32_t off,
                                          TS v) const
    {
        if constexpr (!BUFFER)
        {
            *(TS *) (const_cast<char *>(base) + off + laneOff) = v;
        }
        else if constexpr (sizeof(TS) == 8)
        {
            using V2 = __attribute__((ext_vector_type(2))) unsigned int;
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(V2, v),
                                                  rsrc, (int) laneOff, off,
                                                  0);
        }
        else
        {
            __builtin_amdgcn_raw_buffer_store_b32(
                __builtin_bit_cast(unsigned int, v), rsrc, (int) laneOff,
                off, 0);
        }
    }
};

// One column chunk (problem pIndex, column (bx, by), chunk bz) of one sweep
// on one wave; ringT and ringS are the wave's LDS rings of travel-time
// planes and slowness records.
// GRID: the Cartesian update's branch (uniform or not) and, on uniform
// grids, whether the model's h s suit the roots without range tests;
// MONITOR: the largest decrease is kept for the convergence monitor
// (change != nullptr).  Both are per launch and item, chosen outside the
// step loop so that the loop carries no test of them.
template <typename TS, int DL, bool FACTORED, bool COHERENT, bool MERGED,
          Grid3D GRID, bool MONITOR>
__device__ __forceinline__ void run_column(
    const Problem3D *__restrict__ problems, int pIndex, int bx, int by,
    int bz, int sweep, int initialize, int chunk, int boxPhase,
    TS *__restrict__ T, const TS *__restrict__ S,
    unsigned int *__restrict__ change, TS (*ringT)[ring_slot<TS>()],
    SlownessRing<TS> (*ringS)[kColumnPlane], int lane)
{
    // the slowness ring's slots are compile-time per unrolled step
    static_assert(DL % kSlownessRing == 0, "prefetch depth");
    // bulk instance that also runs the factored-box columns
    constexpr bool kMerged = !FACTORED && MERGED;
    bool boxColumn = false;
    pIndex = __builtin_amdgcn_readfirstlane(pIndex);
    const Problem3D &p = problems[pIndex];
    if (!FACTORED)
    {
        const BoxColumns bc = box_columns(p, sweep, chunk);
        // the full local update in this wave (MERGED), or the planes
        // outside the box while the FACTORED instance runs the others
        boxColumn = bx >= bc.bxLo && bx <= bc.bxHi && by >= bc.byLo &&
                    by <= bc.byHi && bz >= bc.bzLo && bz <= bc.bzHi;
    }
    const int nx = p.nx, ny = p.ny, nz = p.nz;
    const int nTX = p.nTX, nTY = p.nTY;
    const int negX = sweep & 1, negY = (sweep >> 1) & 1, negZ = (sweep >> 2) & 1;
    const Octant o = sweep_octant(p, sweep, initialize);
    // The column's tile (mx, my) in grid order and its first node
    // (X0, Y0) in the permuted frame; a reversed axis starts its tiles at
    // the grid's far end, so X0 may be negative for the last tile.
    const int mx = negX ? nTX - 1 - __builtin_amdgcn_readfirstlane(bx)
                        : __builtin_amdgcn_readfirstlane(bx);
    const int my = negY ? nTY - 1 - __builtin_amdgcn_readfirstlane(by)
                        : __builtin_amdgcn_readfirstlane(by);
    const int X0 = negX ? nx - kColumnTile*(mx + 1) : kColumnTile*mx;
    const int Y0 = negY ? ny - kColumnTile*(my + 1) : kColumnTile*my;
    if (X0 + kColumnTile - 1 < o.jx0 || Y0 + kColumnTile - 1 < o.jy0)
    {
        // column entirely outside the source octant
        return;
    }
    // This item's planes: the chunk's [bz*chunk, (bz+1)*chunk) within the
    // sweep's range, after a read-only first plane (the previous chunk's
    // last, or the plane before the range).
    int zFirst = max(__builtin_amdgcn_readfirstlane(bz)*chunk, o.jz0);
    int zEnd = min((__builtin_amdgcn_readfirstlane(bz) + 1)*chunk, nz);
    if (!kMerged && (FACTORED || boxColumn))
    {
        // a box chunk split in z between the two instances: the FACTORED
        // launch of the split's phase takes the box end, the bulk launch
        // the rest
        const BoxSplitZ bs = box_split_z(nz, p.srcCellZ, p.radius, negZ,
                                         zFirst, zEnd);
        if (FACTORED)
        {
            if (bs.phase != boxPhase) { return; }
            if (bs.phase == 0) { zEnd = bs.cut; }
            else { zFirst = bs.cut; }
        }
        else if (bs.phase == 0) { zFirst = bs.cut; }
        else { zEnd = bs.cut; }
    }
    if (zFirst >= zEnd) { return; }
    const int P0 = zFirst - 1;            // first plane: read only
    const int nPlanes = zEnd - P0;
    const int a = lane & 7, b = lane >> 3;
    const int jx = X0 + a, jy = Y0 + b;
    const bool valid = jx >= 0 && jx < nx && jy >= 0 && jy < ny;
    const bool upd = valid && jx >= o.jx0 && jy >= o.jy0;
    const int ix = negX ? nx - 1 - jx : jx;
    const int iy = negY ? ny - 1 - jy : jy;
    const Sweep3D sw = make_sweep3d(sweep);

    // LDS plane layout: local coordinate (c, r) of the permuted frame,
    // c = jx - X0 + 1, r = jy - Y0 + 1, both in 0..8, at r*9 + c (the
    // upwind halo row and column at r = 0 and c = 0).  A lane's node is
    // (a+1, b+1): its x-1, y-1 and xy-1 neighbours sit at fixed offsets 9,
    // 1 and 0 from (a, b), so one address per ring serves all reads.
    // Slowness records use the same layout with c, r the cell's local
    // indices; the lane's 4 cells of its plane are at (a, b) of the step's
    // record, (a + 1, b) and (a, b + 1) of the next and (a + 1, b + 1) of
    // the one after.
    auto lidx = [](int c, int r) { return r*kColumnHalo + c; };
    // Tile record element e (grid-local x = e % 8, y = e / 8) sits at
    // local (1 + x, 1 + y), mirrored along a reversed axis.
    auto tileSlot = [&](int e)
    {
        const int xl = e % kColumnTile, yl = e/kColumnTile;
        return lidx(1 + (negX ? kColumnTile - 1 - xl : xl),
                    1 + (negY ? kColumnTile - 1 - yl : yl));
    };
    using St = Store<TS>;
    using R = typename St::R;
    // A cell's slowness as it enters the ring: decoded, and times h for the
    // uniform Cartesian update (2 products a step; 7 in the update).
    const bool boxWave = FACTORED || (kMerged && boxColumn);
    const R sScale = boxWave ? (R) 1 : (R) p.dx;
    auto ringCell = [&](TS v)
    {
        const R s = St::slowness(v, p);
        if constexpr (FACTORED || GRID == kNonUniform) { return s; }
        else { return sScale*s; }
    };
    TS *Tp = T + p.tOffset;
    const int64_t tileIndex = (int64_t) my*nTX + mx;
    // Loads per lane and step: tile element `lane`, one halo value (lanes
    // 0..8: the x-halo column c = 0, r = lane; lanes 9..16: the y-halo row
    // r = 0, c = lane - 8; the other lanes repeat lane 16's load into the
    // ring's padding), and brick elements `lane` and 64 + min(lane, 16):
    // the brick variant of the sweep's directions stores its cells in that
    // lane order, so they go to the same ring positions as the travel
    // times.
    // Every prefetch load is unconditional from an in-bounds address;
    // conditional loads would make the compiler wait for them at the merge
    // point and serialise the prefetch.
    const int h = min(lane, kEdgeValues - 1);
    const int dstOwn = tileSlot(lane);
    const int dstHalo = h < kColumnHalo ? lidx(0, h)
                                        : lidx(h - kColumnTile, 0);
    // Halo source: the upwind column's edge records (when that column ran
    // in this sweep: its last node X0 - 1 is at or past the octant start),
    // else the node itself in the tile records.  Per lane: the address at
    // plane P0 and the per-plane stride in bytes.
    const char *haloP0;
    int32_t haloStep;
    {
        const int zP0 = negZ ? nz - 1 - P0 : P0;
        const int dz = negZ ? -1 : 1;
        const bool xHalo = h < kColumnHalo;
        const bool fromEdge = xHalo ? X0 - 1 >= o.jx0 : Y0 - 1 >= o.jy0;
        if (fromEdge)
        {
            const int ux = xHalo ? (negX ? mx + 1 : mx - 1) : mx;
            const int uy = xHalo ? my : (negY ? my + 1 : my - 1);
            const int64_t rec = ((int64_t) uy*nTX + ux)*nz + zP0;
            haloP0 = (const char *) (T + p.eOffset + rec*kEdgeValues + h);
            haloStep = dz*kEdgeValues*(int32_t) sizeof(TS);
        }
        else
        {
            // permuted (X0 - 1, Y0 - 1 + h) or (X0 - 1 + h - 8, Y0 - 1),
            // clamped into the grid (clamped nodes are never read by an
            // update: updated nodes start at index 1 and read index - 1)
            const int hx = xHalo ? X0 - 1 : X0 - 1 + h - kColumnTile;
            const int hy = xHalo ? Y0 - 1 + h : Y0 - 1;
            const int cx = min(max(hx, 0), nx - 1);
            const int cy = min(max(hy, 0), ny - 1);
            const int gx = negX ? nx - 1 - cx : cx;
            const int gy = negY ? ny - 1 - cy : cy;
            haloP0 = (const char *) (Tp + tiled_index(nTX, nz, gx, gy, zP0));
            haloStep = dz*kTileValues*(int32_t) sizeof(TS);
        }
    }
    // Addressing: the column's runs of tile records, edge records and
    // slowness records, each with a wave-uniform byte offset (advanced by
    // one add per step) and a per-lane one (constant).  In the Cartesian
    // bulk instance the runs are buffer resources and the uniform offset is
    // a scalar register, so the per-step address work of these accesses is
    // scalar (the halo address is per lane).
    // Slowness record P0 + m (m >= 0) is read at steps m - 2 .. m and
    // lives in ring slot m % 4.  The prefetch reads records up to
    // P0 + nSteps + DL + 1 <= nz + 2 DL + 14, within the tile's run.
    static_assert(DL <= kMaxPrefetch, "prefetch depth");
    char *colT = (char *) (Tp + tileIndex*nz*kTileValues);
    char *colE = (char *) (T + p.eOffset + tileIndex*nz*kEdgeValues);
    const char *colS = (const char *) (
        S + p.sbOffset + (negX + 2*negY + 4*negZ)*
                             brick_variant_values(nx, ny, nz) +
        tileIndex*brick_records(nz)*kBrickValues);
    // buffer resources in the Cartesian bulk instance only: in the
    // instances with the factored update the resources spill scalar
    // registers and the solves measured no faster
    constexpr bool kBuffer = !FACTORED && !MERGED;
    const ColumnRun<TS, kBuffer> runT(colT, nz*kTileValues);
    const ColumnRun<TS, kBuffer> runE(colE, nz*kEdgeValues);
    const ColumnRun<TS, kBuffer> runS(colS, brick_records(nz)*kBrickValues);
    // byte offsets of plane q's tile and edge records and of slowness
    // record P0 + m in their runs
    auto planeT = [&](int q) -> int32_t
    {
        const int jz = P0 + q;
        const int az = negZ ? nz - 1 - jz : jz;
        return az*kTileValues*(int32_t) sizeof(TS);
    };
    auto planeE = [&](int q) -> int32_t
    {
        const int jz = P0 + q;
        const int az = negZ ? nz - 1 - jz : jz;
        return az*kEdgeValues*(int32_t) sizeof(TS);
    };
    auto recordS = [&](int m) -> int32_t
    {
        return (P0 + m)*kBrickValues*(int32_t) sizeof(TS);
    };
    const uint32_t tB = (uint32_t) lane*sizeof(TS);
    const uint32_t sB0 = (uint32_t) lane*sizeof(TS);
    const uint32_t sB1 = (uint32_t) (kTileValues + h)*sizeof(TS);
    // COHERENT: the halo (the upwind chunks' edge records) always; of the
    // chunk's own tile records only the first plane, which the previous
    // chunk of the column wrote (its other planes were last written by an
    // earlier launch)
    auto loadPlane = [&](int32_t Tz, int32_t Sz, const char *Hz,
                         TS &vT0, TS &vT1, TS &vS0, TS &vS1)
    {
        vT0 = runT.load(tB, Tz);
        vS0 = runS.load(sB0, Sz);
        vT1 = load_time<COHERENT>((const TS *) Hz);
        vS1 = runS.load(sB1, Sz);
    };

    // Slowness records P0 and P0 + 1, which step 0 reads besides the one
    // entering then: loaded first, put in the ring after the prologue.
    TS pS0[2], pS1[2];
#pragma unroll
    for (int m = 0; m < 2; ++m)
    {
        pS0[m] = runS.load(sB0, recordS(m));
        pS1[m] = runS.load(sB1, recordS(m));
    }
    __builtin_amdgcn_sched_barrier(0);
    TS bT0[DL], bT1[DL], bS0[DL], bS1[DL];
    // Prologue: buffer u holds plane u and slowness record P0 + u + 2.  The
    // scheduling barriers keep the buffers in issue order, so the first use
    // of buffer u waits only for the loads issued before it (as in the
    // steady state).
#pragma unroll
    for (int u = 0; u < DL; ++u)
    {
        const int q = min(u, nPlanes - 1);
        loadPlane(planeT(q), recordS(u + 2), haloP0 + (int64_t) q*haloStep,
                  bT0[u], bT1[u], bS0[u], bS1[u]);
        if (COHERENT && u == 0)
        {
            bT0[0] = load_time<true>((const TS *) (colT + planeT(0) + tB));
        }
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int m = 0; m < 2; ++m)
    {
        ringS[m][dstOwn] = ringCell(pS0[m]);
        ringS[m][dstHalo] = ringCell(pS1[m]);
    }
    // Running plane pointers: the next prefetch (plane min(tc + DL,
    // nPlanes - 1), slowness record P0 + tc + DL + 2) and the next
    // write-back (plane clamp(tc - 15, 0, nPlanes - 1)); each advances by
    // at most one plane or record per step.
    const int32_t stepT = (negZ ? -kTileValues : kTileValues)*
                          (int32_t) sizeof(TS);
    const int32_t stepE = (negZ ? -kEdgeValues : kEdgeValues)*
                          (int32_t) sizeof(TS);
    constexpr int32_t stepS = kBrickValues*(int32_t) sizeof(TS);
    int loadQ = min(DL, nPlanes - 1);
    int32_t loadT = planeT(loadQ);
    int32_t loadS = recordS(DL + 2);
    const char *loadH = haloP0 + (int64_t) loadQ*haloStep;
    int wbQ = 0;
    int32_t wbT = planeT(0);
    int32_t wbE = planeE(0);
    // z-neighbours (plane q - 1) of the lane's node, decoded
    R pt4 = (R) kHuge, pt5 = (R) kHuge, pt6 = (R) kHuge, pt7 = (R) kHuge;
    R ps00 = 0, ps10 = 0, ps01 = 0, ps11 = 0;
    R pMin = 0;                           // min(ps00, ps01), uniform grids
    R maxDrop = 0;                        // largest decrease by this lane
    // The node is local (a+1, b+1); oA is (a, b), the xy-1 neighbour.
    constexpr int kB = 1, kC = kColumnHalo, kD = kColumnHalo + 1;
    const int oA = lidx(a, b);
    // Write-back: tile element `lane`, and edge element h (lanes 0..8: the
    // last column c = 8, r = h; lanes 9..16: the last row r = 8, c = h - 8;
    // the other lanes repeat lane 16's store).
    const int wbEdge = h < kColumnHalo ? lidx(kColumnTile, h)
                                       : lidx(h - kColumnTile, kColumnTile);
    const uint32_t eB = (uint32_t) h*sizeof(TS);
    // Steps: every plane passes every lane (plane q is finished at step
    // q + 14) and is written back; rounded up to whole groups of DL so the
    // unrolled loop body has no exit (extra steps only repeat idempotent
    // work: in-bounds loads, no computation, and a re-store of the last
    // plane's final values).
    const int nSteps = ((nPlanes + kColumnSkew + DL - 1)/DL)*DL;
    // Ring slots (planes mod 15): the entering plane's, the lane's plane
    // q = step - (a + b), and the plane being written back.
    int inSlot = 0;
    // the lane's read address: byte offset of (a, b) in its slot, kept in
    // 32 bits and wrapped by an unsigned minimum
    constexpr uint32_t kSlotB = ring_slot<TS>()*sizeof(TS);
    constexpr uint32_t kRingB = kColumnRing*kSlotB;
    uint32_t laneB = (uint32_t) (((kColumnRing - (a + b)) % kColumnRing)*
                                 kSlotB + oA*sizeof(TS));
    const int ab1 = a + b + 1;
    const uint32_t liveSpan = upd ? (uint32_t) (nPlanes - 1) : 0u;
    int wbSlot = 0;
    const int lastSlot = (nPlanes - 1) % kColumnRing;
    // The finished plane of the previous step, stored at the next one.
    // Every store writes final values only (columns of the same launch may
    // read a tile's plane P0 edge records meanwhile), so step 0 stores
    // plane 0 as loaded: the lane's own record element, and for the edge
    // record the value loaded by the lane whose ring position is wbEdge
    // (lane 16's halo value for h = 0).
    TS pendT = bT0[0];
    TS pendE;
    {
        int xe, ye;
        if (h < kColumnHalo)
        {
            xe = negX ? 0 : kColumnTile - 1;
            ye = negY ? kColumnTile - h : h - 1;
        }
        else
        {
            const int c = h - kColumnTile;
            xe = negX ? kColumnTile - c : c - 1;
            ye = negY ? 0 : kColumnTile - 1;
        }
        const int src = h == 0 ? 0 : xe + kColumnTile*ye;
        const TS fromTile = __shfl(bT0[0], src, 64);
        const TS fromHalo = __shfl(bT1[0], kEdgeValues - 1, 64);
        pendE = h == 0 ? fromHalo : fromTile;
    }
    int32_t pendTz = wbT, pendEz = wbE;
    auto nextSlot = [](int s) { return s == kColumnRing - 1 ? 0 : s + 1; };
    for (int t0 = 0; t0 < nSteps; t0 += DL)
    {
#pragma unroll
        for (int u = 0; u < DL; ++u)
        {
            const int tc = t0 + u;
            // (a) the plane prefetched DL steps ago enters the ring.  Past
            // the last plane the repeated loads go to the slot of a plane
            // already written back, never to the last plane's slot, which
            // the clamped write-back keeps re-reading; branch free, so the
            // LDS and memory counters stay exact.
            {
                const int slot = (tc >= nPlanes && inSlot == lastSlot)
                                     ? nextSlot(inSlot) : inSlot;
                TS *dT = ringT[slot];
                SlownessRing<TS> *dS = ringS[(u + 2) % kSlownessRing];
                dT[dstOwn] = bT0[u];
                dS[dstOwn] = ringCell(bS0[u]);
                dT[dstHalo] = bT1[u];
                dS[dstHalo] = ringCell(bS1[u]);
            }
            inSlot = nextSlot(inSlot);
            // (b) prefetch plane tc + DL into the freed registers (past the
            // last plane the load repeats it and is never stored)
            loadPlane(loadT, loadS, loadH, bT0[u], bT1[u], bS0[u], bS1[u]);
            if (loadQ < nPlanes - 1)
            {
                loadQ += 1;
                loadT += stepT;
            }
            // The halo address advances unconditionally (a per-lane select
            // would cost VALU work at every step): past the last plane it
            // reads beyond the column's records, within the field
            // allocation (guard space at its ends), into ring slots that
            // are never used.
            loadH += haloStep;
            loadS += stepS;
            // (d, store) the plane finished in the previous step goes home
            // with its edge records.  A store is issued at every step
            // (plane index clamped to the valid range; unchanged nodes and
            // the tile's padding store their own values), so the prefetch
            // loads always have the same number of memory operations
            // behind them.
            runT.store(tB, pendTz, pendT);
            if constexpr (COHERENT)
            {
                store_time<true>((TS *) (colE + pendEz + eB), pendE);
            }
            else
            {
                runE.store(eB, pendEz, pendE);
            }
            // (c) every lane advances its node on plane tc - (a + b).  The
            // reads and the register shift run on every lane at every step
            // (outside the lane's planes they read unused ring slots and
            // only feed registers that are overwritten before use), so
            // that the unrolled steps rename the registers instead of
            // merging them at a branch.
            const int q = tc - (a + b);
            {
                TS *sT = reinterpret_cast<TS *>(
                    reinterpret_cast<char *>(ringT) + laneB);
                const TS ownCode = sT[kD];
                R tOwn = St::time(ownCode, p);
                const R t1 = St::time(sT[kC], p);
                const R t2 = St::time(sT[0], p);
                const R t3 = St::time(sT[kB], p);
                const R *s0 = ringS[u % kSlownessRing] + oA;
                const R *s1 = ringS[(u + 1) % kSlownessRing] + oA;
                const R *s2 = ringS[(u + 2) % kSlownessRing] + oA;
                const R c00 = s0[0];
                const R c10 = s1[kB];
                const R c01 = s1[kC];
                const R c11 = s2[kD];
                // the wave-uniform choice of operator outside the lanes'
                // branch, so that it stays a scalar branch; live: upd and
                // 0 < q < nPlanes, one unsigned compare
                const bool live = (uint32_t) (tc - ab1) < liveSpan;
                auto keep = [&](R tUpd)
                {
                    const TS c = St::code(tUpd, p);
                    if (c < ownCode)
                    {
                        const R tNew = St::finite_time(c, p);
                        if constexpr (MONITOR)
                        {
                            maxDrop = Math<R>::max(maxDrop, tOwn - tNew);
                        }
                        tOwn = tNew;
                        sT[kD] = c;
                    }
                };
                R nextMin = Math<R>::min(c00, c01);
                if (boxWave)
                {
                    if (live)
                    {
                        const int jz = P0 + q;
                        const int iz = negZ ? nz - 1 - jz : jz;
                        keep(local_update3d<R>(
                            p, sw, ix, iy, iz, ps00, ps10, ps11, ps01, c00,
                            c10, c01, t1, t2, t3, pt4, pt5, pt6, pt7));
                    }
                }
                else if constexpr (GRID != kNonUniform)
                {
                    if (live)
                    {
                        keep(cartesian_uniform3d<R, GRID == kUniformScaled>(
                            ps00, ps10, ps11, ps01, c00, c10, c01, pMin,
                            nextMin, t1, t2, t3, pt4, pt5, pt6, pt7));
                    }
                }
                else if (live)
                {
                    keep(cartesian_nonuniform3d<R>(
                        p, ps00, ps10, ps11, ps01, c00, c10, c01, t1, t2, t3,
                        pt4, pt5, pt6, pt7));
                }
                pt4 = tOwn;
                pt5 = t1;
                pt6 = t2;
                pt7 = t3;
                ps00 = c00;
                ps10 = c10;
                ps01 = c01;
                ps11 = c11;
                pMin = nextMin;
            }
            {
                const uint32_t nb = laneB + kSlotB;
                laneB = min(nb, nb - kRingB);
            }
            // (d, read) plane clamp(tc - 14, 0, nPlanes - 1), which the
            // last lane finished in this step: read after the updates
            lds_order();
            pendT = ringT[wbSlot][dstOwn];
            pendE = ringT[wbSlot][wbEdge];
            pendTz = wbT;
            pendEz = wbE;
            if (tc >= kColumnSkew && wbQ < nPlanes - 1)
            {
                wbQ += 1;
                wbSlot = nextSlot(wbSlot);
                wbT += stepT;
                wbE += stepE;
            }
            // LDS traffic of this step must not be reordered with the next
            // step's: other lanes of the wave consume it.
            lds_order();
            __builtin_amdgcn_wave_barrier();
        }
    }
    // the last finished plane (COHERENT: the next chunk of the column reads
    // it as its first plane; the earlier stores of the same plane wrote the
    // same values)
    store_time<COHERENT>((TS *) (colT + pendTz + tB), pendT);
    store_time<COHERENT>((TS *) (colE + pendEz + eB), pendE);
    // Convergence monitor: the wave's largest decrease, one atomic per
    // column.  Every lane of the wave is still active here (the early
    // returns above are whole-wave).
    if (MONITOR && change != nullptr)
    {
        float d = (float) maxDrop;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1)
        {
            d = fmaxf(d, __shfl_xor(d, off, 64));
        }
        if (lane == 0 && d > 0.0f)
        {
            atomicMax(change, __float_as_uint(d));
        }
    }
}

__device__ __forceinline__ int grid_kind(const Problem3D &p)
{
    return !p.uniform ? kNonUniform : p.scaled ? kUniformScaled : kUniform;
}

// go(grid, monitor) with both as compile-time constants.
template <bool UNIFORM, typename F>
__device__ __forceinline__ void with_grid(int grid, bool monitor, F &&go)
{
    auto with = [&](auto g)
    {
        if (monitor) { go(g, std::true_type{}); }
        else { go(g, std::false_type{}); }
    };
    if constexpr (UNIFORM)
    {
        if (grid == kUniformScaled)
        {
            with(std::integral_constant<Grid3D, kUniformScaled>{});
            return;
        }
        if (grid == kUniform)
        {
            with(std::integral_constant<Grid3D, kUniform>{});
            return;
        }
    }
    with(std::integral_constant<Grid3D, kNonUniform>{});
}

template <typename TS, int WAVES, int DL, bool FACTORED, bool MERGED = false>
__global__ void __launch_bounds__(64*WAVES)
sweep_columns3d(const Problem3D *__restrict__ problems,
                const ColumnItem *__restrict__ items, int nItems, int sweep,
                int initialize, int diagonal, int boxPerDiag, int chunk,
                int boxPhase, TS *__restrict__ T, const TS *__restrict__ S,
                unsigned int *__restrict__ change)
{
    __shared__ TS ringT[WAVES][kColumnRing][ring_slot<TS>()];
    __shared__ SlownessRing<TS> ringS[WAVES][kSlownessRing][kColumnPlane];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int itemIndex = blockIdx.x*WAVES + wave;
    if (itemIndex >= nItems) { return; }
    int pIndex, bx, by, bz;
    if (FACTORED)
    {
        // item = (problem, k): the k-th (bx, by) of the box, at the z-chunk
        // that puts it on this diagonal bx + by + bz
        pIndex = itemIndex/boxPerDiag;
        const int k = itemIndex - pIndex*boxPerDiag;
        const BoxColumns bc = box_columns(problems[pIndex], sweep, chunk);
        const int nbx = bc.bxHi - bc.bxLo + 1, nby = bc.byHi - bc.byLo + 1;
        if (nbx <= 0 || nby <= 0 || k >= nbx*nby) { return; }
        bx = bc.bxLo + k%nbx;
        by = bc.byLo + k/nbx;
        bz = diagonal - bx - by;
        if (bz < bc.bzLo || bz > bc.bzHi) { return; }
    }
    else
    {
        const ColumnItem item = items[itemIndex];
        // a placeholder that keeps the list's XCD interleave: no work
        if (__builtin_amdgcn_readfirstlane(item.problem) < 0) { return; }
        pIndex = item.problem;
        bx = item.bx;
        by = item.by;
        bz = item.bz;
    }
    // the Cartesian update's branch (the factored update tests the grid
    // itself) and the monitor, outside the step loop
    const int grid = FACTORED ? kNonUniform
        : __builtin_amdgcn_readfirstlane(grid_kind(
              problems[__builtin_amdgcn_readfirstlane(pIndex)]));
    auto go = [&](auto g, auto m)
    {
        run_column<TS, DL, FACTORED, false, MERGED, decltype(g)::value,
                   decltype(m)::value>(
            problems, pIndex, bx, by, bz, sweep, initialize, chunk, boxPhase,
            T, S, change, ringT[wave], ringS[wave], lane);
    };
    with_grid<!FACTORED>(grid, change != nullptr, go);
}

// ---------------------------------------------------------------------------
// Work-queue form of a sweep: one launch per sweep (and chain) whose waves
// take column chunks from a counter in the order of the item list (by
// diagonal bx + by + bz) and start each once its upwind chunks
// (bx - 1, by, bz), (bx, by - 1, bz) and (bx, by, bz - 1) have published
// their completion, instead of one launch per diagonal with a barrier
// between diagonals.  A chunk's halo comes from the edge records of its x
// and y upwind chunks and its first plane from its z upwind chunk (the
// diagonal launches order exactly these), so the nodes see the same values
// and the field is the same.  Every item waited for was taken earlier by a
// running wave, so the waits end; each is still bounded in time and, past
// the bound, flags an error and goes on (later waits then return at once),
// so that every wave exits.
// Waves of different XCDs exchange planes through device memory: the
// planes that cross chunks (edge records, the first plane of a chunk, the
// last plane it hands to the next chunk) are read and written with
// agent-scope atomics, which bypass the XCD-local caches, and a chunk
// publishes only after all its stores have completed.  (Agent-scope
// release and acquire fences, which write back and invalidate a whole L2,
// made the sweeps 1.7 times slower.)
// ---------------------------------------------------------------------------
// Every lane runs the queue's control flow (the same address and value in
// all lanes, the loop exits on readfirstlane of the loaded word): a branch
// taken by lane 0 alone at the end of the loop body let the compiler keep
// the other lanes iterating without it, where readfirstlane then read
// theirs.
// A wait is bounded in time (waitTicks of the wall clock, far above the
// longest chain of chunks a sweep can hold up), not in polls: a sweep whose
// last diagonals hold few chunks leaves waves waiting many column times.
__device__ __forceinline__ void wait_published(const ColumnQueue &q, int f)
{
    if (f < 0) { return; }
    uint64_t t0 = 0;
    for (unsigned int spins = 0;; ++spins)
    {
        const unsigned int v = __builtin_amdgcn_readfirstlane(
            __hip_atomic_load(q.flags + f, __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_AGENT));
        if (v >= q.epoch) { return; }
        if ((spins & 63) == 63)
        {
            // the clock starts after the first 64 polls
            const uint64_t now = (uint64_t) wall_clock64();
            if (spins == 63) { t0 = now; }
            const bool failed = __builtin_amdgcn_readfirstlane(
                __hip_atomic_load(q.error, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT)) != 0;
            const bool late = now - t0 > q.waitTicks;
            if (failed || late)
            {
                __hip_atomic_fetch_or(q.error, 1u, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
                return;
            }
        }
        __builtin_amdgcn_s_sleep(2);
    }
}

template <typename TS, int DL>
__global__ void __launch_bounds__(64)
sweep_columns3d_queued(const Problem3D *__restrict__ problems,
                       const ColumnItem *__restrict__ items, int nItems,
                       int sweep, int initialize, int chunk,
                       TS *__restrict__ T, const TS *__restrict__ S,
                       unsigned int *__restrict__ change, ColumnQueue q)
{
    __shared__ TS ringT[kColumnRing][ring_slot<TS>()];
    __shared__ SlownessRing<TS> ringS[kSlownessRing][kColumnPlane];
    const int lane = threadIdx.x & 63;
    for (;;)
    {
        // one item per wave: lane 0 adds 1, the others 0, and every lane
        // reads lane 0's value
        const unsigned int taken = __hip_atomic_fetch_add(
            q.counter, lane == 0 ? 1u : 0u, __ATOMIC_RELAXED,
            __HIP_MEMORY_SCOPE_AGENT);
        const int index = (int) __builtin_amdgcn_readfirstlane(taken);
        if (index >= nItems) { break; }
        const ColumnItem item = items[index];
        const int pIndex = __builtin_amdgcn_readfirstlane(item.problem);
        // a placeholder of the list's XCD interleave: nothing to run or
        // publish (no chunk waits for it)
        if (pIndex < 0) { continue; }
        const int bx = __builtin_amdgcn_readfirstlane(item.bx);
        const int by = __builtin_amdgcn_readfirstlane(item.by);
        const int bz = __builtin_amdgcn_readfirstlane(item.bz);
        const Problem3D &p = problems[pIndex];
        const int nbx = p.nTX, nby = p.nTY;
        const int self = q.flagBase[pIndex] + (bz*nby + by)*nbx + bx;
        // the three flags in one round trip; a wait only for those not
        // yet published
        const int fx = bx > 0 ? self - 1 : self;
        const int fy = by > 0 ? self - nbx : self;
        const int fz = bz > 0 ? self - nbx*nby : self;
        const unsigned int vx = __hip_atomic_load(
            q.flags + fx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned int vy = __hip_atomic_load(
            q.flags + fy, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned int vz = __hip_atomic_load(
            q.flags + fz, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool ready = __builtin_amdgcn_readfirstlane(
            (bx == 0 || vx >= q.epoch) && (by == 0 || vy >= q.epoch) &&
            (bz == 0 || vz >= q.epoch) ? 1 : 0) != 0;
        if (!ready)
        {
            wait_published(q, bx > 0 ? fx : -1);
            wait_published(q, by > 0 ? fy : -1);
            wait_published(q, bz > 0 ? fz : -1);
        }
        // the chunk's travel-time loads are issued after the waits (they
        // follow in program order and the compiler may not hoist them)
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        // the factored-box chunks run in place (MERGED)
        auto go = [&](auto g, auto m)
        {
            run_column<TS, DL, false, true, true, decltype(g)::value,
                       decltype(m)::value>(problems, pIndex, bx, by, bz,
                                           sweep, initialize, chunk, 0, T, S,
                                           change, ringT, ringS, lane);
        };
        with_grid<true>(__builtin_amdgcn_readfirstlane(grid_kind(p)),
                        change != nullptr, go);
        // publish once every store of the chunk has completed
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_s_waitcnt(0);
        __hip_atomic_store(q.flags + self, q.epoch, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Zeroes n words (the queue's flags and counters) with vector stores.
__global__ void __launch_bounds__(256)
clear_words_kernel(unsigned int *__restrict__ w, int64_t n)
{
    for (int64_t i = (int64_t) blockIdx.x*blockDim.x + threadIdx.x; i < n;
         i += (int64_t) gridDim.x*blockDim.x)
    {
        w[i] = 0;
    }
}

// ---------------------------------------------------------------------------
// Tiled layout: slowness bricks and natural-order copies of fields.
// ---------------------------------------------------------------------------
// The 8 brick variants of one model (v = negX + 2 negY + 4 negZ: the
// sweep's directions), each brick_records(nz) records per tile in the column
// kernel's lane order: element l < 64 is the cell at the ring position of
// tile element l (local (1 + x, 1 + y), mirrored along a reversed axis),
// element 64 + h the cell at the halo position of halo lane h (h < 9:
// local (0, h); else (h - 8, 0)).  The cell at local (c, r) of record k is
// grid cell (8 tx - 1 + c', 8 ty - 1 + r', z') with c' = c, or 8 - c along
// a reversed axis, clamped into the grid, and z' the permuted plane
// clamp(k - c - r, 0, ncz - 1), reversed along a reversed z axis.
template <typename TS>
__global__ void __launch_bounds__(256)
tile_slowness_kernel(int nx, int ny, int nz, const TS *__restrict__ s,
                     TS *__restrict__ b)
{
    const int ncx = nx - 1, ncy = ny - 1, ncz = nz - 1;
    const int nTX = tiles_of(nx);
    const int nRec = brick_records(nz);
    const int64_t perVariant = brick_variant_values(nx, ny, nz);
    const int64_t n = kBrickVariants*perVariant;
    for (int64_t i = (int64_t) blockIdx.x*blockDim.x + threadIdx.x; i < n;
         i += (int64_t) gridDim.x*blockDim.x)
    {
        const int v = (int) (i/perVariant);
        const int64_t j = i - v*perVariant;
        const int64_t rec = j/kBrickValues;
        const int l = (int) (j - rec*kBrickValues);
        const int tile = (int) (rec/nRec);
        const int k = (int) (rec - (int64_t) tile*nRec);
        const int ty = tile/nTX, tx = tile - ty*nTX;
        const bool negX = v & 1, negY = v & 2, negZ = v & 4;
        int c, r;
        if (l < kTileValues)
        {
            const int xl = l % kColumnTile, yl = l/kColumnTile;
            c = 1 + (negX ? kColumnTile - 1 - xl : xl);
            r = 1 + (negY ? kColumnTile - 1 - yl : yl);
        }
        else
        {
            const int hl = l - kTileValues;
            c = hl < kColumnHalo ? 0 : hl - kColumnTile;
            r = hl < kColumnHalo ? hl : 0;
        }
        const int cl = negX ? kColumnTile - c : c;
        const int rl = negY ? kColumnTile - r : r;
        const int cx = min(max(tx*kColumnTile - 1 + cl, 0), ncx - 1);
        const int cy = min(max(ty*kColumnTile - 1 + rl, 0), ncy - 1);
        const int pcz = min(max(k - c - r, 0), ncz - 1);
        const int cz = negZ ? ncz - 1 - pcz : pcz;
        b[i] = s[((int64_t) cz*ncy + cy)*ncx + cx];
    }
}

template <typename TS>
__global__ void __launch_bounds__(256)
untile_field_kernel(Problem3D p, const TS *__restrict__ T,
                    TS *__restrict__ out)
{
    const int64_t nxy = (int64_t) p.nx*p.ny;
    const int64_t n = nxy*p.nz;
    const TS *Tp = T + p.tOffset;
    for (int64_t i = (int64_t) blockIdx.x*blockDim.x + threadIdx.x; i < n;
         i += (int64_t) gridDim.x*blockDim.x)
    {
        const int iz = (int) (i/nxy);
        const int rem = (int) (i - (int64_t) iz*nxy);
        const int iy = rem/p.nx;
        const int ix = rem - iy*p.nx;
        out[i] = Tp[tiled_index(p.nTX, p.nz, ix, iy, iz)];
    }
}

// ---------------------------------------------------------------------------
// Model preparation (src/model3d.cpp:45-151 interpolate3d, :316-375).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
nodal_to_cell3d(int nx, int ny, int nz, const double *__restrict__ v,
                int ordering, double *__restrict__ slow)
{
    const int64_t ncx = nx - 1, ncy = ny - 1, ncz = nz - 1;
    const int64_t nCell = ncx*ncy*ncz;
    for (int64_t i = (int64_t) blockIdx.x*blockDim.x + threadIdx.x; i < nCell;
         i += (int64_t) gridDim.x*blockDim.x)
    {
        int64_t iz = i/(ncx*ncy);
        int64_t rem = i - iz*ncx*ncy;
        int64_t iy = rem/ncx;
        int64_t ix = rem - iy*ncx;
        int64_t idx1, idx2, idx3, idx4, idx5, idx6, idx7, idx8;
        if (ordering == 0)
        {
            idx1 = iz*(ncx + 1)*(ncy + 1) + iy*(ncx + 1) + ix;
            idx2 = idx1 + 1;
            idx3 = idx1 + (ncx + 1);
            idx4 = idx3 + 1;
            idx5 = idx1 + (ncx + 1)*(ncy + 1);
            idx6 = idx2 + (ncx + 1)*(ncy + 1);
            idx7 = idx3 + (ncx + 1)*(ncy + 1);
            idx8 = idx4 + (ncx + 1)*(ncy + 1);
        }
        else
        {
            idx1 = ix*(ncz + 1)*(ncy + 1) + iy*(ncz + 1) + iz;
            idx2 = idx1 + 1;
            idx3 = idx1 + (ncz + 1);
            idx4 = idx3 + 1;
            idx5 = idx1 + (ncz + 1)*(ncy + 1);
            idx6 = idx2 + (ncz + 1)*(ncy + 1);
            idx7 = idx3 + (ncz + 1)*(ncy + 1);
            idx8 = idx4 + (ncz + 1)*(ncy + 1);
        }
        double sum1 = v[idx1] + v[idx2];
        double sum2 = v[idx3] + v[idx4];
        double sum3 = v[idx5] + v[idx6];
        double sum4 = v[idx7] + v[idx8];
        slow[i] = 8.0/(sum1 + sum2 + sum3 + sum4);
    }
}

__global__ void __launch_bounds__(256)
cell_velocity_to_slowness3d(int nx, int ny, int nz,
                            const double *__restrict__ v, int ordering,
                            double *__restrict__ slow)
{
    const int64_t ncx = nx - 1, ncy = ny - 1, ncz = nz - 1;
    const int64_t nCell = ncx*ncy*ncz;
    for (int64_t i = (int64_t) blockIdx.x*blockDim.x + threadIdx.x; i < nCell;
         i += (int64_t) gridDim.x*blockDim.x)
    {
        int64_t src = i;
        if (ordering != 0)
        {
            int64_t iz = i/(ncx*ncy);
            int64_t rem = i - iz*ncx*ncy;
            int64_t iy = rem/ncx;
            int64_t ix = rem - iy*ncx;
            src = (ix*ncy + iy)*ncz + iz;
        }
        slow[i] = 1.0/v[src];
    }
}

template <typename TD, typename TSrc>
__global__ void __launch_bounds__(256)
convert_kernel(int64_t n, const TSrc *__restrict__ in, TD *__restrict__ out)
{
    for (int64_t i = (int64_t) blockIdx.x*blockDim.x + threadIdx.x; i < n;
         i += (int64_t) gridDim.x*blockDim.x)
    {
        out[i] = (TD) in[i];
    }
}

// ---------------------------------------------------------------------------
// Model range; scaled-integer storage: slowness codes, decoded fields.
// ---------------------------------------------------------------------------
// Block minima and maxima of v[0..n) into partial[2 blockIdx.x] and
// partial[2 blockIdx.x + 1] (the host reduces them).
__global__ void __launch_bounds__(256)
block_range_kernel(int64_t n, const double *__restrict__ v,
                   double *__restrict__ partial)
{
    __shared__ double lo[256], hi[256];
    double a = v[0], b = a;
    for (int64_t i = (int64_t) blockIdx.x*blockDim.x + threadIdx.x; i < n;
         i += (int64_t) gridDim.x*blockDim.x)
    {
        a = fmin(a, v[i]);
        b = fmax(b, v[i]);
    }
    lo[threadIdx.x] = a;
    hi[threadIdx.x] = b;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1)
    {
        if ((int) threadIdx.x < k)
        {
            lo[threadIdx.x] = fmin(lo[threadIdx.x], lo[threadIdx.x + k]);
            hi[threadIdx.x] = fmax(hi[threadIdx.x], hi[threadIdx.x + k]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0)
    {
        partial[2*blockIdx.x] = lo[0];
        partial[2*blockIdx.x + 1] = hi[0];
    }
}

__global__ void __launch_bounds__(256)
encode_slowness_kernel(int64_t n, const double *__restrict__ in,
                       double scale, uint32_t *__restrict__ out)
{
    for (int64_t i = (int64_t) blockIdx.x*blockDim.x + threadIdx.x; i < n;
         i += (int64_t) gridDim.x*blockDim.x)
    {
        double q = rint(in[i]*scale);
        out[i] = (uint32_t) fmin(fmax(q, 0.0), (double) kTimeMaxCode);
    }
}

// Travel-time codes of every problem to FP64 (blockIdx.y is the problem).
__global__ void __launch_bounds__(256)
decode_times_kernel(const Problem3D *__restrict__ problems,
                    const uint32_t *__restrict__ in, double *__restrict__ out)
{
    const Problem3D &p = problems[blockIdx.y];
    const int64_t n = p.tCount;
    const uint32_t *src = in + p.tOffset;
    double *dst = out + p.tOffset;
    for (int64_t i = (int64_t) blockIdx.x*blockDim.x + threadIdx.x; i < n;
         i += (int64_t) gridDim.x*blockDim.x)
    {
        dst[i] = Store<uint32_t>::time(src[i], p);
    }
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
static inline unsigned grid_for(int64_t n, int block, unsigned cap)
{
    int64_t g = (n + block - 1)/block;
    if (g < 1) { g = 1; }
    return (unsigned) (g < cap ? g : cap);
}

template <typename TS>
hipError_t launch_init3d(const Problem3D *dProblems, int nProblems,
                         int64_t totalCount, TS *T, hipStream_t stream)
{
    hipLaunchKernelGGL(init_travel_times3d<TS>,
                       dim3(grid_for(totalCount/(16/sizeof(TS)) + 1, 256,
                                     16384)),
                       dim3(256), 0, stream, T, totalCount);
    hipLaunchKernelGGL(init_source_corners3d<TS>,
                       dim3((unsigned) ((8*nProblems + 63)/64)), dim3(64), 0,
                       stream, dProblems, nProblems, T);
    return hipGetLastError();
}

template <typename TS>
hipError_t launch_hyperplane3d(const Problem3D *dProblems, int problem,
                               int sweep, int initialize, int level, int kLo,
                               int nPairs, TS *T, const TS *S,
                               unsigned int *change, hipStream_t stream)
{
    if (nPairs <= 0) { return hipSuccess; }
    hipLaunchKernelGGL(sweep_hyperplane3d<TS>,
                       dim3((unsigned) ((nPairs + 255)/256)), dim3(256), 0,
                       stream, dProblems, problem, sweep, initialize, level,
                       kLo, nPairs, T, S, change);
    return hipGetLastError();
}

template <typename TS>
hipError_t launch_columns3d(const Problem3D *dProblems,
                            const ColumnItem *dItems, int nItems, int sweep,
                            int initialize, int diagonal, int boxPerDiag,
                            int chunk, TS *T, const TS *S,
                            unsigned int *change, int depth, bool merged,
                            hipStream_t stream)
{
    if (nItems <= 0) { return hipSuccess; }
    constexpr int W = column_waves<TS>();
    const dim3 grid((unsigned) ((nItems + W - 1)/W)), block(64*W);
    if (merged)
    {
        // prefetch depth 4 only: the factored branch's registers
        hipLaunchKernelGGL((sweep_columns3d<TS, W, 4, false, true>), grid,
                           block, 0, stream, dProblems, dItems, nItems,
                           sweep, initialize, diagonal, boxPerDiag, chunk, 0,
                           T, S, change);
        return hipGetLastError();
    }
    switch (depth)
    {
    case 4:
        hipLaunchKernelGGL((sweep_columns3d<TS, W, 4, false>), grid,
                           block, 0, stream, dProblems, dItems, nItems, sweep,
                           initialize, diagonal, boxPerDiag, chunk, 0, T, S,
                           change);
        break;
    case 8:
        hipLaunchKernelGGL((sweep_columns3d<TS, W, 8, false>), grid,
                           block, 0, stream, dProblems, dItems, nItems, sweep,
                           initialize, diagonal, boxPerDiag, chunk, 0, T, S,
                           change);
        break;
    case 12:
        hipLaunchKernelGGL((sweep_columns3d<TS, W, 12, false>), grid,
                           block, 0, stream, dProblems, dItems, nItems, sweep,
                           initialize, diagonal, boxPerDiag, chunk, 0, T, S,
                           change);
        break;
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <typename TS>
hipError_t launch_factored_columns3d(const Problem3D *dProblems,
                                     int nProblems, int sweep, int initialize,
                                     int diagonal, int boxPerDiag, int chunk,
                                     int phase, TS *T, const TS *S,
                                     unsigned int *change,
                                     hipStream_t stream)
{
    if (boxPerDiag <= 0) { return hipSuccess; }
    int n = nProblems*boxPerDiag;
    hipLaunchKernelGGL((sweep_columns3d<TS, 1, 4, true>),
                       dim3((unsigned) n), dim3(64), 0, stream, dProblems,
                       (const ColumnItem *) nullptr, n, sweep, initialize,
                       diagonal, boxPerDiag, chunk, phase, T, S, change);
    return hipGetLastError();
}

template <typename TS>
hipError_t launch_queued_columns3d(const Problem3D *dProblems,
                                   const ColumnItem *dItems, int nItems,
                                   int sweep, int initialize, int chunk, TS *T,
                                   const TS *S, unsigned int *change,
                                   const ColumnQueue &q, int waves, int depth,
                                   hipStream_t stream)
{
    if (nItems <= 0) { return hipSuccess; }
    static_assert(sizeof(TS) == 8, "the work queue sweeps FP64 fields");
    const dim3 grid((unsigned) std::max(1, std::min(nItems, waves)));
    switch (depth)
    {
    case 4:
        hipLaunchKernelGGL((sweep_columns3d_queued<TS, 4>), grid, dim3(64),
                           0, stream, dProblems, dItems, nItems, sweep,
                           initialize, chunk, T, S, change, q);
        break;
    case 8:
        hipLaunchKernelGGL((sweep_columns3d_queued<TS, 8>), grid, dim3(64),
                           0, stream, dProblems, dItems, nItems, sweep,
                           initialize, chunk, T, S, change, q);
        break;
    case 12:
        hipLaunchKernelGGL((sweep_columns3d_queued<TS, 12>), grid, dim3(64),
                           0, stream, dProblems, dItems, nItems, sweep,
                           initialize, chunk, T, S, change, q);
        break;
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <typename TS>
int column_waves_per_cu(int depth, bool merged)
{
    constexpr int W = column_waves<TS>();
    int blocks = 0;
    hipError_t e = hipSuccess;
    if (merged)
    {
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &blocks, sweep_columns3d<TS, W, 4, false, true>, 64*W, 0);
        return e == hipSuccess && blocks > 0 ? blocks*W : 0;
    }
    switch (depth)
    {
    case 8:
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &blocks, sweep_columns3d<TS, W, 8, false>, 64*W, 0);
        break;
    case 12:
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &blocks, sweep_columns3d<TS, W, 12, false>, 64*W, 0);
        break;
    default:
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &blocks, sweep_columns3d<TS, W, 4, false>, 64*W, 0);
        break;
    }
    return e == hipSuccess && blocks > 0 ? blocks*W : 0;
}

int queued_waves_per_cu(int depth)
{
    int blocks = 0;
    hipError_t e = hipSuccess;
    switch (depth)
    {
    case 8:
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &blocks, sweep_columns3d_queued<double, 8>, 64, 0);
        break;
    case 12:
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &blocks, sweep_columns3d_queued<double, 12>, 64, 0);
        break;
    default:
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &blocks, sweep_columns3d_queued<double, 4>, 64, 0);
        break;
    }
    return e == hipSuccess && blocks > 0 ? blocks : 0;
}

template int column_waves_per_cu<float>(int, bool);
template int column_waves_per_cu<double>(int, bool);
template int column_waves_per_cu<uint32_t>(int, bool);

// A problem descriptor into device memory (the allocation-free solve's
// scratch), with the source cell's slowness read from the model there, so
// that no host copy is needed in either direction.
__global__ void __launch_bounds__(64)
store_problem3d_kernel(Problem3D p, int64_t sourceCell,
                       const double *__restrict__ slowness,
                       Problem3D *__restrict__ dst)
{
    if (threadIdx.x == 0)
    {
        p.srcSlowness = slowness[p.sOffset + sourceCell];
        *dst = p;
    }
}

hipError_t launch_store_problem3d(const Problem3D &p, int64_t sourceCell,
                                  const double *slowness, Problem3D *dst,
                                  hipStream_t stream)
{
    hipLaunchKernelGGL(store_problem3d_kernel, dim3(1), dim3(64), 0, stream,
                       p, sourceCell, slowness, dst);
    return hipGetLastError();
}

hipError_t launch_clear_words(unsigned int *w, int64_t n, hipStream_t stream)
{
    if (n <= 0) { return hipSuccess; }
    hipLaunchKernelGGL(clear_words_kernel, dim3(grid_for(n, 256, 1024)),
                       dim3(256), 0, stream, w, n);
    return hipGetLastError();
}

template <typename TS>
hipError_t launch_tile_slowness(int nx, int ny, int nz, const TS *s, TS *b,
                                hipStream_t stream)
{
    const int64_t n = kBrickVariants*brick_variant_values(nx, ny, nz);
    hipLaunchKernelGGL(tile_slowness_kernel<TS>,
                       dim3(grid_for(n, 256, 16384)), dim3(256), 0, stream,
                       nx, ny, nz, s, b);
    return hipGetLastError();
}

template <typename TS>
hipError_t launch_untile_field(const Problem3D &p, const TS *T, TS *out,
                               hipStream_t stream)
{
    const int64_t n = (int64_t) p.nx*p.ny*p.nz;
    hipLaunchKernelGGL(untile_field_kernel<TS>,
                       dim3(grid_for(n, 256, 16384)), dim3(256), 0, stream,
                       p, T, out);
    return hipGetLastError();
}

hipError_t launch_nodal_to_cell3d(int nx, int ny, int nz, const double *v,
                                  int ordering, double *slow,
                                  hipStream_t stream)
{
    int64_t nCell = (int64_t) (nx - 1)*(ny - 1)*(nz - 1);
    hipLaunchKernelGGL(nodal_to_cell3d, dim3(grid_for(nCell, 256, 8192)),
                       dim3(256), 0, stream, nx, ny, nz, v, ordering, slow);
    return hipGetLastError();
}

hipError_t launch_cell_velocity_to_slowness3d(int nx, int ny, int nz,
                                              const double *v, int ordering,
                                              double *slow,
                                              hipStream_t stream)
{
    int64_t nCell = (int64_t) (nx - 1)*(ny - 1)*(nz - 1);
    hipLaunchKernelGGL(cell_velocity_to_slowness3d,
                       dim3(grid_for(nCell, 256, 8192)), dim3(256), 0, stream,
                       nx, ny, nz, v, ordering, slow);
    return hipGetLastError();
}

hipError_t launch_convert(int64_t n, const double *in, float *out,
                          hipStream_t stream)
{
    hipLaunchKernelGGL((convert_kernel<float, double>),
                       dim3(grid_for(n, 256, 16384)), dim3(256), 0, stream, n,
                       in, out);
    return hipGetLastError();
}

hipError_t launch_convert(int64_t n, const float *in, double *out,
                          hipStream_t stream)
{
    hipLaunchKernelGGL((convert_kernel<double, float>),
                       dim3(grid_for(n, 256, 16384)), dim3(256), 0, stream, n,
                       in, out);
    return hipGetLastError();
}

hipError_t launch_block_range(int64_t n, const double *v, double *partial,
                              int nBlocks, hipStream_t stream)
{
    hipLaunchKernelGGL(block_range_kernel, dim3((unsigned) nBlocks),
                       dim3(256), 0, stream, n, v, partial);
    return hipGetLastError();
}

hipError_t launch_encode_slowness(int64_t n, const double *in, double scale,
                                  uint32_t *out, hipStream_t stream)
{
    hipLaunchKernelGGL(encode_slowness_kernel, dim3(grid_for(n, 256, 16384)),
                       dim3(256), 0, stream, n, in, scale, out);
    return hipGetLastError();
}

hipError_t launch_decode_times(const Problem3D *dProblems, int nProblems,
                               int64_t maxNodes, const uint32_t *in,
                               double *out, hipStream_t stream)
{
    dim3 grid(grid_for(maxNodes, 256, 4096), (unsigned) nProblems);
    hipLaunchKernelGGL(decode_times_kernel, grid, dim3(256), 0, stream,
                       dProblems, in, out);
    return hipGetLastError();
}

template hipError_t launch_init3d<float>(const Problem3D *, int, int64_t,
                                         float *, hipStream_t);
template hipError_t launch_init3d<double>(const Problem3D *, int, int64_t,
                                          double *, hipStream_t);
template hipError_t launch_hyperplane3d<float>(const Problem3D *, int, int,
                                               int, int, int, int, float *,
                                               const float *, unsigned int *, hipStream_t);
template hipError_t launch_hyperplane3d<double>(const Problem3D *, int, int,
                                                int, int, int, int, double *,
                                                const double *, unsigned int *, hipStream_t);
template hipError_t launch_init3d<uint32_t>(const Problem3D *, int, int64_t,
                                            uint32_t *, hipStream_t);
template hipError_t launch_hyperplane3d<uint32_t>(const Problem3D *, int,
                                                  int, int, int, int, int,
                                                  uint32_t *,
                                                  const uint32_t *,
                                                  unsigned int *, hipStream_t);

template hipError_t launch_columns3d<float>(
    const Problem3D *, const ColumnItem *, int, int, int, int, int, int,
    float *, const float *, unsigned int *, int, bool, hipStream_t);
template hipError_t launch_factored_columns3d<float>(
    const Problem3D *, int, int, int, int, int, int, int, float *,
    const float *, unsigned int *, hipStream_t);
template hipError_t launch_queued_columns3d<double>(
    const Problem3D *, const ColumnItem *, int, int, int, int, double *,
    const double *, unsigned int *, const ColumnQueue &, int, int,
    hipStream_t);
template hipError_t launch_columns3d<double>(
    const Problem3D *, const ColumnItem *, int, int, int, int, int, int,
    double *, const double *, unsigned int *, int, bool, hipStream_t);
template hipError_t launch_factored_columns3d<double>(
    const Problem3D *, int, int, int, int, int, int, int, double *,
    const double *, unsigned int *, hipStream_t);
template hipError_t launch_columns3d<uint32_t>(
    const Problem3D *, const ColumnItem *, int, int, int, int, int, int,
    uint32_t *, const uint32_t *, unsigned int *, int, bool, hipStream_t);
template hipError_t launch_factored_columns3d<uint32_t>(
    const Problem3D *, int, int, int, int, int, int, int, uint32_t *,
    const uint32_t *, unsigned int *, hipStream_t);
#define EKX_TILED(TS)                                                        \
    template hipError_t launch_tile_slowness<TS>(int, int, int, const TS *, \
                                                 TS *, hipStream_t);       \
    template hipError_t launch_untile_field<TS>(const Problem3D &,         \
                                                const TS *, TS *,          \
                                                hipStream_t);
EKX_TILED(float)
EKX_TILED(double)
EKX_TILED(uint32_t)
#undef EKX_TILED

} // namespace ekx
