// ekx_device.hpp -- descriptors shared by the host launch code and the HIP
// kernels of the fast-sweeping solver.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace ekx
{

// Sentinel of an unreached node: HUGE in include/private/solver3d.hpp:10 and
// include/private/solver2d.hpp:16.
constexpr double kHuge = 1.e10;

// Tile footprint of the column kernel: one 64-lane wave owns an 8 x 8 block
// of (x, y) nodes and marches through z.
constexpr int kColumnTile = 8;
constexpr int kColumnHalo = kColumnTile + 1;          // 9: tile + upwind halo
constexpr int kColumnPlane = kColumnHalo*kColumnHalo; // 81 values per plane
constexpr int kColumnSkew = 2*(kColumnTile - 1);      // 14: lane a+b spread
// LDS ring of planes per wave.  A plane enters at step q, is read by the
// lanes through step q + 14 and is written back at the end of that step, so
// 15 slots are enough.
constexpr int kColumnRing = kColumnSkew + 1;

__host__ __device__ inline int tiles_of(int n)
{
    return (n + kColumnTile - 1)/kColumnTile;
}

// Tiled field layout of the column kernel.  The nodes of an (x, y) tile of
// 8 x 8 form one run of nz plane records of 64 values (x fastest within a
// record); tiles follow in row-major (tile y, tile x) order and the grid is
// padded to whole tiles.  A column therefore reads and writes one contiguous
// run per sweep, in either z direction.  After a problem's tile records come
// its edge records, one per (tile, plane), of kEdgeValues values: the
// column's most downwind x column of its 9 x 9 working plane (the halo row
// value first, then the 8 tile rows) and its most downwind y row (the 8
// tile columns), as the current sweep leaves them for the next column in x
// and in y.  Slowness bricks hold the 9 x 9 cells around a tile's nodes
// (cells 8 t - 1 .. 8 t + 7 per axis, clamped to the grid) in records of
// 81 values, skewed to the column kernel's steps: in record k of a tile the
// cell at local position (c, r) of the sweep's permuted frame comes from
// permuted cell plane clamp(k - c - r, 0, ncz - 1).  Lane (a, b), working
// on plane z at step g = z + a + b, finds its four cells of the plane in
// records g (position (a, b)), g + 1 ((a + 1, b) and (a, b + 1)) and g + 2
// ((a + 1, b + 1)), so a column keeps only the last few records in LDS
// rather than every plane its lanes span.  A tile has nz + 39 records, one
// contiguous run: records nz + 16 .. nz + 38 (clamped planes) let the
// prefetch run up to 2 x 12 records past the last step without a bound
// check.  There are 8 variants, one per sweep direction (the skew follows
// the permuted frame), each ordered as the column kernel's lanes load
// them.
constexpr int kTileValues = kColumnTile*kColumnTile;    // 64
constexpr int kEdgeValues = 2*kColumnTile + 1;           // 17
constexpr int kBrickValues = kColumnPlane;               // 81
constexpr int kBrickVariants = 8;
// LDS records of slowness per wave: the three a step reads and the one
// entering for the next step.
constexpr int kSlownessRing = 4;
// Elements per travel-time ring slot: the 81-value plane, padded.  At a
// step the lanes of a wave read 15 different slots (lane (a, b) slot
// step - a - b) at positions 9 b + a + {0, 1, 9, 10}; with 81 elements per
// slot the skew cancels the position and up to 16 lanes meet on one LDS
// bank, with these strides at most 2 (4 bytes) or 3 (8 bytes) do, on 32
// banks of 4 bytes.
template <typename TS> constexpr int ring_slot()
{
    return sizeof(TS) == 8 ? 88 : 86;
}
// Element type of the slowness ring: the arithmetic's.  Scaled-integer cells
// are decoded as they enter (2 values a lane and step instead of 4 as they
// are read); the ring's 2.6 KB still leave more waves per CU than the
// registers of the FP64 arithmetic do.
template <typename TS>
using SlownessRing =
    typename std::conditional<sizeof(TS) == 4 &&
                                  !std::is_same<TS, float>::value,
                              double, TS>::type;
// Largest prefetch depth (planes loaded ahead) of the column kernel.
constexpr int kMaxPrefetch = 12;

__host__ __device__ inline int brick_records(int nz)
{
    return nz + kColumnSkew + 2*kMaxPrefetch + 1;
}

// Travel-time elements kept free before the first problem's records and
// after the last one's: the column kernel advances its halo addresses
// without a bound check, so past a chunk's last plane they run up to
// kColumnSkew + 2 kMaxPrefetch planes beyond the records they read (the
// values are never used; a plane holds at most kTileValues of them).
constexpr int64_t kFieldGuard =
    (int64_t) (kColumnSkew + 2*kMaxPrefetch + 1)*kTileValues;

// Elements of one brick variant of an nx x ny x nz node grid.
__host__ __device__ inline int64_t brick_variant_values(int nx, int ny, int nz)
{
    return (int64_t) tiles_of(nx)*tiles_of(ny)*brick_records(nz)*
           kBrickValues;
}

// z-split of a column chunk that overlaps the factored box, when the box
// columns run in their own (factored) launches: the factored launch takes
// the chunk's planes from its first updated plane through the box's last
// permuted plane (phase 0, a prefix, launched before the diagonal's bulk
// launch) or from the box's first permuted plane to the chunk's end (phase
// 1, a suffix, launched after it), whichever is shorter, and the bulk
// launch takes the other planes, which lie outside the box and so need only
// the Cartesian update.  [zFirst, zEnd): the chunk's updated planes; the
// factored part is [zFirst, cut) in phase 0 and [cut, zEnd) in phase 1.
struct BoxSplitZ
{
    int phase, cut;
};

__host__ __device__ inline BoxSplitZ box_split_z(int nz, int srcCellZ,
                                                 int radius, int negZ,
                                                 int zFirst, int zEnd)
{
    const int zLo = srcCellZ - radius < 0 ? 0 : srcCellZ - radius;
    const int zHi = srcCellZ + radius > nz - 1 ? nz - 1 : srcCellZ + radius;
    const int jzLo = negZ ? nz - 1 - zHi : zLo;
    const int jzHi = negZ ? nz - 1 - zLo : zHi;
    BoxSplitZ s;
    s.phase = jzHi + 1 - zFirst <= zEnd - jzLo ? 0 : 1;
    const int c = s.phase == 0 ? jzHi + 1 : jzLo;
    s.cut = c < zFirst ? zFirst : (c > zEnd ? zEnd : c);
    return s;
}

// Index of node (x, y, z) in a tiled field of nTX tiles per row.
__host__ __device__ inline int64_t tiled_index(int nTX, int nz, int x, int y,
                                               int z)
{
    const int64_t tile = (int64_t) (y/kColumnTile)*nTX + x/kColumnTile;
    return (tile*nz + z)*kTileValues + (y % kColumnTile)*kColumnTile +
           x % kColumnTile;
}

// Grid constants of the non-uniform local solver
// (include/private/solver3d.hpp:247-261).
struct NonUniform3D
{
    double dxInv, dyInv, dzInv;
    double dx2Inv, dy2Inv, dz2Inv;
    double dx_dz, dz_dx, dy_dz, dz_dy, dx_dy, dy_dx;
    double dx2_p_dz2_inv, dy2_p_dz2_inv, dx2_p_dy2_inv;
};

// One independent 3D problem (geometry + model + source) of a batch.
struct Problem3D
{
    int nx, ny, nz;
    int radius;                 // factored-eikonal radius (grid points)
    int srcCellX, srcCellY, srcCellZ;
    int uniform;                // dx == dy == dz within 100 eps
    double dx, dy, dz;
    double srcOffX, srcOffY, srcOffZ;  // source - origin (m)
    double srcSlowness;         // slowness of the source cell
    int64_t tOffset;            // first node of this problem's field
    int64_t sOffset;            // first cell of this problem's model
    // Scaled-integer storage (uint32 codes): travel time = code * tStep,
    // slowness = code * sStep; tScale = 1 / tStep.  Unused otherwise.
    double tStep, tScale, sStep;
    NonUniform3D nu;
    // Field layout: tiled (column kernel) or natural (x fastest).  A tiled
    // field is nTX * nTY * nz tile records, then as many edge records
    // starting at eOffset; tCount is the field's whole extent (elements
    // from tOffset).  sbOffset is the first element of the model's
    // slowness bricks.
    int tiled;
    int nTX, nTY;
    // h s of every cell at least 2^-300, no time above HUGE
    // (cartesian_uniform3d, Engine3D::find_ranges)
    int scaled;
    int64_t tCount;
    int64_t eOffset;
    int64_t sbOffset;
};

// Index of node (x, y, z) in problem p's field (relative to tOffset).
__host__ __device__ inline int64_t node_index(const Problem3D &p, int x, int y,
                                              int z)
{
    return p.tiled ? tiled_index(p.nTX, p.nz, x, y, z)
                   : ((int64_t) z*p.ny + y)*p.nx + x;
}

// A column chunk (8 x 8 footprint, one z-chunk) of one problem.
struct ColumnItem
{
    int problem;
    int bx, by, bz;             // column and chunk index, permuted frame
};

// Work queue of one sweep launch in work-queue form: item i of problem p
// publishes the sweep's epoch in flags[flagBase[p] + (bz*nTY + by)*nTX + bx]
// once finished; counter hands out the launch's items in list order; error
// is set when a wait exceeded waitTicks of the device's wall clock (then
// later waits return at once).  Flags and counters are zeroed at the start
// of each sequence of sweeps, whose epochs count from 1.
struct ColumnQueue
{
    const int *flagBase;
    unsigned int *flags;
    unsigned int *counter;
    unsigned int *error;
    unsigned int epoch;
    unsigned int pad;
    uint64_t waitTicks;
};

// Flow kernel (a whole solve in one launch): an 8 x 8 column of a problem,
// its step records (first element of step 0, in either buffer) and its
// mailbox (first element of record 0, in each buffer).  Columns are numbered
// by id, a problem's in row-major (tile y, tile x) order, and their records
// and mailboxes follow each other in that order; the launch places them in
// another (placeholders there have problem -1).
struct FlowColumn
{
    int problem;
    int mx, my;
    int id;
    int64_t rec;
    int64_t mail;
};

// Step records of 64 values: nz + 14 hold nodes; lanes outside the grid's
// planes, the steps' rounding to groups of 4 and the prefetch use up to 28
// records before and 36 after them.
constexpr int kFlowPad = 28;
__host__ __device__ inline int flow_records(int nz)
{
    return nz + kColumnSkew + kFlowPad + 36;
}

// Mailbox records: the corner and the 8 nodes for the x neighbour, then
// those 7 of the y neighbour's 8 nodes that are not among them (the last of
// the x neighbour's is the y neighbour's last too): one 128 byte line in
// FP64.  Record t is read at the reader's step t and written at the writer's
// step t + 7, from 7 records before the first on; the reader's prefetch and
// the rounding of the steps run up to 24 records past nz.
constexpr int kMailValues = 16;
constexpr int kMailBuffers = 4;
constexpr int kMailY = 9;
constexpr int kMailPad = 8;
__host__ __device__ inline int flow_mails(int nz)
{
    return kMailPad + nz + 24;
}

// A receiver located in one problem's grid (Station3D, src/station3d.cpp:
// 158-291): offset from the model origin and the cell that holds it.
struct StationLoc3D
{
    double off[3];
    int cell[3];
    int pad;
};

// One problem of a 2D batch.
struct Problem2D
{
    int nx, nz;
    int radius;
    int srcCellX, srcCellZ;
    int uniform;
    int nSweeps;
    int pad;
    double dx, dz;
    double srcOffX, srcOffZ;
    double srcSlowness;
    double dx_dz, dz_dx, cosTheta, sinTheta;  // solver2d.hpp:41-46
    // quotients of the factored update (h: dx on a uniform grid)
    double dxinv, dzinv, hx2inv, hz2inv;      // 1/dx, 1/dz, 1/dx^2, 1/dz^2
    double twoOverH, twoOverH2, halfOverH2;   // 2/h, 2/h^2, 1/(2 h^2)
    int64_t tOffset;
    int64_t sOffset;
    // band kernel: first values of the skewed travel times and cells
    int64_t wOffset;
    int64_t cOffset;
    int route;                  // Route2D
};

// How a 2D problem is solved: by the level kernel, or by the band kernel
// without or with range tests of its square roots (models out of
// range, Range2D).
enum Route2D { kLevels2d, kBands2d, kBandsAnyRange2d, kRoutes2d };

// Band kernel of the 2D solve: bands of 64 rows, and per band step records
// of 64 travel times (two buffers) and of 65 cells (one set per sweep
// direction).  Lane i is i columns behind lane 0, so nx + 63 steps, rounded
// up to whole groups of 8, pass every column through a band.  Lanes outside
// the grid's columns write too: up to 63 + 7 records on either side of the
// nx + 63 that hold nodes, whose padding also takes the prefetch.
constexpr int kMaxBands2d = 16;
constexpr int kCellRecord2d = 65;
constexpr int kBandPad2d = 72;

__host__ __device__ inline int bands2d(int nz) { return (nz + 63)/64; }

__host__ __device__ inline int band_records2d(int nx)
{
    return nx + 63 + 2*kBandPad2d;
}

// travel-time work of one problem
__host__ __device__ inline int64_t band_values2d(int nx, int nz)
{
    return 2*(int64_t) bands2d(nz)*band_records2d(nx)*64;
}

// bytes of it that a solve touches: both buffers, the lanes with a row
__host__ __device__ inline int64_t band_bytes2d(int nx, int nz)
{
    return 2*(int64_t) nz*(nx + 63)*(int64_t) sizeof(double);
}

// cell records of one band and sweep direction: the steps rounded up to
// whole groups of 8, and the group that the prefetch runs ahead
__host__ __device__ inline int cell_steps2d(int nx)
{
    return (nx + 63 + 7)/8*8 + 8;
}

__host__ __device__ inline int64_t cell_values2d(int nx, int nz)
{
    return 4*(int64_t) bands2d(nz)*cell_steps2d(nx)*kCellRecord2d;
}

// What a launch of the band kernel needs to know of its problems.
struct Plan2D
{
    int problems[kRoutes2d] = {};       // by route
    // of the problems that the band kernel takes: rows of the tallest, bands
    // and bytes of records in all
    int maxNz = 0;
    int64_t bands = 0, recordBytes = 0;
    void add(const Problem2D &p)
    {
        problems[p.route] += 1;
        if (p.route == kLevels2d) { return; }
        maxNz = p.nz > maxNz ? p.nz : maxNz;
        bands += bands2d(p.nz);
        recordBytes += band_bytes2d(p.nx, p.nz);
    }
    int launches() const
    {
        int n = 0;
        for (int k : problems) { n += k > 0; }
        return n;
    }
};

// Grids that the band kernel takes: at most 16 bands (the waves of a
// workgroup), and lane offsets that stay well within 32 bits.
__host__ __device__ inline bool fits_bands2d(int nx, int nz)
{
    return nz <= 64*kMaxBands2d && nx <= 65536;
}

} // namespace ekx
