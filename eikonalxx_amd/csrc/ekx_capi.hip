// ekx_capi.hip -- host implementation of the C ABI declared in
// include/eikonalxx_amd.h.  Owns device memory, builds the launch schedule
// of a solve and replays it from a captured hipGraph.
#include "eikonalxx_amd.h"
#include "ekx_guard.hpp"
#include "ekx_kernels.hpp"
#include "ekx_reads.hpp"
#include "ekx_reservation.hpp"
#include "ekx_storage.hpp"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <map>
#include <mutex>
#include <shared_mutex>
#include <numeric>
#include <string>
#include <tuple>
#include <type_traits>
#include <vector>

using namespace ekx;

namespace
{

// Blocks of the model-maximum reduction (FIXED32 modes).
constexpr size_t kMaxPartials = 1024;
// blocks of the reduction of one model's slowness range
constexpr int kRangeBlocks = 256;
// Column z-chunk depths the launch-shape choice considers (0: whole
// columns), longest first.
constexpr int kChunkCandidates[] = {0, 128, 96, 64, 48, 32, 24, 16, 12, 8};
// Independent launch chains of a batch (one stream each).
constexpr int kMaxChains = 16;


thread_local std::string g_error;

ekx_status fail(ekx_status status, const std::string &message)
{
    g_error = message;
    return status;
}

#define EKX_HIP(expr)                                                        \
    do                                                                       \
    {                                                                        \
        hipError_t e_ = (expr);                                              \
        if (e_ != hipSuccess)                                                \
        {                                                                    \
            return fail(EKX_EHIP, std::string(#expr) + ": " +                \
                                      hipGetErrorString(e_));                \
        }                                                                    \
    } while (0)

#define EKX_CHECK(expr)                                                      \
    do                                                                       \
    {                                                                        \
        ekx_status s_ = (expr);                                              \
        if (s_ != EKX_OK) { return s_; }                                     \
    } while (0)

template <typename T> struct DeviceBuffer
{
    T *ptr = nullptr;
    size_t count = 0;
    DeviceBuffer() = default;
    DeviceBuffer(const DeviceBuffer &) = delete;
    DeviceBuffer &operator=(const DeviceBuffer &) = delete;
    ~DeviceBuffer() { release(); }
    void release()
    {
        if (ptr) { (void) hipFree(ptr); }
        ptr = nullptr;
        count = 0;
    }
    ekx_status allocate(size_t n)
    {
        if (n == count && ptr) { return EKX_OK; }
        release();
        if (n == 0) { return EKX_OK; }
        hipError_t e = hipMalloc((void **) &ptr, n*sizeof(T));
        if (e != hipSuccess)
        {
            ptr = nullptr;
            return fail(EKX_ENOMEM, "hipMalloc of " +
                                        std::to_string(n*sizeof(T)) +
                                        " bytes failed: " +
                                        hipGetErrorString(e));
        }
        count = n;
        return EKX_OK;
    }
};

std::string fmt(double v)
{
    return std::to_string(v);
}

ekx_status check_geometry3d(const ekx_geometry3d *g)
{
    if (!g) { return fail(EKX_EINVAL, "geometry is NULL"); }
    // Geometry3D setters (src/geometry3d.cpp:74-261)
    if (g->nx < 3)
    {
        return fail(EKX_EINVAL, "Number of grid points in x = " +
                                    std::to_string(g->nx) +
                                    " must be at least 3");
    }
    if (g->ny < 3)
    {
        return fail(EKX_EINVAL, "Number of grid points in y = " +
                                    std::to_string(g->ny) +
                                    " must be at least 3");
    }
    if (g->nz < 3)
    {
        return fail(EKX_EINVAL, "Number of grid points in z = " +
                                    std::to_string(g->nz) +
                                    " must be at least 3");
    }
    if (!(g->dx > 0))
    {
        return fail(EKX_EINVAL, "Grid spacing in x = " + fmt(g->dx) +
                                    " must be positive");
    }
    if (!(g->dy > 0))
    {
        return fail(EKX_EINVAL, "Grid spacing in y = " + fmt(g->dy) +
                                    " must be positive");
    }
    if (!(g->dz > 0))
    {
        return fail(EKX_EINVAL, "Grid spacing in z = " + fmt(g->dz) +
                                    " must be positive");
    }
    int64_t n = (int64_t) g->nx*g->ny*g->nz;
    if (n > (int64_t) std::numeric_limits<int32_t>::max())
    {
        return fail(EKX_EINVAL, "a single grid is limited to 2^31-1 nodes");
    }
    return EKX_OK;
}

ekx_status check_options(const ekx_solver_options *o)
{
    if (!o) { return fail(EKX_EINVAL, "options is NULL"); }
    if (o->number_of_sweeps < 0 || o->number_of_sweeps > 65535)
    {
        return fail(EKX_EINVAL, "number_of_sweeps must be in [0, 65535]");
    }
    if (o->precision < EKX_PRECISION_FP64 ||
        o->precision > EKX_PRECISION_FIXED32_POLISH)
    {
        return fail(EKX_EINVAL, "unknown precision");
    }
    if (o->schedule != EKX_SCHEDULE_COMPLETED &&
        o->schedule != EKX_SCHEDULE_SHIPPED)
    {
        return fail(EKX_EINVAL, "unknown schedule");
    }
    if (o->chains < 0 || o->chains > kMaxChains)
    {
        return fail(EKX_EINVAL, "chains must be in [0, " +
                                    std::to_string(kMaxChains) + "]");
    }
    if (o->chunk_planes < 0)
    {
        return fail(EKX_EINVAL, "chunk_planes must be >= 0");
    }
    if (o->launch_order < EKX_LAUNCH_AUTO || o->launch_order > EKX_LAUNCH_QUEUE)
    {
        return fail(EKX_EINVAL, "launch_order must be 0, 1 or 2");
    }
    if (o->prefetch_planes != 0 && o->prefetch_planes != 4 &&
        o->prefetch_planes != 8 && o->prefetch_planes != 12)
    {
        return fail(EKX_EINVAL, "prefetch_planes must be 0, 4, 8 or 12");
    }
    if (o->kernel < EKX_KERNEL_AUTO || o->kernel > EKX_KERNEL_COLUMN)
    {
        return fail(EKX_EINVAL, "unknown kernel");
    }
    if (o->algorithm != EKX_LEVEL_SET_METHOD &&
        o->algorithm != EKX_FAST_SWEEPING_METHOD)
    {
        return fail(EKX_EINVAL, "unknown algorithm");
    }
    return EKX_OK;
}

// Source3D::setLocationIn{X,Y,Z} (src/source3d.cpp:161-291) and the range
// checks of Solver3D::setSource (src/solver3d.cpp:299-325); receivers are
// located the same way (Station3D, src/station3d.cpp:158-291).
struct SourceInfo
{
    double offset[3];
    int cell[3];
    int cellIndex;
};

ekx_status locate_source3d(const ekx_geometry3d &g, double x, double y,
                           double z, SourceInfo &s,
                           const char *what = "source")
{
    // messages are built on the failure paths only: a located source
    // allocates nothing
    auto pos = [&]() { return std::string(" ") + what + " position = "; };
    const double xmax = g.x0 + (g.nx - 1)*g.dx;
    const double ymax = g.y0 + (g.ny - 1)*g.dy;
    const double zmax = g.z0 + (g.nz - 1)*g.dz;
    if (x < g.x0 || x > xmax)
    {
        return fail(EKX_EINVAL, "x" + pos() + fmt(x) +
                                    " must be in range [" + fmt(g.x0) + "," +
                                    fmt(xmax) + "]");
    }
    if (y < g.y0 || y > ymax)
    {
        return fail(EKX_EINVAL, "y" + pos() + fmt(y) +
                                    " must be in range [" + fmt(g.y0) + "," +
                                    fmt(ymax) + "]");
    }
    if (z < g.z0 || z > zmax)
    {
        return fail(EKX_EINVAL, "z" + pos() + fmt(z) +
                                    " must be in range [" + fmt(g.z0) + "," +
                                    fmt(zmax) + "]");
    }
    const int ncx = g.nx - 1, ncy = g.ny - 1, ncz = g.nz - 1;
    s.offset[0] = x - g.x0;
    s.offset[1] = y - g.y0;
    s.offset[2] = z - g.z0;
    s.cell[0] = std::min(ncx - 1, (int) (s.offset[0]/g.dx));
    s.cell[1] = std::min(ncy - 1, (int) (s.offset[1]/g.dy));
    s.cell[2] = std::min(ncz - 1, (int) (s.offset[2]/g.dz));
    s.cellIndex = (s.cell[2]*ncy + s.cell[1])*ncx + s.cell[0];
    return EKX_OK;
}

// Solver3DSweep::initialize uniform test (include/private/solver3d.hpp:35-40)
bool is_uniform3d(const ekx_geometry3d &g)
{
    const double eps100 = std::numeric_limits<double>::epsilon()*100;
    return std::abs(g.dx - g.dy) < eps100 && std::abs(g.dx - g.dz) < eps100;
}

NonUniform3D non_uniform_constants(const ekx_geometry3d &g)
{
    NonUniform3D c;
    const double dx = g.dx, dy = g.dy, dz = g.dz;
    c.dxInv = 1/dx;
    c.dyInv = 1/dy;
    c.dzInv = 1/dz;
    c.dx2Inv = 1/(dx*dx);
    c.dy2Inv = 1/(dy*dy);
    c.dz2Inv = 1/(dz*dz);
    c.dx_dz = dx/dz;
    c.dz_dx = dz/dx;
    c.dy_dz = dy/dz;
    c.dz_dy = dz/dy;
    c.dx_dy = dx/dy;
    c.dy_dx = dy/dx;
    c.dx2_p_dz2_inv = 1/(dx*dx + dz*dz);
    c.dy2_p_dz2_inv = 1/(dy*dy + dz*dz);
    c.dx2_p_dy2_inv = 1/(dx*dx + dy*dy);
    return c;
}

struct HostOctant
{
    int jx0, jy0, jz0;
};

HostOctant host_octant(const Problem3D &p, int sweep, bool initialize)
{
    HostOctant o{1, 1, 1};
    if (initialize)
    {
        int negX = sweep & 1, negY = (sweep >> 1) & 1, negZ = (sweep >> 2) & 1;
        o.jx0 = negX ? std::max(p.nx - 2 - p.srcCellX, 1)
                     : std::max(1, p.srcCellX);
        o.jy0 = negY ? std::max(p.ny - 2 - p.srcCellY, 1)
                     : std::max(1, p.srcCellY);
        o.jz0 = negZ ? std::max(p.nz - 2 - p.srcCellZ, 1)
                     : std::max(1, p.srcCellZ);
    }
    return o;
}

// The column chunks of a sweep that overlap the factored box (box_columns
// in ekx_kernels3d.hip): their columns bx, by in the sweep's visiting
// order, the permuted nodes of their tiles in x and y, and per chunk bz
// its updated planes [zFirst, zEnd) (empty past the octant).
struct HostBoxChunk
{
    int bz, zFirst, zEnd;
};

struct HostBox
{
    int bxLo = 1, bxHi = 0, byLo = 1, byHi = 0;
    int64_t nxs = 0, nys = 0;
    std::vector<HostBoxChunk> chunks;
};

HostBox host_box(const Problem3D &p, int sweep, bool initialize, int chunk)
{
    HostBox b;
    if (p.radius < 0) { return b; }
    const int negX = sweep & 1, negY = (sweep >> 1) & 1;
    const int negZ = (sweep >> 2) & 1;
    int xLo = std::max(p.srcCellX - p.radius, 0);
    int xHi = std::min(p.srcCellX + p.radius, p.nx - 1);
    int yLo = std::max(p.srcCellY - p.radius, 0);
    int yHi = std::min(p.srcCellY + p.radius, p.ny - 1);
    int zLo = std::max(p.srcCellZ - p.radius, 0);
    int zHi = std::min(p.srcCellZ + p.radius, p.nz - 1);
    if (xLo > xHi || yLo > yHi || zLo > zHi) { return b; }
    int jzLo = negZ ? p.nz - 1 - zHi : zLo, jzHi = negZ ? p.nz - 1 - zLo : zHi;
    const HostOctant o = host_octant(p, sweep, initialize);
    // permuted nodes of the tiles holding grid nodes lo..hi (tiles are
    // aligned to the grid: tile t holds 8 t .. 8 t + 7), at or past j0
    auto tileSpan = [](int lo, int hi, int neg, int j0, int n)
    {
        const int tLo = lo/kColumnTile, tHi = hi/kColumnTile;
        const int gLo = tLo*kColumnTile;
        const int gHi = std::min(tHi*kColumnTile + kColumnTile - 1, n - 1);
        const int jLo = std::max(neg ? n - 1 - gHi : gLo, j0);
        const int jHi = neg ? n - 1 - gLo : gHi;
        return std::max(0, jHi - jLo + 1);
    };
    b.nxs = tileSpan(xLo, xHi, negX, o.jx0, p.nx);
    b.nys = tileSpan(yLo, yHi, negY, o.jy0, p.ny);
    const int mxLo = xLo/kColumnTile, mxHi = xHi/kColumnTile;
    const int myLo = yLo/kColumnTile, myHi = yHi/kColumnTile;
    b.bxLo = negX ? p.nTX - 1 - mxHi : mxLo;
    b.bxHi = negX ? p.nTX - 1 - mxLo : mxHi;
    b.byLo = negY ? p.nTY - 1 - myHi : myLo;
    b.byHi = negY ? p.nTY - 1 - myLo : myHi;
    for (int bz = jzLo/chunk; bz <= jzHi/chunk; ++bz)
    {
        const int zFirst = std::max(bz*chunk, o.jz0);
        const int zEnd = std::min((bz + 1)*chunk, p.nz);
        if (zFirst < zEnd) { b.chunks.push_back({bz, zFirst, zEnd}); }
    }
    return b;
}

// Updates a sweep makes with the full local update in the box chunks: the
// whole chunks when the bulk launches run them (merged), else the box end
// that the factored launches take (box_split_z).
int64_t host_box_updates(const Problem3D &p, int sweep, bool initialize,
                         int chunk, bool split)
{
    const HostBox b = host_box(p, sweep, initialize, chunk);
    const int negZ = (sweep >> 2) & 1;
    int64_t planes = 0;
    for (const HostBoxChunk &c : b.chunks)
    {
        if (!split)
        {
            planes += c.zEnd - c.zFirst;
            continue;
        }
        const BoxSplitZ bs = box_split_z(p.nz, p.srcCellZ, p.radius, negZ,
                                         c.zFirst, c.zEnd);
        planes += bs.phase == 0 ? bs.cut - c.zFirst : c.zEnd - bs.cut;
    }
    return b.nxs*b.nys*planes;
}

// Diagonals bx + by + bz on which a sweep's factored launches have work
// for problem p: bit 0 of mask[d] for the launch before the diagonal's bulk
// launch, bit 1 for the one after it (box_split_z).  Columns outside an
// initialisation sweep's octant are included (the kernel skips them).
void host_box_diagonals(const Problem3D &p, int sweep, bool initialize,
                        int chunk, std::vector<uint8_t> &mask)
{
    const HostBox b = host_box(p, sweep, initialize, chunk);
    if (b.nxs == 0 || b.nys == 0) { return; }
    const int negZ = (sweep >> 2) & 1;
    for (const HostBoxChunk &c : b.chunks)
    {
        const BoxSplitZ bs = box_split_z(p.nz, p.srcCellZ, p.radius, negZ,
                                         c.zFirst, c.zEnd);
        const int n = bs.phase == 0 ? bs.cut - c.zFirst : c.zEnd - bs.cut;
        if (n <= 0) { continue; }
        for (int bx = b.bxLo; bx <= b.bxHi; ++bx)
        {
            for (int by = b.byLo; by <= b.byHi; ++by)
            {
                const size_t d = (size_t) (bx + by + c.bz);
                if (d < mask.size()) { mask[d] |= (uint8_t) (1u << bs.phase); }
            }
        }
    }
}

} // namespace

namespace ekx
{
void set_last_error(const std::string &message) { g_error = message; }

void set_last_error_nothrow(const char *message) noexcept
{
    try
    {
        g_error = message;
    }
    catch (...)
    {
        g_error.clear();
    }
}
} // namespace ekx

// ===========================================================================
// Allocation-free solves: the problem descriptors of a call live in this
// device array (one copy per GPU, EKX_NOALLOC_MAX_SOURCES descriptors,
// about 18 KB), whose address on each device is looked up once.
// ===========================================================================
static __device__ __align__(256) Problem3D scratch[EKX_NOALLOC_MAX_SOURCES];

namespace
{
constexpr int kMaxDevices = 64;
std::mutex g_scratchMutex;
Problem3D *g_scratchAddress[kMaxDevices] = {};

// The scratch array's address on the current device (hipGetSymbolAddress
// on the first call with that device current; the symbol's host-side name
// is no device address).
ekx_status scratch_address(Problem3D **out)
{
    int device = 0;
    EKX_HIP(hipGetDevice(&device));
    if (device < 0 || device >= kMaxDevices)
    {
        return fail(EKX_EINVAL, "device index out of range");
    }
    std::lock_guard<std::mutex> lock(g_scratchMutex);
    if (g_scratchAddress[device] == nullptr)
    {
        void *ptr = nullptr;
        EKX_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        g_scratchAddress[device] = static_cast<Problem3D *>(ptr);
    }
    *out = g_scratchAddress[device];
    return EKX_OK;
}
} // namespace

namespace
{
// Held shared by captures in progress: the device cannot be synchronised
// meanwhile.
std::shared_mutex g_captures;
// Waves of flow launches in progress per device.
FlowWaves g_flowWaves[kMaxDevices];
} // namespace

// ===========================================================================
// Engine3D: a batch of 3D problems and the schedule that solves them.
// ===========================================================================
struct Engine3D
{
    ekx_solver_options opt{};
    std::vector<ekx_geometry3d> geometry;
    std::vector<Problem3D> problems;
    std::vector<SourceInfo> sources;
    std::vector<bool> haveSource;
    std::vector<int> modelOf;        // problem -> model
    std::vector<int64_t> modelOffset;
    int64_t totalNodes = 0, totalCells = 0, maxNodes = 0;
    std::vector<int64_t> modelCells;
    // Fields are tiled for the column kernel (tile records and edge
    // records per problem, tCount elements from tOffset) and natural for
    // the hyperplane kernel.  Models: natural cells (S*), and for the
    // column kernel also slowness bricks (SB*, from sbOffset per model).
    bool tiled = true;
    int64_t maxCount = 0, totalBricks = 0;
    std::vector<int64_t> modelBrickOffset;
    DeviceBuffer<double> S64;
    DeviceBuffer<float> S32;
    DeviceBuffer<double> T64;
    DeviceBuffer<float> T32;
    // scaled-integer storage (FIXED32 modes)
    DeviceBuffer<uint32_t> SQ;
    DeviceBuffer<uint32_t> TQ;
    DeviceBuffer<double> SB64;
    DeviceBuffer<float> SB32;
    DeviceBuffer<uint32_t> SBQ;
    // natural-order copy of one problem's field (device pointer access)
    mutable DeviceBuffer<double> natural64;
    mutable DeviceBuffer<float> natural32;
    mutable DeviceBuffer<uint32_t> naturalQ;
    mutable int naturalProblem = -1;
    mutable uint64_t naturalStamp = 0;
    DeviceBuffer<double> partial;
    // smallest and largest slowness of each model
    std::vector<double> modelSMin, modelSMax;
    DeviceBuffer<Problem3D> dProblems;
    DeviceBuffer<ColumnItem> dItems;
    // Column items ordered by chain, then diagonal bx + by: chain c's items
    // of diagonal d are [diagStart[c*(nDiag+1)+d], ...[+d+1]).  A chain is
    // a contiguous range of problems [chainBegin[c], chainBegin[c+1]).
    std::vector<int> diagStart;
    int nDiag = 0;
    int chunkH = 1;      // planes per z-chunk (>= nz: whole columns)
    int nChains = 1;
    // the bulk launches run the box chunks (chunks shorter than
    // kMergedMaxChunk planes)
    bool mergedSmall = false;
    static constexpr int kMergedMaxChunk = 64;
    static constexpr int kMergedMaxChunk64 = 80;    // FP64, default shapes
    // the autotuner's choice (0: none)
    int tunedChunk = 0, tunedChains = 0;
    std::vector<int> chainBegin;
    std::vector<hipStream_t> chainStreams;
    std::vector<hipEvent_t> chainEvents;
    // Upper bound, over any source position, of the column chunks of one
    // problem that overlap its factored box on one diagonal: the box spans
    // at most ceil((2r+1)/8)+1 columns per axis, and each (bx, by) meets a
    // diagonal at one bz at most.
    int boxPerDiag = 0;
    // Work-queue sweeps (launch order QUEUE): per problem the first
    // completion flag of its column chunks (flag of chunk (bx, by, bz):
    // base + (bz*nTY + by)*nTX + bx); queueWords holds the flags, one item
    // counter per chain and sweep of a sequence, then the error word.
    DeviceBuffer<int> dFlagBase;
    DeviceBuffer<unsigned int> queueWords;
    int64_t queueFlags = 0;
    int queueMaxSweeps = 0;
    int queueWaves = 0;          // column waves the device keeps resident
    uint64_t queueWaitTicks = 0; // bound of one dependency wait
    int clockKHz = 0;            // rate of the device's wall clock
    // Flow launches (a whole solve in one launch, every column resident):
    // the columns of all problems in launch order and, per element type
    // swept, two buffers of step records and four of mail; the error word
    // and each column's XCD.  No columns: not for this setup.
    std::vector<FlowColumn> flowColumns;
    DeviceBuffer<FlowColumn> dFlowColumns;
    DeviceBuffer<double> flowRec64, flowMail64;
    DeviceBuffer<float> flowRec32, flowMail32;
    DeviceBuffer<unsigned int> flowWords;
    int flowWaves = 0;           // columns without the placeholders
    int64_t flowRecCount = 0, flowMailCount = 0;
    int flowCapacity = 0;        // waves that the device holds together
    int flowMaxNz = 0;
    int64_t flowSteps = 0;       // flow_chain of all waves
    int64_t flowChain = 0;       // and of the longest
    double flowWaitMs = -1;      // a caller's bound of one wait
    // work counts of the flow launches: with the initialisation sweeps, and
    // of the FP64 polish
    struct Counts
    {
        // what st counts for
        int iterations = -1, chunk = 0;
        uint64_t sourceStamp = 0;
        ekx_solve_stats st{};
    };
    Counts flowCounts[2];
    bool flowUniform = false;
    hipStream_t stream = nullptr;
    hipEvent_t evFork = nullptr;
    hipEvent_t evStart = nullptr, evStop = nullptr;
    // kernel_timing: event pairs around the bulk column launches
    std::vector<hipEvent_t> timingEvents;
    size_t timingUsed = 0;
    bool timing = false;
    // early_exit: the largest decrease of the running iteration (float
    // bits, atomic max), and its host copy
    DeviceBuffer<unsigned int> change;
    unsigned int *changeHost = nullptr;
    // segment events: [0,1] FP32 sweeps, [2,3] FP64 sweeps
    hipEvent_t evSeg[4] = {nullptr, nullptr, nullptr, nullptr};
    // The sweeps of one precision, captured once and replayed per solve.
    struct Segment
    {
        hipGraph_t graph = nullptr;
        hipGraphExec_t exec = nullptr;
        bool valid = false;
        ekx_solve_stats st{};
        uint64_t sourceStamp = 0;       // the sources that st counts for
        void release()
        {
            if (exec) { (void) hipGraphExecDestroy(exec); }
            if (graph) { (void) hipGraphDestroy(graph); }
            exec = nullptr;
            graph = nullptr;
            valid = false;
        }
    };
    // [0] primary sweeps, [1] FP64 polish sweeps; early exit: [2] primary
    // initialisation sweeps, [3] one primary refinement iteration
    Segment segment[4];
    bool haveModel = false;
    bool haveField = false;
    bool fieldIsF64 = true;
    ekx_solve_stats stats{};
    // Count of completed solves: derived results record the solve they
    // were computed from.
    uint64_t solveStamp = 0;
    uint64_t sourceStamp = 0;    // count of moves of a source cell
    // Receivers: nStations per problem, located in every problem's grid
    // (dStations is [problem][station]); their travel times after the
    // solve numbered stationStamp.
    int nStations = 0;
    DeviceBuffer<StationLoc3D> dStations;
    DeviceBuffer<double> stationOut;
    std::vector<double> stationTimes;
    uint64_t stationStamp = 0;
    // Travel-time gradient (3 values per node) of one problem's field.
    DeviceBuffer<double> G;
    int gradientProblem = -1;
    uint64_t gradientStamp = 0;

    ~Engine3D()
    {
        drop_graph();
        if (evStart) { (void) hipEventDestroy(evStart); }
        if (evStop) { (void) hipEventDestroy(evStop); }
        if (evFork) { (void) hipEventDestroy(evFork); }
        for (hipEvent_t &e : timingEvents) { (void) hipEventDestroy(e); }
        for (hipEvent_t &e : chainEvents) { (void) hipEventDestroy(e); }
        for (hipStream_t &c : chainStreams) { (void) hipStreamDestroy(c); }
        if (changeHost) { (void) hipHostFree(changeHost); }
        for (hipEvent_t &e : evSeg)
        {
            if (e) { (void) hipEventDestroy(e); }
        }
        if (stream) { (void) hipStreamDestroy(stream); }
    }

    void drop_graph()
    {
        for (Segment &g : segment) { g.release(); }
    }
    bool early_exit() const
    {
        return opt.early_exit != 0 &&
               opt.schedule == EKX_SCHEDULE_COMPLETED;
    }

    bool sweeps_f64() const
    {
        return opt.precision == EKX_PRECISION_FP64;
    }
    bool fixed32() const
    {
        return opt.precision == EKX_PRECISION_FIXED32 ||
               opt.precision == EKX_PRECISION_FIXED32_POLISH;
    }
    bool polish() const
    {
        return (opt.precision == EKX_PRECISION_FP32_POLISH ||
                opt.precision == EKX_PRECISION_FIXED32_POLISH) &&
               opt.schedule == EKX_SCHEDULE_COMPLETED &&
               opt.number_of_sweeps >= 1;
    }
    int depth() const
    {
        return opt.prefetch_planes > 0 ? opt.prefetch_planes : 4;
    }
    int kernel() const
    {
        return opt.kernel == EKX_KERNEL_AUTO ? EKX_KERNEL_COLUMN : opt.kernel;
    }
    // Sweeps of FP64 fields by the column kernel in work-queue form (its
    // waves run the factored-box chunks in place).
    template <typename TS> bool queued() const
    {
        return kernel() == EKX_KERNEL_COLUMN && sizeof(TS) == 8 &&
               opt.launch_order == EKX_LAUNCH_QUEUE;
    }

    // Whether all sweeps of a solve take that form.
    bool queued_primary() const { return sweeps_f64() && queued<double>(); }

    // Allocates buffers and the column work lists for the given geometries;
    // modelOf maps every problem to one of nModels models.
    ekx_status setup(const ekx_solver_options &o,
                     const std::vector<ekx_geometry3d> &geoms,
                     const std::vector<int> &models, int nModels)
    {
        drop_graph();
        opt = o;
        geometry = geoms;
        modelOf = models;
        const int n = (int) geoms.size();
        problems.assign(n, Problem3D{});
        sources.assign(n, SourceInfo{});
        haveSource.assign(n, false);
        haveModel = false;
        haveField = false;
        stats = ekx_solve_stats{};
        nStations = 0;
        stationTimes.clear();
        gradientProblem = -1;
        tunedChunk = tunedChains = 0;
        if (!stream)
        {
            EKX_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
            EKX_HIP(hipEventCreate(&evStart));
            EKX_HIP(hipEventCreate(&evStop));
            EKX_HIP(hipEventCreateWithFlags(&evFork,
                                            hipEventDisableTiming));
            for (hipEvent_t &e : evSeg) { EKX_HIP(hipEventCreate(&e)); }
        }
        // model offsets (cells)
        modelOffset.assign(nModels, -1);
        modelCells.assign(nModels, 0);
        modelSMin.assign(nModels, 0.0);
        modelSMax.assign(nModels, 0.0);
        EKX_CHECK(partial.allocate((size_t) nModels*2*kRangeBlocks));
        totalCells = 0;
        for (int i = 0; i < n; ++i)
        {
            int m = modelOf[i];
            if (modelOffset[m] < 0)
            {
                modelOffset[m] = totalCells;
                const ekx_geometry3d &g = geoms[i];
                modelCells[m] = (int64_t) (g.nx - 1)*(g.ny - 1)*(g.nz - 1);
                totalCells += modelCells[m];
            }
        }
        tiled = kernel() == EKX_KERNEL_COLUMN;
        modelBrickOffset.assign(nModels, -1);
        totalBricks = 0;
        // guard space before the first and after the last problem's
        // records (the column kernel's unchecked halo addresses)
        totalNodes = tiled ? kFieldGuard : 0;
        maxNodes = 0;
        maxCount = 0;
        for (int i = 0; i < n; ++i)
        {
            const ekx_geometry3d &g = geoms[i];
            Problem3D &p = problems[i];
            p.tiled = tiled ? 1 : 0;
            p.nTX = tiles_of(g.nx);
            p.nTY = tiles_of(g.ny);
            p.scaled = 0;
            const int64_t nTiles = (int64_t) p.nTX*p.nTY;
            const int m = modelOf[i];
            if (modelBrickOffset[m] < 0)
            {
                modelBrickOffset[m] = totalBricks;
                totalBricks += kBrickVariants*
                               brick_variant_values(g.nx, g.ny, g.nz);
            }
            p.sbOffset = modelBrickOffset[m];
            p.nx = g.nx;
            p.ny = g.ny;
            p.nz = g.nz;
            p.radius = o.factored_radius;
            p.uniform = is_uniform3d(g) ? 1 : 0;
            p.dx = g.dx;
            p.dy = g.dy;
            p.dz = g.dz;
            p.tOffset = totalNodes;
            p.sOffset = modelOffset[modelOf[i]];
            p.nu = non_uniform_constants(g);
            int64_t nodes = (int64_t) g.nx*g.ny*g.nz;
            p.tCount = tiled ? nTiles*g.nz*(kTileValues + kEdgeValues) : nodes;
            p.eOffset = p.tOffset + (tiled ? nTiles*g.nz*kTileValues : 0);
            totalNodes += p.tCount;
            maxNodes = std::max(maxNodes, nodes);
            maxCount = std::max(maxCount, p.tCount);
        }
        if (tiled) { totalNodes += kFieldGuard; }
        naturalProblem = -1;
        EKX_CHECK(S64.allocate((size_t) totalCells));
        const bool fp32 = !sweeps_f64() && !fixed32();
        if (fp32) { EKX_CHECK(S32.allocate((size_t) totalCells)); }
        else { S32.release(); }
        // bricks of the element types the sweeps read
        if (tiled && (sweeps_f64() || polish()))
        {
            EKX_CHECK(SB64.allocate((size_t) totalBricks));
        }
        else { SB64.release(); }
        if (tiled && fp32) { EKX_CHECK(SB32.allocate((size_t) totalBricks)); }
        else { SB32.release(); }
        if (tiled && fixed32())
        {
            EKX_CHECK(SBQ.allocate((size_t) totalBricks));
        }
        else { SBQ.release(); }
        if (fixed32())
        {
            EKX_CHECK(SQ.allocate((size_t) totalCells));
            EKX_CHECK(TQ.allocate((size_t) totalNodes));
            EKX_HIP(hipMemsetAsync(TQ.ptr, 0, TQ.count*sizeof(uint32_t),
                                   stream));
        }
        else
        {
            SQ.release();
            TQ.release();
        }
        if (sweeps_f64() || polish())
        {
            EKX_CHECK(T64.allocate((size_t) totalNodes));
            EKX_HIP(hipMemsetAsync(T64.ptr, 0, T64.count*sizeof(double),
                                   stream));
        }
        else { T64.release(); }
        if (fp32)
        {
            EKX_CHECK(T32.allocate((size_t) totalNodes));
            EKX_HIP(hipMemsetAsync(T32.ptr, 0, T32.count*sizeof(float),
                                   stream));
        }
        else { T32.release(); }
        fieldIsF64 = sweeps_f64() || polish();
        EKX_CHECK(dProblems.allocate((size_t) n));
        if (early_exit())
        {
            EKX_CHECK(change.allocate(1));
            if (!changeHost)
            {
                EKX_HIP(hipHostMalloc((void **) &changeHost,
                                      sizeof(unsigned int),
                                      hipHostMallocDefault));
            }
        }
        else { change.release(); }
        EKX_CHECK(build_schedule());
        EKX_CHECK(setup_flow());
        EKX_HIP(hipStreamSynchronize(stream));
        return EKX_OK;
    }

    // Flow launches serve the default launch shape (a caller who names one
    // gets it) of the completed schedule in FP64 and FP32 arithmetic on
    // FP64 and FP32 fields (mail keeps its tag in the sign bit, which the
    // scaled integers use), for problems that each fit the device's resident
    // waves.  There the sweeps are a chain of dependent steps, which a launch
    // per diagonal lengthens: 257 x 257 x 193 FP64 50.9 ms by diagonals, 14.3
    // ms in one launch.
    // With more columns than waves the problems follow each other through
    // the device, the longest chains first: a column waits only for columns
    // of its own problem, and workgroups of an XCD start in launch order, so
    // the first unfinished problem always becomes resident as a whole.  That
    // is faster than the diagonals
    // until these have enough columns to fill the chip: measured on FP64
    // grids of 64 to 200 nodes a side, by the ratio of all the waves' steps
    // to what the device runs in the longest chain: 1.2 27.5 -> 15.3 ms, 2.0
    // 61.4 -> 33.0, 2.6 69.9 -> 63.6, 3.3 37.1 -> 32.4, 3.75 27.3 -> 26.0,
    // 4.0 67.3 -> 72.7, 5.0 38.7 -> 45.0.  So up to 7/2.
    // Memory that the device does not have for the buffers is no error: the
    // diagonals need none of it.
    static constexpr int64_t kFlowLoad2 = 7;

    // The bound of one wait in a flow launch of nSweeps sweeps, in the
    // device's wall clock.  With every column resident a wait lasts a few
    // traversals of a problem at most; otherwise a column may wait until the
    // problems before its own have done all their sweeps, which is the
    // launch's whole time.  At 4 us a step (0.5 to 1.5 measured), 4 traversals,
    // and at least 250 ms, so that a device shared with other work does not
    // trip it.
    uint64_t flow_wait_ticks(int nSweeps) const
    {
        if (flowWaitMs >= 0) { return (uint64_t) (clockKHz*flowWaitMs); }
        constexpr double kStepMs = 4e-3;
        double steps = 2*(double) flowChain;
        if (flowWaves > flowCapacity) { steps += nSweeps*flow_steps(); }
        return (uint64_t) (clockKHz*std::max(250.0, kStepMs*steps));
    }

    // Steps that a sweep of the launch takes.
    double flow_steps() const
    {
        const double chain = 0.5*(double) flowChain;
        return flowWaves > flowCapacity
                   ? 0.5*(double) flowSteps/flowCapacity + chain : chain;
    }

    ekx_status set_wait_bound(double ms)
    {
        if (ms > 1e9)
        {
            return fail(EKX_EINVAL, "wait bound must be at most 1e9 ms");
        }
        flowWaitMs = ms;
        return EKX_OK;
    }

    // Twice the steps that a wave of problem p spends in a sweep, waits for
    // the hops to its columns included (a hop is 10.6 steps; x reverses in
    // every sweep, y in every second).
    static int64_t flow_chain(const Problem3D &p)
    {
        return 2*(p.nz + kColumnSkew) + 21*(p.nTX - 1) + 11*(p.nTY - 1);
    }

    ekx_status setup_flow()
    {
        flowColumns.clear();
        flowWaitMs = -1;
        flowCounts[0] = flowCounts[1] = Counts{};
        const ekx_solver_options &o = opt;
        const bool wanted =
            kernel() == EKX_KERNEL_COLUMN && !fixed32() && !early_exit() &&
            o.schedule == EKX_SCHEDULE_COMPLETED && o.kernel_timing == 0 &&
            o.launch_order == EKX_LAUNCH_AUTO && o.chunk_planes == 0 &&
            o.chains == 0 && o.prefetch_planes == 0;
        int device = 0, cus = 0;
        int64_t most = 0;               // columns of one problem
        int uniform = 0;
        flowMaxNz = 0;
        flowSteps = flowChain = 0;
        for (const Problem3D &p : problems)
        {
            const int64_t columns = (int64_t) p.nTX*p.nTY;
            most = std::max(most, columns);
            flowSteps += columns*flow_chain(p);
            flowChain = std::max(flowChain, flow_chain(p));
            uniform += p.uniform;
            flowMaxNz = std::max(flowMaxNz, p.nz);
        }
        flowUniform = uniform > 0;
        bool fits = wanted &&
                    (uniform == 0 || uniform == (int) problems.size());
        if (fits && hipGetDevice(&device) == hipSuccess &&
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount,
                                  device) == hipSuccess)
        {
            int perCU = 1 << 20;
            if (sweeps_f64() || polish())
            {
                perCU = flow_waves_per_cu<double>(flowUniform);
            }
            if (!sweeps_f64())
            {
                perCU = std::min(perCU, flow_waves_per_cu<float>(flowUniform));
            }
            flowCapacity = perCU*cus;
            fits = most <= flowCapacity &&
                   2*flowSteps <= kFlowLoad2*flowCapacity*flowChain;
        }
        else { fits = false; }
        int64_t rec = 0, mail = 0;
        std::vector<FlowColumn> list;
        for (size_t i = 0; fits && i < problems.size(); ++i)
        {
            const Problem3D &p = problems[i];
            for (int my = 0; my < p.nTY; ++my)
            {
                for (int mx = 0; mx < p.nTX; ++mx)
                {
                    list.push_back(FlowColumn{
                        (int) i, mx, my, (int) list.size(), rec + kFlowPad*kTileValues,
                        mail + kMailPad*kMailValues});
                    rec += (int64_t) flow_records(p.nz)*kTileValues;
                    mail += (int64_t) flow_mails(p.nz)*kMailValues;
                }
            }
        }
        std::vector<FlowColumn> placed;
        if (fits) { placed = place_columns(list); }
        // (byte offsets into a mail buffer are 32 bits)
        fits = fits && mail*8 < ((int64_t) 1 << 31);
        flowRecCount = rec;
        flowMailCount = mail;
        const bool f64 = fits && (sweeps_f64() || polish());
        const bool f32 = fits && !sweeps_f64();
        const bool have =
            flowRec64.allocate(f64 ? 2*(size_t) rec : 0) == EKX_OK &&
            flowMail64.allocate(f64 ? kMailBuffers*(size_t) mail : 0) == EKX_OK &&
            flowRec32.allocate(f32 ? 2*(size_t) rec : 0) == EKX_OK &&
            flowMail32.allocate(f32 ? kMailBuffers*(size_t) mail : 0) == EKX_OK &&
            dFlowColumns.allocate(fits ? placed.size() : 0) == EKX_OK &&
            flowWords.allocate(fits ? 1 + list.size() : 0) == EKX_OK;
        if (!fits || !have)
        {
            if (!have) { (void) hipGetLastError(); }
            release_flow();
            return EKX_OK;
        }
        flowColumns = placed;
        flowWaves = (int) list.size();
        EKX_HIP(hipMemcpyAsync(dFlowColumns.ptr, flowColumns.data(),
                               placed.size()*sizeof(FlowColumn),
                               hipMemcpyHostToDevice, stream));
        return EKX_OK;
    }

    // The launch order of the columns.  Workgroups (one column each) go to
    // the 8 XCDs round-robin by index, and on an XCD to one CU after the
    // other, then to the next SIMD of each.  So a problem's columns are cut
    // into contiguous runs, one per XCD, so that most neighbours exchange
    // their mail through one L2; a run of up to a column per CU stays on one
    // XCD (33 x 29 x 25, 20 columns: 0.68 ms per iteration on one XCD, 0.72
    // on eight), a longer one is cheaper spread (129^3, 289 columns: 1.62 ms
    // on three, 1.51 on eight).  Within a run x first: columns that share a
    // CU are then far apart in x, and seldom busy together (257 x 257 x 193:
    // 3.46 ms; in rows of y, where they are neighbours on a diagonal, 4.54).
    // What runs where changes no result.
    std::vector<FlowColumn> place_columns(
        const std::vector<FlowColumn> &list) const
    {
        constexpr size_t kXcds = 8, kCusPerXcd = 32;
        // each problem's columns, the longest chain first
        std::vector<size_t> begin(problems.size() + 1, 0);
        for (const FlowColumn &c : list) { ++begin[c.problem + 1]; }
        std::partial_sum(begin.begin(), begin.end(), begin.begin());
        std::vector<int> byChain(problems.size());
        std::iota(byChain.begin(), byChain.end(), 0);
        std::stable_sort(byChain.begin(), byChain.end(), [&](int a, int b)
                         { return flow_chain(problems[a]) >
                                  flow_chain(problems[b]); });
        std::vector<FlowColumn> onXcd[kXcds];
        for (int i : byChain)
        {
            size_t first = begin[i];
            const size_t end = begin[i + 1], n = end - first;
            const size_t per = std::max((n + kXcds - 1)/kXcds,
                                        std::min(n, kCusPerXcd));
            // the least loaded XCDs first
            size_t order[kXcds];
            for (size_t x = 0; x < kXcds; ++x) { order[x] = x; }
            std::stable_sort(order, order + kXcds, [&](size_t a, size_t b)
                             { return onXcd[a].size() < onXcd[b].size(); });
            for (size_t x = 0; first < end; ++x)
            {
                const size_t m = std::min(per, end - first);
                std::vector<FlowColumn> &to = onXcd[order[x]];
                to.insert(to.end(), list.begin() + first,
                          list.begin() + first + m);
                std::stable_sort(to.end() - m, to.end(),
                                 [](const FlowColumn &a, const FlowColumn &b)
                                 { return a.mx < b.mx; });
                first += m;
            }
        }
        size_t longest = 0;
        for (const auto &l : onXcd) { longest = std::max(longest, l.size()); }
        std::vector<FlowColumn> placed(kXcds*longest,
                                       FlowColumn{-1, 0, 0, 0, 0, 0});
        for (size_t x = 0; x < kXcds; ++x)
        {
            for (size_t k = 0; k < onXcd[x].size(); ++k)
            {
                placed[k*kXcds + x] = onXcd[x][k];
            }
        }
        return placed;
    }

    void release_flow()
    {
        flowColumns.clear();
        dFlowColumns.release();
        flowRec64.release();
        flowMail64.release();
        flowRec32.release();
        flowMail32.release();
        flowWords.release();
    }

    // Whether this solve can run as flow launches; takes their waves: as if
    // every XCD had as many as the one with most, so that the columns of
    // launches that run together are resident on each.  Beside other threads'
    // it waits for its turn, as long as the solve by diagonals takes (four
    // times its own time, at 0.6 us a step), and then goes by diagonals: 257 x
    // 257 x 97 on 3 threads, ms a solve: 12.6 when it went there at once, 8.2
    // so, 11.3 all by diagonals; on 8 threads 15.0, 10.0 and 16.1.
    bool take_flow(FlowReservation &r, int nSweeps) const
    {
        if (flowColumns.empty()) { return false; }
        for (const Problem3D &p : problems)
        {
            if (!p.scaled) { return false; }
        }
        int device = 0;
        return hipGetDevice(&device) == hipSuccess && device >= 0 &&
               device < kMaxDevices &&
               r.take(g_flowWaves[device],
                      std::min((int) flowColumns.size(), flowCapacity),
                      flowCapacity, std::chrono::duration<double>(
                          4*0.6e-6*nSweeps*flow_steps()));
    }

    template <typename TS> DeviceBuffer<TS> &flow_records_buffer()
    {
        if constexpr (sizeof(TS) == 8) { return flowRec64; }
        else { return flowRec32; }
    }
    template <typename TS> DeviceBuffer<TS> &flow_mail_buffer()
    {
        if constexpr (sizeof(TS) == 8) { return flowMail64; }
        else { return flowMail32; }
    }

    // The sweeps of one precision segment in one launch, from the source
    // initialisation (doInit) or from the tiled field, to the tiled field.
    template <typename TS>
    ekx_status run_flow(TS *T, bool doInit, int iterations,
                        ekx_solve_stats &st)
    {
        const int n = (int) flowColumns.size();
        TS *rec = flow_records_buffer<TS>().ptr;
        TS *mail = flow_mail_buffer<TS>().ptr;
        const int nInit = doInit ? 8 : 0;
        const int nSweeps = nInit + 8*iterations;
        // the segment's counts, which follow the sources' cells (counting
        // 24 sweeps of 4096 problems takes 2 ms)
        Counts &c = flowCounts[doInit ? 0 : 1];
        if (c.iterations != iterations || c.chunk != chunkH ||
            c.sourceStamp != sourceStamp)
        {
            c = Counts{iterations, chunkH, sourceStamp, ekx_solve_stats{}};
            count_segment<TS>(doInit, iterations, c.st);
        }
        st.updates += c.st.updates;
        st.updates_fp64 += c.st.updates_fp64;
        st.updates_factored += c.st.updates_factored;
        st.iterations_run += iterations;
        EKX_HIP(launch_clear_words(flowWords.ptr + (doInit ? 0 : 1),
                                   flowWaves + (doInit ? 1 : 0), stream));
        EKX_HIP(launch_clear_words(
            reinterpret_cast<unsigned int *>(mail),
            kMailBuffers*flowMailCount*
                (int64_t) (sizeof(TS)/sizeof(unsigned int)),
            stream));
        if (doInit)
        {
            EKX_HIP(launch_flow_init<TS>(dProblems.ptr, dFlowColumns.ptr, n,
                                         flowMaxNz, rec, stream));
        }
        else
        {
            EKX_HIP(launch_flow_copy<TS>(dProblems.ptr, dFlowColumns.ptr, n,
                                         flowMaxNz, 0, true, rec, T, stream));
        }
        EKX_HIP(launch_flow3d<TS>(
            dProblems.ptr, dFlowColumns.ptr, n, nInit, nSweeps, rec,
            flowRecCount, mail, flowMailCount, bricks<TS>(), flowUniform,
            flowWords.ptr, flowWords.ptr + 1, flow_wait_ticks(nSweeps),
            stream));
        EKX_HIP(launch_flow_copy<TS>(
            dProblems.ptr, dFlowColumns.ptr, n, flowMaxNz, nSweeps & 7, false,
            rec + (nSweeps & 1)*flowRecCount, T, stream));
        st.kernel_launches += 1;
        if (sizeof(TS) == 8) { st.kernel_launches_fp64 += 1; }
        return EKX_OK;
    }

    // Appends one diagonal's items to the list in an XCD-aware order.
    // Workgroups go to the 8 XCDs round-robin by index, each XCD with its
    // own L2: the items are sorted by column position (bz, by, bx), then
    // problem, dealt into 8 contiguous, equal runs, one per XCD, and
    // interleaved block by block (W items per workgroup), so that the
    // problems of a chain that share a model read each column's slowness
    // bricks on one XCD, at most two where a run ends.  Runs that come out
    // short are padded with placeholder items (problem -1) that the
    // kernels skip.
    void xcd_order(std::vector<ColumnItem> &d,
                   std::vector<ColumnItem> &out) const
    {
        constexpr int kXcds = 8;
        const int W = sweeps_f64() ? column_waves<double>()
                    : fixed32()    ? column_waves<uint32_t>()
                                   : column_waves<float>();
        const int n = (int) d.size();
        if (n == 0) { return; }
        std::stable_sort(d.begin(), d.end(),
                         [](const ColumnItem &a, const ColumnItem &b)
                         {
                             if (a.bz != b.bz) { return a.bz < b.bz; }
                             if (a.by != b.by) { return a.by < b.by; }
                             return a.bx < b.bx;
                         });
        // run x: items [x*per, min((x+1)*per, n)), per a whole number of
        // workgroups
        const int blocks = (n + W - 1)/W;
        const int perBlocks = (blocks + kXcds - 1)/kXcds;
        const int per = perBlocks*W;
        const ColumnItem none{-1, 0, 0, 0};
        for (int m = 0; m < perBlocks; ++m)
        {
            for (int x = 0; x < kXcds; ++x)
            {
                for (int w = 0; w < W; ++w)
                {
                    const int i = x*per + m*W + w;
                    out.push_back(i < n ? d[i] : none);
                }
            }
        }
        // trailing placeholders carry no work: drop them
        while (!out.empty() && out.back().problem < 0) { out.pop_back(); }
    }

    int default_chains() const
    {
        const int n = (int) geometry.size();
        return opt.chains > 0 ? std::min(opt.chains, n)
                              : (n >= 16 ? std::min(4, n) : 1);
    }

    // The launch schedule of the current options: chains, the z-chunk
    // depth and the column-chunk work lists by chain and diagonal.
    ekx_status build_schedule()
    {
        // Chains: contiguous ranges of problems with about equal work
        // (node count).  One chain unless the batch is large enough to
        // keep several independent launch sequences busy.
        const ekx_solver_options &o = opt;
        const std::vector<ekx_geometry3d> &geoms = geometry;
        const int n = (int) geoms.size();
        int64_t naturalNodes = 0;
        for (const ekx_geometry3d &g : geoms)
        {
            naturalNodes += (int64_t) g.nx*g.ny*g.nz;
        }
        nChains = tunedChains > 0 ? std::min(tunedChains, n)
                                  : default_chains();
        if (kernel() != EKX_KERNEL_COLUMN) { nChains = 1; }
        chainBegin.assign(1, 0);
        {
            int64_t done = 0;
            for (int i = 0; i < n; ++i)
            {
                const ekx_geometry3d &g = geoms[i];
                done += (int64_t) g.nx*g.ny*g.nz;
                int c = (int) chainBegin.size();      // chain being filled
                if (c < nChains &&
                    done*nChains >= naturalNodes*(int64_t) c && i + 1 < n)
                {
                    chainBegin.push_back(i + 1);
                }
            }
            chainBegin.push_back(n);
            nChains = (int) chainBegin.size() - 1;
        }
        while ((int) chainStreams.size() < nChains)
        {
            hipStream_t cs = nullptr;
            hipEvent_t ce = nullptr;
            EKX_HIP(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
            EKX_HIP(hipEventCreateWithFlags(&ce, hipEventDisableTiming));
            chainStreams.push_back(cs);
            chainEvents.push_back(ce);
        }
        // Column-chunk work lists by chain, then diagonal bx + by + bz.
        int maxNz = 0;
        for (int i = 0; i < n; ++i) { maxNz = std::max(maxNz, geoms[i].nz); }
        // The bulk launches also run the box columns when the chunks are
        // short (short launches, where a second launch per diagonal costs
        // more than the lower occupancy of that instance); with long chunks
        // (the tables' whole columns) the launches are long and occupancy
        // counts.  The chunk depth is chosen for that instance's
        // occupancy and kept when the separate instances take over: asked
        // again at their higher occupancy the size-class rule would pick
        // shorter chunks, which measured slower.
        chunkH = tunedChunk > 0       ? std::min(tunedChunk, maxNz)
                 : o.chunk_planes > 0 ? std::min(o.chunk_planes, maxNz)
                                      : even_chunk(auto_chunk(geoms, maxNz),
                                                   maxNz);
        // (64 FP64 sources on 385 x 385 x 193, chunks of 65: 164 ms with
        // launches of their own for the box, 154 without; FP32 108 and 115)
        mergedSmall = chunkH < kMergedMaxChunk ||
                      (sweeps_f64() && o.chunk_planes == 0 &&
                       o.prefetch_planes == 0 && chunkH < kMergedMaxChunk64);
        nDiag = 0;
        for (int i = 0; i < n; ++i)
        {
            const ekx_geometry3d &g = geoms[i];
            int nbx = (g.nx + kColumnTile - 1)/kColumnTile;
            int nby = (g.ny + kColumnTile - 1)/kColumnTile;
            int nbz = (g.nz + chunkH - 1)/chunkH;
            nDiag = std::max(nDiag, nbx + nby + nbz - 2);
        }
        std::vector<ColumnItem> flat;
        diagStart.clear();
        for (int c = 0; c < nChains; ++c)
        {
            std::vector<std::vector<ColumnItem>> perDiag(nDiag);
            for (int i = chainBegin[c]; i < chainBegin[c + 1]; ++i)
            {
                const ekx_geometry3d &g = geoms[i];
                int nbx = (g.nx + kColumnTile - 1)/kColumnTile;
                int nby = (g.ny + kColumnTile - 1)/kColumnTile;
                int nbz = (g.nz + chunkH - 1)/chunkH;
                for (int bz = 0; bz < nbz; ++bz)
                {
                    for (int by = 0; by < nby; ++by)
                    {
                        for (int bx = 0; bx < nbx; ++bx)
                        {
                            perDiag[bx + by + bz].push_back(
                                ColumnItem{i, bx, by, bz});
                        }
                    }
                }
            }
            for (auto &d : perDiag)
            {
                diagStart.push_back((int) flat.size());
                xcd_order(d, flat);
            }
            diagStart.push_back((int) flat.size());
        }
        boxPerDiag = 0;
        if (o.factored_radius >= 0)
        {
            // a box 2r+1 nodes wide touches at most ceil((2r+1)/8)+1
            // columns per axis
            int span = (2*o.factored_radius + 1 + kColumnTile - 1)/kColumnTile
                     + 1;
            for (int i = 0; i < n; ++i)
            {
                const ekx_geometry3d &g = geoms[i];
                int nbx = (g.nx + kColumnTile - 1)/kColumnTile;
                int nby = (g.ny + kColumnTile - 1)/kColumnTile;
                boxPerDiag = std::max(boxPerDiag,
                                      std::min(span, nbx)*std::min(span, nby));
            }
        }
        EKX_CHECK(dItems.allocate(flat.size()));
        EKX_HIP(hipMemcpyAsync(dItems.ptr, flat.data(),
                               flat.size()*sizeof(ColumnItem),
                               hipMemcpyHostToDevice, stream));
        // work-queue flags: one per column chunk of every problem
        std::vector<int> flagBase(n);
        int64_t nFlags = 0;
        for (int i = 0; i < n; ++i)
        {
            const ekx_geometry3d &g = geoms[i];
            flagBase[i] = (int) nFlags;
            nFlags += (int64_t) ((g.nx + kColumnTile - 1)/kColumnTile)*
                      ((g.ny + kColumnTile - 1)/kColumnTile)*
                      ((g.nz + chunkH - 1)/chunkH);
        }
        if (nFlags > INT32_MAX)
        {
            return fail(EKX_EINVAL, "too many column chunks for one batch");
        }
        queueFlags = nFlags;
        queueMaxSweeps = 8*(std::max(o.number_of_sweeps, 1) + 1);
        EKX_CHECK(dFlagBase.allocate(flagBase.size()));
        EKX_HIP(hipMemcpyAsync(dFlagBase.ptr, flagBase.data(),
                               flagBase.size()*sizeof(int),
                               hipMemcpyHostToDevice, stream));
        const size_t words = (size_t) queueFlags +
                             (size_t) nChains*queueMaxSweeps + 1;
        EKX_CHECK(queueWords.allocate(words));
        EKX_HIP(hipMemsetAsync(queueWords.ptr, 0, words*sizeof(unsigned int),
                               stream));
        {
            int device = 0, cus = 256, v = 0;
            if (hipGetDevice(&device) == hipSuccess &&
                hipDeviceGetAttribute(&v,
                                      hipDeviceAttributeMultiprocessorCount,
                                      device) == hipSuccess && v > 0)
            {
                cus = v;
            }
            // the work-queue kernel's resident waves (LDS rings and
            // registers bound them)
            const int perCU = queued_waves_per_cu(depth());
            queueWaves = (perCU > 0 ? perCU : 8)*cus;
            // The bound of one dependency wait, in the device's wall clock
            // (rate in kHz): at least 250 ms, and 4 times a whole sweep of
            // the largest chain at 1e9 node updates per second (a wait can
            // only last as long as the chunks queued before it take, and
            // the sweeps run at 1e10 and more), so that a device shared
            // with other work does not trip it.  A wait past the bound
            // makes the solve fail with EKX_EHIP and its field is void.
            if (hipDeviceGetAttribute(&clockKHz,
                                      hipDeviceAttributeWallClockRate,
                                      device) != hipSuccess || clockKHz <= 0)
            {
                clockKHz = 100000;
            }
            int64_t chainNodes = 0;
            for (int c = 0; c < nChains; ++c)
            {
                int64_t nodes = 0;
                for (int i = chainBegin[c]; i < chainBegin[c + 1]; ++i)
                {
                    const ekx_geometry3d &g = geoms[i];
                    nodes += (int64_t) g.nx*g.ny*g.nz;
                }
                chainNodes = std::max(chainNodes, nodes);
            }
            const double ms = std::max(250.0, 4.0e-6*(double) chainNodes);
            queueWaitTicks = (uint64_t) ((double) clockKHz*ms);
        }
        return EKX_OK;
    }

    // The error word of the work queue: set when a dependency wait of a
    // sweep exceeded its bound (the launch then finished with unordered
    // chunks).  Read after a synchronised solve, then cleared.
    ekx_status check_queue_error()
    {
        if (!queued<double>() || queueWords.ptr == nullptr) { return EKX_OK; }
        unsigned int err = 0;
        unsigned int *w = queueWords.ptr + queueFlags +
                          (size_t) nChains*queueMaxSweeps;
        EKX_CHECK(copy_out(&err, w, sizeof(err)));
        if (err != 0)
        {
            EKX_HIP(launch_clear_words(w, 1, stream));
            EKX_HIP(hipStreamSynchronize(stream));
            return fail(EKX_EHIP, "column work queue: a dependency wait "
                                  "exceeded its bound");
        }
        return EKX_OK;
    }

    // The work queue of chain c's sweep number `epoch` (1-based) of the
    // current sequence.
    ColumnQueue column_queue(int c, unsigned int epoch) const
    {
        ColumnQueue q;
        q.flagBase = dFlagBase.ptr;
        q.flags = queueWords.ptr;
        q.counter = queueWords.ptr + queueFlags +
                    (size_t) c*queueMaxSweeps + (epoch - 1);
        q.error = queueWords.ptr + queueFlags +
                  (size_t) nChains*queueMaxSweeps;
        q.epoch = epoch;
        q.pad = 0;
        q.waitTicks = queueWaitTicks;
        return q;
    }

    // A chosen depth made even: as many chunks, all of about the same
    // depth (193 planes in chunks of 64 end with one of a single plane: 64
    // sources on 385 x 385 x 193, FP64, 1 iteration: 198 ms, in chunks of
    // 49 156; 97 planes, FIXED32, 64 sources on 193 x 193: chunks of 32 47
    // ms, of 25 43).  Shorter chunks than 24 planes differ by little.
    static int even_chunk(int h, int maxNz)
    {
        if (h < 24 || h >= maxNz) { return h; }
        const int chunks = (maxNz + h - 1)/h;
        return (maxNz + chunks - 1)/chunks;
    }

    // Planes per z-chunk when the caller leaves the choice
    // (chunk_planes = 0), by size class: the longest of whole columns, 128,
    // 96, 64, 48, 32, 24, 16, 12 or 8 planes whose column diagonals hold on
    // average at least a number of times the column waves the device keeps
    // resident of the bulk instance that also runs the box chunks: 1.5 up to
    // 96 planes, 3 up to 128, above that 2.5 in FP64, 4 in FP32 and 3.5 in
    // scaled integers, whose steps are shorter against a launch's ends.
    // Shorter chunks put more column-chunks on each diagonal (a sweep's
    // dependency chain is nbx + nby + nbz - 2 launches) at the price of
    // the 15-step lane skew at both ends of every chunk.  Measured on the
    // MI355X, 3 iterations, ms of whole columns / chunks of half their planes
    // (/ of a third), with the ratio of whole columns (processes differ by up
    // to 4%, the shapes within one by less than 1%):
    // 385 x 385 x 193   FP64          FP32          scaled integers
    //   128 (1.5)       727 664 677   468 395 387   780 642 633
    //   192 (2.3)       954 946       568 537       929 887
    //   224 (2.7)       1068 1084
    //   256 (3.1)       1200 1217     685 678       1167 1143
    //   320 (3.9)       1464 1520                   1370 1401
    //   384 (4.6)       1739 1804     956 926       1622 1669
    //     (again)                     915 952
    //   512 (6.2)                     1168 1239
    // 257 x 257 x 257
    //   300 (2.5)       860 861       530 478       853 798
    //   600 (4.9)                     845 833       1477 1495
    // 201 x 201 x 120 (whole: 128 or less)
    //   500 (3.2)       451 490       267 342       435 514
    // 193 x 193 x 110
    //   300 (1.9)       278 268       197 194       302 280
    // A 64-problem batch of 96..320-point grids runs fastest with 32 planes,
    // a single 257 x 257 x 193 or 129^3 grid with 8 (4.5x and 3x faster than
    // whole columns); every choice gives the same field.
    int auto_chunk(const std::vector<ekx_geometry3d> &geoms, int maxNz) const
    {
        int device = 0, cus = 256;
        if (hipGetDevice(&device) == hipSuccess)
        {
            int v = 0;
            if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount,
                                      device) == hipSuccess && v > 0)
            {
                cus = v;
            }
        }
        // resident column waves per CU of the precision's bulk kernel
        int perCU = sweeps_f64()
                        ? column_waves_per_cu<double>(depth(), true)
                  : fixed32()
                        ? column_waves_per_cu<uint32_t>(depth(), true)
                        : column_waves_per_cu<float>(depth(), true);
        if (perCU <= 0) { perCU = 8; }
        const double resident = (double) cus*perCU;
        const double deep = sweeps_f64() ? 2.5 : fixed32() ? 3.5 : 4.0;
        for (int c : kChunkCandidates)
        {
            const int h = c == 0 ? maxNz : std::min(c, maxNz);
            double items = 0;
            int diags = 1;
            for (const ekx_geometry3d &g : geoms)
            {
                const int nbx = tiles_of(g.nx), nby = tiles_of(g.ny);
                const int nbz = (g.nz + h - 1)/h;
                items += (double) nbx*nby*nbz;
                diags = std::max(diags, nbx + nby + nbz - 2);
            }
            const double want = h > 128 ? deep : h > 96 ? 3.0 : 1.5;
            if (items/diags >= want*resident) { return h; }
        }
        return std::min(8, maxNz);
    }

    // Uploads one model (cell slowness, double) to its slot.
    ekx_status upload_model(int model, const double *slowness, int64_t n)
    {
        drop_graph();
        EKX_HIP(hipMemcpyAsync(S64.ptr + modelOffset[model], slowness,
                               (size_t) n*sizeof(double),
                               hipMemcpyHostToDevice, stream));
        return EKX_OK;
    }

    // The slowness range of every model, and whether it suits the update
    // without range tests of its roots (cartesian_uniform3d); scaled
    // integers decode to zero or to at least sMax / (2^32 - 2), half a step
    // less before rounding.
    ekx_status find_ranges()
    {
        const size_t per = 2*(size_t) kRangeBlocks;
        for (size_t m = 0; m < modelCells.size(); ++m)
        {
            EKX_HIP(launch_block_range(modelCells[m], S64.ptr + modelOffset[m],
                                       partial.ptr + m*per, kRangeBlocks,
                                       stream));
        }
        std::vector<double> host(modelCells.size()*per);
        EKX_HIP(hipMemcpyAsync(host.data(), partial.ptr,
                               host.size()*sizeof(double),
                               hipMemcpyDeviceToHost, stream));
        EKX_HIP(hipStreamSynchronize(stream));
        for (size_t m = 0; m < modelCells.size(); ++m)
        {
            modelSMin[m] = host[m*per];
            modelSMax[m] = host[m*per + 1];
            for (size_t k = m*per; k < (m + 1)*per; k += 2)
            {
                modelSMin[m] = std::min(modelSMin[m], host[k]);
                modelSMax[m] = std::max(modelSMax[m], host[k + 1]);
            }
        }
        for (size_t i = 0; i < problems.size(); ++i)
        {
            Problem3D &p = problems[i];
            const double hi = modelSMax[modelOf[i]];
            const double lo = std::min(modelSMin[modelOf[i]], hi*0x1p-33);
            // unequal spacings: the planes' determinants are of the size of
            // (h s)^2 for their larger spacing, the 3D one of (s / h)^2
            const double least = std::min(p.dx, std::min(p.dy, p.dz));
            const double most = std::max(p.dx, std::max(p.dy, p.dz));
            // (and no time at the source cell's corners above HUGE, which an
            // invalid candidate of the branch-free updates would lower)
            p.scaled = least*lo >= 0x1p-300 &&
                       (p.dx + p.dy + p.dz)*hi <= kHuge &&
                       (p.uniform || (lo >= most*0x1p-340 &&
                                      hi <= least*0x1p500)) ? 1 : 0;
        }
        return EKX_OK;
    }

    ekx_status finish_models()
    {
        EKX_CHECK(find_ranges());
        if (S32.ptr)
        {
            EKX_HIP(launch_convert(totalCells, S64.ptr, S32.ptr, stream));
        }
        if (SQ.ptr)
        {
            // Per model: the largest slowness fixes the code step
            // (s = code * sMax / (2^32 - 2)), then the model is encoded.
            for (size_t m = 0; m < modelCells.size(); ++m)
            {
                const double *sm = S64.ptr + modelOffset[m];
                const double sMax = modelSMax[m];
                if (!(sMax > 0.0) || !std::isfinite(sMax))
                {
                    return fail(EKX_EINVAL, "slowness model must be positive "
                                            "and finite");
                }
                double step = sMax/(double) kTimeMaxCode;
                EKX_HIP(launch_encode_slowness(modelCells[m], sm, 1.0/step,
                                               SQ.ptr + modelOffset[m],
                                               stream));
            }
        }
        if (tiled)
        {
            // slowness bricks of every model, in each element type swept
            for (size_t m = 0; m < modelCells.size(); ++m)
            {
                const ekx_geometry3d *g = nullptr;
                for (size_t i = 0; i < problems.size() && !g; ++i)
                {
                    if (modelOf[i] == (int) m) { g = &geometry[i]; }
                }
                if (!g) { continue; }
                const int64_t so = modelOffset[m], bo = modelBrickOffset[m];
                if (SB64.ptr)
                {
                    EKX_HIP(launch_tile_slowness<double>(
                        g->nx, g->ny, g->nz, S64.ptr + so, SB64.ptr + bo,
                        stream));
                }
                if (SB32.ptr)
                {
                    EKX_HIP(launch_tile_slowness<float>(
                        g->nx, g->ny, g->nz, S32.ptr + so, SB32.ptr + bo,
                        stream));
                }
                if (SBQ.ptr)
                {
                    EKX_HIP(launch_tile_slowness<uint32_t>(
                        g->nx, g->ny, g->nz, SQ.ptr + so, SBQ.ptr + bo,
                        stream));
                }
            }
        }
        EKX_HIP(hipStreamSynchronize(stream));
        haveModel = true;
        haveField = false;
        return EKX_OK;
    }

    // Whether captured launches depend on the source cells: the hyperplane
    // kernel's levels do, and the diagonals that get factored launches (the
    // work queue, which runs the box in place, has none).  13440 launches:
    // 129 ms a solve, 152 when they are captured again.
    bool captures_source() const
    {
        if (kernel() == EKX_KERNEL_HYPERPLANE) { return true; }
        return !mergedSmall && boxPerDiag > 0 && !queued_primary();
    }

    // Fills the source fields of the problem descriptors (the source cell
    // slowness is read from the device copy of the model).
    ekx_status prepare_sources()
    {
        const int n = (int) problems.size();
        std::vector<double> sSrc(n, 0.0);
        for (int i = 0; i < n; ++i)
        {
            Problem3D &p = problems[i];
            const SourceInfo &s = sources[i];
            EKX_HIP(hipMemcpyAsync(&sSrc[i],
                                   S64.ptr + p.sOffset + s.cellIndex,
                                   sizeof(double), hipMemcpyDeviceToHost,
                                   stream));
        }
        EKX_HIP(hipStreamSynchronize(stream));
        bool moved = false;
        for (int i = 0; i < n; ++i)
        {
            Problem3D &p = problems[i];
            const SourceInfo &s = sources[i];
            moved = moved || p.srcCellX != s.cell[0] ||
                    p.srcCellY != s.cell[1] || p.srcCellZ != s.cell[2];
            p.srcCellX = s.cell[0];
            p.srcCellY = s.cell[1];
            p.srcCellZ = s.cell[2];
            p.srcOffX = s.offset[0];
            p.srcOffY = s.offset[1];
            p.srcOffZ = s.offset[2];
            p.srcSlowness = sSrc[i];
            if (SQ.ptr) { set_fixed32_steps(i); }
        }
        if (moved) { sourceStamp += 1; }
        if (moved && captures_source()) { drop_graph(); }
        EKX_HIP(hipMemcpyAsync(dProblems.ptr, problems.data(),
                               problems.size()*sizeof(Problem3D),
                               hipMemcpyHostToDevice, stream));
        return EKX_OK;
    }

    // Code steps of problem i in the FIXED32 modes.  Every finite travel
    // time of the scheme is at most sMax times the largest Manhattan
    // distance from the source to a node, plus a few cells: the local
    // update never exceeds its smallest face neighbour + h * sMax
    // (the 1D operators of finiteDifference), the initialisation sweeps
    // reach every node through such a chain from the source cell, whose
    // corners hold sSrc * |x - xs|, and refinement sweeps only lower
    // values.  The slack of 8 cells also absorbs the half-step rounding of
    // the stored codes along a chain.
    void set_fixed32_steps(int i)
    {
        Problem3D &p = problems[i];
        const ekx_geometry3d &g = geometry[i];
        const double sMax = modelSMax[modelOf[i]];
        const double lx = (g.nx - 1)*g.dx, ly = (g.ny - 1)*g.dy;
        const double lz = (g.nz - 1)*g.dz;
        const double mx = std::max(p.srcOffX, lx - p.srcOffX);
        const double my = std::max(p.srcOffY, ly - p.srcOffY);
        const double mz = std::max(p.srcOffZ, lz - p.srcOffZ);
        const double hMax = std::max(g.dx, std::max(g.dy, g.dz));
        const double tBound = sMax*(mx + my + mz + 8*hMax);
        p.tStep = tBound/(double) kTimeMaxCode;
        p.tScale = 1.0/p.tStep;
        p.sStep = sMax/(double) kTimeMaxCode;
    }

    // The factored-box columns need their own launch unless the bulk
    // instance runs them: with chunks shorter than kMergedMaxChunk planes
    // (single grids and uneven batches, whose diagonals are short launches,
    // where a second launch per diagonal costs more than the bulk
    // instance's extra registers).
    template <typename TS> bool separate_factored() const
    {
        return !mergedSmall;
    }

    // kernel_timing times every bulk column launch (the dominant kernel).
    template <typename TS> bool timed_sweep(bool) const { return timing; }

    // Work counters of one sweep over every problem.
    template <typename TS>
    void count_sweep(int sweep, bool initialize, ekx_solve_stats &st) const
    {
        for (const Problem3D &p : problems)
        {
            HostOctant o = host_octant(p, sweep, initialize);
            int64_t upd = (int64_t) (p.nx - o.jx0)*(p.ny - o.jy0)*
                          (p.nz - o.jz0);
            st.updates += upd;
            if (sizeof(TS) == 8) { st.updates_fp64 += upd; }
            if (kernel() == EKX_KERNEL_COLUMN)
            {
                const int64_t box = host_box_updates(
                    p, sweep, initialize, chunkH, separate_factored<TS>());
                st.updates_factored += box;
                if (timed_sweep<TS>(initialize))
                {
                    st.timed_updates += separate_factored<TS>() ? upd - box
                                                                : upd;
                }
            }
        }
    }

    template <typename TS>
    ekx_status enqueue_sweep(int sweep, bool initialize, TS *T, const TS *S,
                             unsigned int epoch, ekx_solve_stats &st)
    {
        int64_t launches = 0;
        ekx_status rc = enqueue_sweep_launches<TS>(sweep, initialize, T, S,
                                                   epoch, launches);
        st.kernel_launches += launches;
        if (sizeof(TS) == 8) { st.kernel_launches_fp64 += launches; }
        return rc;
    }

    // Slowness bricks of element type TS (the column kernel's model).
    template <typename TS> const TS *bricks() const
    {
        if constexpr (sizeof(TS) == 8) { return SB64.ptr; }
        else if constexpr (std::is_same<TS, float>::value) { return SB32.ptr; }
        else { return SBQ.ptr; }
    }

    // Per diagonal, the phases of the factored launches of a sweep over
    // problems [p0, p0 + np) (host_box_diagonals); none when the bulk
    // launches run the box chunks.
    template <typename TS>
    std::vector<uint8_t> box_diagonals(int p0, int np, int sweep,
                                       bool initialize) const
    {
        std::vector<uint8_t> mask((size_t) nDiag, 0);
        if (!separate_factored<TS>() || boxPerDiag <= 0) { return mask; }
        for (int i = p0; i < p0 + np; ++i)
        {
            host_box_diagonals(problems[i], sweep, initialize, chunkH, mask);
        }
        return mask;
    }

    // One sweep of chain c on its own stream: per diagonal, the bulk
    // launch over the chain's items, with the box ends of the box chunks
    // of the chain's problems in factored launches before (phase 0) and
    // after it (phase 1).
    template <typename TS>
    ekx_status enqueue_chain_sweep(int c, int sweep, bool initialize, TS *T,
                                   unsigned int epoch, int64_t &launches)
    {
        hipStream_t cs = chainStreams[c];
        const TS *SB = bricks<TS>();
        const int p0 = chainBegin[c];
        const int np = chainBegin[c + 1] - p0;
        const int *ds = diagStart.data() + (size_t) c*(nDiag + 1);
        if (queued<TS>())
        {
            EKX_CHECK(enqueue_queued_sweep<TS>(c, sweep, initialize, T,
                                               epoch, cs, launches));
            return EKX_OK;
        }
        const std::vector<uint8_t> phases =
            box_diagonals<TS>(p0, np, sweep, initialize);
        for (int d = 0; d < nDiag; ++d)
        {
            const int count = ds[d + 1] - ds[d];
            EKX_CHECK(enqueue_diagonal<TS>(d, dItems.ptr + ds[d], count,
                                           dProblems.ptr + p0, np, phases[d],
                                           sweep, initialize, T, SB, cs,
                                           launches));
        }
        return EKX_OK;
    }

    // One diagonal d on stream s: the factored launch of phase 0, the bulk
    // launch over `count` items, the factored launch of phase 1 (the
    // factored launches over problems [pp, pp + np), where `phases` has
    // work).
    template <typename TS>
    ekx_status enqueue_diagonal(int d, const ColumnItem *items, int count,
                                const Problem3D *pp, int np,
                                unsigned phases, int sweep, bool initialize,
                                TS *T, const TS *SB, hipStream_t s,
                                int64_t &launches)
    {
        for (int phase = 0; phase < 2; ++phase)
        {
            if (phase == 1 && count > 0)
            {
                if (timed_sweep<TS>(initialize))
                {
                    EKX_CHECK(record_timing_event(s));
                }
                EKX_HIP(launch_columns3d<TS>(
                    dProblems.ptr, items, count, sweep, initialize ? 1 : 0,
                    d, boxPerDiag, chunkH, T, SB, change.ptr, depth(),
                    !separate_factored<TS>(), s));
                if (timed_sweep<TS>(initialize))
                {
                    EKX_CHECK(record_timing_event(s));
                }
                launches += 1;
            }
            if (phases & (1u << phase))
            {
                EKX_HIP(launch_factored_columns3d<TS>(
                    pp, np, sweep, initialize ? 1 : 0, d, boxPerDiag, chunkH,
                    phase, T, SB, change.ptr, s));
                launches += 1;
            }
        }
        return EKX_OK;
    }

    // One sweep of chain c in work-queue form: one launch over the chain's
    // items, all diagonals.
    template <typename TS>
    ekx_status enqueue_queued_sweep(int c, int sweep, bool initialize, TS *T,
                                    unsigned int epoch, hipStream_t s,
                                    int64_t &launches)
    {
        if (epoch < 1 || (int) epoch > queueMaxSweeps)
        {
            return fail(EKX_EINVAL, "work queue: too many sweeps in one "
                                    "sequence");
        }
        const int *ds = diagStart.data() + (size_t) c*(nDiag + 1);
        const int count = ds[nDiag] - ds[0];
        if (count <= 0) { return EKX_OK; }
        if (timed_sweep<TS>(initialize)) { EKX_CHECK(record_timing_event(s)); }
        EKX_HIP(launch_queued_columns3d<TS>(
            dProblems.ptr, dItems.ptr + ds[0], count, sweep,
            initialize ? 1 : 0, chunkH, T, bricks<TS>(), change.ptr,
            column_queue(c, epoch), std::max(1, queueWaves/nChains), depth(),
            s));
        if (timed_sweep<TS>(initialize)) { EKX_CHECK(record_timing_event(s)); }
        launches += 1;
        return EKX_OK;
    }

    template <typename TS>
    ekx_status enqueue_sweep_launches(int sweep, bool initialize, TS *T,
                                      const TS *S, unsigned int epoch,
                                      int64_t &launches)
    {
        const int n = (int) problems.size();
        if (kernel() == EKX_KERNEL_COLUMN && queued<TS>())
        {
            return enqueue_queued_sweep<TS>(0, sweep, initialize, T, epoch,
                                            stream, launches);
        }
        if (kernel() == EKX_KERNEL_HYPERPLANE)
        {
            for (int i = 0; i < n; ++i)
            {
                const Problem3D &p = problems[i];
                HostOctant o = host_octant(p, sweep, initialize);
                const int lastLevel = (p.nx - 1) + (p.ny - 1) + (p.nz - 1);
                for (int L = o.jx0 + o.jy0 + o.jz0; L <= lastLevel; ++L)
                {
                    int kLo = std::max(o.jz0, L - (p.nx - 1) - (p.ny - 1));
                    int kHi = std::min(p.nz - 1, L - o.jx0 - o.jy0);
                    if (kLo > kHi) { continue; }
                    int nPairs = (kHi - kLo + 1)*(p.ny - o.jy0);
                    EKX_HIP(launch_hyperplane3d<TS>(
                        dProblems.ptr, i, sweep, initialize ? 1 : 0, L, kLo,
                        nPairs, T, S, change.ptr, stream));
                    launches += 1;
                }
            }
        }
        else
        {
            const TS *SB = bricks<TS>();
            const std::vector<int> &ds = diagStart;
            const std::vector<uint8_t> phases =
                box_diagonals<TS>(0, n, sweep, initialize);
            for (int d = 0; d < nDiag; ++d)
            {
                EKX_CHECK(enqueue_diagonal<TS>(d, dItems.ptr + ds[d],
                                               ds[d + 1] - ds[d],
                                               dProblems.ptr, n, phases[d],
                                               sweep, initialize, T, SB,
                                               stream, launches));
            }
        }
        return EKX_OK;
    }

    // Records the next event of the timing pool on stream s.
    ekx_status record_timing_event(hipStream_t s)
    {
        if (timingUsed == timingEvents.size())
        {
            hipEvent_t e = nullptr;
            EKX_HIP(hipEventCreate(&e));
            timingEvents.push_back(e);
        }
        EKX_HIP(hipEventRecord(timingEvents[timingUsed], s));
        timingUsed += 1;
        return EKX_OK;
    }

    // The sweeps of one precision segment (sweep, initialisation sweep) and
    // the refinement iterations among them.
    std::vector<std::pair<int, bool>> sweep_list(bool doInit,
                                                 int &iterations) const
    {
        std::vector<std::pair<int, bool>> list;
        if (doInit)
        {
            if (opt.schedule == EKX_SCHEDULE_SHIPPED)
            {
                // src/solver3d.cpp:451-463 (FSM); level set: nothing.
                if (opt.algorithm == EKX_FAST_SWEEPING_METHOD)
                {
                    list = {{0, true}, {1, true}};
                }
                iterations = 0;
            }
            else
            {
                for (int s = 0; s < 8; ++s) { list.push_back({s, true}); }
            }
        }
        for (int k = 0; k < iterations; ++k)
        {
            for (int s = 0; s < 8; ++s) { list.push_back({s, false}); }
        }
        return list;
    }

    template <typename TS>
    void count_segment(bool doInit, int iterations, ekx_solve_stats &st) const
    {
        for (const auto &sw : sweep_list(doInit, iterations))
        {
            count_sweep<TS>(sw.first, sw.second, st);
        }
    }

    template <typename TS>
    ekx_status enqueue_phase_sweeps(TS *T, const TS *S, bool doInit,
                                    int iterations, ekx_solve_stats &st)
    {
        count_segment<TS>(doInit, iterations, st);
        const std::vector<std::pair<int, bool>> list =
            sweep_list(doInit, iterations);
        if (queued<TS>())
        {
            // a new sequence of work-queue sweeps: flags and counters back
            // to zero, epochs count from 1
            EKX_HIP(launch_clear_words(queueWords.ptr,
                                       queueFlags + (int64_t) nChains*
                                                        queueMaxSweeps,
                                       stream));
        }
        if (nChains == 1)
        {
            unsigned int epoch = 0;
            for (const auto &sw : list)
            {
                EKX_CHECK(enqueue_sweep<TS>(sw.first, sw.second, T, S,
                                            ++epoch, st));
            }
        }
        else
        {
            // Chains run their whole sweep list independently: fork from
            // the main stream, join back at the end.
            int64_t launches = 0;
            EKX_HIP(hipEventRecord(evFork, stream));
            for (int c = 0; c < nChains; ++c)
            {
                EKX_HIP(hipStreamWaitEvent(chainStreams[c], evFork, 0));
                unsigned int epoch = 0;
                for (const auto &sw : list)
                {
                    EKX_CHECK(enqueue_chain_sweep<TS>(c, sw.first, sw.second,
                                                      T, ++epoch, launches));
                }
                EKX_HIP(hipEventRecord(chainEvents[c], chainStreams[c]));
            }
            for (int c = 0; c < nChains; ++c)
            {
                EKX_HIP(hipStreamWaitEvent(stream, chainEvents[c], 0));
            }
            st.kernel_launches += launches;
            if (sizeof(TS) == 8) { st.kernel_launches_fp64 += launches; }
        }
        st.iterations_run += iterations;
        return EKX_OK;
    }

    // Runs the sweeps of one precision segment: replayed from its captured
    // graph (captured on first use) or issued directly.
    template <typename TS>
    ekx_status run_segment(int k, TS *T, const TS *S, bool doInit,
                           int iterations, ekx_solve_stats &st)
    {
        ekx_solve_stats local{};
        if (opt.use_graph && !timing)
        {
            Segment &g = segment[k];
            if (!g.valid)
            {
                g.release();
                std::shared_lock<std::shared_mutex> capturing(g_captures);
                EKX_HIP(hipStreamBeginCapture(stream,
                                              hipStreamCaptureModeThreadLocal));
                ekx_status s = enqueue_phase_sweeps<TS>(T, S, doInit,
                                                        iterations, local);
                hipGraph_t captured = nullptr;
                hipError_t e = hipStreamEndCapture(stream, &captured);
                capturing.unlock();
                if (s != EKX_OK)
                {
                    if (captured) { (void) hipGraphDestroy(captured); }
                    return s;
                }
                EKX_HIP(e);
                g.graph = captured;
                if (local.kernel_launches > 0)
                {
                    EKX_HIP(hipGraphInstantiate(&g.exec, g.graph, nullptr,
                                                nullptr, 0));
                }
                g.st = local;
                g.sourceStamp = sourceStamp;
                g.valid = true;
            }
            else if (g.sourceStamp != sourceStamp)
            {
                // the octants and the box moved with the sources
                count_segment<TS>(doInit, iterations, local);
                g.st.updates = local.updates;
                g.st.updates_fp64 = local.updates_fp64;
                g.st.updates_factored = local.updates_factored;
                g.sourceStamp = sourceStamp;
            }
            local = g.st;
            if (g.exec) { EKX_HIP(hipGraphLaunch(g.exec, stream)); }
        }
        else
        {
            EKX_CHECK(enqueue_phase_sweeps<TS>(T, S, doInit, iterations,
                                               local));
        }
        st.updates += local.updates;
        st.updates_fp64 += local.updates_fp64;
        st.updates_factored += local.updates_factored;
        st.kernel_launches += local.kernel_launches;
        st.kernel_launches_fp64 += local.kernel_launches_fp64;
        st.iterations_run += local.iterations_run;
        st.timed_updates += local.timed_updates;
        return EKX_OK;
    }

    // The sweeps of the first precision segment: one captured block, or,
    // with early exit, the initialisation sweeps and then one refinement
    // iteration at a time until an iteration's largest decrease is at most
    // the tolerance.  kernel_timing times the bulk launches of this
    // segment (issued eagerly).
    template <typename TS>
    ekx_status run_primary(TS *T, const TS *S, int iterations,
                           ekx_solve_stats &st)
    {
        timing = opt.kernel_timing != 0;
        timingUsed = 0;
        if (!early_exit())
        {
            EKX_CHECK(run_segment<TS>(0, T, S, true, iterations, st));
        }
        else
        {
            EKX_CHECK(run_segment<TS>(2, T, S, true, 0, st));
            for (int k = 0; k < iterations; ++k)
            {
                EKX_HIP(hipMemsetAsync(change.ptr, 0, sizeof(unsigned int),
                                       stream));
                EKX_CHECK(run_segment<TS>(3, T, S, false, 1, st));
                EKX_HIP(hipMemcpyAsync(changeHost, change.ptr,
                                       sizeof(unsigned int),
                                       hipMemcpyDeviceToHost, stream));
                EKX_HIP(hipStreamSynchronize(stream));
                float c = 0;
                std::memcpy(&c, changeHost, sizeof(float));
                st.last_iteration_change = c;
                if (c <= opt.convergence_tolerance) { break; }
            }
        }
        timing = false;
        return EKX_OK;
    }

    // One short solve for the autotuner: the initialisation sweeps and one
    // refinement iteration, run as later solves run (in one launch, or the
    // captured graph, unless use_graph is off): once to capture, then timed;
    // device ms.
    template <typename TS>
    ekx_status trial_run(TS *T, const TS *S, bool flow, float &ms)
    {
        const int nProb = (int) problems.size();
        ekx_solve_stats st{};
        timing = false;
        for (int pass = 0; pass < 2; ++pass)
        {
            EKX_HIP(hipEventRecord(evStart, stream));
            if constexpr (std::is_same<TS, uint32_t>::value) { flow = false; }
            else if (flow) { EKX_CHECK(run_flow<TS>(T, true, 1, st)); }
            if (!flow)
            {
                EKX_HIP(launch_init3d<TS>(dProblems.ptr, nProb, totalNodes, T,
                                          stream));
                EKX_CHECK(run_segment<TS>(0, T, S, true, 1, st));
            }
            EKX_HIP(hipEventRecord(evStop, stream));
            EKX_HIP(hipEventSynchronize(evStop));
            EKX_CHECK(check_queue_error());
        }
        EKX_HIP(hipEventElapsedTime(&ms, evStart, evStop));
        return EKX_OK;
    }

    ekx_status trial_ms(bool flow, float &ms)
    {
        EKX_CHECK(prepare_sources());
        if (sweeps_f64())
        {
            return trial_run<double>(T64.ptr, S64.ptr, flow, ms);
        }
        if (fixed32())
        {
            return trial_run<uint32_t>(TQ.ptr, SQ.ptr, flow, ms);
        }
        return trial_run<float>(T32.ptr, S32.ptr, flow, ms);
    }

    // Time of the solve in one launch; ms < 0: this setup has none, or it
    // gave up (and is given up for later solves too).
    ekx_status trial_flow(float &ms)
    {
        ms = -1;
        FlowReservation r;
        if (!take_flow(r, 16)) { return EKX_OK; }
        EKX_CHECK(trial_ms(true, ms));
        unsigned int err = 0;
        EKX_CHECK(copy_out(&err, flowWords.ptr, sizeof(err)));
        if (err != 0)
        {
            release_flow();
            ms = -1;
        }
        return EKX_OK;
    }

    // The schedule of a launch shape (0, 0: the default).
    ekx_status use_shape(int chunk, int chains)
    {
        tunedChunk = chunk;
        tunedChains = chains;
        drop_graph();
        return build_schedule();
    }

    // Measured choice of the launch shape (no reference counterpart): times
    // a short solve for z-chunk depths around the size-class default (the
    // default and its neighbours in auto_chunk's list) and 1, 2 or 4
    // chains, and the solve in one launch where the setup has it, and keeps
    // the fastest for later solves.  Fields do not depend on the choice; the
    // field of the last solve is discarded.
    ekx_status autotune(int &chunkOut, int &chainsOut)
    {
        if (!haveModel)
        {
            return fail(EKX_ESTATE, "Velocity model not set");
        }
        for (size_t i = 0; i < problems.size(); ++i)
        {
            if (!haveSource[i])
            {
                return fail(EKX_ESTATE, "Source location not set");
            }
        }
        if (kernel() == EKX_KERNEL_COLUMN)
        {
            int maxNz = 0;
            for (const ekx_geometry3d &g : geometry)
            {
                maxNz = std::max(maxNz, g.nz);
            }
            std::vector<int> depths;
            for (int c : kChunkCandidates)
            {
                const int h = even_chunk(c == 0 ? maxNz : std::min(c, maxNz),
                                         maxNz);
                if (depths.empty() || h < depths.back()) { depths.push_back(h); }
            }
            const int h0 = even_chunk(auto_chunk(geometry, maxNz), maxNz);
            size_t k0 = 0;
            while (k0 + 1 < depths.size() && depths[k0] != h0) { ++k0; }
            std::vector<int> tryDepth;
            for (size_t k = (k0 > 0 ? k0 - 1 : 0);
                 k <= std::min(k0 + 1, depths.size() - 1); ++k)
            {
                tryDepth.push_back(depths[k]);
            }
            const int n = (int) problems.size();
            std::vector<int> tryChains;
            for (int c : {1, 2, 4})
            {
                if (c <= n) { tryChains.push_back(c); }
            }
            float best = 0;
            int bestDepth = h0, bestChains = 1;
            bool first = true;
            // the default shape first; another replaces the best only when
            // it is more than 3% faster (trial times vary by about that)
            const int c0 = default_chains();
            std::vector<std::pair<int, int>> shapes{{h0, c0}};
            for (int d : tryDepth)
            {
                for (int c : tryChains)
                {
                    if (d != h0 || c != c0) { shapes.push_back({d, c}); }
                }
            }
            const int chunkBefore = tunedChunk, chainsBefore = tunedChains;
            for (const auto &shape : shapes)
            {
                ekx_status rc = use_shape(shape.first, shape.second);
                float ms = 0;
                if (rc == EKX_OK) { rc = trial_ms(false, ms); }
                if (rc != EKX_OK)
                {
                    (void) use_shape(chunkBefore, chainsBefore);
                    return rc;
                }
                if (first || ms < 0.97f*best)
                {
                    best = ms;
                    bestDepth = shape.first;
                    bestChains = shape.second;
                    first = false;
                }
            }
            EKX_CHECK(use_shape(bestDepth, bestChains));
            float flowMs = -1;
            EKX_CHECK(trial_flow(flowMs));
            if (flowMs > 0 && best < 0.97f*flowMs) { release_flow(); }
        }
        haveField = false;
        chunkOut = chunkH;
        chainsOut = nChains;
        return EKX_OK;
    }

    ekx_status solve()
    {
        timing = false;
        if (!haveModel)
        {
            return fail(EKX_ESTATE, "Velocity model not set");
        }
        for (size_t i = 0; i < problems.size(); ++i)
        {
            if (!haveSource[i])
            {
                return fail(EKX_ESTATE, "Source location not set");
            }
        }
        haveField = false;
        EKX_CHECK(prepare_sources());
        bool flowFailed = false;
        {
            FlowReservation r;
            if (take_flow(r, 8*(1 + opt.number_of_sweeps)))
            {
                EKX_CHECK(solve_fields(true, flowFailed));
            }
            else { EKX_CHECK(solve_fields(false, flowFailed)); }
        }
        // A wait of the flow launch exceeded its bound (the device is shared
        // with work that keeps columns out): once more by diagonals, and so
        // every later solve of this setup, which would wait out the bound
        // again otherwise.
        if (flowFailed)
        {
            release_flow();
            EKX_CHECK(solve_fields(false, flowFailed));
        }
        haveField = true;
        solveStamp += 1;
        if (nStations > 0) { EKX_CHECK(compute_stations()); }
        return EKX_OK;
    }

    // The sweeps of a solve, as flow launches or by diagonals; flowFailed: a
    // flow launch flagged an error and the field is void.
    ekx_status solve_fields(bool flow, bool &flowFailed)
    {
        flowFailed = false;
        ekx_solve_stats st{};
        st.last_iteration_change = -1;
        const int nIt = opt.number_of_sweeps;
        const int nProb = (int) problems.size();
        const int itPrimary = polish() ? nIt - 1 : nIt;
        bool polished = false;
        EKX_HIP(hipEventRecord(evStart, stream));
        if (sweeps_f64())
        {
            if (!flow)
            {
                EKX_HIP(launch_init3d<double>(dProblems.ptr, nProb,
                                              totalNodes, T64.ptr, stream));
            }
            EKX_HIP(hipEventRecord(evSeg[0], stream));
            if (flow) { EKX_CHECK(run_flow<double>(T64.ptr, true, nIt, st)); }
            else
            {
                EKX_CHECK(run_primary<double>(T64.ptr, S64.ptr, nIt, st));
            }
            EKX_HIP(hipEventRecord(evSeg[1], stream));
        }
        else if (fixed32())
        {
            EKX_HIP(launch_init3d<uint32_t>(dProblems.ptr, nProb, totalNodes,
                                            TQ.ptr, stream));
            EKX_HIP(hipEventRecord(evSeg[0], stream));
            EKX_CHECK(run_primary<uint32_t>(TQ.ptr, SQ.ptr, itPrimary, st));
            EKX_HIP(hipEventRecord(evSeg[1], stream));
        }
        else
        {
            if (!flow)
            {
                EKX_HIP(launch_init3d<float>(dProblems.ptr, nProb,
                                             totalNodes, T32.ptr, stream));
            }
            EKX_HIP(hipEventRecord(evSeg[0], stream));
            if (flow)
            {
                EKX_CHECK(run_flow<float>(T32.ptr, true, itPrimary, st));
            }
            else
            {
                EKX_CHECK(run_primary<float>(T32.ptr, S32.ptr, itPrimary,
                                             st));
            }
            EKX_HIP(hipEventRecord(evSeg[1], stream));
        }
        if (polish())
        {
            if (fixed32())
            {
                EKX_HIP(launch_decode_times(dProblems.ptr, nProb, maxCount,
                                            TQ.ptr, T64.ptr, stream));
            }
            else
            {
                EKX_HIP(launch_convert(totalNodes, T32.ptr, T64.ptr, stream));
            }
            EKX_HIP(hipEventRecord(evSeg[2], stream));
            if (flow) { EKX_CHECK(run_flow<double>(T64.ptr, false, 1, st)); }
            else
            {
                EKX_CHECK(run_segment<double>(1, T64.ptr, S64.ptr, false, 1,
                                              st));
            }
            EKX_HIP(hipEventRecord(evSeg[3], stream));
            polished = true;
        }
        EKX_HIP(hipEventRecord(evStop, stream));
        EKX_HIP(hipEventSynchronize(evStop));
        EKX_HIP(hipGetLastError());
        EKX_CHECK(check_queue_error());
        if (flow)
        {
            unsigned int err = 0;
            EKX_CHECK(copy_out(&err, flowWords.ptr, sizeof(err)));
            flowFailed = err != 0;
            if (flowFailed) { return EKX_OK; }
        }
        float ms = 0;
        EKX_HIP(hipEventElapsedTime(&ms, evStart, evStop));
        st.last_solve_ms = ms;
        EKX_HIP(hipEventElapsedTime(&ms, evSeg[0], evSeg[1]));
        if (sweeps_f64()) { st.sweep_ms_fp64 = ms; }
        else { st.sweep_ms_fp32 = ms; }
        if (polished)
        {
            EKX_HIP(hipEventElapsedTime(&ms, evSeg[2], evSeg[3]));
            st.sweep_ms_fp64 = ms;
        }
        if (timingUsed > 0)
        {
            double total = 0;
            for (size_t i = 0; i + 1 < timingUsed; i += 2)
            {
                EKX_HIP(hipEventElapsedTime(&ms, timingEvents[i],
                                            timingEvents[i + 1]));
                total += ms;
            }
            st.timed_kernel_ms = total;
            st.timed_launches = (int64_t) (timingUsed/2);
            // timed_updates: counted per timed sweep by count_sweep
        }
        st.tiled = tiled ? 1 : 0;
        st.chunk_planes = kernel() == EKX_KERNEL_COLUMN ? chunkH : 0;
        st.chains = nChains;
        stats = st;
        return EKX_OK;
    }

    ekx_status copy_out(void *dst, const void *src, size_t bytes) const
    {
        EKX_HIP(read_back(dst, src, bytes, stream));
        return EKX_OK;
    }

    // Runs f(T) with the device field in the type it is stored in.
    template <typename F> ekx_status with_field(F &&f) const
    {
        if (fieldIsF64) { return f(T64.ptr); }
        if (TQ.ptr) { return f((const uint32_t *) TQ.ptr); }
        return f((const float *) T32.ptr);
    }

    // Locates the receivers in every problem's grid.
    ekx_status set_stations(int n, const double *x, const double *y,
                            const double *z)
    {
        if (n < 0 || (n > 0 && (!x || !y || !z)))
        {
            return fail(EKX_EINVAL, "invalid station arrays");
        }
        const size_t np = problems.size();
        std::vector<StationLoc3D> locs(np*(size_t) n);
        for (size_t k = 0; k < np; ++k)
        {
            for (int i = 0; i < n; ++i)
            {
                SourceInfo s;
                EKX_CHECK(locate_source3d(geometry[k], x[i], y[i], z[i], s,
                                          "station"));
                StationLoc3D &l = locs[k*(size_t) n + i];
                for (int a = 0; a < 3; ++a)
                {
                    l.off[a] = s.offset[a];
                    l.cell[a] = s.cell[a];
                }
                l.pad = 0;
            }
        }
        nStations = 0;
        stationTimes.clear();
        if (n > 0)
        {
            EKX_CHECK(dStations.allocate(locs.size()));
            EKX_CHECK(stationOut.allocate(locs.size()));
            EKX_HIP(hipMemcpyAsync(dStations.ptr, locs.data(),
                                   locs.size()*sizeof(StationLoc3D),
                                   hipMemcpyHostToDevice, stream));
            EKX_HIP(hipStreamSynchronize(stream));
        }
        nStations = n;
        if (haveField && n > 0) { EKX_CHECK(compute_stations()); }
        return EKX_OK;
    }

    // Interpolates the solved fields at the receivers and copies the
    // [problem][station] table to the host.
    ekx_status compute_stations()
    {
        const int np = (int) problems.size();
        EKX_CHECK(with_field([&](auto *T) -> ekx_status {
            using TS = std::remove_cv_t<std::remove_pointer_t<
                decltype(T)>>;
            EKX_HIP(launch_stations3d<TS>(dProblems.ptr, np, dStations.ptr,
                                          nStations, T, stationOut.ptr,
                                          stream));
            return EKX_OK;
        }));
        stationTimes.assign((size_t) np*nStations, 0.0);
        EKX_HIP(hipMemcpyAsync(stationTimes.data(), stationOut.ptr,
                               stationTimes.size()*sizeof(double),
                               hipMemcpyDeviceToHost, stream));
        EKX_HIP(hipStreamSynchronize(stream));
        stationStamp = solveStamp;
        return EKX_OK;
    }

    ekx_status copy_station_times(int problem, int n, double *out) const
    {
        if (!haveField || stationStamp != solveStamp)
        {
            return fail(EKX_ESTATE, "Travel time field not yet computed");
        }
        if (n != nStations || (n > 0 && !out))
        {
            return fail(EKX_EINVAL, "output must hold one value per "
                                    "station (" +
                                        std::to_string(nStations) + ")");
        }
        const double *src = stationTimes.data() + (size_t) problem*n;
        std::copy(src, src + n, out);
        return EKX_OK;
    }

    // Travel-time gradient of one problem into G (src/gradient.hpp).
    ekx_status compute_gradient(int problem)
    {
        if (!haveField)
        {
            return fail(EKX_ESTATE, "Travel time field not yet computed");
        }
        if (gradientProblem == problem && gradientStamp == solveStamp)
        {
            return EKX_OK;
        }
        const ekx_geometry3d &g = geometry[problem];
        const size_t nGrid = (size_t) g.nx*g.ny*g.nz;
        size_t need = 0;
        for (const ekx_geometry3d &q : geometry)
        {
            need = std::max(need, (size_t) q.nx*q.ny*q.nz);
        }
        gradientProblem = -1;
        EKX_CHECK(G.allocate(3*std::max(need, nGrid)));
        EKX_CHECK(with_field([&](auto *T) -> ekx_status {
            using TS = std::remove_cv_t<std::remove_pointer_t<
                decltype(T)>>;
            EKX_HIP(launch_gradient3d<TS>(dProblems.ptr, problem,
                                          problems[problem], T, G.ptr,
                                          stream));
            return EKX_OK;
        }));
        EKX_HIP(hipStreamSynchronize(stream));
        gradientProblem = problem;
        gradientStamp = solveStamp;
        return EKX_OK;
    }

    bool have_gradient(int problem) const
    {
        return haveField && gradientProblem == problem &&
               gradientStamp == solveStamp;
    }

    ekx_status copy_gradient(int problem, int64_t n, double *out) const
    {
        if (!have_gradient(problem))
        {
            return fail(EKX_ESTATE, "Travel time gradient field not yet "
                                    "computed");
        }
        const ekx_geometry3d &g = geometry[problem];
        const int64_t nOut = 3*(int64_t) g.nx*g.ny*g.nz;
        if (n != nOut || !out)
        {
            return fail(EKX_EINVAL, "output must hold 3 x " +
                                        std::to_string(nOut/3) +
                                        " values");
        }
        EKX_CHECK(copy_out(out, G.ptr, (size_t) n*sizeof(double)));
        return EKX_OK;
    }

    // Device pointer to problem's field in natural order, in its stored
    // type: the field itself, or (tiled) a copy kept until the next solve.
    template <typename TS>
    ekx_status natural_field(int problem, const TS *T, const TS **out) const
    {
        const Problem3D &p = problems[problem];
        if (!tiled)
        {
            *out = T + p.tOffset;
            return EKX_OK;
        }
        DeviceBuffer<TS> *buf;
        if constexpr (sizeof(TS) == 8) { buf = &natural64; }
        else if constexpr (std::is_same<TS, float>::value)
        {
            buf = &natural32;
        }
        else { buf = &naturalQ; }
        if (naturalProblem != problem || naturalStamp != solveStamp ||
            !buf->ptr)
        {
            naturalProblem = -1;
            // one buffer, kept for later reads (a release and an allocation
            // per solve were 0.5 ms on 257 x 257 x 193)
            const void *kept = buf;
            if (kept != &natural64) { natural64.release(); }
            if (kept != &natural32) { natural32.release(); }
            if (kept != &naturalQ) { naturalQ.release(); }
            EKX_CHECK(buf->allocate((size_t) maxNodes));
            EKX_HIP(launch_untile_field<TS>(p, T, buf->ptr, stream));
            EKX_HIP(hipStreamSynchronize(stream));
            naturalProblem = problem;
            naturalStamp = solveStamp;
        }
        *out = buf->ptr;
        return EKX_OK;
    }

    ekx_status copy_field(int problem, int64_t n, double *out) const
    {
        if (!haveField)
        {
            return fail(EKX_ESTATE, "Travel time field not yet computed");
        }
        const ekx_geometry3d &g = geometry[problem];
        int64_t nGrid = (int64_t) g.nx*g.ny*g.nz;
        if (n != nGrid)
        {
            return fail(EKX_EINVAL, "output length " + std::to_string(n) +
                                        " must equal the number of grid "
                                        "points " + std::to_string(nGrid));
        }
        if (!out) { return fail(EKX_EINVAL, "output is NULL"); }
        if (fieldIsF64)
        {
            const double *src = nullptr;
            EKX_CHECK(natural_field<double>(problem, T64.ptr, &src));
            EKX_CHECK(copy_out(out, src, (size_t) n*sizeof(double)));
        }
        else if (TQ.ptr)
        {
            // the decoding of Store<uint32_t>::time
            const uint32_t *src = nullptr;
            EKX_CHECK(natural_field<uint32_t>(problem, TQ.ptr, &src));
            std::vector<uint32_t> tmp((size_t) n);
            EKX_CHECK(copy_out(tmp.data(), src,
                               (size_t) n*sizeof(uint32_t)));
            const double step = problems[problem].tStep;
            for (int64_t i = 0; i < n; ++i)
            {
                uint32_t c = tmp[(size_t) i];
                out[i] = c == kTimeHugeCode ? kHuge : (double) c*step;
            }
        }
        else
        {
            const float *src = nullptr;
            EKX_CHECK(natural_field<float>(problem, T32.ptr, &src));
            std::vector<float> tmp((size_t) n);
            EKX_CHECK(copy_out(tmp.data(), src,
                               (size_t) n*sizeof(float)));
            for (int64_t i = 0; i < n; ++i) { out[i] = tmp[(size_t) i]; }
        }
        return EKX_OK;
    }
};

// ---------------------------------------------------------------------------
// Generated layered Gaussian models (ekx_layered_gaussian)
// ---------------------------------------------------------------------------
ekx_status check_layered_gaussian(const ekx_layered_gaussian *m)
{
    if (!m) { return fail(EKX_EINVAL, "model is NULL"); }
    if (m->n_layers < 1 || !m->layer_velocity)
    {
        return fail(EKX_EINVAL, "a model needs at least one layer velocity");
    }
    for (int k = 0; k < m->n_layers; ++k)
    {
        if (!(m->layer_velocity[k] > 0) || !std::isfinite(m->layer_velocity[k]))
        {
            return fail(EKX_EINVAL, "Non-positive velocities detected");
        }
    }
    if (!(m->amplitude >= 0) || !std::isfinite(m->amplitude))
    {
        return fail(EKX_EINVAL, "amplitude must be >= 0");
    }
    if (!(m->correlation_length >= 0) ||
        !std::isfinite(m->correlation_length))
    {
        return fail(EKX_EINVAL, "correlation length must be >= 0");
    }
    return EKX_OK;
}

// Nodal velocities of the model into device memory dV (nx*ny*nz values,
// natural order), on stream s (synchronised on return).
ekx_status generate_layered_gaussian(const ekx_geometry3d &g,
                                     const ekx_layered_gaussian &m,
                                     double *dV, hipStream_t s)
{
    const int64_t n = (int64_t) g.nx*g.ny*g.nz;
    DeviceBuffer<double> a, b, w, partial, layers;
    EKX_CHECK(a.allocate((size_t) n));
    EKX_CHECK(b.allocate((size_t) n));
    EKX_CHECK(partial.allocate(kMaxPartials));
    EKX_CHECK(layers.allocate((size_t) m.n_layers));
    EKX_HIP(hipMemcpyAsync(layers.ptr, m.layer_velocity,
                           (size_t) m.n_layers*sizeof(double),
                           hipMemcpyHostToDevice, s));
    EKX_HIP(launch_gaussian_noise(n, m.seed, a.ptr, s));
    const double d[3] = {g.dx, g.dy, g.dz};
    std::vector<double> taps;
    for (int axis = 0; axis < 3; ++axis)
    {
        // sigma = l / (2 d) nodes, radius int(4 sigma + 0.5)
        const double sigma = m.correlation_length/(2.0*d[axis]);
        const int radius = (int) (4.0*sigma + 0.5);
        if (radius < 1) { continue; }
        taps.assign((size_t) (2*radius + 1), 0.0);
        double sum = 0.0;
        for (int k = -radius; k <= radius; ++k)
        {
            const double x = k/sigma;
            taps[(size_t) (k + radius)] = std::exp(-0.5*x*x);
            sum += taps[(size_t) (k + radius)];
        }
        for (double &t : taps) { t /= sum; }
        EKX_CHECK(w.allocate(taps.size()));
        EKX_HIP(hipMemcpyAsync(w.ptr, taps.data(), taps.size()*sizeof(double),
                               hipMemcpyHostToDevice, s));
        EKX_HIP(launch_filter_axis(g.nx, g.ny, g.nz, axis, radius, w.ptr,
                                   a.ptr, b.ptr, s));
        EKX_HIP(hipStreamSynchronize(s));    // taps are reused per axis
        std::swap(a.ptr, b.ptr);
    }
    std::vector<double> host(kMaxPartials);
    auto reduce = [&](const double *v, double mean, int power,
                      double &out) -> ekx_status
    {
        EKX_HIP(launch_moment(n, v, mean, power, partial.ptr, kMaxPartials,
                              s));
        EKX_HIP(hipMemcpyAsync(host.data(), partial.ptr,
                               kMaxPartials*sizeof(double),
                               hipMemcpyDeviceToHost, s));
        EKX_HIP(hipStreamSynchronize(s));
        out = power == 0 ? host[0] : 0.0;
        for (double x : host) { out = power == 0 ? std::min(out, x) : out + x; }
        return EKX_OK;
    };
    double sum = 0, ss = 0;
    EKX_CHECK(reduce(a.ptr, 0.0, 1, sum));
    const double mean = sum/(double) n;
    EKX_CHECK(reduce(a.ptr, mean, 2, ss));
    double sd = std::sqrt(ss/(double) n);
    if (!(sd > 0)) { sd = 1.0; }
    EKX_HIP(launch_layered_velocity(g.nx, g.ny, g.nz, m.n_layers, layers.ptr,
                                    m.amplitude, mean, sd, a.ptr, dV, s));
    double vmin = 0;
    EKX_CHECK(reduce(dV, 0.0, 0, vmin));
    if (!(vmin > 0))
    {
        return fail(EKX_EINVAL, "Non-positive velocities detected (the "
                                "amplitude is too large for the field)");
    }
    return EKX_OK;
}

// ===========================================================================
// C ABI
// ===========================================================================
struct ekx_solver3d
{
    Engine3D engine;
    ekx_geometry3d geometry{};
    bool initialized = false;
};

struct ekx_batch3d
{
    Engine3D engine;
    bool initialized = false;
};

extern "C" {

const char *ekx_last_error(void) { return g_error.c_str(); }

const char *ekx_version(void) { return "0.1.0"; }

void ekx_solver_options_default(ekx_solver_options *o)
{
    if (!o) { return; }
    o->number_of_sweeps = 5;
    o->factored_radius = 3;
    o->algorithm = EKX_LEVEL_SET_METHOD;
    o->verbosity = 0;
    o->convergence_tolerance = 1.e-5;
    o->precision = EKX_PRECISION_FP64;
    o->schedule = EKX_SCHEDULE_COMPLETED;
    o->kernel = EKX_KERNEL_AUTO;
    o->early_exit = 0;
    o->use_graph = 1;
    o->kernel_timing = 0;
    o->chains = 0;
    o->prefetch_planes = 0;
    o->chunk_planes = 0;
    o->launch_order = EKX_LAUNCH_AUTO;
}

ekx_status ekx_device_count(int *count)
{
    return guarded([&]() -> ekx_status
    {
        if (!count) { return fail(EKX_EINVAL, "count is NULL"); }
        int n = 0;
        hipError_t e = hipGetDeviceCount(&n);
        if (e != hipSuccess) { n = 0; }
        *count = n;
        return EKX_OK;
    });
}

ekx_status ekx_device_synchronize(void)
{
    return guarded([&]() -> ekx_status
    {
        // (not while a solver captures on another thread)
        std::unique_lock<std::shared_mutex> quiet(g_captures);
        EKX_HIP(hipDeviceSynchronize());
        return EKX_OK;
    });
}

// ----------------------------- Solver3D -----------------------------------
ekx_status ekx_solver3d_create(ekx_solver3d **solver)
{
    return guarded([&]() -> ekx_status
    {
        if (!solver) { return fail(EKX_EINVAL, "solver is NULL"); }
        *solver = new (std::nothrow) ekx_solver3d();
        if (!*solver) { return fail(EKX_ENOMEM, "out of host memory"); }
        return EKX_OK;
    });
}

void ekx_solver3d_destroy(ekx_solver3d *solver) { delete solver; }

ekx_status ekx_solver3d_initialize(ekx_solver3d *h,
                                   const ekx_solver_options *options,
                                   const ekx_geometry3d *geometry)
{
    return guarded([&]() -> ekx_status
    {
        if (!h) { return fail(EKX_EINVAL, "solver is NULL"); }
        h->initialized = false;
        EKX_CHECK(check_options(options));
        EKX_CHECK(check_geometry3d(geometry));
        h->geometry = *geometry;
        EKX_CHECK(h->engine.setup(*options, {*geometry}, {0}, 1));
        h->initialized = true;
        return EKX_OK;
    });
}

int ekx_solver3d_is_initialized(const ekx_solver3d *h)
{
    return h && h->initialized ? 1 : 0;
}

static ekx_status require_initialized(const ekx_solver3d *h)
{
    if (!h) { return fail(EKX_EINVAL, "solver is NULL"); }
    if (!h->initialized) { return fail(EKX_ESTATE, "Class not initialized"); }
    return EKX_OK;
}

ekx_status ekx_solver3d_set_slowness(ekx_solver3d *h, int64_t n,
                                     const double *slowness)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        h->engine.haveModel = false;
        h->engine.haveField = false;
        const ekx_geometry3d &g = h->geometry;
        int64_t nCell = (int64_t) (g.nx - 1)*(g.ny - 1)*(g.nz - 1);
        if (n != nCell)
        {
            return fail(EKX_EINVAL, "Number of cells = " + std::to_string(n) +
                                        " must equal " + std::to_string(nCell));
        }
        if (!slowness) { return fail(EKX_EINVAL, "slowness is NULL"); }
        for (int64_t i = 0; i < n; ++i)
        {
            if (!(slowness[i] > 0))
            {
                return fail(EKX_EINVAL, "Non-positive slowness detected");
            }
        }
        EKX_CHECK(h->engine.upload_model(0, slowness, n));
        return h->engine.finish_models();
    });
}

ekx_status ekx_model3d_layered_gaussian(const ekx_geometry3d *geometry,
                                        const ekx_layered_gaussian *model,
                                        int64_t n, double *velocity)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(check_geometry3d(geometry));
        EKX_CHECK(check_layered_gaussian(model));
        const ekx_geometry3d &g = *geometry;
        const int64_t nGrid = (int64_t) g.nx*g.ny*g.nz;
        if (n != nGrid || !velocity)
        {
            return fail(EKX_EINVAL, "output must hold the " +
                                        std::to_string(nGrid) + " grid points");
        }
        hipStream_t s = nullptr;
        EKX_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
        DeviceBuffer<double> dv;
        ekx_status rc = dv.allocate((size_t) n);
        if (rc == EKX_OK) { rc = generate_layered_gaussian(g, *model, dv.ptr, s); }
        if (rc == EKX_OK)
        {
            hipError_t e = hipMemcpyAsync(velocity, dv.ptr,
                                          (size_t) n*sizeof(double),
                                          hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) { e = hipStreamSynchronize(s); }
            if (e != hipSuccess)
            {
                rc = fail(EKX_EHIP, std::string("hipMemcpyAsync: ") +
                                        hipGetErrorString(e));
            }
        }
        (void) hipStreamDestroy(s);
        return rc;
    });
}

ekx_status ekx_solver3d_set_layered_gaussian_model(
    ekx_solver3d *h, const ekx_layered_gaussian *model)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        h->engine.haveModel = false;
        h->engine.haveField = false;
        EKX_CHECK(check_layered_gaussian(model));
        const ekx_geometry3d &g = h->geometry;
        Engine3D &e = h->engine;
        e.drop_graph();
        DeviceBuffer<double> dv;
        EKX_CHECK(dv.allocate((size_t) g.nx*g.ny*g.nz));
        EKX_CHECK(generate_layered_gaussian(g, *model, dv.ptr, e.stream));
        EKX_HIP(launch_nodal_to_cell3d(g.nx, g.ny, g.nz, dv.ptr,
                                       EKX_ORDERING_NATURAL, e.S64.ptr,
                                       e.stream));
        EKX_HIP(hipStreamSynchronize(e.stream));
        return e.finish_models();
    });
}

ekx_status ekx_solver3d_set_nodal_velocities(ekx_solver3d *h, int64_t n,
                                             const double *v, int ordering)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        h->engine.haveModel = false;
        h->engine.haveField = false;
        const ekx_geometry3d &g = h->geometry;
        int64_t nGrid = (int64_t) g.nx*g.ny*g.nz;
        if (n != nGrid)
        {
            return fail(EKX_EINVAL, "Number of grid points = " +
                                        std::to_string(n) + " must equal " +
                                        std::to_string(nGrid));
        }
        if (!v) { return fail(EKX_EINVAL, "velocities is NULL"); }
        if (ordering != EKX_ORDERING_NATURAL && ordering != EKX_ORDERING_XYZ)
        {
            return fail(EKX_EINVAL, "unknown ordering");
        }
        // Model3D::setNodalVelocities rejects v <= 0 (src/model3d.cpp:303-307)
        for (int64_t i = 0; i < n; ++i)
        {
            if (!(v[i] > 0))
            {
                return fail(EKX_EINVAL, "Non-positive velocities detected");
            }
        }
        Engine3D &e = h->engine;
        e.drop_graph();
        DeviceBuffer<double> dv;
        EKX_CHECK(dv.allocate((size_t) n));
        EKX_HIP(hipMemcpyAsync(dv.ptr, v, (size_t) n*sizeof(double),
                               hipMemcpyHostToDevice, e.stream));
        EKX_HIP(launch_nodal_to_cell3d(g.nx, g.ny, g.nz, dv.ptr, ordering,
                                       e.S64.ptr, e.stream));
        EKX_HIP(hipStreamSynchronize(e.stream));
        return e.finish_models();
    });
}

ekx_status ekx_solver3d_set_cell_velocities(ekx_solver3d *h, int64_t n,
                                            const double *v, int ordering)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        h->engine.haveModel = false;
        h->engine.haveField = false;
        const ekx_geometry3d &g = h->geometry;
        int64_t nCell = (int64_t) (g.nx - 1)*(g.ny - 1)*(g.nz - 1);
        if (n != nCell)
        {
            return fail(EKX_EINVAL, "Number of cells = " + std::to_string(n) +
                                        " must equal " + std::to_string(nCell));
        }
        if (!v) { return fail(EKX_EINVAL, "velocities is NULL"); }
        if (ordering != EKX_ORDERING_NATURAL && ordering != EKX_ORDERING_XYZ)
        {
            return fail(EKX_EINVAL, "unknown ordering");
        }
        for (int64_t i = 0; i < n; ++i)
        {
            if (!(v[i] > 0))
            {
                return fail(EKX_EINVAL, "Non-positive velocities detected");
            }
        }
        Engine3D &e = h->engine;
        e.drop_graph();
        DeviceBuffer<double> dv;
        EKX_CHECK(dv.allocate((size_t) n));
        EKX_HIP(hipMemcpyAsync(dv.ptr, v, (size_t) n*sizeof(double),
                               hipMemcpyHostToDevice, e.stream));
        EKX_HIP(launch_cell_velocity_to_slowness3d(g.nx, g.ny, g.nz, dv.ptr,
                                                   ordering, e.S64.ptr,
                                                   e.stream));
        EKX_HIP(hipStreamSynchronize(e.stream));
        return e.finish_models();
    });
}

int ekx_solver3d_have_velocity_model(const ekx_solver3d *h)
{
    return h && h->initialized && h->engine.haveModel ? 1 : 0;
}

ekx_status ekx_solver3d_set_source(ekx_solver3d *h, double x, double y,
                                   double z)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        h->engine.haveSource[0] = false;
        h->engine.haveField = false;
        SourceInfo s;
        EKX_CHECK(locate_source3d(h->geometry, x, y, z, s));
        h->engine.sources[0] = s;
        h->engine.haveSource[0] = true;
        return EKX_OK;
    });
}

int ekx_solver3d_have_source(const ekx_solver3d *h)
{
    return h && h->initialized && h->engine.haveSource[0] ? 1 : 0;
}

ekx_status ekx_solver3d_get_source_cell(const ekx_solver3d *h,
                                        double offset[3], int cell[3],
                                        int *cell_index)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        if (!h->engine.haveSource[0])
        {
            return fail(EKX_ESTATE, "Source location not set");
        }
        const SourceInfo &s = h->engine.sources[0];
        for (int k = 0; k < 3; ++k)
        {
            if (offset) { offset[k] = s.offset[k]; }
            if (cell) { cell[k] = s.cell[k]; }
        }
        if (cell_index) { *cell_index = s.cellIndex; }
        return EKX_OK;
    });
}

ekx_status ekx_solver3d_solve(ekx_solver3d *h)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        return h->engine.solve();
    });
}

ekx_status ekx_solver3d_set_wait_bound(ekx_solver3d *h, double ms)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        return h->engine.set_wait_bound(ms);
    });
}

ekx_status ekx_solver3d_autotune(ekx_solver3d *h, int *chunk_planes,
                                 int *chains)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        int c = 0, n = 0;
        EKX_CHECK(h->engine.autotune(c, n));
        if (chunk_planes) { *chunk_planes = c; }
        if (chains) { *chains = n; }
        return EKX_OK;
    });
}

int ekx_solver3d_have_travel_time_field(const ekx_solver3d *h)
{
    return h && h->initialized && h->engine.haveField ? 1 : 0;
}

ekx_status ekx_solver3d_get_travel_times(const ekx_solver3d *h, int64_t n,
                                         double *out)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        return h->engine.copy_field(0, n, out);
    });
}

ekx_status ekx_solver3d_get_travel_times_f32(const ekx_solver3d *h,
                                             int64_t n, float *out)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        const Engine3D &e = h->engine;
        const ekx_geometry3d &g = h->geometry;
        int64_t nGrid = (int64_t) g.nx*g.ny*g.nz;
        if (n != nGrid || !out)
        {
            return fail(EKX_EINVAL, "output must hold the " +
                                        std::to_string(nGrid) + " grid points");
        }
        if (e.T32.ptr && !e.fieldIsF64)
        {
            if (!e.haveField)
            {
                return fail(EKX_ESTATE, "Travel time field not yet computed");
            }
            const float *src = nullptr;
            EKX_CHECK(e.natural_field<float>(0, e.T32.ptr, &src));
            EKX_CHECK(e.copy_out(out, src, (size_t) n*sizeof(float)));
            return EKX_OK;
        }
        std::vector<double> tmp((size_t) n);
        EKX_CHECK(e.copy_field(0, n, tmp.data()));
        for (int64_t i = 0; i < n; ++i) { out[i] = (float) tmp[(size_t) i]; }
        return EKX_OK;
    });
}

ekx_status ekx_solver3d_get_travel_times_device(const ekx_solver3d *h,
                                                const void **ptr,
                                                int *element_size)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        if (!h->engine.haveField)
        {
            return fail(EKX_ESTATE, "Travel time field not yet computed");
        }
        const Engine3D &e = h->engine;
        if (!e.fieldIsF64 && !e.T32.ptr)
        {
            return fail(EKX_ESTATE, "a FIXED32 field is stored as scaled "
                                    "integers; copy it with "
                                    "ekx_solver3d_get_travel_times");
        }
        if (ptr)
        {
            if (e.fieldIsF64)
            {
                const double *src = nullptr;
                EKX_CHECK(e.natural_field<double>(0, e.T64.ptr, &src));
                *ptr = src;
            }
            else
            {
                const float *src = nullptr;
                EKX_CHECK(e.natural_field<float>(0, e.T32.ptr, &src));
                *ptr = src;
            }
        }
        if (element_size) { *element_size = e.fieldIsF64 ? 8 : 4; }
        return EKX_OK;
    });
}

ekx_status ekx_solver3d_set_stations(ekx_solver3d *h, int n,
                                     const double *x, const double *y,
                                     const double *z)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        return h->engine.set_stations(n, x, y, z);
    });
}

ekx_status ekx_solver3d_get_number_of_stations(const ekx_solver3d *h,
                                               int *n)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        if (!n) { return fail(EKX_EINVAL, "n is NULL"); }
        *n = h->engine.nStations;
        return EKX_OK;
    });
}

ekx_status ekx_solver3d_get_travel_times_at_stations(const ekx_solver3d *h,
                                                     int n, double *out)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        return h->engine.copy_station_times(0, n, out);
    });
}

ekx_status ekx_solver3d_compute_travel_time_gradient_field(ekx_solver3d *h)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        return h->engine.compute_gradient(0);
    });
}

int ekx_solver3d_have_travel_time_gradient_field(const ekx_solver3d *h)
{
    return h && h->initialized && h->engine.have_gradient(0) ? 1 : 0;
}

ekx_status ekx_solver3d_get_travel_time_gradient_field(
    const ekx_solver3d *h, int64_t n, double *out)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        return h->engine.copy_gradient(0, n, out);
    });
}

ekx_status ekx_solver3d_get_travel_time_gradient_field_device(
    const ekx_solver3d *h, const double **ptr)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        if (!h->engine.have_gradient(0))
        {
            return fail(EKX_ESTATE, "Travel time gradient field not yet "
                                    "computed");
        }
        if (!ptr) { return fail(EKX_EINVAL, "ptr is NULL"); }
        *ptr = h->engine.G.ptr;
        return EKX_OK;
    });
}

ekx_status ekx_solver3d_get_stats(const ekx_solver3d *h,
                                  ekx_solve_stats *stats)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        if (!stats) { return fail(EKX_EINVAL, "stats is NULL"); }
        *stats = h->engine.stats;
        return EKX_OK;
    });
}

ekx_status ekx_solver3d_get_stream(const ekx_solver3d *h, void **stream)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_initialized(h));
        if (!stream) { return fail(EKX_EINVAL, "stream is NULL"); }
        *stream = (void *) h->engine.stream;
        return EKX_OK;
    });
}

// ------------------------------ Batch3D -----------------------------------
ekx_status ekx_batch3d_create(ekx_batch3d **batch)
{
    return guarded([&]() -> ekx_status
    {
        if (!batch) { return fail(EKX_EINVAL, "batch is NULL"); }
        *batch = new (std::nothrow) ekx_batch3d();
        if (!*batch) { return fail(EKX_ENOMEM, "out of host memory"); }
        return EKX_OK;
    });
}

void ekx_batch3d_destroy(ekx_batch3d *batch) { delete batch; }

ekx_status ekx_batch3d_initialize(ekx_batch3d *h,
                                  const ekx_solver_options *options,
                                  int n, const ekx_problem3d *problems)
{
    return guarded([&]() -> ekx_status
    {
        if (!h) { return fail(EKX_EINVAL, "batch is NULL"); }
        h->initialized = false;
        EKX_CHECK(check_options(options));
        if (n < 1 || !problems)
        {
            return fail(EKX_EINVAL, "a batch needs at least one problem");
        }
        std::vector<ekx_geometry3d> geoms((size_t) n);
        std::vector<int> modelOf((size_t) n);
        std::map<std::tuple<const double *, int, int, int>, int> models;
        std::vector<const double *> modelPtr;
        for (int i = 0; i < n; ++i)
        {
            const ekx_problem3d &pr = problems[i];
            EKX_CHECK(check_geometry3d(&pr.geometry));
            if (!pr.slowness)
            {
                return fail(EKX_EINVAL, "problem " + std::to_string(i) +
                                            ": slowness is NULL");
            }
            geoms[i] = pr.geometry;
            auto key = std::make_tuple(pr.slowness, pr.geometry.nx,
                                       pr.geometry.ny, pr.geometry.nz);
            auto it = models.find(key);
            if (it == models.end())
            {
                int m = (int) modelPtr.size();
                models.emplace(key, m);
                modelPtr.push_back(pr.slowness);
                modelOf[i] = m;
            }
            else { modelOf[i] = it->second; }
        }
        Engine3D &e = h->engine;
        EKX_CHECK(e.setup(*options, geoms, modelOf, (int) modelPtr.size()));
        std::vector<bool> uploaded(modelPtr.size(), false);
        for (int i = 0; i < n; ++i)
        {
            int m = modelOf[i];
            if (uploaded[m]) { continue; }
            const ekx_geometry3d &g = geoms[i];
            int64_t nCell = (int64_t) (g.nx - 1)*(g.ny - 1)*(g.nz - 1);
            const double *s = modelPtr[m];
            for (int64_t k = 0; k < nCell; ++k)
            {
                if (!(s[k] > 0))
                {
                    return fail(EKX_EINVAL, "problem " + std::to_string(i) +
                                                ": non-positive slowness");
                }
            }
            EKX_CHECK(e.upload_model(m, s, nCell));
            uploaded[m] = true;
        }
        EKX_CHECK(e.finish_models());
        for (int i = 0; i < n; ++i)
        {
            SourceInfo s;
            EKX_CHECK(locate_source3d(geoms[i], problems[i].source[0],
                                      problems[i].source[1],
                                      problems[i].source[2], s));
            e.sources[i] = s;
            e.haveSource[i] = true;
        }
        h->initialized = true;
        return EKX_OK;
    });
}

static ekx_status require_batch(const ekx_batch3d *h)
{
    if (!h) { return fail(EKX_EINVAL, "batch is NULL"); }
    if (!h->initialized) { return fail(EKX_ESTATE, "Class not initialized"); }
    return EKX_OK;
}

ekx_status ekx_batch3d_set_source(ekx_batch3d *h, int problem, double x,
                                  double y, double z)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_batch(h));
        Engine3D &e = h->engine;
        if (problem < 0 || problem >= (int) e.problems.size())
        {
            return fail(EKX_EINVAL, "problem index out of range");
        }
        e.haveField = false;
        e.haveSource[problem] = false;
        SourceInfo s;
        EKX_CHECK(locate_source3d(e.geometry[problem], x, y, z, s));
        e.sources[problem] = s;
        e.haveSource[problem] = true;
        return EKX_OK;
    });
}

ekx_status ekx_batch3d_solve(ekx_batch3d *h)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_batch(h));
        return h->engine.solve();
    });
}

ekx_status ekx_batch3d_set_wait_bound(ekx_batch3d *h, double ms)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_batch(h));
        return h->engine.set_wait_bound(ms);
    });
}

ekx_status ekx_batch3d_autotune(ekx_batch3d *h, int *chunk_planes, int *chains)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_batch(h));
        int c = 0, n = 0;
        EKX_CHECK(h->engine.autotune(c, n));
        if (chunk_planes) { *chunk_planes = c; }
        if (chains) { *chains = n; }
        return EKX_OK;
    });
}

ekx_status ekx_batch3d_get_travel_times(const ekx_batch3d *h, int problem,
                                        int64_t n, double *out)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_batch(h));
        if (problem < 0 || problem >= (int) h->engine.problems.size())
        {
            return fail(EKX_EINVAL, "problem index out of range");
        }
        return h->engine.copy_field(problem, n, out);
    });
}

static ekx_status check_problem(const ekx_batch3d *h, int problem)
{
    if (problem < 0 || problem >= (int) h->engine.problems.size())
    {
        return fail(EKX_EINVAL, "problem index out of range");
    }
    return EKX_OK;
}

ekx_status ekx_batch3d_set_stations(ekx_batch3d *h, int n, const double *x,
                                    const double *y, const double *z)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_batch(h));
        return h->engine.set_stations(n, x, y, z);
    });
}

ekx_status ekx_batch3d_get_travel_times_at_stations(const ekx_batch3d *h,
                                                    int problem, int n,
                                                    double *out)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_batch(h));
        EKX_CHECK(check_problem(h, problem));
        return h->engine.copy_station_times(problem, n, out);
    });
}

ekx_status ekx_batch3d_get_station_table(const ekx_batch3d *h, int64_t n,
                                         double *out)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_batch(h));
        const Engine3D &e = h->engine;
        const int64_t want = (int64_t) e.problems.size()*e.nStations;
        if (!e.haveField || e.stationStamp != e.solveStamp)
        {
            return fail(EKX_ESTATE, "Travel time field not yet computed");
        }
        if (n != want || (n > 0 && !out))
        {
            return fail(EKX_EINVAL, "output must hold problems x stations = " +
                                        std::to_string(want) + " values");
        }
        std::copy(e.stationTimes.begin(), e.stationTimes.end(), out);
        return EKX_OK;
    });
}

ekx_status ekx_batch3d_compute_travel_time_gradient_field(ekx_batch3d *h,
                                                          int problem)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_batch(h));
        EKX_CHECK(check_problem(h, problem));
        return h->engine.compute_gradient(problem);
    });
}

ekx_status ekx_batch3d_get_travel_time_gradient_field(const ekx_batch3d *h,
                                                      int problem, int64_t n,
                                                      double *out)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_batch(h));
        EKX_CHECK(check_problem(h, problem));
        return h->engine.copy_gradient(problem, n, out);
    });
}

ekx_status ekx_batch3d_get_stats(const ekx_batch3d *h,
                                 ekx_solve_stats *stats)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_batch(h));
        if (!stats) { return fail(EKX_EINVAL, "stats is NULL"); }
        *stats = h->engine.stats;
        return EKX_OK;
    });
}

ekx_status ekx_batch3d_get_stream(const ekx_batch3d *h, void **stream)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(require_batch(h));
        if (!stream) { return fail(EKX_EINVAL, "stream is NULL"); }
        *stream = (void *) h->engine.stream;
        return EKX_OK;
    });
}

// ------------------------- allocation-free solve ----------------------------
ekx_status ekx_solve3d_noalloc(const ekx_solver_options *options,
                               const ekx_geometry3d *geometry, int n_sources,
                               const double *sources_xyz,
                               const double *d_slowness,
                               double *d_travel_times, void *stream)
{
    return guarded([&]() -> ekx_status
    {
        EKX_CHECK(check_options(options));
        EKX_CHECK(check_geometry3d(geometry));
        if (n_sources < 1 || n_sources > EKX_NOALLOC_MAX_SOURCES)
        {
            return fail(EKX_EINVAL, "n_sources = " +
                                        std::to_string(n_sources) +
                                        " must be in [1, " +
                                        std::to_string(
                                            EKX_NOALLOC_MAX_SOURCES) + "]");
        }
        if (!sources_xyz || !d_slowness || !d_travel_times)
        {
            return fail(EKX_EINVAL, "sources, slowness and travel times "
                                    "must not be NULL");
        }
        if (options->precision != EKX_PRECISION_FP64)
        {
            return fail(EKX_EINVAL, "the allocation-free solve is FP64");
        }
        if (options->kernel == EKX_KERNEL_COLUMN)
        {
            return fail(EKX_EINVAL, "the allocation-free solve runs the "
                                    "hyperplane kernel (the column kernel "
                                    "needs its tiled workspace)");
        }
        if (options->early_exit != 0)
        {
            return fail(EKX_EINVAL, "early exit needs a host round trip "
                                    "per iteration; not available "
                                    "without allocation");
        }
        Problem3D *dp = nullptr;
        EKX_CHECK(scratch_address(&dp));
        const ekx_geometry3d &g = *geometry;
        const int64_t nGrid = (int64_t) g.nx*g.ny*g.nz;
        hipStream_t s = static_cast<hipStream_t>(stream);
        // descriptors: natural layout, source k's field at k nGrid, the
        // source-cell slowness filled in on the device
        Problem3D host[EKX_NOALLOC_MAX_SOURCES];
        for (int k = 0; k < n_sources; ++k)
        {
            SourceInfo si;
            EKX_CHECK(locate_source3d(g, sources_xyz[3*k],
                                      sources_xyz[3*k + 1],
                                      sources_xyz[3*k + 2], si));
            Problem3D &p = host[k];
            p = Problem3D{};
            p.nx = g.nx;
            p.ny = g.ny;
            p.nz = g.nz;
            p.radius = options->factored_radius;
            p.srcCellX = si.cell[0];
            p.srcCellY = si.cell[1];
            p.srcCellZ = si.cell[2];
            p.uniform = is_uniform3d(g) ? 1 : 0;
            p.dx = g.dx;
            p.dy = g.dy;
            p.dz = g.dz;
            p.srcOffX = si.offset[0];
            p.srcOffY = si.offset[1];
            p.srcOffZ = si.offset[2];
            p.tOffset = k*nGrid;
            p.sOffset = 0;
            p.nu = non_uniform_constants(g);
            p.tiled = 0;
            p.nTX = tiles_of(g.nx);
            p.nTY = tiles_of(g.ny);
            p.tCount = nGrid;
            EKX_HIP(launch_store_problem3d(p, si.cellIndex, d_slowness,
                                           dp + k, s));
        }
        // Solver3DImpl::initializeTravelTimes, then the schedule of
        // Engine3D::enqueue_phase_sweeps on the hyperplane kernel
        EKX_HIP(launch_init3d<double>(dp, n_sources, n_sources*nGrid,
                                      d_travel_times, s));
        auto sweepAll = [&](int sweep, bool initialize) -> ekx_status
        {
            for (int k = 0; k < n_sources; ++k)
            {
                const Problem3D &p = host[k];
                const HostOctant o = host_octant(p, sweep, initialize);
                const int lastLevel = (p.nx - 1) + (p.ny - 1) + (p.nz - 1);
                for (int L = o.jx0 + o.jy0 + o.jz0; L <= lastLevel; ++L)
                {
                    const int kLo = std::max(o.jz0,
                                             L - (p.nx - 1) - (p.ny - 1));
                    const int kHi = std::min(p.nz - 1, L - o.jx0 - o.jy0);
                    if (kLo > kHi) { continue; }
                    const int nPairs = (kHi - kLo + 1)*(p.ny - o.jy0);
                    EKX_HIP(launch_hyperplane3d<double>(
                        dp, k, sweep, initialize ? 1 : 0, L, kLo, nPairs,
                        d_travel_times, d_slowness, nullptr, s));
                }
            }
            return EKX_OK;
        };
        if (options->schedule == EKX_SCHEDULE_SHIPPED)
        {
            // src/solver3d.cpp:451-463 (FSM); level set: nothing
            if (options->algorithm == EKX_FAST_SWEEPING_METHOD)
            {
                EKX_CHECK(sweepAll(0, true));
                EKX_CHECK(sweepAll(1, true));
            }
            return EKX_OK;
        }
        for (int sw = 0; sw < 8; ++sw) { EKX_CHECK(sweepAll(sw, true)); }
        for (int it = 0; it < options->number_of_sweeps; ++it)
        {
            for (int sw = 0; sw < 8; ++sw) { EKX_CHECK(sweepAll(sw, false)); }
        }
        return EKX_OK;
    });
}

} // extern "C"
