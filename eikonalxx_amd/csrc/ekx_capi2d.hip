// ekx_capi2d.hip -- C ABI of the 2D solver (include/eikonalxx_amd.h).
#include "eikonalxx_amd.h"
#include "ekx_guard.hpp"
#include "ekx_kernels.hpp"
#include "ekx_reads.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <string>
#include <vector>

using namespace ekx;

// The 3D translation unit owns the per-thread error message.
namespace ekx
{
void set_last_error(const std::string &message);
}

namespace
{

ekx_status fail2(ekx_status status, const std::string &message)
{
    ekx::set_last_error(message);
    return status;
}

#define EKX2_HIP(expr)                                                       \
    do                                                                       \
    {                                                                        \
        hipError_t e_ = (expr);                                              \
        if (e_ != hipSuccess)                                                \
        {                                                                    \
            return fail2(EKX_EHIP, std::string(#expr) + ": " +               \
                                       hipGetErrorString(e_));               \
        }                                                                    \
    } while (0)

#define EKX2_CHECK(expr)                                                     \
    do                                                                       \
    {                                                                        \
        ekx_status s_ = (expr);                                              \
        if (s_ != EKX_OK) { return s_; }                                     \
    } while (0)

template <typename T> struct Buf
{
    T *ptr = nullptr;
    size_t count = 0;
    Buf() = default;
    Buf(const Buf &) = delete;
    Buf &operator=(const Buf &) = delete;
    ~Buf() { release(); }
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
            return fail2(EKX_ENOMEM, std::string("hipMalloc failed: ") +
                                         hipGetErrorString(e));
        }
        count = n;
        return EKX_OK;
    }
};

// The band kernel's buffers, in one allocation: skewed travel times (work)
// and skewed cells; none (both counts 0) for grids that it does not take.
// Memory that the device does not have is no error: the solve then runs the
// level kernel, which needs neither.
struct Bands2D
{
    Buf<double> all;
    double *work = nullptr, *cells = nullptr;
    bool allocate(int64_t workValues, int64_t cellValues)
    {
        work = cells = nullptr;
        if (all.allocate((size_t) (workValues + cellValues)) != EKX_OK)
        {
            (void) hipGetLastError();
            all.release();
            return false;
        }
        if (all.ptr)
        {
            work = all.ptr;
            cells = all.ptr + workValues;
        }
        return true;
    }
};

// Slowness range of a model, and whether the band kernel's square roots
// without range tests cover it on a grid: h s at least 2^-345 (2^-700 <= hs0
// hs0), and no time at the source cell's corners above HUGE.
struct Range2D
{
    double lo = std::numeric_limits<double>::infinity(), hi = 0;
    // (in pairs and four at a time: one chain of minima was half of
    // set_slowness, 0.5 of 0.76 ms on 366 000 cells)
    void add(const double *v, int64_t n)
    {
        using Pair = double __attribute__((ext_vector_type(2)));
        constexpr int kPairs = 4;
        Pair a[kPairs], b[kPairs];
        for (int k = 0; k < kPairs; ++k) { a[k] = lo, b[k] = hi; }
        int64_t i = 0;
        for (; i + 2*kPairs <= n; i += 2*kPairs)
        {
#pragma unroll
            for (int k = 0; k < kPairs; ++k)
            {
                Pair x;
                std::memcpy(&x, v + i + 2*k, sizeof(x));
                a[k] = x < a[k] ? x : a[k];
                b[k] = x > b[k] ? x : b[k];
            }
        }
        for (; i < n; ++i)
        {
            lo = std::min(lo, v[i]);
            hi = std::max(hi, v[i]);
        }
        for (int k = 0; k < kPairs; ++k)
        {
            lo = std::min(lo, std::min(a[k].x, a[k].y));
            hi = std::max(hi, std::max(b[k].x, b[k].y));
        }
    }
    bool scaled(const ekx_geometry2d &g) const
    {
        return std::min(g.dx, g.dz)*lo >= 0x1p-345 &&
               (g.dx + g.dz)*hi <= kHuge;
    }
};

// Host to device on the handle's own stream, and its end: on the default
// stream it fails while another thread's solver captures.
ekx_status upload2d(void *dst, const void *src, size_t bytes,
                    hipStream_t stream)
{
    EKX2_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream));
    EKX2_HIP(hipStreamSynchronize(stream));
    return EKX_OK;
}

// (201 x 201, out of range: 2.8 ms by levels in LDS, 3.1 by levels in
// memory, 1.5 by bands with range tests, 1.2 without)
int route2d(bool bands, bool scaled)
{
    return !bands ? kLevels2d : scaled ? kBands2d : kBandsAnyRange2d;
}

std::string f2s(double v) { return std::to_string(v); }

struct Loc2D
{
    double off[2];
    int cell[2];
};

// Source2D / Station2D location -> offset and cell (src/source2d.cpp,
// src/station2d.cpp:155-158, 210-213).
ekx_status locate2d(const ekx_geometry2d &g, double x, double z, Loc2D &l,
                    const char *what)
{
    const double xmax = g.x0 + (g.nx - 1)*g.dx;
    const double zmax = g.z0 + (g.nz - 1)*g.dz;
    if (x < g.x0 || x > xmax)
    {
        return fail2(EKX_EINVAL, std::string("x ") + what + " position = " +
                                     f2s(x) + " must be in range [" +
                                     f2s(g.x0) + "," + f2s(xmax) + "]");
    }
    if (z < g.z0 || z > zmax)
    {
        return fail2(EKX_EINVAL, std::string("z ") + what + " position = " +
                                     f2s(z) + " must be in range [" +
                                     f2s(g.z0) + "," + f2s(zmax) + "]");
    }
    l.off[0] = x - g.x0;
    l.off[1] = z - g.z0;
    l.cell[0] = std::min(g.nx - 2, (int) (l.off[0]/g.dx));
    l.cell[1] = std::min(g.nz - 2, (int) (l.off[1]/g.dz));
    return EKX_OK;
}

} // namespace

// Solver2DSweep::initialize (include/private/solver2d.hpp:29-46): the
// problem constants of a geometry.
static Problem2D problem2d(const ekx_geometry2d &g, const ekx_solver_options &o)
{
    Problem2D p{};
    p.nx = g.nx;
    p.nz = g.nz;
    p.radius = o.factored_radius;
    p.nSweeps = o.number_of_sweeps;
    p.uniform = std::abs(g.dx - g.dz) <
                std::numeric_limits<double>::epsilon()*100 ? 1 : 0;
    p.dx = g.dx;
    p.dz = g.dz;
    p.dx_dz = g.dx/g.dz;
    p.dz_dx = g.dz/g.dx;
    p.cosTheta = g.dx/std::hypot(g.dx, g.dz);
    p.sinTheta = g.dz/std::hypot(g.dx, g.dz);
    p.dxinv = 1/g.dx;
    p.dzinv = 1/g.dz;
    p.hx2inv = 1/(g.dx*g.dx);
    p.hz2inv = 1/(g.dz*g.dz);
    p.twoOverH = 2/g.dx;
    p.twoOverH2 = 2/(g.dx*g.dx);
    p.halfOverH2 = 1/(2*(g.dx*g.dx));
    return p;
}

// Geometry2D setters (src/geometry2d.cpp)
static ekx_status check_geometry2d(const ekx_geometry2d &g)
{
    if (g.nx < 3 || g.nz < 3)
    {
        return fail2(EKX_EINVAL, "Number of grid points must be at least 3");
    }
    if (!(g.dx > 0) || !(g.dz > 0))
    {
        return fail2(EKX_EINVAL, "Grid spacing must be positive");
    }
    if ((int64_t) g.nx*g.nz > (int64_t) std::numeric_limits<int>::max())
    {
        return fail2(EKX_EINVAL, "grid too large");
    }
    return EKX_OK;
}

// Local updates of one solve: 4 initialization sweeps over the source
// quadrants, then nSweeps x 4 refinement sweeps.
static int64_t updates2d(const Problem2D &p)
{
    int64_t u = 0;
    for (int s = 0; s < 4; ++s)
    {
        int negX = s & 1, negZ = (s >> 1) & 1;
        int jx0 = negX ? std::max(p.nx - 2 - p.srcCellX, 1)
                       : std::max(p.srcCellX, 1);
        int jz0 = negZ ? std::max(p.nz - 2 - p.srcCellZ, 1)
                       : std::max(p.srcCellZ, 1);
        u += (int64_t) (p.nx - jx0)*(p.nz - jz0);
    }
    return u + (int64_t) p.nSweeps*4*(p.nx - 1)*(p.nz - 1);
}

struct ekx_solver2d
{
    ekx_solver_options opt{};
    ekx_geometry2d geometry{};
    Problem2D problem{};
    Loc2D source{};
    std::vector<Loc2D> stations;
    Buf<double> S, T, stationOut, stationX, stationZ;
    Bands2D bands;                  // none: level kernel
    Buf<int> stationCX, stationCZ;
    Buf<Problem2D> dProblem;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    bool initialized = false, haveModel = false, haveSource = false;
    bool haveField = false;
    bool scaled = false;            // the model suits the band kernel
    std::vector<double> stationTimes;
    // travel-time gradient (2 values per node) of the current field
    Buf<double> G;
    bool haveGradient = false;
    ekx_solve_stats stats{};
    ~ekx_solver2d()
    {
        if (ev0) { (void) hipEventDestroy(ev0); }
        if (ev1) { (void) hipEventDestroy(ev1); }
        if (stream) { (void) hipStreamDestroy(stream); }
    }
};

// The band kernel's cells from the model in S.
static ekx_status skew_model(ekx_solver2d *h)
{
    if (h->bands.cells)
    {
        EKX2_HIP(launch_skew_cells2d(h->geometry.nx, h->geometry.nz,
                                     h->S.ptr, h->bands.cells, h->stream));
    }
    return EKX_OK;
}

static ekx_status require2d(const ekx_solver2d *h)
{
    if (!h) { return fail2(EKX_EINVAL, "solver is NULL"); }
    if (!h->initialized)
    {
        return fail2(EKX_ESTATE, "Class not initialized");
    }
    return EKX_OK;
}

extern "C" {

ekx_status ekx_solver2d_create(ekx_solver2d **solver)
{
    return guarded([&]() -> ekx_status
    {
        if (!solver) { return fail2(EKX_EINVAL, "solver is NULL"); }
        *solver = new (std::nothrow) ekx_solver2d();
        if (!*solver) { return fail2(EKX_ENOMEM, "out of host memory"); }
        return EKX_OK;
    });
}

void ekx_solver2d_destroy(ekx_solver2d *solver) { delete solver; }

ekx_status ekx_solver2d_initialize(ekx_solver2d *h,
                                   const ekx_solver_options *options,
                                   const ekx_geometry2d *g)
{
    return guarded([&]() -> ekx_status
    {
        if (!h) { return fail2(EKX_EINVAL, "solver is NULL"); }
        h->initialized = false;
        h->haveModel = h->haveSource = h->haveField = false;
        if (!options || !g)
        {
            return fail2(EKX_EINVAL, "options and geometry must not be NULL");
        }
        if (options->number_of_sweeps < 0 || options->number_of_sweeps > 65535)
        {
            return fail2(EKX_EINVAL, "number_of_sweeps must be in [0, 65535]");
        }
        EKX2_CHECK(check_geometry2d(*g));
        h->opt = *options;
        h->geometry = *g;
        if (!h->stream)
        {
            EKX2_HIP(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
            EKX2_HIP(hipEventCreate(&h->ev0));
            EKX2_HIP(hipEventCreate(&h->ev1));
        }
        Problem2D &p = h->problem;
        p = problem2d(*g, *options);
        p.tOffset = 0;
        p.sOffset = 0;
        EKX2_CHECK(h->S.allocate((size_t) (g->nx - 1)*(g->nz - 1)));
        EKX2_CHECK(h->T.allocate((size_t) g->nx*g->nz));
        EKX2_CHECK(h->dProblem.allocate(1));
        const bool bands = fits_bands2d(g->nx, g->nz);
        h->bands.allocate(bands ? band_values2d(g->nx, g->nz) : 0,
                          bands ? cell_values2d(g->nx, g->nz) : 0);
        p.wOffset = 0;
        p.cOffset = 0;
        EKX2_HIP(hipMemsetAsync(h->T.ptr, 0, h->T.count*sizeof(double),
                                h->stream));
        EKX2_HIP(hipStreamSynchronize(h->stream));
        h->stations.clear();
        h->stationTimes.clear();
        h->initialized = true;
        return EKX_OK;
    });
}

ekx_status ekx_solver2d_set_slowness(ekx_solver2d *h, int64_t n,
                                     const double *s)
{
    return guarded([&]() -> ekx_status
    {
        EKX2_CHECK(require2d(h));
        h->haveModel = false;
        h->haveField = false;
        int64_t nCell = (int64_t) (h->geometry.nx - 1)*(h->geometry.nz - 1);
        if (n != nCell || !s)
        {
            return fail2(EKX_EINVAL, "Number of cells = " + std::to_string(n) +
                                         " must equal " + std::to_string(nCell));
        }
        Range2D range;
        range.add(s, n);
        if (!(range.lo > 0))
        {
            return fail2(EKX_EINVAL, "Non-positive slowness detected");
        }
        h->scaled = range.scaled(h->geometry);
        EKX2_HIP(hipMemcpyAsync(h->S.ptr, s, (size_t) n*sizeof(double),
                                hipMemcpyHostToDevice, h->stream));
        EKX2_CHECK(skew_model(h));
        EKX2_HIP(hipStreamSynchronize(h->stream));
        h->haveModel = true;
        return EKX_OK;
    });
}

ekx_status ekx_solver2d_set_nodal_velocities(ekx_solver2d *h, int64_t n,
                                             const double *v, int ordering)
{
    return guarded([&]() -> ekx_status
    {
        EKX2_CHECK(require2d(h));
        h->haveModel = false;
        h->haveField = false;
        int64_t nGrid = (int64_t) h->geometry.nx*h->geometry.nz;
        if (n != nGrid || !v)
        {
            return fail2(EKX_EINVAL, "Number of grid points = " +
                                         std::to_string(n) + " must equal " +
                                         std::to_string(nGrid));
        }
        if (ordering != EKX_ORDERING_NATURAL && ordering != EKX_ORDERING_XYZ)
        {
            return fail2(EKX_EINVAL, "unknown ordering");
        }
        Range2D velocity;
        velocity.add(v, n);
        if (!(velocity.lo > 0))
        {
            return fail2(EKX_EINVAL, "Non-positive velocities detected");
        }
        // (a cell's slowness is 4 over the sum of its corners' velocities)
        Range2D range;
        range.lo = 1/velocity.hi;
        range.hi = 1/velocity.lo;
        h->scaled = range.scaled(h->geometry);
        Buf<double> dv;
        EKX2_CHECK(dv.allocate((size_t) n));
        EKX2_HIP(hipMemcpyAsync(dv.ptr, v, (size_t) n*sizeof(double),
                                hipMemcpyHostToDevice, h->stream));
        EKX2_HIP(launch_nodal_to_cell2d(h->geometry.nx, h->geometry.nz, dv.ptr,
                                        ordering, h->S.ptr, h->stream));
        EKX2_CHECK(skew_model(h));
        EKX2_HIP(hipStreamSynchronize(h->stream));
        h->haveModel = true;
        return EKX_OK;
    });
}

ekx_status ekx_solver2d_set_source(ekx_solver2d *h, double x, double z)
{
    return guarded([&]() -> ekx_status
    {
        EKX2_CHECK(require2d(h));
        h->haveSource = false;
        h->haveField = false;
        Loc2D l;
        EKX2_CHECK(locate2d(h->geometry, x, z, l, "source"));
        h->source = l;
        h->haveSource = true;
        return EKX_OK;
    });
}

ekx_status ekx_solver2d_set_stations(ekx_solver2d *h, int n, const double *x,
                                     const double *z)
{
    return guarded([&]() -> ekx_status
    {
        EKX2_CHECK(require2d(h));
        if (n < 0 || (n > 0 && (!x || !z)))
        {
            return fail2(EKX_EINVAL, "invalid station arrays");
        }
        std::vector<Loc2D> locs((size_t) n);
        for (int i = 0; i < n; ++i)
        {
            EKX2_CHECK(locate2d(h->geometry, x[i], z[i], locs[i], "station"));
        }
        h->stations = locs;
        h->stationTimes.clear();
        std::vector<double> xo(n), zo(n);
        std::vector<int> cx(n), cz(n);
        for (int i = 0; i < n; ++i)
        {
            xo[i] = locs[i].off[0];
            zo[i] = locs[i].off[1];
            cx[i] = locs[i].cell[0];
            cz[i] = locs[i].cell[1];
        }
        size_t m = (size_t) std::max(n, 1);
        EKX2_CHECK(h->stationX.allocate(m));
        EKX2_CHECK(h->stationZ.allocate(m));
        EKX2_CHECK(h->stationCX.allocate(m));
        EKX2_CHECK(h->stationCZ.allocate(m));
        EKX2_CHECK(h->stationOut.allocate(m));
        if (n > 0)
        {
            EKX2_CHECK(upload2d(h->stationX.ptr, xo.data(), n*sizeof(double),
                                h->stream));
            EKX2_CHECK(upload2d(h->stationZ.ptr, zo.data(), n*sizeof(double),
                                h->stream));
            EKX2_CHECK(upload2d(h->stationCX.ptr, cx.data(), n*sizeof(int),
                                h->stream));
            EKX2_CHECK(upload2d(h->stationCZ.ptr, cz.data(), n*sizeof(int),
                                h->stream));
        }
        return EKX_OK;
    });
}

ekx_status ekx_solver2d_solve(ekx_solver2d *h)
{
    return guarded([&]() -> ekx_status
    {
        EKX2_CHECK(require2d(h));
        h->haveField = false;
        if (!h->haveModel)
        {
            return fail2(EKX_ESTATE, "Velocity model not set");
        }
        if (!h->haveSource)
        {
            return fail2(EKX_ESTATE, "Source location not set");
        }
        Problem2D &p = h->problem;
        p.srcCellX = h->source.cell[0];
        p.srcCellZ = h->source.cell[1];
        p.srcOffX = h->source.off[0];
        p.srcOffZ = h->source.off[1];
        p.route = route2d(h->bands.work != nullptr, h->scaled);
        Plan2D plan;
        plan.add(p);
        // (the source cell's slowness comes from the device's model)
        EKX2_HIP(launch_store_problem2d(
            p, h->S.ptr + (size_t) p.srcCellZ*(h->geometry.nx - 1) +
                   p.srcCellX,
            h->dProblem.ptr, h->stream));
        EKX2_HIP(hipEventRecord(h->ev0, h->stream));
        EKX2_HIP(launch_solve2d(h->dProblem.ptr, 1, plan, h->T.ptr, h->S.ptr,
                                h->bands.work, h->bands.cells, h->stream));
        EKX2_HIP(hipEventRecord(h->ev1, h->stream));
        const int ns = (int) h->stations.size();
        if (ns > 0)
        {
            EKX2_HIP(launch_stations2d(h->dProblem.ptr, ns, h->stationX.ptr,
                                       h->stationZ.ptr, h->stationCX.ptr,
                                       h->stationCZ.ptr, h->T.ptr,
                                       h->stationOut.ptr, h->stream));
        }
        EKX2_HIP(hipStreamSynchronize(h->stream));
        EKX2_HIP(hipGetLastError());
        h->stationTimes.assign((size_t) ns, 0.0);
        if (ns > 0)
        {
            EKX2_HIP(read_back(h->stationTimes.data(), h->stationOut.ptr,
                               ns*sizeof(double), h->stream));
        }
        float ms = 0;
        EKX2_HIP(hipEventElapsedTime(&ms, h->ev0, h->ev1));
        ekx_solve_stats st{};
        st.updates = updates2d(p);
        st.updates_fp64 = st.updates;
        st.kernel_launches = 1;
        st.iterations_run = p.nSweeps;
        st.last_solve_ms = ms;
        h->stats = st;
        h->haveField = true;
        h->haveGradient = false;
        return EKX_OK;
    });
}

ekx_status ekx_solver2d_get_travel_times(const ekx_solver2d *h, int64_t n,
                                         double *out)
{
    return guarded([&]() -> ekx_status
    {
        EKX2_CHECK(require2d(h));
        int64_t nGrid = (int64_t) h->geometry.nx*h->geometry.nz;
        if (n != nGrid || !out)
        {
            return fail2(EKX_EINVAL, "output must hold the " +
                                         std::to_string(nGrid) + " grid points");
        }
        EKX2_HIP(read_back(out, h->T.ptr, (size_t) n*sizeof(double),
                           h->stream));
        return EKX_OK;
    });
}

ekx_status ekx_solver2d_get_travel_times_at_stations(const ekx_solver2d *h,
                                                     int n, double *out)
{
    return guarded([&]() -> ekx_status
    {
        EKX2_CHECK(require2d(h));
        if (!h->haveField)
        {
            return fail2(EKX_ESTATE, "Travel time field not yet computed");
        }
        if (n != (int) h->stationTimes.size() || (n > 0 && !out))
        {
            return fail2(EKX_EINVAL, "output must hold one value per station");
        }
        for (int i = 0; i < n; ++i) { out[i] = h->stationTimes[(size_t) i]; }
        return EKX_OK;
    });
}

// Solver2D::computeTravelTimeGradientField (src/solver2d.cpp:866-879).
ekx_status ekx_solver2d_compute_travel_time_gradient_field(ekx_solver2d *h)
{
    return guarded([&]() -> ekx_status
    {
        EKX2_CHECK(require2d(h));
        if (!h->haveField)
        {
            return fail2(EKX_ESTATE, "Travel time field not yet computed");
        }
        if (h->haveGradient) { return EKX_OK; }
        const ekx_geometry2d &g = h->geometry;
        if (g.nx < 3 || g.nz < 3)
        {
            return fail2(EKX_EINVAL, "At least 3 grid points in x and z for "
                                     "central difference");
        }
        EKX2_CHECK(h->G.allocate(2*(size_t) g.nx*g.nz));
        EKX2_HIP(launch_gradient2d(h->dProblem.ptr, g.nx, g.nz, h->T.ptr,
                                   h->G.ptr, h->stream));
        EKX2_HIP(hipStreamSynchronize(h->stream));
        h->haveGradient = true;
        return EKX_OK;
    });
}

int ekx_solver2d_have_travel_time_gradient_field(const ekx_solver2d *h)
{
    return h && h->initialized && h->haveField && h->haveGradient ? 1 : 0;
}

ekx_status ekx_solver2d_get_travel_time_gradient_field(const ekx_solver2d *h,
                                                       int64_t n,
                                                       double *out)
{
    return guarded([&]() -> ekx_status
    {
        EKX2_CHECK(require2d(h));
        if (!h->haveField || !h->haveGradient)
        {
            return fail2(EKX_ESTATE, "Travel time gradient field not yet "
                                     "computed");
        }
        const int64_t want = 2*(int64_t) h->geometry.nx*h->geometry.nz;
        if (n != want || !out)
        {
            return fail2(EKX_EINVAL, "output must hold 2 x " +
                                         std::to_string(want/2) + " values");
        }
        EKX2_HIP(read_back(out, h->G.ptr, (size_t) n*sizeof(double),
                           h->stream));
        return EKX_OK;
    });
}

ekx_status ekx_solver2d_get_stats(const ekx_solver2d *h,
                                  ekx_solve_stats *stats)
{
    return guarded([&]() -> ekx_status
    {
        EKX2_CHECK(require2d(h));
        if (!stats) { return fail2(EKX_EINVAL, "stats is NULL"); }
        *stats = h->stats;
        return EKX_OK;
    });
}

} // extern "C"

// Many independent 2D problems solved by one launch, one workgroup each
// (no reference counterpart; each problem's field equals that of a
// Solver2D with the same geometry, model and source).
struct ekx_batch2d
{
    ekx_solver_options opt{};
    std::vector<ekx_geometry2d> geoms;
    std::vector<Problem2D> problems;
    Buf<double> S, T;
    // travel times of a slice's problems, cells of every model; none: level
    // kernel
    Bands2D bands;
    Buf<Problem2D> dProblems;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // problems solved by one launch, which the slices after it share the
    // band kernel's travel times with
    struct Slice
    {
        int first = 0, problems = 0;
        Plan2D plan;
    };
    std::vector<Slice> slices;
    bool initialized = false, haveField = false;
    ekx_solve_stats stats{};
    ~ekx_batch2d()
    {
        if (ev0) { (void) hipEventDestroy(ev0); }
        if (ev1) { (void) hipEventDestroy(ev1); }
        if (stream) { (void) hipStreamDestroy(stream); }
    }
};

// Cuts a batch into slices whose skewed travel times fit `values`, of about
// the same size each, and sets the problems' first values in their slice;
// returns the values that the largest needs (0: some problem does not fit).
static int64_t cut_slices(ekx_batch2d &b, int64_t values)
{
    int64_t total = 0, most = 0;
    auto need = [](const Problem2D &p)
    {
        return fits_bands2d(p.nx, p.nz) ? band_values2d(p.nx, p.nz) : 0;
    };
    for (const Problem2D &p : b.problems)
    {
        total += need(p);
        most = std::max(most, need(p));
    }
    if (most > values) { return 0; }
    // a slice begins with the first problem past its share of the total, or
    // with the one that does not fit into the slice before
    const int64_t slices = std::max<int64_t>(1, (total + values - 1)/values);
    int64_t start = 0, used = 0, largest = 0, slice = 0;
    b.slices.assign(1, ekx_batch2d::Slice{});
    for (int i = 0; i < (int) b.problems.size(); ++i)
    {
        Problem2D &p = b.problems[i];
        const int64_t at = total > 0 ? start*slices/total : 0;
        const bool full = used + need(p) > values;
        if ((at > slice || full) && b.slices.back().problems > 0)
        {
            b.slices.push_back(ekx_batch2d::Slice{});
            b.slices.back().first = i;
            used = 0;
        }
        slice = std::max(slice, full ? at + 1 : at);
        p.wOffset = used;
        used += need(p);
        start += need(p);
        b.slices.back().problems += 1;
        largest = std::max(largest, used);
    }
    return largest;
}

static ekx_status require_batch2d(const ekx_batch2d *h)
{
    if (!h) { return fail2(EKX_EINVAL, "batch is NULL"); }
    if (!h->initialized)
    {
        return fail2(EKX_ESTATE, "Class not initialized");
    }
    return EKX_OK;
}

extern "C" {

ekx_status ekx_batch2d_create(ekx_batch2d **batch)
{
    return guarded([&]() -> ekx_status
    {
        if (!batch) { return fail2(EKX_EINVAL, "batch is NULL"); }
        *batch = new (std::nothrow) ekx_batch2d();
        if (!*batch) { return fail2(EKX_ENOMEM, "out of host memory"); }
        return EKX_OK;
    });
}

void ekx_batch2d_destroy(ekx_batch2d *batch) { delete batch; }

ekx_status ekx_batch2d_initialize(ekx_batch2d *h,
                                  const ekx_solver_options *options, int n,
                                  const ekx_problem2d *in)
{
    return guarded([&]() -> ekx_status
    {
        if (!h) { return fail2(EKX_EINVAL, "batch is NULL"); }
        h->initialized = h->haveField = false;
        if (!options || !in || n < 1)
        {
            return fail2(EKX_EINVAL, "options and at least one problem needed");
        }
        if (options->number_of_sweeps < 0 || options->number_of_sweeps > 65535)
        {
            return fail2(EKX_EINVAL, "number_of_sweeps must be in [0, 65535]");
        }
        if (!h->stream)
        {
            EKX2_HIP(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
            EKX2_HIP(hipEventCreate(&h->ev0));
            EKX2_HIP(hipEventCreate(&h->ev1));
        }
        h->opt = *options;
        h->geoms.assign(n, ekx_geometry2d{});
        h->problems.assign(n, Problem2D{});
        // models: one device copy per distinct host pointer
        std::vector<const double *> models;
        std::vector<int64_t> modelOffset, cellOffset;
        std::vector<Range2D> ranges;
        int64_t tTotal = 0, sTotal = 0, cTotal = 0;
        std::vector<char> scaled(n, 0);
        for (int i = 0; i < n; ++i)
        {
            const ekx_geometry2d &g = in[i].geometry;
            EKX2_CHECK(check_geometry2d(g));
            if (!in[i].slowness)
            {
                return fail2(EKX_EINVAL, "problem " + std::to_string(i) +
                                             ": slowness is NULL");
            }
            const int64_t nCell = (int64_t) (g.nx - 1)*(g.nz - 1);
            Loc2D src;
            EKX2_CHECK(locate2d(g, in[i].source[0], in[i].source[1], src,
                                "source"));
            Problem2D p = problem2d(g, *options);
            p.srcCellX = src.cell[0];
            p.srcCellZ = src.cell[1];
            p.srcOffX = src.off[0];
            p.srcOffZ = src.off[1];
            p.srcSlowness = in[i].slowness[(size_t) src.cell[1]*(g.nx - 1) +
                                           src.cell[0]];
            size_t m = std::find(models.begin(), models.end(), in[i].slowness)
                     - models.begin();
            if (m == models.size())
            {
                // a new model: every cell positive (checked once per model)
                Range2D range;
                range.add(in[i].slowness, nCell);
                if (!(range.lo > 0))
                {
                    return fail2(EKX_EINVAL, "problem " + std::to_string(i) +
                                                 ": slowness must be "
                                                 "positive");
                }
                models.push_back(in[i].slowness);
                ranges.push_back(range);
                modelOffset.push_back(sTotal);
                sTotal += nCell;
                cellOffset.push_back(cTotal);
                cTotal += fits_bands2d(g.nx, g.nz)
                              ? cell_values2d(g.nx, g.nz) : 0;
            }
            else
            {
                // a shared model needs the same grid
                for (int j = 0; j < i; ++j)
                {
                    if (in[j].slowness != in[i].slowness) { continue; }
                    if (in[j].geometry.nx != g.nx || in[j].geometry.nz != g.nz)
                    {
                        return fail2(EKX_EINVAL, "problems sharing a model must "
                                                 "share its grid");
                    }
                    break;
                }
            }
            p.sOffset = modelOffset[m];
            p.tOffset = tTotal;
            tTotal += (int64_t) g.nx*g.nz;
            p.cOffset = cellOffset[m];
            scaled[i] = ranges[m].scaled(g);
            h->geoms[i] = g;
            h->problems[i] = p;
        }
        EKX2_CHECK(h->S.allocate((size_t) sTotal));
        EKX2_CHECK(h->T.allocate((size_t) tTotal));
        EKX2_CHECK(h->dProblems.allocate((size_t) n));
        // The skewed times, five fields a problem, are kept for as many
        // problems as 4 GiB hold (2571 of 201 x 201, ten rounds of the
        // device), or fewer where
        // the device has less.
        bool bands = false;
        for (int64_t values = (int64_t) 1 << 29; !bands; values /= 2)
        {
            const int64_t largest = cut_slices(*h, values);
            if (largest == 0) { break; }
            bands = h->bands.allocate(largest, cTotal);
        }
        if (!bands) { h->slices.assign(1, {0, n, Plan2D{}}); }
        for (ekx_batch2d::Slice &slice : h->slices)
        {
            for (int i = slice.first; i < slice.first + slice.problems; ++i)
            {
                Problem2D &p = h->problems[i];
                p.route = route2d(bands && fits_bands2d(p.nx, p.nz),
                                  scaled[i] != 0);
                slice.plan.add(p);
            }
        }
        for (size_t m = 0; m < models.size(); ++m)
        {
            ekx_geometry2d g{};
            for (int i = 0; i < n; ++i)
            {
                if (in[i].slowness == models[m])
                {
                    g = in[i].geometry;
                    break;
                }
            }
            const int64_t nCell = (int64_t) (g.nx - 1)*(g.nz - 1);
            EKX2_HIP(hipMemcpyAsync(h->S.ptr + modelOffset[m], models[m],
                                    (size_t) nCell*sizeof(double),
                                    hipMemcpyHostToDevice, h->stream));
            if (bands && fits_bands2d(g.nx, g.nz))
            {
                EKX2_HIP(launch_skew_cells2d(
                    g.nx, g.nz, h->S.ptr + modelOffset[m],
                    h->bands.cells + cellOffset[m], h->stream));
            }
        }
        EKX2_HIP(hipMemcpyAsync(h->dProblems.ptr, h->problems.data(),
                                (size_t) n*sizeof(Problem2D),
                                hipMemcpyHostToDevice, h->stream));
        EKX2_HIP(hipStreamSynchronize(h->stream));
        h->initialized = true;
        return EKX_OK;
    });
}

ekx_status ekx_batch2d_solve(ekx_batch2d *h)
{
    return guarded([&]() -> ekx_status
    {
        EKX2_CHECK(require_batch2d(h));
        EKX2_HIP(hipEventRecord(h->ev0, h->stream));
        ekx_solve_stats st{};
        for (const ekx_batch2d::Slice &s : h->slices)
        {
            EKX2_HIP(launch_solve2d(h->dProblems.ptr + s.first, s.problems,
                                    s.plan, h->T.ptr, h->S.ptr,
                                    h->bands.work, h->bands.cells,
                                    h->stream));
            st.kernel_launches += s.plan.launches();
        }
        EKX2_HIP(hipEventRecord(h->ev1, h->stream));
        EKX2_HIP(hipEventSynchronize(h->ev1));
        float ms = 0;
        EKX2_HIP(hipEventElapsedTime(&ms, h->ev0, h->ev1));
        for (const Problem2D &p : h->problems) { st.updates += updates2d(p); }
        st.updates_fp64 = st.updates;
        st.iterations_run = h->opt.number_of_sweeps;
        st.last_solve_ms = ms;
        h->stats = st;
        h->haveField = true;
        return EKX_OK;
    });
}

ekx_status ekx_batch2d_get_travel_times(const ekx_batch2d *h, int problem,
                                        int64_t n, double *out)
{
    return guarded([&]() -> ekx_status
    {
        EKX2_CHECK(require_batch2d(h));
        if (problem < 0 || problem >= (int) h->problems.size())
        {
            return fail2(EKX_EINVAL, "problem index out of range");
        }
        if (!h->haveField)
        {
            return fail2(EKX_ESTATE, "Travel time field not yet computed");
        }
        const Problem2D &p = h->problems[problem];
        const int64_t nGrid = (int64_t) p.nx*p.nz;
        if (n != nGrid || !out)
        {
            return fail2(EKX_EINVAL, "output must hold the " +
                                         std::to_string(nGrid) + " grid points");
        }
        EKX2_HIP(read_back(out, h->T.ptr + p.tOffset,
                           (size_t) n*sizeof(double), h->stream));
        return EKX_OK;
    });
}

ekx_status ekx_batch2d_get_stats(const ekx_batch2d *h, ekx_solve_stats *stats)
{
    return guarded([&]() -> ekx_status
    {
        EKX2_CHECK(require_batch2d(h));
        if (!stats) { return fail2(EKX_EINVAL, "stats is NULL"); }
        *stats = h->stats;
        return EKX_OK;
    });
}

} // extern "C"
