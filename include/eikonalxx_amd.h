/*
 * eikonalxx_amd.h -- C ABI of the MI355X (gfx950) fast-sweeping eikonal
 * solver.  Plain pointers and sizes only; no C++ or device types cross
 * this boundary.  All travel-time fields are nodal, x fastest, then y,
 * then z (the reference's include/private/grid.hpp:27-34); slowness
 * fields are cell based with the same ordering over cells
 * (src/model3d.cpp:90).
 *
 * Every entry point returns an ekx_status; ekx_last_error() returns the
 * message of the last failure on the calling thread.  No exception crosses
 * the ABI: EKX_EINVAL corresponds to the reference's std::invalid_argument
 * and EKX_ESTATE to its std::runtime_error (call-order violations).
 *
 * Handles are not thread safe; use one handle per host thread.  Each handle
 * owns one HIP stream and its device buffers.
 *
 * Citations are to files of uofuseismo/eikonalxx.
 */
#ifndef EIKONALXX_AMD_H
#define EIKONALXX_AMD_H
#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define EKX_API __attribute__((visibility("default")))

typedef enum
{
    EKX_OK = 0,
    EKX_EINVAL = 1,   /* invalid argument (std::invalid_argument) */
    EKX_ESTATE = 2,   /* wrong call order (std::runtime_error)     */
    EKX_EHIP = 3,     /* HIP runtime failure                        */
    EKX_ENOMEM = 4    /* device or host allocation failed           */
} ekx_status;

/* include/eikonalxx/enums.hpp:44 */
typedef enum
{
    EKX_LEVEL_SET_METHOD = 0,
    EKX_FAST_SWEEPING_METHOD = 1
} ekx_algorithm;

/* include/eikonalxx/enums.hpp:23 (Ordering3D) / :7 (Ordering2D) */
typedef enum
{
    EKX_ORDERING_NATURAL = 0, /* x fastest (ZYX / ZX) */
    EKX_ORDERING_XYZ = 1      /* z fastest (XYZ / XZ) */
} ekx_ordering;

/* Arithmetic of a solve (no reference counterpart: the reference only
 * instantiates Solver3D<double>, src/solver3d.cpp:626). */
typedef enum
{
    EKX_PRECISION_FP64 = 0,        /* every sweep in double                */
    EKX_PRECISION_FP32_POLISH = 1, /* FP32 sweeps, FP64 near the source,
                                      final iteration (8 sweeps) in FP64   */
    EKX_PRECISION_FP32 = 2,        /* FP32 sweeps, FP64 near the source    */
    EKX_PRECISION_FIXED32 = 3,     /* travel times and slowness stored as
                                      32-bit scaled integers (step ~1e-9 of
                                      the problem's travel-time bound),
                                      FP64 arithmetic                      */
    EKX_PRECISION_FIXED32_POLISH = 4 /* FIXED32, final iteration in FP64   */
} ekx_precision;

/* Sweep schedule of Solver3D::solve.  COMPLETED: 8 initialisation sweeps
 * then number_of_sweeps x 8 refinement sweeps (the schedule of
 * Solver2D::solve, src/solver2d.cpp:514-539, and of the commented-out lines
 * src/solver3d.cpp:465-485).  SHIPPED: what src/solver3d.cpp:451-499 runs
 * today (fast sweeping: initialisation sweeps 1 and 2 only; level set:
 * source initialisation only). */
typedef enum
{
    EKX_SCHEDULE_COMPLETED = 0,
    EKX_SCHEDULE_SHIPPED = 1
} ekx_schedule;

/* Device kernel family for the 3D sweeps.  Both are exact topological
 * orderings of the serial fast-sweeping loop and give identical results. */
typedef enum
{
    EKX_KERNEL_AUTO = 0,
    EKX_KERNEL_HYPERPLANE = 1, /* one launch per i+j+k hyperplane        */
    EKX_KERNEL_COLUMN = 2      /* 8x8 columns, skewed z pipeline in LDS,
                                  one launch per column diagonal         */
} ekx_kernel;

/* Launch order of the column kernel's sweeps (FP64 fields). */
typedef enum
{
    EKX_LAUNCH_AUTO = 0,
    EKX_LAUNCH_DIAGONALS = 1,  /* one launch per diagonal bx+by+bz        */
    EKX_LAUNCH_QUEUE = 2       /* one launch per sweep, chunks from a work
                                  queue in dependency order; each
                                  dependency wait is bounded in time (at
                                  least 250 ms, more for large batches):
                                  past the bound the solve returns
                                  EKX_EHIP and its field must be discarded */
} ekx_launch_order;

/* SolverOptions (include/eikonalxx/solverOptions.hpp:54-97, defaults
 * src/solverOptions.cpp:5-21) plus the device-side choices. */
typedef struct
{
    int number_of_sweeps;          /* refinement iterations, default 5     */
    int factored_radius;           /* grid points, default 3, <0 disables  */
    int algorithm;                 /* ekx_algorithm, default level set     */
    int verbosity;                 /* 0 error .. 3 debug                   */
    double convergence_tolerance;  /* seconds, default 1e-5                */
    int precision;                 /* ekx_precision, default FP64          */
    int schedule;                  /* ekx_schedule, default COMPLETED      */
    int kernel;                    /* ekx_kernel, default AUTO             */
    int early_exit;                /* 0 (default): always run every
                                      iteration, as the reference does (its
                                      tolerance is never tested);
                                      1: stop the refinement iterations once
                                      no update of an iteration lowered a
                                      travel time by more than
                                      convergence_tolerance (3D only)       */
    int use_graph;                 /* 1 (default): replay solves from a
                                      captured hipGraph                     */
    int kernel_timing;             /* 1: issue the launches eagerly and time
                                      every bulk column-kernel launch of the
                                      first precision segment with HIP
                                      events (ekx_solve_stats.timed_*)      */
    int chains;                    /* batches: independent launch chains
                                      (groups of problems on their own
                                      streams, no barrier between them);
                                      0 (default) chooses                  */
    int prefetch_planes;           /* column kernel: z-planes loaded ahead
                                      of the compute, 4, 8 or 12; 0
                                      (default) chooses.  Chunks shorter
                                      than 64 planes (their bulk launches
                                      also run the factored-box columns)
                                      always prefetch 4                    */
    int chunk_planes;              /* column kernel: z-planes per chunk of
                                      a column (chunks run on diagonals
                                      bx+by+bz, shortening the dependency
                                      chain of a sweep); 0 (default): chosen
                                      by size class (whole columns for
                                      large batches, down to 8 planes for
                                      one grid); results do not depend on
                                      it                                   */
    int launch_order;              /* column kernel, FP64 fields: 1: one
                                      launch per diagonal of column chunks;
                                      2: one launch per sweep whose waves
                                      take the chunks from a work queue in
                                      diagonal order and start each once
                                      its upwind chunks are done; 0
                                      (default) chooses: with chunk_planes,
                                      chains and prefetch_planes 0 too,
                                      COMPLETED solves in FP64, FP32 and
                                      FP32_POLISH run as one launch (a
                                      resident wave per column) unless the
                                      diagonals would fill the device;
                                      else one launch per diagonal.
                                      Results do not depend on it          */
} ekx_solver_options;

/* Geometry3D (include/eikonalxx/geometry3d.hpp:50-160). */
typedef struct
{
    int nx, ny, nz;       /* grid points, each >= 3 */
    double dx, dy, dz;    /* grid spacing (m), > 0  */
    double x0, y0, z0;    /* origin (m)             */
} ekx_geometry3d;

/* Geometry2D (include/eikonalxx/geometry2d.hpp). */
typedef struct
{
    int nx, nz;
    double dx, dz;
    double x0, z0;
} ekx_geometry2d;

/* Work and timing of the last solve on a handle. */
typedef struct
{
    int64_t updates;              /* local-solver evaluations: every node
                                     inside a sweep's update range        */
    int64_t updates_fp64;         /* of which evaluated in FP64 sweeps     */
    int64_t updates_factored;     /* of which with the full local update
                                     of the factored-box chunks (column
                                     kernel only)                         */
    int64_t kernel_launches;      /* sweep kernel launches                 */
    int64_t kernel_launches_fp64; /* of which FP64 sweep launches          */
    int64_t timed_launches;       /* bulk column launches timed
                                     (kernel_timing)                       */
    int64_t timed_updates;        /* updates done by the timed launches    */
    int32_t iterations_run;       /* refinement iterations actually run    */
    int32_t tiled;                /* 1: fields in the column kernel's tiled
                                     layout (device copies in natural
                                     order are made on request)           */
    int32_t chunk_planes;         /* column kernel: z-planes per column
                                     chunk (the size-class choice when the
                                     option is 0) of the launches per
                                     diagonal; a solve in one launch
                                     (kernel_launches 1, with polish 2) has
                                     them ready and uses none             */
    int32_t chains;               /* their launch chains                   */
    double timed_kernel_ms;       /* summed durations of the timed launches */
    double last_iteration_change; /* early_exit: largest decrease of one
                                     update in the last refinement
                                     iteration (s); -1 otherwise           */
    double last_solve_ms;         /* device time of the whole last solve   */
    double sweep_ms_fp32;         /* device time of the sweep launches on
                                     4-byte storage (FP32 or FIXED32)      */
    double sweep_ms_fp64;         /* device time of the FP64 sweep launches */
} ekx_solve_stats;

/* ---------------------------------------------------------------------- */
EKX_API const char *ekx_last_error(void);
EKX_API const char *ekx_version(void);
/* SolverOptions::SolverOptions defaults (src/solverOptions.cpp:5-21). */
EKX_API void ekx_solver_options_default(ekx_solver_options *options);
/* Number of visible HIP devices; 0 on a host without a GPU. */
EKX_API ekx_status ekx_device_count(int *count);
/* Blocks until all work of this process on the current device is done. */
EKX_API ekx_status ekx_device_synchronize(void);

/* ---------------------------- Solver3D ---------------------------------
 * Replaces EikonalXX::Solver3D<double> (include/eikonalxx/solver3d.hpp:
 * 19-177, src/solver3d.cpp). */
typedef struct ekx_solver3d ekx_solver3d;

/* Solver3D::Solver3D (src/solver3d.cpp:109-113). */
EKX_API ekx_status ekx_solver3d_create(ekx_solver3d **solver);
/* Solver3D::~Solver3D (src/solver3d.cpp:116-117). */
EKX_API void ekx_solver3d_destroy(ekx_solver3d *solver);
/* Solver3D::initialize(SolverOptions, Geometry3D)
 * (solver3d.hpp:40-41, src/solver3d.cpp:148-194). */
EKX_API ekx_status ekx_solver3d_initialize(ekx_solver3d *solver,
                                           const ekx_solver_options *options,
                                           const ekx_geometry3d *geometry);
/* Solver3D::isInitialized (src/solver3d.cpp:197-201). */
EKX_API int ekx_solver3d_is_initialized(const ekx_solver3d *solver);
/* Solver3D::setVelocityModel(Model3D) with the model's cell slowness
 * (Model3D::getSlownessPointer, src/model3d.cpp:401-409;
 * Solver3D::setVelocityModel src/solver3d.cpp:212-249).  n_cells must be
 * (nx-1)(ny-1)(nz-1); every slowness must be positive. */
EKX_API ekx_status ekx_solver3d_set_slowness(ekx_solver3d *solver,
                                             int64_t n_cells,
                                             const double *slowness);
/* Model3D::setNodalVelocities then Solver3D::setVelocityModel
 * (src/model3d.cpp:285-314, interpolate3d :45-151); the nodal to cell
 * conversion runs on the device. */
EKX_API ekx_status ekx_solver3d_set_nodal_velocities(ekx_solver3d *solver,
                                                     int64_t n_grid,
                                                     const double *velocity,
                                                     int ordering);
/* Model3D::setCellularVelocities then Solver3D::setVelocityModel
 * (src/model3d.cpp:316-375). */
EKX_API ekx_status ekx_solver3d_set_cell_velocities(ekx_solver3d *solver,
                                                    int64_t n_cells,
                                                    const double *velocity,
                                                    int ordering);
/* Solver3D::haveVelocityModel (src/solver3d.cpp:275-279). */
EKX_API int ekx_solver3d_have_velocity_model(const ekx_solver3d *solver);
/* Solver3D::setSource(std::tuple<double,double,double>)
 * (solver3d.hpp:97, src/solver3d.cpp:282-341 with Source3D
 * src/source3d.cpp:161-291). */
EKX_API ekx_status ekx_solver3d_set_source(ekx_solver3d *solver, double x,
                                           double y, double z);
/* Solver3D::haveSource (src/solver3d.cpp:385-389). */
EKX_API int ekx_solver3d_have_source(const ekx_solver3d *solver);
/* Source3D offsets and cell of the current source (src/source3d.cpp:
 * 192-208, 247-263, 309-325, 143-158). */
EKX_API ekx_status ekx_solver3d_get_source_cell(const ekx_solver3d *solver,
                                                double offset[3],
                                                int cell[3], int *cell_index);
/* Solver3D::solve (solver3d.hpp:127, src/solver3d.cpp:391-500). */
EKX_API ekx_status ekx_solver3d_solve(ekx_solver3d *solver);
/* No reference counterpart; for callers that solve many times on one
 * setup.  Times short trial solves (the initialisation sweeps and one
 * refinement iteration) for column z-chunk depths around the size-class
 * default and for 1, 2 or 4 launch chains, and for the solve in one launch
 * where the options allow it, and keeps the fastest for later solves.
 * Fields do not depend on the shape.  Needs the model and the source set;
 * discards the current field.  chunk_planes and chains (each may be NULL)
 * receive the choice for launches per diagonal, which a solve in one launch
 * does not use. */
EKX_API ekx_status ekx_solver3d_autotune(ekx_solver3d *solver,
                                         int *chunk_planes, int *chains);
/* No reference counterpart.  Longest time (ms) that a wave of a solve in one
 * launch (launch_order 0) waits for another: past it the solve is repeated
 * by launches per diagonal, as are all later solves until the next
 * initialize, which also restores the default.  Negative: the default, at
 * least 250 ms and more where problems wait for others to finish.  For
 * devices shared with other processes, where columns can be kept out. */
EKX_API ekx_status ekx_solver3d_set_wait_bound(ekx_solver3d *solver,
                                               double ms);
/* Solver3D::haveTravelTimeField (src/solver3d.cpp:510-514). */
EKX_API int ekx_solver3d_have_travel_time_field(const ekx_solver3d *solver);
/* Solver3D::getTravelTimeField (solver3d.hpp:137, src/solver3d.cpp:
 * 503-507): copies the nx*ny*nz field (natural order) into out. */
EKX_API ekx_status ekx_solver3d_get_travel_times(const ekx_solver3d *solver,
                                                 int64_t n, double *out);
/* Same field as float (the stored precision of the FP32 modes). */
EKX_API ekx_status ekx_solver3d_get_travel_times_f32(
    const ekx_solver3d *solver, int64_t n, float *out);
/* Device pointer of the travel-time field in natural order (x fastest;
 * borrowed until the next solve or initialize), and its element size (4:
 * float, 8: double).  With the column kernel, whose fields are tiled, this
 * is a natural-order copy made on the first request after a solve.  A
 * FIXED32 field
 * without polish is stored as scaled integers and is not exposed here
 * (EKX_ESTATE); read it with ekx_solver3d_get_travel_times.  Corresponds to
 * Solver3D::getTravelTimeFieldPointer (src/solver3d.cpp:516-525). */
EKX_API ekx_status ekx_solver3d_get_travel_times_device(
    const ekx_solver3d *solver, const void **device_ptr,
    int *element_size);
/* Solver3D::setStations (solver3d.hpp:113, src/solver3d.cpp:555-609):
 * receiver locations, absolute x, y and z, each inside the model (the
 * checks of Station3D::setLocationIn*, src/station3d.cpp:158-291).  The
 * reference only stores 3D stations; here every solve also interpolates
 * its field at them (as Solver2D does, src/solver2d.cpp:106-167, on three
 * axes), and a call after a solve interpolates the current field. */
EKX_API ekx_status ekx_solver3d_set_stations(ekx_solver3d *solver, int n,
                                             const double *x,
                                             const double *y,
                                             const double *z);
/* Solver3D::getStations().size(). */
EKX_API ekx_status ekx_solver3d_get_number_of_stations(
    const ekx_solver3d *solver, int *n);
/* The 3D counterpart of Solver2D::getTravelTimesAtStations
 * (solver2d.hpp:148): trilinear interpolation of the field at each
 * station, the analytic time of the source cell's slowness for a station
 * in the source cell.  n must equal the number of stations. */
EKX_API ekx_status ekx_solver3d_get_travel_times_at_stations(
    const ekx_solver3d *solver, int n, double *out);
/* The 3D counterpart of Solver2D::computeTravelTimeGradientField
 * (solver2d.hpp:127, src/solver2d.cpp:866-879, src/gradient.hpp): central
 * differences inside, second-order one-sided ones on the faces, the
 * analytic gradient at the corners of the source cell. */
EKX_API ekx_status ekx_solver3d_compute_travel_time_gradient_field(
    ekx_solver3d *solver);
/* Solver3D::haveTravelTimeGradientField (solver3d.hpp:163). */
EKX_API int ekx_solver3d_have_travel_time_gradient_field(
    const ekx_solver3d *solver);
/* Solver3D::getTravelTimeGradientField (solver3d.hpp:153): 3 x nx*ny*nz
 * values, (dT/dx, dT/dy, dT/dz) per node in natural order. */
EKX_API ekx_status ekx_solver3d_get_travel_time_gradient_field(
    const ekx_solver3d *solver, int64_t n, double *out);
/* Solver3D::getTravelTimeGradientFieldPointer (solver3d.hpp:160), as a
 * device pointer borrowed until the next solve or gradient call. */
EKX_API ekx_status ekx_solver3d_get_travel_time_gradient_field_device(
    const ekx_solver3d *solver, const double **device_ptr);
EKX_API ekx_status ekx_solver3d_get_stats(const ekx_solver3d *solver,
                                          ekx_solve_stats *stats);
/* The handle's HIP stream (hipStream_t), for callers that time or order
 * work around a solve. */
EKX_API ekx_status ekx_solver3d_get_stream(const ekx_solver3d *solver,
                                           void **stream);

/* ------------------------- Generated models ----------------------------
 * No reference counterpart (the reference reads models from the caller): a
 * velocity model of n_layers equal-thickness layers in z (layer k holds
 * nodes iz with floor(iz n_layers / nz) = k), each node's layer velocity
 * times (1 + amplitude G), G a unit-variance Gaussian random field with
 * covariance ~ exp(-r^2 / l^2): white noise from (seed, node index) through
 * a splitmix64 counter hash and the Box-Muller transform, filtered per axis
 * by a Gaussian of sigma = l / (2 d) nodes truncated at 4 sigma with
 * half-sample-symmetric boundaries (x, then y, then z), shifted and scaled
 * to zero mean and unit population variance.  Generated on the GPU. */
typedef struct
{
    int n_layers;
    const double *layer_velocity;  /* host, n_layers values (m/s), top first */
    double amplitude;              /* relative perturbation, >= 0          */
    double correlation_length;     /* l in m; 0: white noise               */
    uint64_t seed;
} ekx_layered_gaussian;

/* Nodal velocities (natural order, nx*ny*nz values) into host memory.
 * EKX_EINVAL if a velocity would be <= 0. */
EKX_API ekx_status ekx_model3d_layered_gaussian(
    const ekx_geometry3d *geometry, const ekx_layered_gaussian *model,
    int64_t n_grid, double *velocity);
/* Generates the model in device memory and sets it as the solver's model
 * (nodal velocities to cell slowness on the device, src/model3d.cpp:45-151),
 * with no host copy of the field. */
EKX_API ekx_status ekx_solver3d_set_layered_gaussian_model(
    ekx_solver3d *solver, const ekx_layered_gaussian *model);

/* ------------------------------ Batch3D --------------------------------
 * Many independent 3D solves in one schedule of launches (no reference
 * counterpart: the reference solves one source per Solver3D).  A problem
 * is (geometry, slowness, source).  Problems whose slowness pointers and
 * geometries are identical share one device copy of the model. */
typedef struct
{
    ekx_geometry3d geometry;
    const double *slowness;   /* host, (nx-1)(ny-1)(nz-1) cells */
    double source[3];         /* absolute (x, y, z) in m        */
} ekx_problem3d;

typedef struct ekx_batch3d ekx_batch3d;

EKX_API ekx_status ekx_batch3d_create(ekx_batch3d **batch);
EKX_API void ekx_batch3d_destroy(ekx_batch3d *batch);
EKX_API ekx_status ekx_batch3d_initialize(ekx_batch3d *batch,
                                          const ekx_solver_options *options,
                                          int n_problems,
                                          const ekx_problem3d *problems);
/* Moves problem i's source (same checks as ekx_solver3d_set_source). */
EKX_API ekx_status ekx_batch3d_set_source(ekx_batch3d *batch, int problem,
                                          double x, double y, double z);
EKX_API ekx_status ekx_batch3d_solve(ekx_batch3d *batch);
/* The launch-shape autotuner of ekx_solver3d_autotune for a batch (no
 * reference counterpart): candidate z-chunk depths around the size-class
 * default times 1, 2 or 4 chains, each timed on a short solve of the whole
 * batch; the fastest is kept. */
EKX_API ekx_status ekx_batch3d_autotune(ekx_batch3d *batch,
                                        int *chunk_planes, int *chains);
/* As ekx_solver3d_set_wait_bound. */
EKX_API ekx_status ekx_batch3d_set_wait_bound(ekx_batch3d *batch, double ms);
EKX_API ekx_status ekx_batch3d_get_travel_times(const ekx_batch3d *batch,
                                                int problem, int64_t n,
                                                double *out);
/* Receivers shared by every problem (each must lie inside every problem's
 * model): after each solve the batch holds a problems x stations table of
 * travel times, e.g. the station-reciprocal tables of a locator when the
 * problems' sources are the stations. */
EKX_API ekx_status ekx_batch3d_set_stations(ekx_batch3d *batch, int n,
                                            const double *x,
                                            const double *y,
                                            const double *z);
EKX_API ekx_status ekx_batch3d_get_travel_times_at_stations(
    const ekx_batch3d *batch, int problem, int n, double *out);
/* The whole table, [problem][station]; n = problems x stations. */
EKX_API ekx_status ekx_batch3d_get_station_table(const ekx_batch3d *batch,
                                                 int64_t n, double *out);
/* Gradient of one problem's field (one problem held at a time). */
EKX_API ekx_status ekx_batch3d_compute_travel_time_gradient_field(
    ekx_batch3d *batch, int problem);
EKX_API ekx_status ekx_batch3d_get_travel_time_gradient_field(
    const ekx_batch3d *batch, int problem, int64_t n, double *out);
EKX_API ekx_status ekx_batch3d_get_stats(const ekx_batch3d *batch,
                                         ekx_solve_stats *stats);
EKX_API ekx_status ekx_batch3d_get_stream(const ekx_batch3d *batch,
                                          void **stream);

/* ---------------------------- Solver2D ---------------------------------
 * Replaces EikonalXX::Solver2D<double> (include/eikonalxx/solver2d.hpp,
 * src/solver2d.cpp); the fast-sweeping schedule of src/solver2d.cpp:
 * 462-565. */
typedef struct ekx_solver2d ekx_solver2d;

EKX_API ekx_status ekx_solver2d_create(ekx_solver2d **solver);
EKX_API void ekx_solver2d_destroy(ekx_solver2d *solver);
/* Solver2D::initialize (src/solver2d.cpp:250-302). */
EKX_API ekx_status ekx_solver2d_initialize(ekx_solver2d *solver,
                                           const ekx_solver_options *options,
                                           const ekx_geometry2d *geometry);
/* Solver2D::setVelocityModel with Model2D's cell slowness
 * (src/solver2d.cpp:413-441). */
EKX_API ekx_status ekx_solver2d_set_slowness(ekx_solver2d *solver,
                                             int64_t n_cells,
                                             const double *slowness);
/* Model2D::setNodalVelocities (src/model2d.cpp:46-127) then
 * Solver2D::setVelocityModel. */
EKX_API ekx_status ekx_solver2d_set_nodal_velocities(ekx_solver2d *solver,
                                                     int64_t n_grid,
                                                     const double *velocity,
                                                     int ordering);
/* Solver2D::setSource(std::pair<double,double>) (src/solver2d.cpp:
 * 351-392). */
EKX_API ekx_status ekx_solver2d_set_source(ekx_solver2d *solver, double x,
                                           double z);
/* Solver2D::setStations (receiver locations, absolute x and z). */
EKX_API ekx_status ekx_solver2d_set_stations(ekx_solver2d *solver, int n,
                                             const double *x,
                                             const double *z);
/* Solver2D::solve (src/solver2d.cpp:462-565), including the bilinear
 * interpolation at the stations (:106-167). */
EKX_API ekx_status ekx_solver2d_solve(ekx_solver2d *solver);
EKX_API ekx_status ekx_solver2d_get_travel_times(const ekx_solver2d *solver,
                                                 int64_t n, double *out);
/* Solver2D::getTravelTimesAtStations. */
EKX_API ekx_status ekx_solver2d_get_travel_times_at_stations(
    const ekx_solver2d *solver, int n, double *out);
/* Solver2D::computeTravelTimeGradientField (solver2d.hpp:127,
 * src/solver2d.cpp:866-879, src/gradient.hpp). */
EKX_API ekx_status ekx_solver2d_compute_travel_time_gradient_field(
    ekx_solver2d *solver);
/* Solver2D::haveTravelTimeGradientField (src/solver2d.cpp:919-922). */
EKX_API int ekx_solver2d_have_travel_time_gradient_field(
    const ekx_solver2d *solver);
/* Solver2D::getTravelTimeGradientField (src/solver2d.cpp:925-932):
 * 2 x nx*nz values, (dT/dx, dT/dz) per node. */
EKX_API ekx_status ekx_solver2d_get_travel_time_gradient_field(
    const ekx_solver2d *solver, int64_t n, double *out);
EKX_API ekx_status ekx_solver2d_get_stats(const ekx_solver2d *solver,
                                          ekx_solve_stats *stats);

/* Many independent 2D problems (geometry, model, source each; problems
 * passing the same slowness pointer share one device copy of it) solved
 * by one launch, one workgroup per problem.  No reference counterpart:
 * problem i's field equals that of a Solver2D (ekx_solver2d_*) with the
 * same inputs. */
typedef struct
{
    ekx_geometry2d geometry;
    const double *slowness;   /* host, (nx-1)(nz-1) cells, x fastest */
    double source[2];         /* absolute (x, z) in m                */
} ekx_problem2d;

typedef struct ekx_batch2d ekx_batch2d;

EKX_API ekx_status ekx_batch2d_create(ekx_batch2d **batch);
EKX_API void ekx_batch2d_destroy(ekx_batch2d *batch);
EKX_API ekx_status ekx_batch2d_initialize(ekx_batch2d *batch,
                                          const ekx_solver_options *options,
                                          int n_problems,
                                          const ekx_problem2d *problems);
EKX_API ekx_status ekx_batch2d_solve(ekx_batch2d *batch);
EKX_API ekx_status ekx_batch2d_get_travel_times(const ekx_batch2d *batch,
                                                int problem, int64_t n,
                                                double *out);
EKX_API ekx_status ekx_batch2d_get_stats(const ekx_batch2d *batch,
                                         ekx_solve_stats *stats);

/* ---- Allocation-free solve ------------------------------------------- */
/* No counterpart in the reference: an entry point for callers that cannot
 * allocate device memory (code under HIP graph capture, serving loops,
 * harnesses that forbid hipMalloc).  The FP64 batch solve of n_sources
 * sources on one model (as ekx_batch3d_solve with kernel
 * EKX_KERNEL_HYPERPLANE: same fields, bit for bit) from device buffers the
 * caller owns: d_slowness, the (nx-1)(ny-1)(nz-1) cell slownesses in
 * natural order, and d_travel_times, n_sources fields of nx*ny*nz nodes in
 * natural order, field k the k-th source's.  sources_xyz: 3 host doubles
 * per source.  Enqueued on stream (a hipStream_t; NULL: the null stream)
 * without waiting for it.  It allocates nothing: the problem descriptors
 * go to a static device array of EKX_NOALLOC_MAX_SOURCES entries (about
 * 18 KB per GPU, held until the process ends), so n_sources beyond that is
 * an EKX_EINVAL error, and calls that overlap on one GPU (other streams or
 * threads) race on it.  FP64 only, no early exit, kernel AUTO or
 * HYPERPLANE; both schedules. */
#define EKX_NOALLOC_MAX_SOURCES 64
EKX_API ekx_status ekx_solve3d_noalloc(const ekx_solver_options *options,
                                       const ekx_geometry3d *geometry,
                                       int n_sources,
                                       const double *sources_xyz,
                                       const double *d_slowness,
                                       double *d_travel_times, void *stream);

#ifdef __cplusplus
}
#endif
#endif
