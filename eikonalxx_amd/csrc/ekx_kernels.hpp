// ekx_kernels.hpp -- host-side launchers of the HIP kernels.
#pragma once
#include "ekx_device.hpp"

namespace ekx
{

// Waves per workgroup of the column kernel.  Each wave owns a 15-slot
// travel-time ring and a 4-record slowness ring (6.5 KB for 4-byte
// elements, 13.2 KB for FP64), so LDS (160 KB per CU) bounds residency at
// 24 or 12 waves per CU; small blocks let the dispatcher reach that bound.
template <typename TS> constexpr int column_waves()
{
    return sizeof(TS) == 4 ? 2 : 1;
}

// Resident waves per CU of the bulk column kernel (prefetch depth 4, 8 or
// 12; merged: the instance that also runs the box columns) and of
// the work-queue kernel, from the occupancy API; 0 if it fails.
template <typename TS> int column_waves_per_cu(int depth, bool merged);
int queued_waves_per_cu(int depth);

// HUGE everywhere in the fields of all problems (totalCount elements from
// T, the problems' fields back to back), then the analytic times at each
// source cell's corners.
template <typename TS>
hipError_t launch_init3d(const Problem3D *dProblems, int nProblems,
                         int64_t totalCount, TS *T, hipStream_t stream);
template <typename TS>
hipError_t launch_hyperplane3d(const Problem3D *dProblems, int problem,
                               int sweep, int initialize, int level, int kLo,
                               int nPairs, TS *T, const TS *S,
                               unsigned int *change, hipStream_t stream);
// One diagonal bx + by + bz of column chunks (8 x 8 columns cut into
// z-chunks of `chunk` planes), Cartesian operators: the diagonal's items,
// except the chunks overlapping a factored box (boxPerDiag > 0).  depth:
// planes prefetched ahead of the compute (4, 8 or 12).  T: tiled fields
// (with their edge records); S: slowness bricks.  merged: the launch also
// runs the box chunks, with the full local update, and
// launch_factored_columns3d is not needed.
template <typename TS>
hipError_t launch_columns3d(const Problem3D *dProblems,
                            const ColumnItem *dItems, int nItems, int sweep,
                            int initialize, int diagonal, int boxPerDiag,
                            int chunk, TS *T, const TS *S,
                            unsigned int *change, int depth, bool merged,
                            hipStream_t stream);
// The box end of the same diagonal's chunks that overlap a factored box
// (box_split_z): up to boxPerDiag per problem (the box's columns in x and
// y), full local update, the chunks whose split has this phase.  Phase 0
// goes before the diagonal's bulk launch (launch_columns3d without merged,
// which takes the rest of those chunks), phase 1 after it.
template <typename TS>
hipError_t launch_factored_columns3d(const Problem3D *dProblems,
                                     int nProblems, int sweep, int initialize,
                                     int diagonal, int boxPerDiag, int chunk,
                                     int phase, TS *T, const TS *S,
                                     unsigned int *change,
                                     hipStream_t stream);
// A whole sweep of one chain's items (the diagonal launches' lists,
// concatenated in diagonal order) in work-queue form: `waves` waves (the
// chain's share of the resident ones) take the items in order and start each once its upwind chunks have
// published completion in q (the factored-box chunks included; FP64
// fields only).
template <typename TS>
hipError_t launch_queued_columns3d(const Problem3D *dProblems,
                                   const ColumnItem *dItems, int nItems,
                                   int sweep, int initialize, int chunk, TS *T,
                                   const TS *S, unsigned int *change,
                                   const ColumnQueue &q, int waves, int depth,
                                   hipStream_t stream);
// Flow kernel: resident waves per CU; the first sweep's records; records
// from (toRecords) or to the tiled fields, in the order of sweep `sweep`;
// nSweeps sweeps, the first nInit of them initialisation sweeps, from
// rec (step records of sweep 0 in the first of two buffers of recCount
// elements) to the buffer nSweeps & 1, in the order of sweep nSweeps & 7.
// mail: kMailBuffers buffers of mailCount elements, zero before the launch.
// Every model must be in range (Problem3D::scaled), every grid uniform or
// every one not, every problem's columns no more than the resident waves, and
// the columns of each XCD (blocks of one index modulo 8) in the same order of
// problems; error is set when a wait exceeded waitTicks.
template <typename TS> int flow_waves_per_cu(bool uniform);
template <typename TS>
hipError_t launch_flow_init(const Problem3D *dProblems,
                            const FlowColumn *dColumns, int nColumns,
                            int maxNz, TS *rec, hipStream_t stream);
template <typename TS>
hipError_t launch_flow_copy(const Problem3D *dProblems,
                            const FlowColumn *dColumns, int nColumns,
                            int maxNz, int sweep, bool toRecords, TS *rec,
                            TS *T, hipStream_t stream);
template <typename TS>
hipError_t launch_flow3d(const Problem3D *dProblems,
                         const FlowColumn *dColumns, int nColumns, int nInit,
                         int nSweeps, TS *rec, int64_t recCount, TS *mail,
                         int64_t mailCount, const TS *bricks, bool uniform,
                         unsigned int *error, unsigned int *xcc,
                         uint64_t waitTicks, hipStream_t stream);
// Zeroes n words of device memory (a kernel, so that captured graphs hold
// no memset node).
hipError_t launch_clear_words(unsigned int *w, int64_t n, hipStream_t stream);
// Writes descriptor p to dst in device memory, its srcSlowness read on the
// device from slowness[p.sOffset + sourceCell].
hipError_t launch_store_problem3d(const Problem3D &p, int64_t sourceCell,
                                  const double *slowness, Problem3D *dst,
                                  hipStream_t stream);
// Tiled layout: the slowness bricks of one model (natural cells s of an
// nx x ny x nz node grid) into b, and a natural-order copy (nx*ny*nz
// values) of problem p's tiled field (T: the whole buffer).
template <typename TS>
hipError_t launch_tile_slowness(int nx, int ny, int nz, const TS *s, TS *b,
                                hipStream_t stream);
template <typename TS>
hipError_t launch_untile_field(const Problem3D &p, const TS *T, TS *out,
                               hipStream_t stream);
// Sweep launches take `change`: NULL, or a device word that receives (as
// float bits, by atomic max) the largest decrease any update of the launch
// made -- the convergence monitor of the early-exit option.
hipError_t launch_nodal_to_cell3d(int nx, int ny, int nz, const double *v,
                                  int ordering, double *slow,
                                  hipStream_t stream);
hipError_t launch_cell_velocity_to_slowness3d(int nx, int ny, int nz,
                                              const double *v, int ordering,
                                              double *slow,
                                              hipStream_t stream);
// Block minima and maxima of a model (2 nBlocks values).  Scaled-integer
// storage: the model's slowness codes round(s * scale), and every problem's travel-time
// codes decoded to FP64.
hipError_t launch_block_range(int64_t n, const double *v, double *partial,
                              int nBlocks, hipStream_t stream);
hipError_t launch_encode_slowness(int64_t n, const double *in, double scale,
                                  uint32_t *out, hipStream_t stream);
hipError_t launch_decode_times(const Problem3D *dProblems, int nProblems,
                               int64_t maxCount, const uint32_t *in,
                               double *out, hipStream_t stream);
hipError_t launch_convert(int64_t n, const double *in, float *out,
                          hipStream_t stream);
hipError_t launch_convert(int64_t n, const float *in, double *out,
                          hipStream_t stream);

// Travel times at stations: out[k*nStations + i] for problem k, station i
// (locations per problem, same layout).
template <typename TS>
hipError_t launch_stations3d(const Problem3D *dProblems, int nProblems,
                             const StationLoc3D *dLocs, int nStations,
                             const TS *T, double *out, hipStream_t stream);
// Travel-time gradient of one problem: 3 values per node (host: the same
// problem's descriptor, for the grid size).
template <typename TS>
hipError_t launch_gradient3d(const Problem3D *dProblems, int problem,
                             const Problem3D &host, const TS *T,
                             double *grad, hipStream_t stream);
hipError_t launch_gradient2d(const Problem2D *dProblem, int nx, int nz,
                             const double *T, double *grad,
                             hipStream_t stream);

// Generated models (ekx_model3d.hip): Gaussian white noise from (seed,
// node index); one axis of a separable filter with 2*radius+1 taps and
// half-sample-symmetric boundaries; block partial sums (power 1), sums of
// squared deviations from mean (power 2) or minima (power 0); layered
// velocity times (1 + amplitude (g - mean) / sd).
hipError_t launch_gaussian_noise(int64_t n, uint64_t seed, double *out,
                                 hipStream_t stream);
hipError_t launch_filter_axis(int nx, int ny, int nz, int axis, int radius,
                              const double *w, const double *in, double *out,
                              hipStream_t stream);
hipError_t launch_moment(int64_t n, const double *v, double mean, int power,
                         double *partial, int nPartial, hipStream_t stream);
hipError_t launch_layered_velocity(int nx, int ny, int nz, int nLayers,
                                   const double *layerV, double amplitude,
                                   double mean, double sd, const double *g,
                                   double *v, hipStream_t stream);

// The whole 2D solve, one workgroup per problem, one launch per route that
// the plan (of these problems) holds.  work and cells: the band kernel's
// buffers (Problem2D::wOffset, cOffset; grids within fits_bands2d).
hipError_t launch_solve2d(const Problem2D *dProblems, int nProblems,
                          const Plan2D &plan, double *T, const double *S,
                          double *work, const double *cells,
                          hipStream_t stream);
// Writes a problem's descriptor, with the slowness at `cell` as its source's.
hipError_t launch_store_problem2d(const Problem2D &p, const double *cell,
                                  Problem2D *dst, hipStream_t stream);
// The band kernel's cell records of one model (cell_values2d values).
hipError_t launch_skew_cells2d(int nx, int nz, const double *s, double *out,
                               hipStream_t stream);
hipError_t launch_stations2d(const Problem2D *dProblem, int n,
                             const double *xOff, const double *zOff,
                             const int *cellX, const int *cellZ,
                             const double *T, double *out,
                             hipStream_t stream);
hipError_t launch_nodal_to_cell2d(int nx, int nz, const double *v,
                                  int ordering, double *slow,
                                  hipStream_t stream);

} // namespace ekx
