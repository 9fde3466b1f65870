// ekx_flow3d.hip -- a whole 3D solve in one launch: every column of 8 x 8
// nodes belongs to one wave for all sweeps, and the columns of a sweep
// pipeline through mailboxes instead of launches.
//
// The order of the updates is that of the column kernel (a node's upwind
// neighbours of the sweep are done before it), so the field is the same.
#include "ekx_kernels.hpp"
#include "ekx_local3d.hpp"
#include "ekx_storage.hpp"
#include "ekx_sweep3d.hpp"

#include <algorithm>

namespace ekx
{

// ---------------------------------------------------------------------------
// Flow kernel.  One 64-lane wave owns an 8 x 8 (x, y) column.  In a sweep's
// permuted frame lane (a, b) works at step t on plane t - a - b.  Its x and
// y neighbours were updated one step before by the neighbouring lanes (LDS,
// a ring of 4 steps), its z neighbour one step before by itself.
//
// Between columns: at step t a column publishes the values its downwind
// neighbours need at their step t - 7: lanes (7, b) for x, lanes (a, 7) for
// y, and the corner (7, -1) for x.  They are 16 mailbox values of one record,
// one store.
// Each sweep of four has its own buffer, and each value carries a tag in its
// sign bit (times are not negative) that alternates with every fourth sweep,
// so a value is its own arrival flag: the reader loads kMailAhead steps ahead
// and loads again while a tag is old.  Four buffers are what that takes: of
// any two neighbours one is upwind of the other in x in every second sweep,
// in y in two sweeps of four, and a column waits for both its upwind columns
// in every sweep.  So when it starts sweep s, its neighbours have read what
// it sent in sweep s - 4 and have sent sweep s - 4 themselves: nothing unread
// is overwritten, and an old value has the other tag.  (With two buffers a
// column that ran two sweeps ahead of its y neighbour read the neighbour's
// mail of four sweeps before.)
//
// Old times are step records (64 values a step, in the step and lane order
// of the sweep that reads them); a sweep writes the other buffer in the
// order of the next sweep, so no plane is staged through LDS.  A lane
// outside the grid's planes writes a padding element.
//
// Mail is stored to L2, which is where a reader on the same XCD finds it
// (its loads pass over the L1), and through to memory as well where a reader
// is on another XCD: columns tell each other at the start where they run.
// The launch order makes most neighbours share an XCD.  A hop from column to
// column takes 8 steps and 1.3 us through L2, 2.7 us through memory (64 x 8
// x 193: 1.22 ms per iteration with all mail through memory, 1.03 now).
//
// What bounds it: the chain of dependent steps.  A sweep needs
// nz + 14 + lag (bx + by) of them, where lag is 8 plus the mail's flight,
// and the next sweep starts where the last one ended, so only the reversed axes'
// lags add up.  A wave has its SIMD nearly to itself, so a step costs its
// instruction count: branch-free updates, and group kinds for what a group
// of 4 steps can meet.
//
// One 257 x 257 x 193 grid, FP64, 3 iterations: 50.9 ms with one launch per
// diagonal of 8-plane chunks (89 a sweep), 14.3 ms here.  A step takes 0.46
// us alone (170 instructions of 5 cycles, and the wait for LDS), more where
// waves share a CU (4: 0.52 us) or a SIMD (the younger one 0.7 us).
//
// A column waits for columns of its own problem only, so every column of a
// problem must become resident: the host launches it only for problems that
// each fit the device, and reserves their waves.  Problems beyond the resident
// waves follow the earlier ones: the columns of each XCD are in problem order,
// and its workgroups start in that order, so the first unfinished problem is
// resident as a whole.  Where that does not hold (a device shared with other
// work), each wait is bounded in wall-clock time, and past the bound flags an
// error, after which no wave waits any more and the host solves with the
// diagonals.
// ---------------------------------------------------------------------------
constexpr int kFlowAhead = 4;       // steps that records are loaded ahead
// Steps that mail is loaded ahead: each one more is one step more a hop
// (129^3: 1.50 ms per iteration, 1.65 with 2).
constexpr int kMailAhead = 1;
constexpr int kFlowRing = 4;
// The lane that sends the corner: the lanes from here on hold the mail of
// node (7, -1).
constexpr int kCornerLane = 2*kColumnTile;

template <typename TS> using Global = __attribute__((address_space(1))) TS;

template <typename TS> struct TagBits;
template <> struct TagBits<double>
{
    static __device__ __forceinline__ uint32_t high(double v)
    { return (uint32_t) (__builtin_bit_cast(uint64_t, v) >> 32); }
    static __device__ __forceinline__ double with_high(double v, uint32_t hi)
    {
        return __builtin_bit_cast(
            double, ((uint64_t) hi << 32) |
                        (uint32_t) __builtin_bit_cast(uint64_t, v));
    }
};
template <> struct TagBits<float>
{
    static __device__ __forceinline__ uint32_t high(float v)
    { return __builtin_bit_cast(uint32_t, v); }
    static __device__ __forceinline__ float with_high(float, uint32_t hi)
    { return __builtin_bit_cast(float, hi); }
};

// v with its sign replaced by the tag (0 or the sign bit)
template <typename TS>
__device__ __forceinline__ TS tagged(TS v, uint32_t tag)
{
    using B = TagBits<TS>;
    return B::with_high(v, (B::high(v) & 0x7FFFFFFFu) | tag);
}

// A region of device memory as a buffer resource: a 32-bit lane offset and a
// scalar one, in bytes, so that a step's address work is scalar.  COHERENT
// accesses are mail's: loads that pass over L1, stores that go through L2 to
// where the other XCDs see them.
template <typename TS>
struct FlowBuffer
{
    // raw buffer data format of gfx9 (32-bit elements, no swizzle)
    static constexpr int kFlags = 0x00020000;
    static constexpr int kAgent = 16;               // sc1
    __amdgpu_buffer_rsrc_t rsrc;
    __device__ __forceinline__ void set(const void *base, int64_t bytes)
    {
        const uint64_t p = (uint64_t) base;
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t) p);
        const uint32_t hi = __builtin_amdgcn_readfirstlane(
            (uint32_t) (p >> 32));
        rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void *) (((uint64_t) hi << 32) | lo), (short) 0,
            __builtin_amdgcn_readfirstlane((uint32_t) bytes), kFlags);
    }
    template <bool COHERENT = false>
    __device__ __forceinline__ TS load(uint32_t lane, uint32_t scalar) const
    {
        constexpr int kAux = COHERENT ? kAgent : 0;
        if constexpr (sizeof(TS) == 8)
        {
            return __builtin_bit_cast(
                TS, __builtin_amdgcn_raw_buffer_load_b64(
                        rsrc, (int) lane, (int) scalar, kAux));
        }
        else
        {
            return __builtin_bit_cast(
                TS, __builtin_amdgcn_raw_buffer_load_b32(
                        rsrc, (int) lane, (int) scalar, kAux));
        }
    }
    template <bool COHERENT>
    __device__ __forceinline__ void store(uint32_t lane, uint32_t scalar,
                                          TS v) const
    {
        constexpr int kAux = COHERENT ? kAgent : 0;
        if constexpr (sizeof(TS) == 8)
        {
            using V2 = __attribute__((ext_vector_type(2))) unsigned int;
            __builtin_amdgcn_raw_buffer_store_b64(
                __builtin_bit_cast(V2, v), rsrc, (int) lane, (int) scalar,
                kAux);
        }
        else
        {
            __builtin_amdgcn_raw_buffer_store_b32(
                __builtin_bit_cast(unsigned int, v), rsrc, (int) lane,
                (int) scalar, kAux);
        }
    }
};

// LDS values pass between the lanes of one wave, whose LDS instructions run
// in order: the compiler must keep them in program order, no wait is needed.
__device__ __forceinline__ void wave_lds_order()
{
    __asm__ __volatile__("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

// Bytes from one step's record to the next.
template <typename TS>
constexpr uint32_t kRecordBytes = kTileValues*sizeof(TS);
template <typename TS>
constexpr uint32_t kBrickBytes = kBrickValues*sizeof(TS);
template <typename TS>
constexpr uint32_t kMailBytes = kMailValues*sizeof(TS);

enum FlowGroup { kFlowFull, kFlowAny, kFlowIdle, kFlowBox };

// One column in one sweep.
template <typename TS>
struct FlowSweep
{
    // wave-uniform
    const Problem3D &p;
    int negX, negY, negZ;
    int nz, jz0;
    FlowBuffer<TS> old, cells, mail;
    // byte offsets of the records of step t + kFlowAhead, of the mail of
    // step t + kMailAhead, and of the record that step t writes (from xOff
    // and yOff, which are 7 records back)
    uint32_t oldS, cellS, mailInS, mailOutS;
    int outStep;
    int remote;             // a reader of this column's mail on another XCD
    uint32_t tag;
    unsigned int *error;
    uint64_t waitTicks;
    TS (*ring)[ring_slot<TS>()];
    // per lane
    int lane, ab, ix, iy;
    Global<TS> *out;                        // the result of step t
    uint32_t oldOff, mailOff, sendOff;  // byte offsets
    uint32_t off00, off10, off01, off11;
    bool need;              // the lane's mail has a sender
    bool sender;
    uint32_t liveSpan;
    TS floor;
    int haloPos, haloSlot;  // ring position, and steps back of its slot
    // step state
    int t;
    TS T0[kFlowAhead], C00[kFlowAhead], C10[kFlowAhead], C01[kFlowAhead],
        C11[kFlowAhead], H[kFlowRing];
    TS pt4, pt5, pt6, pt7, ps00, ps10, ps01, ps11, pMin;
    FactoredGrid fg;
    FactoredDistances dist;                 // of the step before, in the box
    bool failed;
};

// The natural indices of the lane's node in plane q.
struct FlowPlace
{
    int ix, iy, iz;
};

template <typename TS>
__device__ __forceinline__ FlowPlace flow_place(const FlowSweep<TS> &f, int q)
{
    FlowPlace n{f.ix, f.iy, f.negZ ? f.nz - 1 - q : q};
    // opaque, so that what the factored update derives from them is not
    // kept in registers across all the loops
    __asm__ __volatile__("" : "+v"(n.ix), "+v"(n.iy));
    return n;
}

// The lane's mail of the record at byte offset m, once every lane's has the
// sweep's tag.
template <typename TS>
__device__ __forceinline__ TS wait_mail(FlowSweep<TS> &f, uint32_t m)
{
    uint64_t t0 = 0;
    TS v;
    for (unsigned int spins = 1;; ++spins)
    {
        __asm__ __volatile__("" ::: "memory");
        v = f.mail.template load<true>(f.mailOff, m);
        const bool old = f.need &&
            ((TagBits<TS>::high(v) ^ f.tag) & 0x80000000u) != 0;
        if (__builtin_amdgcn_ballot_w64(old) == 0) { break; }
        if ((spins & 63) == 0)
        {
            const uint64_t now = (uint64_t) wall_clock64();
            if (spins == 64) { t0 = now; }
            const bool stop = __builtin_amdgcn_readfirstlane(
                __hip_atomic_load(f.error, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT)) != 0;
            if (stop || now - t0 > f.waitTicks)
            {
                __hip_atomic_fetch_or(f.error, 1u, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
                f.need = false;
                f.failed = true;
                break;
            }
        }
    }
    return v;
}

// What step t + u takes from the registers loaded ahead.
template <typename TS>
struct FlowLoads
{
    TS h, t0, c00, c10, c01, c11;
};

// The loads of step u of the group, and the loads ahead into the freed
// registers (u: a constant).
template <typename TS>
__device__ __forceinline__ FlowLoads<TS> take_loads(FlowSweep<TS> &f, int u)
{
    const FlowLoads<TS> l{f.H[u], f.T0[u], f.C00[u], f.C10[u], f.C01[u],
                          f.C11[u]};
    f.H[(u + kMailAhead) & (kFlowRing - 1)] = f.mail.template load<true>(
        f.mailOff + u*kMailBytes<TS>, f.mailInS);
    f.T0[u] = f.old.load(f.oldOff + u*kRecordBytes<TS>, f.oldS);
    f.C00[u] = f.cells.load(f.off00 + u*kBrickBytes<TS>, f.cellS);
    f.C10[u] = f.cells.load(f.off10 + u*kBrickBytes<TS>, f.cellS);
    f.C01[u] = f.cells.load(f.off01 + u*kBrickBytes<TS>, f.cellS);
    f.C11[u] = f.cells.load(f.off11 + u*kBrickBytes<TS>, f.cellS);
    return l;
}

// Step u of the group.  GRID: the Cartesian update's branch; BOX: the column
// overlaps the factored box (cells kept as they are, not times h); WAIT: the
// group still receives mail.
template <typename TS, Grid3D GRID, bool BOX, FlowGroup KIND, bool WAIT>
__device__ __forceinline__ void flow_step(FlowSweep<TS> &f,
                                          const FlowGrid<TS> &g, int u,
                                          FlowLoads<TS> l)
{
    constexpr bool kScaledCells = GRID != kNonUniform && !BOX;
    constexpr int kMask = kFlowRing - 1;
    const int a = f.lane & 7, b = f.lane >> 3;
    const int oA = b*kColumnHalo + a;
    // (a) the halo of this step into the ring: next to the values of the
    // step before (the corner: of two steps before)
    if constexpr (WAIT)
    {
        const bool old = f.need &&
            ((TagBits<TS>::high(l.h) ^ f.tag) & 0x80000000u) != 0;
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(old) != 0, 0))
        {
            l.h = wait_mail(f, f.mailInS + (u - kMailAhead)*
                                               (int) kMailBytes<TS>);
        }
    }
    f.ring[(u + kFlowRing - f.haloSlot) & kMask][f.haloPos] = tagged(l.h, 0u);
    wave_lds_order();
    const TS t1 = f.ring[(u + 3) & kMask][oA + kColumnHalo];
    const TS t3 = f.ring[(u + 3) & kMask][oA + 1];
    const TS t2 = f.ring[(u + 2) & kMask][oA];
    const TS t0 = l.t0;
    TS c00 = l.c00, c10 = l.c10, c01 = l.c01, c11 = l.c11;
    if constexpr (kScaledCells)
    {
        c00 *= g.dx;
        c10 *= g.dx;
        c01 *= g.dx;
        c11 *= g.dx;
    }
    // (b) the update
    TS cur = t0;
    TS nextMin = Math<TS>::min(c00, c01);
    if constexpr (KIND != kFlowIdle)
    {
        TS v;
        if constexpr (GRID == kNonUniform)
        {
            v = cartesian_nonuniform3d_flat<TS>(
                g, f.ps00, f.ps10, f.ps11, f.ps01, c00, c10, c01, t1, t2, t3,
                f.pt4, f.pt5, f.pt6, f.pt7);
        }
        else if constexpr (kScaledCells)
        {
            v = cartesian_uniform3d_flat<TS>(
                f.ps00, f.ps10, f.ps11, f.ps01, c00, c10, c01, f.pMin,
                nextMin, t1, t2, t3, f.pt4, f.pt5, f.pt6, f.pt7);
        }
        else
        {
            TS hs47;
            v = cartesian_uniform3d_flat<TS>(
                g.dx*f.ps00, g.dx*f.ps10, g.dx*f.ps11, g.dx*f.ps01, g.dx*c00,
                g.dx*c10, g.dx*c01, g.dx*f.pMin, hs47, t1, t2, t3, f.pt4,
                f.pt5, f.pt6, f.pt7);
        }
        if constexpr (KIND == kFlowFull)
        {
            cur = Math<TS>::min(Math<TS>::max(v, f.floor), t0);
        }
        else
        {
            const int q = f.t + u - f.ab;
            const bool live = (uint32_t) (q - f.jz0) < f.liveSpan;
            if constexpr (KIND == kFlowBox)
            {
                const FlowPlace n = flow_place(f, q);
                const Sweep3D sw =
                    make_sweep3d(f.negX + 2*f.negY + 4*f.negZ);
                const FactoredDistances d =
                    factored_distances(f.fg, sw, n.ix, n.iy, n.iz);
                const bool in = live &&
                    in_factored_box(f.p, n.ix, n.iy, n.iz);
                if (__builtin_amdgcn_ballot_w64(in) != 0)
                {
                    double w;
                    if constexpr (GRID == kNonUniform)
                    {
                        w = factored_nonuniform3d_flat(
                            f.fg, sw, d, f.dist, n.ix, n.iy, n.iz, f.ps00,
                            f.ps10, f.ps11, f.ps01, c00, c10, c01, t1, t2,
                            t3, f.pt4, f.pt5, f.pt6, f.pt7);
                    }
                    else
                    {
                        const double h = sizeof(TS) == 8 ? (double) g.dx
                                                         : f.fg.dx;
                        w = factored_uniform3d_flat(
                            f.fg, sw, d, f.dist, n.ix, n.iy, n.iz, f.ps00,
                            h*f.ps00, h*f.ps10, h*f.ps11, h*f.ps01, h*c00,
                            h*c10, h*c01, t1, t2, t3, f.pt4, f.pt5, f.pt6,
                            f.pt7);
                    }
                    v = in ? (TS) w : v;
                }
                f.dist = d;
            }
            cur = live & (v < t0) ? v : t0;
        }
    }
    f.ring[u][oA + kColumnHalo + 1] = cur;
    wave_lds_order();
    // (c) the result for the next sweep, and the mail
    *f.out = cur;
    f.out += f.outStep;
    if (f.sender)
    {
        const TS sent = tagged(f.lane == kCornerLane ? l.h : cur, f.tag);
        const uint32_t s = f.mailOutS + u*kMailBytes<TS>;
        f.mail.template store<false>(f.sendOff, s, sent);
        if (f.remote) { f.mail.template store<true>(f.sendOff, s, sent); }
    }
    f.pt4 = cur;
    f.pt5 = t1;
    f.pt6 = t2;
    f.pt7 = t3;
    f.ps00 = c00;
    f.ps10 = c10;
    f.ps01 = c01;
    f.ps11 = c11;
    f.pMin = nextMin;
}

// One group of steps.
template <typename TS, Grid3D GRID, bool BOX, FlowGroup KIND, bool WAIT>
__device__ __forceinline__ void flow_steps(FlowSweep<TS> &f,
                                           const FlowGrid<TS> &g)
{
#pragma unroll
    for (int u = 0; u < kFlowAhead; ++u)
    {
        const FlowLoads<TS> l = take_loads(f, u);
        flow_step<TS, GRID, BOX, KIND, WAIT>(f, g, u, l);
    }
    f.t += kFlowAhead;
    f.oldS += kFlowAhead*kRecordBytes<TS>;
    f.cellS += kFlowAhead*kBrickBytes<TS>;
    f.mailInS += kFlowAhead*kMailBytes<TS>;
    f.mailOutS += kFlowAhead*kMailBytes<TS>;
}

// Groups [from, to) of one kind.
template <typename TS, Grid3D GRID, bool BOX, FlowGroup KIND, bool WAIT>
__device__ __forceinline__ void flow_run(FlowSweep<TS> &f,
                                         const FlowGrid<TS> &g, int from,
                                         int to)
{
    if constexpr (KIND == kFlowBox)
    {
        const FlowPlace n = flow_place(f, f.t - 1 - f.ab);
        f.dist = factored_distances(
            f.fg, make_sweep3d(f.negX + 2*f.negY + 4*f.negZ), n.ix, n.iy,
            n.iz);
    }
#pragma unroll 1
    for (int i = from; i < to; ++i)
    {
        flow_steps<TS, GRID, BOX, KIND, WAIT>(f, g);
    }
}

template <typename TS, Grid3D GRID, bool BOX>
__device__ __forceinline__ void flow_column(FlowSweep<TS> &f,
                                            const FlowGrid<TS> &g, int groups,
                                            bool anyRow, int boxLo, int boxHi)
{
    // Runs of groups of one kind: idle before idleEnd, full in [fullLo,
    // fullHi), lanes in the box in [boxFirst, boxEnd); no mail is received
    // in the last two groups (past plane nz - 1 on every halo lane).
    const int waitEnd = groups - 2;
    const int idleEnd = anyRow ? f.jz0/kFlowAhead : groups;
    const int fullLo = (f.jz0 + kColumnSkew + kFlowAhead - 1)/kFlowAhead;
    const int fullHi = f.nz/kFlowAhead;
    int boxFirst = groups, boxEnd = groups;
    if (BOX && boxLo <= boxHi)
    {
        boxFirst = max(boxLo, 0)/kFlowAhead;
        boxEnd = boxHi/kFlowAhead + 1;
    }
    for (int i = 0; i < groups;)
    {
        int end = groups;
        if (i < waitEnd) { end = min(end, waitEnd); }
        if (i < idleEnd) { end = min(end, idleEnd); }
        if (i < fullLo) { end = min(end, fullLo); }
        if (i < fullHi) { end = min(end, fullHi); }
        if (BOX && i < boxFirst) { end = min(end, boxFirst); }
        if (BOX && i < boxEnd) { end = min(end, boxEnd); }
        if (i >= waitEnd)
        {
            // the tail: lanes leave the planes (and may be in the box)
            flow_run<TS, GRID, BOX, BOX ? kFlowBox : kFlowAny, false>(f, g,
                                                                     i, end);
        }
        else if (i < idleEnd)
        {
            flow_run<TS, GRID, BOX, kFlowIdle, true>(f, g, i, end);
        }
        else if (BOX && i >= boxFirst && i < boxEnd)
        {
            flow_run<TS, GRID, BOX, BOX ? kFlowBox : kFlowAny, true>(f, g, i,
                                                                    end);
        }
        else if (i >= fullLo && i < fullHi)
        {
            flow_run<TS, GRID, BOX, kFlowFull, true>(f, g, i, end);
        }
        else
        {
            flow_run<TS, GRID, BOX, kFlowAny, true>(f, g, i, end);
        }
        i = end;
    }
}

// Element of a slowness brick record at local cell position (c, r) of the
// sweep's frame (the order that tile_slowness_kernel stores).
__device__ __forceinline__ uint32_t brick_element(int c, int r, int negX,
                                                  int negY)
{
    const int xl = negX ? kColumnTile - c : c - 1;
    const int yl = negY ? kColumnTile - r : r - 1;
    return c == 0 ? kTileValues + r
                  : (r == 0 ? kTileValues + kColumnTile + c
                            : yl*kColumnTile + xl);
}

// Publishes the XCD that this column runs on and returns which neighbours
// run on the same one (bits: +x, -x, +y, -y), for which L2 is coherent.
__device__ __forceinline__ unsigned int local_neighbours(
    unsigned int *xcc, int id, bool hasE, bool hasW, bool hasN, bool hasS,
    int nTX, unsigned int *error, uint64_t waitTicks, bool &need)
{
    constexpr int kXccId = 20;              // hardware register XCC_ID
    const unsigned int mine =
        1 + __builtin_amdgcn_s_getreg(kXccId | (3 << 11));
    const int lane = threadIdx.x & 63;
    if (lane == 0)
    {
        __hip_atomic_store(xcc + id, mine, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    const bool has = lane == 0 ? hasE : lane == 1 ? hasW
                   : lane == 2 ? hasN : lane == 3 ? hasS : false;
    const int other = id + (lane == 0 ? 1 : lane == 1 ? -1
                            : lane == 2 ? nTX : lane == 3 ? -nTX : 0);
    const uint64_t t0 = (uint64_t) wall_clock64();
    for (;;)
    {
        unsigned int v = 0;
        if (has)
        {
            v = __hip_atomic_load(xcc + other, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
        }
        if (__builtin_amdgcn_ballot_w64(has && v == 0) == 0)
        {
            return (unsigned int) __builtin_amdgcn_ballot_w64(!has ||
                                                              v == mine);
        }
        const bool stop = __builtin_amdgcn_readfirstlane(
            __hip_atomic_load(error, __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_AGENT)) != 0;
        if (stop || (uint64_t) wall_clock64() - t0 > waitTicks)
        {
            __hip_atomic_fetch_or(error, 1u, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
            need = false;
            return 0;
        }
    }
}

// GRID: every problem's grid.  Two waves per SIMD: 2048 columns on 256 CUs.
template <typename TS, Grid3D GRID>
__global__ void __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(2, 2)))
sweep_flow3d(const Problem3D *__restrict__ problems,
             const FlowColumn *__restrict__ columns, int nInit, int nSweeps,
             TS *rec, int64_t recCount, TS *mail, int64_t mailCount,
             const TS *__restrict__ bricks, unsigned int *error,
             unsigned int *xcc, uint64_t waitTicks)
{
    __shared__ TS ring[kFlowRing][ring_slot<TS>()];
    const FlowColumn col = columns[blockIdx.x];
    if (col.problem < 0) { return; }
    const Problem3D &p = problems[__builtin_amdgcn_readfirstlane(col.problem)];
    const int lane = threadIdx.x & 63;
    const int a = lane & 7, b = lane >> 3;
    const int nx = p.nx, ny = p.ny, nz = p.nz, nTX = p.nTX, nTY = p.nTY;
    const int mx = __builtin_amdgcn_readfirstlane(col.mx);
    const int my = __builtin_amdgcn_readfirstlane(col.my);
    const FlowGrid<TS> grid = flow_grid<TS>(p);
    const int64_t tileIndex = (int64_t) my*nTX + mx;
    const int64_t perMail = (int64_t) flow_mails(nz)*kMailValues;
    // groups of steps: every plane through every lane, one step to spare
    // so that the last two groups receive nothing
    const int groups = (nz + kColumnSkew + 1 + kFlowAhead - 1)/kFlowAhead;
    bool need = true;       // false once a wait has failed
    const unsigned int local = local_neighbours(
        xcc, col.id, mx + 1 < nTX, mx > 0, my + 1 < nTY, my > 0, nTX, error,
        waitTicks, need);
    for (int s = 0; s < nSweeps; ++s)
    {
        const int sweep = s & 7;
        const int negX = sweep & 1, negY = (sweep >> 1) & 1;
        const int negZ = (sweep >> 2) & 1;
        const int next = (s + 1) & 7;
        const Octant o = sweep_octant(p, sweep, s < nInit);
        const int X0 = negX ? nx - kColumnTile*(mx + 1) : kColumnTile*mx;
        const int Y0 = negY ? ny - kColumnTile*(my + 1) : kColumnTile*my;
        const int jx = X0 + a, jy = Y0 + b;
        const bool upd = jx >= o.jx0 && jx < nx && jy >= o.jy0 && jy < ny;
        const bool anyRow = __builtin_amdgcn_ballot_w64(upd) != 0;
        // the result of plane q goes to the next sweep's lane (a', b') of
        // the same node, at its step q' + a' + b'
        const int a2 = kColumnTile - 1 - a;         // x always reverses
        const int b2 = ((sweep ^ next) & 2) ? kColumnTile - 1 - b : b;
        const bool flipZ = ((sweep ^ next) & 4) != 0;
        const int t2 = (flipZ ? nz - 1 + a + b : -a - b) + a2 + b2;
        // upwind columns
        const bool hasX = negX ? mx + 1 < nTX : mx > 0;
        const bool hasY = negY ? my + 1 < nTY : my > 0;
        const int64_t upX = hasX ? (negX ? 1 : -1) : 0;
        const int64_t upY = hasY ? (negY ? nTX : -nTX) : 0;
        const int h = min(lane, 2*kColumnTile);
        const bool xHalo = h <= kColumnTile;
        const int64_t selfMail = col.mail;
        const int64_t fromMail = selfMail + (xHalo ? upX : upY)*perMail;
        constexpr int64_t kSize = sizeof(TS);
        const int64_t recBytes = flow_records(nz)*kTileValues*kSize;
        const TS *variant = bricks + p.sbOffset +
            (int64_t) sweep*brick_variant_values(nx, ny, nz) +
            tileIndex*brick_records(nz)*kBrickValues;
        FlowSweep<TS> f{p};
        f.negX = negX;
        f.negY = negY;
        f.negZ = negZ;
        f.nz = nz;
        f.jz0 = o.jz0;
        f.old.set(rec + (s & 1)*recCount + col.rec - kFlowPad*kTileValues,
                  recBytes);
        f.cells.set(variant, brick_records(nz)*kBrickValues*kSize);
        f.mail.set(mail + (s & 3)*mailCount, mailCount*kSize);
        f.oldS = kFlowPad*kRecordBytes<TS>;
        f.cellS = f.mailInS = f.mailOutS = 0;
        f.out = (Global<TS> *) rec + ((s + 1) & 1)*recCount + col.rec +
                (int64_t) t2*kTileValues + kColumnTile*b2 + a2;
        f.outStep = flipZ ? -kTileValues : kTileValues;
        f.tag = (s & 4) ? 0u : 0x80000000u;
        f.error = error;
        f.waitTicks = waitTicks;
        f.ring = ring;
        f.lane = lane;
        f.ab = a + b;
        f.ix = negX ? nx - 1 - jx : jx;
        f.iy = negY ? ny - 1 - jy : jy;
        auto bytes = [](int64_t v) { return (uint32_t) (v*kSize); };
        f.oldOff = bytes(lane);
        f.mailOff = bytes(fromMail +
                          (xHalo ? h : h == kCornerLane ? kColumnTile
                                 : kMailY + h - kColumnTile - 1));
        f.sender = a == kColumnTile - 1 || b == kColumnTile - 1 ||
                   lane == kCornerLane;
        f.remote = 1 - (int) ((local >> negX) & (local >> (2 + negY)) & 1);
        f.sendOff = bytes(selfMail - (kColumnTile - 1)*kMailValues +
                          (lane == kCornerLane    ? 0
                           : a == kColumnTile - 1 ? 1 + b : kMailY + a));
        f.off00 = bytes(brick_element(a, b, negX, negY));
        f.off10 = bytes(kBrickValues + brick_element(a + 1, b, negX, negY));
        f.off01 = bytes(kBrickValues + brick_element(a, b + 1, negX, negY));
        f.off11 = bytes(2*kBrickValues +
                        brick_element(a + 1, b + 1, negX, negY));
        f.need = need && (xHalo ? hasX : hasY);
        f.liveSpan = upd ? (uint32_t) (nz - o.jz0) : 0u;
        f.floor = upd ? -(TS) kHuge : 4*(TS) kHuge;
        f.haloPos = xHalo ? h*kColumnHalo : h - kColumnTile;
        f.haloSlot = h == 0 ? 2 : 1;
        f.t = 0;
        f.pt4 = f.pt5 = f.pt6 = f.pt7 = (TS) kHuge;
        f.ps00 = f.ps10 = f.ps01 = f.ps11 = f.pMin = 0;
        f.failed = false;
        // the first records (step 0 .. kFlowAhead - 1) and mail
#pragma unroll
        for (int u = 0; u < kFlowAhead; ++u)
        {
            f.T0[u] = f.old.load(f.oldOff + u*kRecordBytes<TS>, f.oldS);
            f.C00[u] = f.cells.load(f.off00 + u*kBrickBytes<TS>, 0);
            f.C10[u] = f.cells.load(f.off10 + u*kBrickBytes<TS>, 0);
            f.C01[u] = f.cells.load(f.off01 + u*kBrickBytes<TS>, 0);
            f.C11[u] = f.cells.load(f.off11 + u*kBrickBytes<TS>, 0);
        }
#pragma unroll
        for (int u = 0; u < kMailAhead; ++u)
        {
            f.H[u] = f.mail.template load<true>(
                f.mailOff + u*kMailBytes<TS>, 0);
        }
        f.oldS += kFlowAhead*kRecordBytes<TS>;
        f.cellS += kFlowAhead*kBrickBytes<TS>;
        f.mailInS += kMailAhead*kMailBytes<TS>;
        // the steps at which lanes of this column are in the factored box
        int boxLo = 1, boxHi = 0;
        if (p.radius >= 0)
        {
            auto range = [&](int cell, int n, int neg, int &lo, int &hi)
            {
                const int l = max(cell - p.radius, 0);
                const int u = min(cell + p.radius, n - 1);
                lo = neg ? n - 1 - u : l;
                hi = neg ? n - 1 - l : u;
            };
            int xLo, xHi, yLo, yHi, zLo, zHi;
            range(p.srcCellX, nx, negX, xLo, xHi);
            range(p.srcCellY, ny, negY, yLo, yHi);
            range(p.srcCellZ, nz, negZ, zLo, zHi);
            const int aLo = max(xLo - X0, 0), aHi = min(xHi - X0, 7);
            const int bLo = max(yLo - Y0, 0), bHi = min(yHi - Y0, 7);
            if (aLo <= aHi && bLo <= bHi && zLo <= zHi)
            {
                boxLo = zLo + aLo + bLo;
                boxHi = zHi + aHi + bHi;
            }
        }
        const bool box = boxLo <= boxHi && anyRow;
        if (box)
        {
            f.fg = factored_grid<GRID != kNonUniform>(p);
            flow_column<TS, GRID, true>(f, grid, groups, anyRow, boxLo,
                                        boxHi);
        }
        else
        {
            flow_column<TS, GRID, false>(f, grid, groups, anyRow, 1, 0);
        }
        // a lane without a sender in this sweep may have one in the next:
        // only a failed wait ends the waiting
        need = need && __builtin_amdgcn_readfirstlane(
                           f.failed ? 1 : 0) == 0;
        // the next sweep reads this one's records, by other lanes: the
        // stores first
        __asm__ __volatile__("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0);
        __asm__ __volatile__("" ::: "memory");
    }
}

// ---------------------------------------------------------------------------
// Step records <-> the tiled field.
// ---------------------------------------------------------------------------
// Grid node of a column's plane q and lane in the order of sweep `sweep`.
struct FlowNode
{
    int x, y, z;
};

__device__ __forceinline__ FlowNode flow_node(const Problem3D &p,
                                              const FlowColumn &c, int sweep,
                                              int q, int lane)
{
    const int a = lane & 7, b = lane >> 3;
    FlowNode n;
    n.x = kColumnTile*c.mx + ((sweep & 1) ? kColumnTile - 1 - a : a);
    n.y = kColumnTile*c.my + ((sweep & 2) ? kColumnTile - 1 - b : b);
    n.z = (sweep & 4) ? p.nz - 1 - q : q;
    return n;
}

// Before the first sweep: HUGE, and the analytic times at the corners of
// each source cell (Solver3DImpl::initializeTravelTimes,
// src/solver3d.cpp:21-84).  Block (x): column; threads: lanes of 4 planes.
template <typename TS>
__global__ void __launch_bounds__(256)
flow_init_kernel(const Problem3D *__restrict__ problems,
                 const FlowColumn *__restrict__ columns, TS *__restrict__ rec)
{
    const FlowColumn c = columns[blockIdx.x];
    if (c.problem < 0) { return; }
    const Problem3D &p = problems[c.problem];
    const int lane = threadIdx.x & 63;
    const bool source = p.srcCellX + 1 >= kColumnTile*c.mx &&
                        p.srcCellX < kColumnTile*(c.mx + 1) &&
                        p.srcCellY + 1 >= kColumnTile*c.my &&
                        p.srcCellY < kColumnTile*(c.my + 1);
    for (int q = blockIdx.y*4 + (threadIdx.x >> 6); q < p.nz;
         q += 4*gridDim.y)
    {
        TS v = (TS) kHuge;
        if (source)
        {
            const FlowNode n = flow_node(p, c, 0, q, lane);
            const int ox = n.x - p.srcCellX, oy = n.y - p.srcCellY;
            const int oz = n.z - p.srcCellZ;
            if ((unsigned) ox <= 1u && (unsigned) oy <= 1u &&
                (unsigned) oz <= 1u)
            {
                v = (TS) analytic_time3d(n.x, n.y, n.z, p.dx, p.dy, p.dz,
                                         p.srcOffX, p.srcOffY, p.srcOffZ,
                                         p.srcSlowness);
            }
        }
        rec[c.rec + (int64_t) (q + (lane & 7) + (lane >> 3))*kTileValues +
            lane] = v;
    }
}

// TO_RECORDS: the tiled field into step records of sweep `sweep`, else back.
template <typename TS, bool TO_RECORDS>
__global__ void __launch_bounds__(256)
flow_copy_kernel(const Problem3D *__restrict__ problems,
                 const FlowColumn *__restrict__ columns, int sweep,
                 TS *__restrict__ rec, TS *__restrict__ T)
{
    const FlowColumn c = columns[blockIdx.x];
    if (c.problem < 0) { return; }
    const Problem3D &p = problems[c.problem];
    const int lane = threadIdx.x & 63;
    for (int q = blockIdx.y*4 + (threadIdx.x >> 6); q < p.nz;
         q += 4*gridDim.y)
    {
        const FlowNode n = flow_node(p, c, sweep, q, lane);
        const int64_t r = c.rec +
            (int64_t) (q + (lane & 7) + (lane >> 3))*kTileValues + lane;
        const int64_t e = p.tOffset + tiled_index(p.nTX, p.nz, n.x, n.y, n.z);
        if (TO_RECORDS) { rec[r] = T[e]; }
        else { T[e] = rec[r]; }
    }
}

static dim3 flow_grid_dim(int nColumns, int maxNz)
{
    const int y = std::max(1, std::min((maxNz + 3)/4, 16384/nColumns + 1));
    return dim3((unsigned) nColumns, (unsigned) y);
}

template <typename TS>
hipError_t launch_flow_init(const Problem3D *dProblems,
                            const FlowColumn *dColumns, int nColumns,
                            int maxNz, TS *rec, hipStream_t stream)
{
    hipLaunchKernelGGL(flow_init_kernel<TS>, flow_grid_dim(nColumns, maxNz),
                       dim3(256), 0, stream, dProblems, dColumns, rec);
    return hipGetLastError();
}

template <typename TS>
hipError_t launch_flow_copy(const Problem3D *dProblems,
                            const FlowColumn *dColumns, int nColumns,
                            int maxNz, int sweep, bool toRecords, TS *rec,
                            TS *T, hipStream_t stream)
{
    const dim3 grid = flow_grid_dim(nColumns, maxNz);
    if (toRecords)
    {
        hipLaunchKernelGGL((flow_copy_kernel<TS, true>), grid, dim3(256), 0,
                           stream, dProblems, dColumns, sweep, rec, T);
    }
    else
    {
        hipLaunchKernelGGL((flow_copy_kernel<TS, false>), grid, dim3(256), 0,
                           stream, dProblems, dColumns, sweep, rec, T);
    }
    return hipGetLastError();
}

template <typename TS>
hipError_t launch_flow3d(const Problem3D *dProblems,
                         const FlowColumn *dColumns, int nColumns, int nInit,
                         int nSweeps, TS *rec, int64_t recCount, TS *mail,
                         int64_t mailCount, const TS *bricks, bool uniform,
                         unsigned int *error, unsigned int *xcc,
                         uint64_t waitTicks,
                         hipStream_t stream)
{
    if (nColumns <= 0 || nSweeps <= 0) { return hipErrorInvalidValue; }
    const dim3 grid((unsigned) nColumns);
    if (uniform)
    {
        hipLaunchKernelGGL((sweep_flow3d<TS, kUniformScaled>), grid, dim3(64),
                           0, stream, dProblems, dColumns, nInit, nSweeps,
                           rec, recCount, mail, mailCount, bricks, error,
                           xcc, waitTicks);
    }
    else
    {
        hipLaunchKernelGGL((sweep_flow3d<TS, kNonUniform>), grid, dim3(64), 0,
                           stream, dProblems, dColumns, nInit, nSweeps, rec,
                           recCount, mail, mailCount, bricks, error,
                           xcc, waitTicks);
    }
    return hipGetLastError();
}

template <typename TS> int flow_waves_per_cu(bool uniform)
{
    int blocks = 0;
    const hipError_t e = uniform
        ? hipOccupancyMaxActiveBlocksPerMultiprocessor(
              &blocks, sweep_flow3d<TS, kUniformScaled>, 64, 0)
        : hipOccupancyMaxActiveBlocksPerMultiprocessor(
              &blocks, sweep_flow3d<TS, kNonUniform>, 64, 0);
    return e == hipSuccess && blocks > 0 ? blocks : 0;
}

#define EKX_FLOW(TS)                                                         \
    template int flow_waves_per_cu<TS>(bool);                                \
    template hipError_t launch_flow_init<TS>(const Problem3D *,              \
                                             const FlowColumn *, int, int,   \
                                             TS *, hipStream_t);             \
    template hipError_t launch_flow_copy<TS>(const Problem3D *,              \
                                             const FlowColumn *, int, int,   \
                                             int, bool, TS *, TS *,          \
                                             hipStream_t);                   \
    template hipError_t launch_flow3d<TS>(const Problem3D *,                 \
                                          const FlowColumn *, int, int, int, \
                                          TS *, int64_t, TS *, int64_t,      \
                                          const TS *, bool, unsigned int *,  \
                                          unsigned int *, uint64_t,          \
                                          hipStream_t);
EKX_FLOW(double)
EKX_FLOW(float)
#undef EKX_FLOW

} // namespace ekx
