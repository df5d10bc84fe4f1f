// resident.h -- per-system descriptors of the workgroup-resident drivers
// (resident.hip).
#pragma once

#include "sol_internal.h"
#include "slice_map.h"

namespace sol {

// RES_STOPPED: the step met a stop reason of stop_mask (SOL_STOP_OUTPUT,
// SOL_STOP_EVENT), recorded in reason; the host resumes with RES_RUNNING.
// RES_SYNC_ERROR: a grid-wide step decision (GridSync) did not complete.
enum { RES_RUNNING = 0, RES_DONE = 1, RES_UNDERFLOW = 2, RES_MAXITER = 3, RES_STOPPED = 4, RES_SYNC_ERROR = 5 };
constexpr int kResidentMaxBodies = 2000;   // LDS: 64 B per body

// One system: its bodies are [base, base + n) of the concatenated arrays.
// Time-line fields follow TimeLine (Solaris/TimeLine.h); clip switches on
// the Simulator's step clipping and small-number flush, flush_count is the
// caller loop's accepted-step count modulo 100.  With clip, stop_mask
// (SOL_STOP_OUTPUT | SOL_STOP_EVENT) makes the system stop after a step at
// which an output is due or an event threshold (e3 = 1/ejection^3,
// h3 = 1/hitCentrum^3, coll = collision factor; 0 = off) is crossed.
struct ResSystem {
    int32_t n, nm, end_a, end_b;
    int32_t base, barycentric, clip, status;
    int32_t millenium, flush_count;
    double t, h_next, h_did, body_h, eps;
    double elapsed, last_save, last_nsteps, length, output;
    int64_t steps, attempts;
    double e3, h3, coll;
    int32_t stop_mask, reason;
    // a slice of a larger system (GridSync): bodies [0, src) are the
    // system's first bodies, the others are bodies shift + i of it
    // (shift = 0 for a whole system); drag acts on the system's bodies
    // [drag_lo, drag_hi), migration on its massive bodies [1, nm) (Type II
    // on [mig_lo, giant_end), the giants)
    int32_t src, shift, drag_lo, drag_hi;
    int32_t mig_lo, giant_end;
};

// Grid-wide step decisions for one system integrated as slices, one
// workgroup each (every slice holds the system's sources, so the slices
// evolve the sources identically): each workgroup publishes its error
// maximum and event flag of an attempt in its own entry of vals / flags
// (double-buffered by the parity of the combine), meets the others at a
// barrier (count, gen) and reads every entry.  All accesses are
// system-scope atomics: the L2 caches of the device's chiplets are not
// coherent with each other for ordinary device memory.  A barrier that does
// not complete within sync_ticks of the real-time counter sets error and
// every workgroup stops.
constexpr int kGridMaxSlices = 512;
struct GridSync {
    uint32_t count, pad0[31];      // one cache line each
    uint32_t gen, pad1[31];
    uint32_t error, pad2[31];
    unsigned long long vals[2][kGridMaxSlices];
    uint32_t flags[2][kGridMaxSlices];
};

// Structure-of-arrays storage over all systems: component c of body b at
// [c * tot + b]; stage l >= 1 derivatives at fst + (l-1) * 6 * tot.
struct ResArrays {
    int64_t tot;
    double *y0, *y, *acc0, *yscale, *err, *fst, *mass, *rm3, *nnd;
    int32_t *nni;
    const double *radius;     // read by the collision check only
    // RK4 only, both optional: the step size of each step of the launch
    // (h_seq[step], step counted from the launch's first), and the stage
    // states Y1..Y4 of each step at stages_out + (step * 4 + s) * 6 * tot
    const double *h_seq;
    double *stages_out;
    // gas (gas_on): drag every stage, migration at each Driver call's first
    // evaluation, cached; per-body parameters in the systems' body order
    // (mig_do1, mig_do2: Type I / Type II computed at all)
    const double *density, *cd, *gs, *ge, *stop;
    int32_t *migt;
    // optional: the caches of the multi-kernel path (system layout,
    // component stride cache_stride), left as that path leaves them: the
    // migration of the Driver's first evaluation and the drag of the last
    // evaluation
    double *migc, *dragc;
    int64_t cache_stride;
    GasDev gas;
    int32_t gas_on, mig_do1, mig_do2, nsync;
    GridSync *sync;           // non-null: the workgroups are slices of one system
    uint64_t sync_ticks;      // real-time-counter ticks a grid-wide wait lasts before it gives up
};

int resident_block_size(int n);
size_t resident_lds_bytes(int nmax);
// lds_limit: LDS bytes a workgroup may use for the optional LDS-held stage
// derivatives (0: none; the ensemble passes 0 to keep its occupancy).
void launch_resident(hipStream_t st, int integ, ResSystem *systems, int nsys, const ResArrays &A, int max_steps,
                     int block, int nmax, size_t lds_limit);

// What the persistent form reads of its queue: the counter its workgroups take
// systems by, how many there are, and the accepted steps each is run for at
// most.  On the device, so that a captured launch serves every queue.
struct QueueWords { int32_t head, nsys, max_steps, pad; };

// The persistent form: `grid` workgroups of `block` threads take systems
// from the queue order[0 .. q->nsys) (through the counter q->head, which
// the launch zeroes first with a one-thread kernel, so the pair can be
// captured in a graph) and run each for up to q->max_steps accepted steps.
// Bodies per thread: resident_queue_bpt(block, nmax), at most 4.  With one
// body per thread (nmax <= block, blocks of up to 768 threads) each
// system's bodies get up to 1 << max_lsh lanes each, which split the
// source loop.
int resident_queue_bpt(int block, int nmax);
// lf = 4 (RKF78, one body per thread, blocks of up to 640 threads): F0 and
// F3-F5 in LDS, resident_queue_lds_f(nmax) more bytes of it.
void launch_resident_queue(hipStream_t st, int integ, ResSystem *systems, const int32_t *order, QueueWords *q,
                           const ResArrays &A, int grid, int block, int nmax, int max_lsh = 0, int lf = 0);
// Workgroups of that launch one CU holds at once.
int resident_queue_occupancy(int integ, int block, int nmax, int lf = 0);
size_t resident_queue_lds_f(int nmax);

// One system as nslices workgroups of `block` (<= 256) threads, one body
// per thread (A.sync set, A.nsync = nslices), each with its own ResSystem;
// nslices must not exceed resident_grid_capacity, so that all are resident
// at once; the GridSync is zeroed first.  Stage derivatives are kept in LDS as far as lds_limit
// bytes allow (all but the last stage's, or RKF78's four most-read).
// Returns the launch status.
hipError_t launch_resident_grid(hipStream_t st, int integ, ResSystem *systems, int nslices, const ResArrays &A,
                                int max_steps, int block, int nmax, size_t lds_limit);
// Largest number of slices such a launch can hold on this device (0 when
// it cannot be launched).
int resident_grid_capacity(int integ, int block, int nmax, size_t lds_limit, int cu_count, bool gas);

// The system-layout arrays (component stride np) the slices come from and
// go back to; density == nullptr: no gas parameters (and migt untouched).
struct SliceArrays {
    double *y0, *y, *acc0, *yscale, *err, *rm3, *nnd;
    int32_t *nni, *migt;
    const double *mass, *radius, *density, *cd, *gs, *ge, *stop;
};
void launch_slice_scatter(hipStream_t st, const SliceMap &m, const SliceArrays &sys, const ResArrays &A);
void launch_slice_gather(hipStream_t st, const SliceMap &m, const SliceArrays &sys, const ResArrays &A);

}  // namespace sol
