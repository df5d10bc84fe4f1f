// ensemble.cpp -- batched integration of independent small systems
// (sol_ensemble_* in include/solaris_amd.h).
//
// Every system occupies a 64-aligned range of the structure-of-arrays
// storage and one ResSystem descriptor.  One persistent launch of the
// workgroup-resident kernel (resident.hip, k_resident_queue) integrates
// them all: each workgroup takes the next system from a device-side queue
// (an atomic counter over an order array, the systems with the most work
// expected first), runs its Driver loop with the caller loop's clipping
// for up to a bounded number of accepted steps, and takes the next, so
// systems of every size and step count share one launch and the many
// short ones fill in around the few long ones.  The launch shape (threads
// per system, and with it bodies per thread) is picked by timing the
// candidates on a short probe of the systems themselves, whose states are
// restored afterwards (sol_ensemble_tune; sol_ensemble_run tunes first when
// this has not been done).
//
// A run lasts as long as its slowest system, and a system's step takes a
// time that grows with its size (one body per lane, each summing over all
// sources).  The systems of at least wide_min bodies therefore go to a
// second queue, launched beside the first on a second stream, whose
// workgroups of wide_block threads give each body of a system up to
// 1 << wide_lsh lanes that split its source loop.  Each queue's launch (the
// counter reset and the kernel) is captured once in a HIP graph of its own
// and replayed until every system is done.
//
// Once the systems still running fit the device at several workgroups each,
// those with many sources go on in the mesh form (run_mesh), so that the last
// few do not take their steps on one CU each.  So which form a step of theirs is
// summed in, and with it its last digits, depends on the systems beside them.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "sol_internal.h"
#include "resident.h"
#include "mesh.h"
#include "unit_lease.h"

using namespace sol;

namespace {
thread_local std::string g_ens_create_error;
}  // namespace

struct sol_ensemble {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;
    int nsys = 0;
    std::vector<sol_nbodies> nb;
    std::vector<int> slot_of, sys_of;   // external index <-> slot (bucket order)
    std::vector<int64_t> base;          // per slot
    int64_t tot = 0;
    std::vector<double> ipe;            // interactions per evaluation, per slot
    // host mirrors
    std::vector<double> y0_h, mass_h;
    std::vector<ResSystem> sys_h;
    // y_dirty: the host states (and masses) were changed and must go up
    // (set only after download(), so the host copy is current); sys_dirty:
    // the host descriptors were changed; stale: the device states have
    // moved on since the last download()
    bool y_dirty = true, sys_dirty = true, stale = false;
    // device
    ResSystem *sys_d = nullptr;
    double *y0 = nullptr, *y = nullptr, *acc0 = nullptr, *yscale = nullptr, *errv = nullptr, *fst = nullptr;
    double *mass = nullptr, *rm3 = nullptr, *nnd = nullptr;
    int32_t *nni = nullptr;
    // the persistent launch: the queues of slots (queue_d: the two queues'
    // words, the narrow queue's slots, and from count_n on the wide one's), its
    // shape (block threads per system, grid workgroups) and the candidates
    // the tuner times
    int32_t *queue_d = nullptr;
    std::vector<int32_t> queue_h;
    std::vector<int32_t> order_h;        // the narrow queue
    std::vector<int32_t> order_w;        // the wide queue
    int count_n = 0, count_w = 0;        // systems of each, running or not
    int nmax = 0, cu_count = 256;
    int nmax_n = 0, nmax_w = 0;          // largest system of each queue
    int block = 0, grid = 0;
    // the wide queue (wide_block 0: every system in the narrow queue)
    int wide_block = 512, wide_lsh = 1, wide_min = 97, grid_w = 0;
    size_t lds_per_block = 65536;        // the device's LDS per workgroup
    hipStream_t stream2 = nullptr;
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    bool tuned = false;
    std::vector<int> cand;
    std::vector<double> cand_ms;
    hipGraphExec_t graph = nullptr, graph_w = nullptr;   // the narrow and the wide queue's launch
    int graph_integ = -1, graph_block = 0, graphw_integ = -1;      // what they were captured for
    int64_t launches = 0, graph_launches = 0;
    std::vector<int64_t> last_steps;     // per slot: steps of the previous launch
    // the mesh form for the last systems (mesh.h): their descriptors while it
    // runs, its copy of the states, k^2 m, positions, parts and exchange words
    // (mesh_state null: no system of the ensemble can take it, or off)
    bool mesh_off = false;
    int mesh_failures = 0;               // launches that gave up; two turn it off
    double wait_s = 2.0;                 // seconds a wait of it lasts before it gives up
    uint64_t rtc_hz = 100000000;
    double *mesh_state = nullptr, *mesh_gm = nullptr, *mesh_pos = nullptr;
    ResSystem *mesh_sys = nullptr;
    MeshPart *mesh_part = nullptr;
    int32_t *mesh_part_of = nullptr;
    MeshSync *mesh_sync = nullptr;
    std::vector<double> gm_h;

    int fail(int code, const std::string &m) { err = m; return code; }
};

#define ECHECK(e, call)                                                                          \
    do {                                                                                         \
        hipError_t r_ = (call);                                                                  \
        if (r_ != hipSuccess) return (e)->fail(SOL_ERR_DEVICE, std::string(#call " failed: ") + hipGetErrorString(r_)); \
    } while (0)

namespace {

// Where the slots start in an ensemble's queue_d.
constexpr int kQueueSlots = 2 * sizeof(QueueWords) / sizeof(int32_t);

// Accepted steps of a run's first launch.
constexpr int kFirstSteps = 16;

int nmassive(const sol_nbodies &b) { return b.central_body + b.giant_planet + b.rocky_planet + b.proto_planet; }

// interactions per evaluation with the reference's astrocentric ranges
double interactions(const sol_nbodies &b)
{
    const int nm = nmassive(b), n = b.total;
    const int ea = nm + b.super_planetesimal, eb = nm;
    double s = 0.0;
    const int na = nm - 1, nbk = n - nm;
    if (na > 0) s += (double)na * (1.0 + std::max(ea - 1, 0)) - (double)std::max(0, std::min(nm, ea) - 1);
    if (nbk > 0) s += (double)nbk * (1.0 + std::max(eb - 1, 0));
    return s;
}

template <typename T>
int ealloc(sol_ensemble *e, T **p, size_t n)
{
    void *q = nullptr;
    ECHECK(e, hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T)));
    // (on the ensemble's stream, which is not ordered after the default one)
    ECHECK(e, hipMemsetAsync(q, 0, std::max<size_t>(n, 1) * sizeof(T), e->stream));
    *p = static_cast<T *>(q);
    return SOL_OK;
}

ResArrays arrays(sol_ensemble *e)
{
    ResArrays A{};
    A.tot = e->tot;
    A.y0 = e->y0; A.y = e->y; A.acc0 = e->acc0; A.yscale = e->yscale; A.err = e->errv; A.fst = e->fst;
    A.mass = e->mass; A.rm3 = e->rm3; A.nnd = e->nnd; A.nni = e->nni;
    return A;
}

int upload(sol_ensemble *e)
{
    if (e->y_dirty) {
        ECHECK(e, hipMemcpyAsync(e->y0, e->y0_h.data(), e->y0_h.size() * sizeof(double), hipMemcpyHostToDevice,
                                 e->stream));
        ECHECK(e, hipMemcpyAsync(e->mass, e->mass_h.data(), e->mass_h.size() * sizeof(double),
                                 hipMemcpyHostToDevice, e->stream));
        if (e->mesh_state) {
            e->gm_h.resize(e->mass_h.size());
            for (size_t i = 0; i < e->mass_h.size(); ++i) e->gm_h[i] = kGauss2 * e->mass_h[i];
            ECHECK(e, hipMemcpyAsync(e->mesh_gm, e->gm_h.data(), e->gm_h.size() * sizeof(double),
                                     hipMemcpyHostToDevice, e->stream));
        }
    }
    if (e->sys_dirty)
        ECHECK(e, hipMemcpyAsync(e->sys_d, e->sys_h.data(), e->sys_h.size() * sizeof(ResSystem),
                                 hipMemcpyHostToDevice, e->stream));
    ECHECK(e, hipStreamSynchronize(e->stream));
    e->y_dirty = e->sys_dirty = false;
    return SOL_OK;
}

int download(sol_ensemble *e)
{
    if (!e->stale) return SOL_OK;
    ECHECK(e, hipMemcpyAsync(e->y0_h.data(), e->y0, e->y0_h.size() * sizeof(double), hipMemcpyDeviceToHost, e->stream));
    ECHECK(e, hipStreamSynchronize(e->stream));
    e->stale = false;
    return SOL_OK;
}

// Workgroups of one launch: every CU full at the shape's occupancy, or one
// per queued system if there are fewer.
int grid_for(sol_ensemble *e, int ik, int block, int nrun)
{
    const int per_cu = resident_queue_occupancy(ik, block, e->nmax_n);
    return std::max(1, std::min(nrun, e->cu_count * per_cu));
}

bool is_wide(const sol_ensemble *e, int s) { return e->wide_block > 0 && e->sys_h[s].n >= e->wide_min; }

// Queue orders for the next launch: the running systems of each queue that
// have not had their steps (the narrow one only when `narrow_only`), the most work expected first
// (n^2 times the steps the system took in the previous launch, n^2 alone
// before the first), so that the long ones start early.  steps: the accepted
// steps of the launches that take them.
int make_order(sol_ensemble *e, int steps, bool narrow_only = false, const std::vector<char> *had = nullptr)
{
    e->order_h.clear();
    e->order_w.clear();
    for (int s = 0; s < e->nsys; ++s) {
        if (e->sys_h[s].status != RES_RUNNING || (had && (*had)[s])) continue;
        if (!is_wide(e, s)) e->order_h.push_back(s);
        else if (!narrow_only) e->order_w.push_back(s);
    }
    auto cost = [&](int s) {
        const double n = e->sys_h[s].n;
        return n * n * (double)std::max<int64_t>(1, e->last_steps[s]);
    };
    auto by_cost = [&](int a, int b) { return cost(a) > cost(b); };
    std::stable_sort(e->order_h.begin(), e->order_h.end(), by_cost);
    std::stable_sort(e->order_w.begin(), e->order_w.end(), by_cost);
    if (e->order_h.empty() && e->order_w.empty()) return SOL_OK;
    const QueueWords words[2] = {{0, (int32_t)e->order_h.size(), steps, 0}, {0, (int32_t)e->order_w.size(), steps, 0}};
    std::memcpy(e->queue_h.data(), words, sizeof words);
    std::copy(e->order_h.begin(), e->order_h.end(), e->queue_h.begin() + kQueueSlots);
    std::copy(e->order_w.begin(), e->order_w.end(), e->queue_h.begin() + kQueueSlots + e->count_n);
    ECHECK(e, hipMemcpyAsync(e->queue_d, e->queue_h.data(), e->queue_h.size() * sizeof(int32_t), hipMemcpyHostToDevice,
                             e->stream));
    return SOL_OK;
}

// Enqueues one queue's launch (the counter reset and the kernel) on st, with
// workgroups for all its systems, running or not: what is left of them and
// their steps are in the queue's words.
void enqueue_one(sol_ensemble *e, hipStream_t st, int ik, int block, bool wide, const ResArrays &A)
{
    QueueWords *words = reinterpret_cast<QueueWords *>(e->queue_d);
    const int32_t *slots = e->queue_d + kQueueSlots;
    if (wide) {
        // RKF78: the four most-read stage derivatives in LDS where they fit
        // (one wide workgroup per CU: its registers leave room for no other)
        const int lf = ik == INTEG_RKF78 && resident_lds_bytes(e->nmax_w) + resident_queue_lds_f(e->nmax_w) + 4096 <=
                                                e->lds_per_block ? 4 : 0;
        const int per_cu = resident_queue_occupancy(ik, e->wide_block, e->nmax_w, lf);
        e->grid_w = std::max(1, std::min(e->count_w, e->cu_count * per_cu));
        launch_resident_queue(st, ik, e->sys_d, slots + e->count_n, words + 1, A, e->grid_w, e->wide_block, e->nmax_w,
                              e->wide_lsh, lf);
    } else {
        e->grid = grid_for(e, ik, block, e->count_n);
        launch_resident_queue(st, ik, e->sys_d, slots, words, A, e->grid, block, e->nmax_n);
    }
}

// Captures one queue's launch into *exec (again for another integrator or
// launch shape only).
int capture_one(sol_ensemble *e, hipGraphExec_t *exec, int ik, int block, bool wide, const ResArrays &A)
{
    if (*exec) { (void)hipGraphExecDestroy(*exec); *exec = nullptr; }
    hipGraph_t g;
    ECHECK(e, hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
    enqueue_one(e, e->stream, ik, block, wide, A);
    hipError_t le = hipGetLastError();
    hipError_t ce = hipStreamEndCapture(e->stream, &g);
    if (le != hipSuccess || ce != hipSuccess) return e->fail(SOL_ERR_DEVICE, "graph capture failed");
    ECHECK(e, hipGraphInstantiate(exec, g, nullptr, nullptr, 0));
    (void)hipGraphDestroy(g);
    return SOL_OK;
}

// One persistent launch per queue over the systems that make_order queued;
// through the captured graphs when `graph` is set.
// The wide queue runs on the ensemble's stream, the narrow one beside it
// on the second stream (forked from the first and joined back), so the
// two kernels share the device: each queue's launch is a graph of its own,
// since the branches of one graph were found to run one after the other.
int launch_queue(sol_ensemble *e, int ik, int block, bool graph)
{
    const int nn = (int)e->order_h.size(), nw = (int)e->order_w.size();
    const ResArrays A = arrays(e);
    ++e->launches;
    if (graph) {
        if (nn > 0 && (!e->graph || e->graph_integ != ik || e->graph_block != block)) {
            if (int r = capture_one(e, &e->graph, ik, block, false, A)) return r;
            e->graph_integ = ik; e->graph_block = block;
        }
        if (nw > 0 && (!e->graph_w || e->graphw_integ != ik)) {
            if (int r = capture_one(e, &e->graph_w, ik, block, true, A)) return r;
            e->graphw_integ = ik;
        }
    }
    const bool both = nn > 0 && nw > 0;
    if (both) {
        ECHECK(e, hipEventRecord(e->ev_fork, e->stream));
        ECHECK(e, hipStreamWaitEvent(e->stream2, e->ev_fork, 0));
    }
    if (nw > 0) {
        if (graph) ECHECK(e, hipGraphLaunch(e->graph_w, e->stream));
        else enqueue_one(e, e->stream, ik, block, true, A);
    }
    if (nn > 0) {
        hipStream_t sn = both ? e->stream2 : e->stream;
        if (graph) ECHECK(e, hipGraphLaunch(e->graph, sn));
        else enqueue_one(e, sn, ik, block, false, A);
    }
    if (both) {
        ECHECK(e, hipEventRecord(e->ev_join, e->stream2));
        ECHECK(e, hipStreamWaitEvent(e->stream, e->ev_join, 0));
    }
    ECHECK(e, hipGetLastError());
    if (graph) ++e->graph_launches;
    return SOL_OK;
}

int read_systems(sol_ensemble *e)
{
    ECHECK(e, hipMemcpyAsync(e->sys_h.data(), e->sys_d, e->sys_h.size() * sizeof(ResSystem), hipMemcpyDeviceToHost,
                             e->stream));
    ECHECK(e, hipStreamSynchronize(e->stream));
    return SOL_OK;
}

// The mesh form (mesh.hip) takes systems whose larger class of bodies has at
// least this many sources: per RKF78 attempt in the queue and in the mesh form
// 33 bodies take 48 and 47 us, 49 bodies 54 and 48, 66 69 and 50, 97 63 and
// 51, 129 104 and 54, 193 138 and 56, 257 324 and 69.
constexpr int kMeshMinSources = 48;

bool mesh_takes(const ResSystem &S) { return std::max(S.end_a, S.end_b) >= kMeshMinSources; }

// Runs `steps` accepted steps of the running systems that the mesh form
// takes, over several workgroups each, if all of them fit the device at once;
// `had` marks them, and the caller's next queue launch leaves them out.  A
// run lasts as long as its slowest systems, which leave most of the device
// idle once the others are done: 1,024 systems over two days, of 3 to 257
// bodies and 9 steps in the mean, have 31 to 49 systems of more than 16 steps
// and need up to 504; 46 to 145 ms with the queue alone, 25 to 53 with these
// in the mesh form.  (Several launches of it in turn for more systems than
// fit gained nothing over the queue.)
int run_mesh(sol_ensemble *e, int ik, int steps, std::vector<char> &had)
{
    had.assign((size_t)e->nsys, 0);
    if (!e->mesh_state || e->mesh_off) return SOL_OK;
    std::vector<int> slots;
    int max_n = 0;
    for (int s = 0; s < e->nsys; ++s)
        if (e->sys_h[s].status == RES_RUNNING && mesh_takes(e->sys_h[s])) {
            slots.push_back(s);
            max_n = std::max(max_n, e->sys_h[s].n);
        }
    if (slots.empty() || (int)slots.size() > e->cu_count) return SOL_OK;
    // the smallest share of bodies per workgroup with which they fit
    auto groups_of = [&](int s, int share) {
        const ResSystem &S = e->sys_h[s];
        return mesh_groups(S.n, S.nm, S.end_a, S.end_b, share);
    };
    int share = 7, groups = 0;
    for (;; share += 8) {
        if (share > kMeshMaxShare) return SOL_OK;
        groups = 0;
        int most = 0;
        for (int s : slots) {
            const int g = groups_of(s, share);
            groups += g;
            most = std::max(most, g);
        }
        if (most <= kMeshMaxGroups && groups <= e->cu_count &&
            groups <= mesh_capacity(ik, max_n, share, e->cu_count)) break;
    }
    std::vector<MeshPart> parts;
    std::vector<int32_t> part_of;
    std::vector<int64_t> before;
    for (int s : slots) {
        const int g = groups_of(s, share);
        parts.push_back(MeshPart{s, (int32_t)part_of.size(), g, share});
        part_of.insert(part_of.end(), (size_t)g, (int32_t)parts.size() - 1);
        before.push_back(e->sys_h[s].steps);
    }
    ECHECK(e, hipMemcpyAsync(e->mesh_part, parts.data(), parts.size() * sizeof(MeshPart), hipMemcpyHostToDevice,
                             e->stream));
    ECHECK(e, hipMemcpyAsync(e->mesh_part_of, part_of.data(), part_of.size() * sizeof(int32_t),
                             hipMemcpyHostToDevice, e->stream));
    ECHECK(e, hipMemcpyAsync(e->mesh_sys, e->sys_d, (size_t)e->nsys * sizeof(ResSystem), hipMemcpyDeviceToDevice,
                             e->stream));
    MeshArgs A{};
    A.systems = e->mesh_sys;
    A.parts = e->mesh_part; A.part_of = e->mesh_part_of;
    A.sync = e->mesh_sync;
    A.pos = e->mesh_pos; A.gm = e->mesh_gm;
    A.tot = e->tot;
    A.y0_in = e->y0; A.mass = e->mass;
    A.y0 = e->mesh_state; A.y = e->y; A.acc0 = e->acc0; A.yscale = e->yscale; A.err = e->errv;
    A.rm3 = e->rm3; A.nnd = e->nnd; A.nni = e->nni;
    A.ticks = (uint64_t)(e->wait_s * (double)e->rtc_hz);
    {
        const UnitLease lease(e->device, groups, e->cu_count);
        ECHECK(e, launch_mesh(e->stream, ik, A, (int)parts.size(), groups, max_n, share, steps));
        ECHECK(e, launch_mesh_commit(e->stream, A, (int)parts.size(), e->sys_d, e->y0));
        if (int r = read_systems(e)) return r;
    }
    // a system whose workgroups were not all resident has kept its state, and
    // the queue takes it
    bool lost = false;
    for (size_t p = 0; p < parts.size(); ++p) {
        const ResSystem &S = e->sys_h[parts[p].system];
        const bool ran = S.status != RES_RUNNING || S.steps != before[p];
        had[parts[p].system] = ran;
        lost |= !ran;
    }
    if (lost && ++e->mesh_failures >= 2) e->mesh_off = true;
    return SOL_OK;
}

int ensemble_integ(int32_t integrator)
{
    return integrator == SOL_RUNGE_KUTTA_FEHLBERG78 ? INTEG_RKF78 : integrator == SOL_RUNGE_KUTTA4 ? INTEG_RK4
         : integrator == SOL_DORMAND_PRINCE ? INTEG_DP : -1;
}

// Times every candidate shape of the narrow queue on probe_steps accepted
// steps of its running systems from their current states, restoring states
// and descriptors after each, and keeps the fastest.
int tune(sol_ensemble *e, int ik, double eps, int probe_steps)
{
    for (auto &S : e->sys_h) S.eps = eps;
    e->sys_dirty = true;
    if (int r = upload(e)) return r;
    const size_t ny = 6 * (size_t)e->tot;
    double *y0_save = nullptr;
    ResSystem *sys_save = nullptr;
    ECHECK(e, hipMalloc(&y0_save, ny * sizeof(double)));
    ECHECK(e, hipMalloc(&sys_save, e->sys_h.size() * sizeof(ResSystem)));
    ECHECK(e, hipMemcpyAsync(y0_save, e->y0, ny * sizeof(double), hipMemcpyDeviceToDevice, e->stream));
    ECHECK(e, hipMemcpyAsync(sys_save, e->sys_d, e->sys_h.size() * sizeof(ResSystem), hipMemcpyDeviceToDevice,
                             e->stream));
    // the probe times the narrow queue's shapes on its own systems
    int r = make_order(e, probe_steps, true);
    e->cand_ms.assign(e->cand.size(), 0.0);
    hipEvent_t t0 = nullptr, t1 = nullptr;
    if (!r && (hipEventCreate(&t0) != hipSuccess || hipEventCreate(&t1) != hipSuccess))
        r = e->fail(SOL_ERR_DEVICE, "hipEventCreate failed");
    double best = -1.0;
    for (size_t k = 0; !r && k < e->cand.size() && !e->order_h.empty(); ++k) {
        (void)hipEventRecord(t0, e->stream);
        r = launch_queue(e, ik, e->cand[k], false);
        (void)hipEventRecord(t1, e->stream);
        if (!r && hipEventSynchronize(t1) != hipSuccess) r = e->fail(SOL_ERR_DEVICE, "tuning launch failed");
        float ms = 0.0f;
        (void)hipEventElapsedTime(&ms, t0, t1);
        e->cand_ms[k] = ms;
        if (!r && (best < 0.0 || ms < best)) { best = ms; e->block = e->cand[k]; }
        // restore
        if (!r && (hipMemcpyAsync(e->y0, y0_save, ny * sizeof(double), hipMemcpyDeviceToDevice, e->stream) !=
                       hipSuccess ||
                   hipMemcpyAsync(e->sys_d, sys_save, e->sys_h.size() * sizeof(ResSystem),
                                  hipMemcpyDeviceToDevice, e->stream) != hipSuccess))
            r = e->fail(SOL_ERR_DEVICE, "restoring the probed systems failed");
    }
    (void)hipStreamSynchronize(e->stream);
    if (t0) (void)hipEventDestroy(t0);
    if (t1) (void)hipEventDestroy(t1);
    (void)hipFree(y0_save);
    (void)hipFree(sys_save);
    e->launches = 0;
    if (!r) e->tuned = true;
    return r;
}

}  // namespace

extern "C" {

const char *sol_ensemble_last_error(const sol_ensemble *e) { return e ? e->err.c_str() : g_ens_create_error.c_str(); }

int sol_ensemble_create(sol_ensemble **out, int32_t nsys, const sol_nbodies *nbs, int32_t device)
{
    if (!out || !nbs || nsys <= 0) { g_ens_create_error = "bad argument"; return SOL_ERR_ARGUMENT; }
    *out = nullptr;
    for (int k = 0; k < nsys; ++k) {
        const sol_nbodies &b = nbs[k];
        const int sum = b.central_body + b.giant_planet + b.rocky_planet + b.proto_planet + b.super_planetesimal +
                        b.planetesimal + b.test_particle;
        if (b.total < 2 || sum != b.total || b.central_body != 1 || b.total > kResidentMaxBodies) {
            g_ens_create_error = "system " + std::to_string(k) + ": counts must add up to total, one central body, "
                                 "2 <= total <= " + std::to_string(kResidentMaxBodies);
            return SOL_ERR_ARGUMENT;
        }
    }
    if (hipSetDevice(device) != hipSuccess) { g_ens_create_error = "hipSetDevice failed"; return SOL_ERR_DEVICE; }
    size_t lds_per_block = 0;
    {
        // the resident kernel's LDS (64 B per body of the largest system)
        // must fit a workgroup's share, with 2 KB left for its fixed arrays
        hipDeviceProp_t prop;
        if (hipGetDeviceProperties(&prop, device) != hipSuccess) {
            g_ens_create_error = "hipGetDeviceProperties failed";
            return SOL_ERR_DEVICE;
        }
        int nmax = 0;
        for (int k = 0; k < nsys; ++k) nmax = std::max(nmax, nbs[k].total);
        if (resident_lds_bytes(nmax) + 2048 > prop.sharedMemPerBlock) {
            g_ens_create_error = "systems of " + std::to_string(nmax) + " bodies need " +
                                 std::to_string(resident_lds_bytes(nmax)) + " B of LDS per workgroup; the device has " +
                                 std::to_string(prop.sharedMemPerBlock);
            return SOL_ERR_ARGUMENT;
        }
        lds_per_block = prop.sharedMemPerBlock;
    }
    sol_ensemble *e = new sol_ensemble();
    e->device = device;
    e->lds_per_block = lds_per_block;
    e->nsys = nsys;
    e->nb.assign(nbs, nbs + nsys);
    // storage in the caller's system order
    e->slot_of.assign(nsys, 0);
    e->sys_of.assign(nsys, 0);
    e->base.assign(nsys, 0);
    e->ipe.assign(nsys, 0.0);
    e->last_steps.assign(nsys, 0);
    int64_t off = 0;
    for (int k = 0; k < nsys; ++k) {
        e->slot_of[k] = k;
        e->sys_of[k] = k;
        e->base[k] = off;
        e->ipe[k] = interactions(nbs[k]);
        off += (nbs[k].total + 63) / 64 * 64;
        e->nmax = std::max(e->nmax, nbs[k].total);
    }
    e->tot = off;
    {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && cus > 0)
            e->cu_count = cus;
    }
    // the wide queue: SOLARIS_AMD_ENSEMBLE_WIDE = "block,lanes_log2,min_bodies" or "0" (off)
    if (const char *w = std::getenv("SOLARIS_AMD_ENSEMBLE_WIDE")) {
        int b = 0, l = 0, m = 0;
        const int got = std::sscanf(w, "%d,%d,%d", &b, &l, &m);
        e->wide_block = got >= 1 ? std::max(0, std::min(768, b / 64 * 64)) : 0;
        if (got >= 2) e->wide_lsh = std::max(0, std::min(4, l));
        if (got >= 3) e->wide_min = std::max(2, m);
    }
    for (int k = 0; k < nsys; ++k) {
        if (e->wide_block > 0 && nbs[k].total >= e->wide_min) e->nmax_w = std::max(e->nmax_w, nbs[k].total);
        else e->nmax_n = std::max(e->nmax_n, nbs[k].total);
    }
    // a wide queue needs one body per thread slot
    if (e->nmax_w > e->wide_block) {
        e->wide_block = 0;
        e->nmax_n = e->nmax;
        e->nmax_w = 0;
    }
    for (int k = 0; k < nsys; ++k) e->count_w += e->wide_block > 0 && nbs[k].total >= e->wide_min ? 1 : 0;
    e->count_n = nsys - e->count_w;
    e->queue_h.assign((size_t)kQueueSlots + nsys, 0);
    // launch shapes the tuner times for the narrow queue: the exact fit
    // (one body per thread up to 640 bodies) and the multiples of 64 below
    // it that hold the largest system at two or four bodies per thread
    const int nq = std::max(2, e->nmax_n);
    const int fit = resident_block_size(nq);
    for (int c : {64, 128, 192, 256, 320, 384, 512})
        if (c < fit && 4 * c >= nq) e->cand.push_back(c);
    e->cand.push_back(fit);
    e->block = fit;
    if (const char *fix = std::getenv("SOLARIS_AMD_ENSEMBLE_BLOCK")) {
        int b = std::max(64, std::min(640, std::atoi(fix) / 64 * 64));
        if (4 * b < nq) b = (nq + 3) / 4 / 64 * 64 + 64;
        e->block = b;
        e->cand.assign(1, b);
        e->tuned = true;
    }
    const size_t tot = (size_t)e->tot;
    int r = SOL_OK;
    if (hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) != hipSuccess ||
        hipStreamCreateWithFlags(&e->stream2, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&e->ev_fork, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&e->ev_join, hipEventDisableTiming) != hipSuccess) {
        g_ens_create_error = "creating the ensemble's streams failed";
        sol_ensemble_destroy(e);
        return SOL_ERR_DEVICE;
    }
    if ((r = ealloc(e, &e->sys_d, nsys)) || (r = ealloc(e, &e->y0, 6 * tot)) || (r = ealloc(e, &e->y, 6 * tot)) ||
        (r = ealloc(e, &e->acc0, 6 * tot)) || (r = ealloc(e, &e->yscale, 6 * tot)) ||
        (r = ealloc(e, &e->errv, 6 * tot)) || (r = ealloc(e, &e->fst, 12 * 6 * tot)) ||
        (r = ealloc(e, &e->mass, tot)) || (r = ealloc(e, &e->rm3, tot)) || (r = ealloc(e, &e->nnd, tot)) ||
        (r = ealloc(e, &e->nni, tot)) || (r = ealloc(e, &e->queue_d, e->queue_h.size()))) {
        g_ens_create_error = e->err;
        sol_ensemble_destroy(e);
        return r;
    }
    bool mesh = false;
    for (int k = 0; k < nsys; ++k) {
        ResSystem S{};
        S.n = nbs[k].total;
        S.nm = nmassive(nbs[k]);
        S.end_a = S.nm + nbs[k].super_planetesimal;
        S.end_b = S.nm;
        mesh |= mesh_takes(S);
    }
    if (const char *w = std::getenv("SOLARIS_AMD_NO_GRID")) mesh &= w[0] != '1';
    if (const char *w = std::getenv("SOLARIS_AMD_GRID_WAIT")) e->wait_s = std::max(0.0, std::atof(w));
    {
        int khz = 0;
        if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device) == hipSuccess && khz > 0)
            e->rtc_hz = (uint64_t)khz * 1000;
    }
    const size_t most = (size_t)e->cu_count;      // parts, and workgroups, of a mesh launch
    if (mesh && ((r = ealloc(e, &e->mesh_state, 6 * tot)) || (r = ealloc(e, &e->mesh_gm, tot)) ||
                 (r = ealloc(e, &e->mesh_pos, 6 * tot)) || (r = ealloc(e, &e->mesh_sys, nsys)) ||
                 (r = ealloc(e, &e->mesh_part, most)) || (r = ealloc(e, &e->mesh_part_of, most)) ||
                 (r = ealloc(e, &e->mesh_sync, most)))) {
        g_ens_create_error = e->err;
        sol_ensemble_destroy(e);
        return r;
    }
    e->y0_h.assign(6 * tot, 0.0);
    e->mass_h.assign(tot, 0.0);
    e->sys_h.assign(nsys, ResSystem{});
    for (int s = 0; s < nsys; ++s) {
        const sol_nbodies &b = nbs[s];
        ResSystem &S = e->sys_h[s];
        S.n = b.total;
        S.nm = nmassive(b);
        S.end_a = S.nm + b.super_planetesimal;
        S.end_b = S.nm;
        S.base = (int32_t)e->base[s];
        S.status = RES_DONE;   // until set
        S.clip = 1;
    }
    *out = e;
    return SOL_OK;
}

int sol_ensemble_destroy(sol_ensemble *e)
{
    if (!e) return SOL_OK;
    (void)hipSetDevice(e->device);
    if (e->stream) (void)hipStreamSynchronize(e->stream);
    if (e->graph) (void)hipGraphExecDestroy(e->graph);
    if (e->graph_w) (void)hipGraphExecDestroy(e->graph_w);
    void *ptrs[] = {e->sys_d, e->y0,  e->y,   e->acc0, e->yscale,  e->errv,  e->fst,
                    e->mass,  e->rm3, e->nnd, e->nni,  e->queue_d,
                    e->mesh_state, e->mesh_gm, e->mesh_pos, e->mesh_sys, e->mesh_part, e->mesh_part_of,
                    e->mesh_sync};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    if (e->ev_fork) (void)hipEventDestroy(e->ev_fork);
    if (e->ev_join) (void)hipEventDestroy(e->ev_join);
    if (e->stream2) (void)hipStreamDestroy(e->stream2);
    if (e->stream) (void)hipStreamDestroy(e->stream);
    delete e;
    return SOL_OK;
}

int sol_ensemble_set_system(sol_ensemble *e, int32_t k, const sol_body_params *p, const double *y0,
                            const sol_timeline *tl)
{
    if (!e || !p || !y0 || !tl || k < 0 || k >= e->nsys) return SOL_ERR_ARGUMENT;
    if (download(e)) return SOL_ERR_DEVICE;
    const int s = e->slot_of[k];
    const int n = e->nb[k].total;
    const int64_t b = e->base[s], tot = e->tot;
    if (p->type)
        for (int i = 1; i < n; ++i)
            if (p->type[i] < p->type[i - 1]) return e->fail(SOL_ERR_ARGUMENT, "bodies are not sorted by type");
    for (int i = 0; i < n; ++i) {
        e->mass_h[b + i] = p->mass ? p->mass[i] : 0.0;
        for (int c = 0; c < 6; ++c) e->y0_h[c * tot + b + i] = y0[6 * (size_t)i + c];
    }
    ResSystem &S = e->sys_h[s];
    S.status = RES_RUNNING;
    S.t = tl->time; S.h_next = tl->hNext; S.h_did = tl->hDid; S.length = tl->length; S.output = tl->output;
    S.elapsed = tl->elapsedTime; S.last_save = tl->lastSave; S.last_nsteps = tl->lastNSteps;
    S.millenium = tl->millenium;
    S.flush_count = tl->flush_count;
    S.steps = 0; S.attempts = 0;
    e->last_steps[s] = 0;
    e->y_dirty = e->sys_dirty = true;
    return SOL_OK;
}

int sol_ensemble_tune(sol_ensemble *e, int32_t integrator, double eps, int32_t probe_steps)
{
    if (!e || probe_steps < 1) return SOL_ERR_ARGUMENT;
    const int ik = ensemble_integ(integrator);
    if (ik < 0) return e->fail(SOL_ERR_UNSUPPORTED, "integrator not provided");
    ECHECK(e, hipSetDevice(e->device));
    if (const char *fix = std::getenv("SOLARIS_AMD_ENSEMBLE_BLOCK")) { (void)fix; return SOL_OK; }
    return tune(e, ik, eps, probe_steps);
}

int sol_ensemble_get_info(const sol_ensemble *e, sol_ensemble_info *info)
{
    if (!e || !info) return SOL_ERR_ARGUMENT;
    *info = sol_ensemble_info{};
    info->block = e->block;
    info->bodies_per_thread = resident_queue_bpt(e->block, std::max(2, e->nmax_n));
    info->wide_block = e->wide_block;
    info->wide_lanes = e->wide_block > 0 ? 1 << e->wide_lsh : 0;
    info->wide_min_bodies = e->wide_block > 0 ? e->wide_min : 0;
    info->wide_grid = e->grid_w;
    for (int s = 0; s < e->nsys; ++s) info->wide_systems += is_wide(e, s) ? 1 : 0;
    info->grid = e->grid;
    info->tuned = e->tuned ? 1 : 0;
    info->launches = e->launches;
    info->graph_launches = e->graph_launches;
    const int nc = (int)std::min<size_t>(e->cand.size(), 8);
    info->candidates = nc;
    for (int k = 0; k < nc; ++k) {
        info->candidate_block[k] = e->cand[k];
        info->candidate_ms[k] = k < (int)e->cand_ms.size() ? e->cand_ms[k] : 0.0;
    }
    return SOL_OK;
}

int sol_ensemble_run(sol_ensemble *e, int32_t integrator, double eps, int64_t max_steps, sol_run_stats *stats)
{
    if (!e) return SOL_ERR_ARGUMENT;
    const int ik = ensemble_integ(integrator);
    if (ik < 0) return e->fail(SOL_ERR_UNSUPPORTED, "integrator not provided");
    ECHECK(e, hipSetDevice(e->device));
    if (!e->tuned) {
        if (int r = tune(e, ik, eps, 8)) return r;
    }
    for (auto &S : e->sys_h) S.eps = eps;
    e->sys_dirty = true;
    if (int r = upload(e)) return r;
    std::vector<int64_t> s0(e->nsys), a0(e->nsys);
    for (int s = 0; s < e->nsys; ++s) { s0[s] = e->sys_h[s].steps; a0[s] = e->sys_h[s].attempts; }
    // accepted steps per system per launch: about 0.25 s of the largest
    // system's Driver loop (13 stage evaluations of ~3,000 + 12 n cycles)
    const double per_step = 13.0 * (3000.0 + 12.0 * e->nmax) / 2.1e9;
    int chunk = (int)std::max<int64_t>(16, std::min<int64_t>(20000, (int64_t)(0.25 / per_step)));
    // (of the mesh form, whose launches hold their compute units, about 0.2 s)
    if (e->mesh_state && !e->mesh_off) chunk = std::min(chunk, mesh_chunk(e->nmax));
    if (max_steps > 0) chunk = (int)std::min<int64_t>(chunk, max_steps);
    // where the last systems may take the mesh form, the launches start short
    // and grow, so that few running systems are soon noticed (run_mesh)
    int next = e->mesh_state && !e->mesh_off ? std::min(chunk, kFirstSteps) : chunk;
    std::vector<char> had((size_t)e->nsys, 0);
    hipEvent_t t0, t1;
    ECHECK(e, hipEventCreate(&t0));
    ECHECK(e, hipEventCreate(&t1));
    ECHECK(e, hipEventRecord(t0, e->stream));
    int64_t done_steps = 0;
    for (;;) {
        int k = next;
        next = std::min(2 * next, chunk);
        if (max_steps > 0) k = (int)std::min<int64_t>(k, max_steps - done_steps);
        std::vector<int64_t> before(e->nsys);
        for (int s = 0; s < e->nsys; ++s) before[s] = e->sys_h[s].steps;
        if (done_steps > 0)
            if (int r = run_mesh(e, ik, k, had)) return r;
        if (int r = make_order(e, k, false, &had)) return r;
        if (!e->order_h.empty() || !e->order_w.empty()) {
            if (int r = launch_queue(e, ik, e->block, true)) return r;
            if (int r = read_systems(e)) return r;
        }
        done_steps += k;
        for (int s = 0; s < e->nsys; ++s) e->last_steps[s] = e->sys_h[s].steps - before[s];
        const bool any = std::any_of(e->sys_h.begin(), e->sys_h.end(), [](const ResSystem &S) { return S.status == RES_RUNNING; });
        if (!any) break;
        if (max_steps > 0 && done_steps >= max_steps) break;
    }
    ECHECK(e, hipEventRecord(t1, e->stream));
    ECHECK(e, hipEventSynchronize(t1));
    float ms = 0.0f;
    (void)hipEventElapsedTime(&ms, t0, t1);
    (void)hipEventDestroy(t0);
    (void)hipEventDestroy(t1);
    e->stale = true;
    if (stats) {
        const int per = ik == INTEG_RKF78 ? 12 : ik == INTEG_RK4 ? 3 : 8;
        *stats = sol_run_stats{};
        for (int s = 0; s < e->nsys; ++s) {
            const int64_t st = e->sys_h[s].steps - s0[s], at = e->sys_h[s].attempts - a0[s];
            stats->accepted_steps += st;
            stats->attempts += at;
            const int64_t ev = st + at * per;
            stats->force_evaluations += ev;
            stats->interactions += (double)ev * e->ipe[s];
        }
        stats->device_ms = ms;
        stats->path = SOL_PATH_RESIDENT;
    }
    return SOL_OK;
}

int sol_ensemble_get_system(sol_ensemble *e, int32_t k, double *y0, sol_timeline *tl, int32_t *status,
                            int64_t *steps)
{
    if (!e || k < 0 || k >= e->nsys) return SOL_ERR_ARGUMENT;
    ECHECK(e, hipSetDevice(e->device));
    if (int r = download(e)) return r;
    const int s = e->slot_of[k];
    const int n = e->nb[k].total;
    const int64_t b = e->base[s], tot = e->tot;
    if (y0)
        for (int i = 0; i < n; ++i)
            for (int c = 0; c < 6; ++c) y0[6 * (size_t)i + c] = e->y0_h[c * tot + b + i];
    const ResSystem &S = e->sys_h[s];
    if (tl) {
        tl->time = S.t; tl->hNext = S.h_next; tl->hDid = S.h_did; tl->length = S.length; tl->output = S.output;
        tl->elapsedTime = S.elapsed; tl->lastSave = S.last_save; tl->lastNSteps = S.last_nsteps;
        tl->millenium = S.millenium;
        tl->flush_count = S.flush_count;
    }
    if (status) *status = S.status;
    if (steps) *steps = S.steps;
    return SOL_OK;
}

}  // extern "C"
