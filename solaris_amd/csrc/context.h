// context.h -- the context object behind the sol_context handle of
// include/solaris_amd.h, shared by context.cpp (forces, drivers) and
// adjoint.cpp (the RK4 adjoint).
#pragma once

#include <algorithm>
#include <cstdarg>
#include <cstddef>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "sol_internal.h"
#include "resident.h"
#include "mesh.h"
#include "quad.h"

namespace sol {
struct AdjointState;

// What a run of the mesh form reads first, in one copy, and what comes back
// of it and of the quad form: the descriptor up to the exchange's error word
// (the first of either form's words: a wait gave up).
struct MeshRun {
    ResSystem system;
    MeshPart part;
    union Words { MeshSync mesh; QuadSync quad; };
    alignas(128) Words words;
};
constexpr size_t kMeshRunBack = offsetof(MeshRun, words) + sizeof(uint32_t);
}  // namespace sol

struct sol_context {
    int device = 0;
    hipStream_t stream = nullptr;
    hipStream_t stream2 = nullptr;                       // the nearest-neighbour search beside the pair sum
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    sol_nbodies nb{};
    int n = 0, np = 0, nblk = 0, n_massive = 0;
    int barycentric = 0;
    int precision = SOL_PRECISION_FP64;
    double softening = 0.0;
    int end_massive = -1, end_other = -1;
    bool has_gas = false, gas_dead = false;
    sol_gas_component gas{};
    sol::GasDev gasdev{};
    int eval_drag = 1, eval_mig1 = 1, eval_mig2 = 1;
    int cu_count = 256;
    int waves_per_simd = 8;
    int chunk = 256;
    sol::PairPlan plan{};
    double interactions_per_eval = 0.0;
    std::string err;

    // device buffers
    double *mass = nullptr, *gm = nullptr, *radius = nullptr, *density = nullptr, *cd = nullptr;
    double *gs = nullptr, *ge = nullptr, *stop = nullptr;
    int32_t *type = nullptr, *migt = nullptr;
    double *y0 = nullptr, *y = nullptr, *acc0 = nullptr, *yscale = nullptr, *error = nullptr;
    double *fst = nullptr, *cin = nullptr, *aos = nullptr;
    double4 *J = nullptr;
    float4 *J32 = nullptr;     // allocated when the mixed form is selected
    sol::NNGrid grid{};       // nearest-neighbour search of the symmetric path
    double *part = nullptr, *nnr2 = nullptr;
    int32_t *nnidx = nullptr;
    double *ind = nullptr;
    double *rm3 = nullptr, *nnd = nullptr;
    int32_t *nni = nullptr;
    double *migc = nullptr, *dragc = nullptr;
    double *errblk = nullptr, *scal = nullptr, *coef = nullptr, *integ = nullptr;
    unsigned char *pinned = nullptr;   // one allocation: mesh_h, res_h, h_scal, io_h
    double *h_scal = nullptr;   // pinned: [0] h, [1] t, [2] error max
    double *integ_h = nullptr;  // pinned, 12 * np: the integrals' rows and the masses (made on first use)
    // pinned: the arrays of a call, which the kernels read and write in place
    // (those that do not fit are copied to and from aos)
    double *io_h = nullptr;
    size_t io_bytes = 0;
    size_t part_slots = 0;
    std::vector<void *> allocs;
    // workgroup-resident drivers (resident.hip) for small systems
    sol::ResSystem *res_d = nullptr, *res_h = nullptr;
    bool resident_disabled = false;
    size_t lds_limit = 65536;
    // few-source systems too large for one workgroup: slices of the system
    // over one cooperative grid (resident.hip), in their own slice-layout
    // buffers (gbuf: 111 doubles per slot, gibuf: 2 int32)
    bool grid_disabled = false;
    int grid_block = 0;           // slice threads; 0: chosen per system
    int grid_min_bodies = 129, quad_min_bodies = 2;
    sol::ResSystem *grid_sys_d = nullptr;
    std::vector<sol::ResSystem> grid_sys_h;
    int grid_sys_cap = 0;
    double *gbuf = nullptr;
    int32_t *gibuf = nullptr;
    int64_t gbuf_tot = 0;
    sol::GridSync *gsync = nullptr;
    double grid_wait_s = 2.0;        // seconds a grid-wide wait lasts before it gives up
    uint64_t rtc_hz = 100000000;     // the device's real-time counter
    int grid_failures = 0;           // grid runs that gave up; two turn the grid form off
    int grid_capacity[18] = {-1, -1, -1, -1, -1, -1, -1, -1, -1,
                             -1, -1, -1, -1, -1, -1, -1, -1, -1};   // per integrator, gas, slice size
    // systems over several workgroups that exchange positions (mesh.hip) or,
    // with few sources, step decisions only (quad.hip): the arrays a run writes, which change places with the context's own at its end
    // (a run that could not complete leaves those untouched)
    struct Mesh {
        double *y0 = nullptr, *y = nullptr, *acc0 = nullptr, *yscale = nullptr, *error = nullptr;
        double *rm3 = nullptr, *nnd = nullptr;
        int32_t *nni = nullptr;
        double *pos = nullptr;
        // with gas: migration and drag (prev: as the run's last launch left them)
        int32_t *migt = nullptr, *migt_prev = nullptr;
        double *migc = nullptr, *migc_prev = nullptr, *dragc = nullptr;
        sol::MeshRun *run = nullptr;
        int32_t *part_of = nullptr;
    } mesh;
    sol::MeshRun *mesh_h = nullptr;          // pinned: a run's words to the device ([0]) and back ([1])
    // workgroups the device holds (-1: not asked yet): mesh form by integrator
    // and share, quad form by integrator and pulls per lane, with gas also places
    int mesh_caps[3][4], quad_caps[3][3], quad_gas_caps[3][3][2];
    // profiling (sol_profile)
    bool profiling = false;
    std::vector<hipEvent_t> ev_pool;
    struct Timed { hipEvent_t a, b; int kind; double inter; };
    std::vector<Timed> timed;
    size_t ev_used = 0;
    sol_kernel_profile prof{};
    double pair_inter_per_launch = 0.0;
    // symmetric pair sum of the self-interacting block (pairs.hip) and the
    // one-directional plan of the remaining ranges
    sol::SymPlan sym{};
    sol::PairPlan plan_rest{};
    double sym_inter_per_launch = 0.0, rest_inter_per_launch = 0.0;
    double *apart = nullptr, *bpart = nullptr;
    size_t apart_cap = 0, bpart_cap = 0;
    bool sym_disabled = false;
    bool side_outputs = true;     // sol_compute tracks nearest neighbours (sol_set_side_outputs)
    // event thresholds of sol_integrate_until (sol_set_events): 1/ejection^3,
    // 1/hitCentrum^3 and the collision factor, each 0 when off
    double ev_e3 = 0.0, ev_h3 = 0.0, ev_factor = 0.0;
    int32_t *ev_flag = nullptr;   // device: any event at the last accepted step
    // recorded forward pass of the RK4 adjoint (adjoint.cpp)
    sol::AdjointState *adj = nullptr;

    int fail(int code, const char *fmt, ...)
    {
        char buf[512];
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(buf, sizeof(buf), fmt, ap);
        va_end(ap);
        err = buf;
        return code;
    }
};

// The end of a call that queues work: one that fails in between waits for what
// it has queued on either stream, as its kernels read and write pinned memory
// that the next call fills, and the neighbour search may not have been joined.
class CallEnd {
public:
    explicit CallEnd(sol_context *c) : c_(c) {}
    ~CallEnd()
    {
        if (!failed_) return;
        (void)hipStreamSynchronize(c_->stream);
        if (c_->stream2) (void)hipStreamSynchronize(c_->stream2);
    }
    CallEnd(const CallEnd &) = delete;
    CallEnd &operator=(const CallEnd &) = delete;
    // r is the call's result
    int operator()(int r)
    {
        failed_ = r != SOL_OK;
        return r;
    }

private:
    sol_context *c_;
    bool failed_ = true;
};

#define HIPCHECK(ctx, call)                                                                    \
    do {                                                                                       \
        hipError_t e_ = (call);                                                                \
        if (e_ != hipSuccess)                                                                  \
            return (ctx)->fail(SOL_ERR_DEVICE, "%s failed: %s (%s:%d)", #call,                \
                               hipGetErrorString(e_), __FILE__, __LINE__);                     \
    } while (0)

namespace sol {

// Device allocation owned by the context (freed by sol_destroy), zeroed.
template <typename T>
int dalloc(sol_context *c, T **p, size_t count)
{
    void *q = nullptr;
    HIPCHECK(c, hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T)));
    // on the context's stream: a fill on the default stream is not waited for,
    // and would not be ordered before the kernels of a non-blocking one
    HIPCHECK(c, hipMemsetAsync(q, 0, std::max<size_t>(count, 1) * sizeof(T), c->stream));
    c->allocs.push_back(q);
    *p = static_cast<T *>(q);
    return SOL_OK;
}

// Several arrays in one allocation, which the first of them starts.  Each
// allocation takes time of its own to make, to fill and to give back: a context
// of 515 bodies made and destroyed takes 565 us with 33 of them and 400 with
// three, of a disk of 16,385 865 us with 47 and 545 with five.
class ArrayBlock {
public:
    template <typename T>
    void add(T **p, size_t count)
    {
        items_.push_back({p, bytes_});
        bytes_ += (std::max<size_t>(count, 1) * sizeof(T) + kPage - 1) / kPage * kPage;
    }
    size_t bytes() const { return bytes_; }
    void place(void *block)
    {
        for (const Item &i : items_) {
            void *at = static_cast<unsigned char *>(block) + i.at;
            std::memcpy(i.p, &at, sizeof at);
        }
    }
    // Owned by the context (freed by sol_destroy), zeroed.  Leaves the pointers
    // alone when it fails.
    int make(sol_context *c)
    {
        unsigned char *q = nullptr;
        if (int r = dalloc(c, &q, bytes_)) return r;
        place(q);
        return SOL_OK;
    }

private:
    static constexpr size_t kPage = 4096;      // (at 256 bytes a mixed step of 32,769 bodies is 1.2% slower)
    struct Item { void *p; size_t at; };       // the pointer's place, and its array's in the block
    std::vector<Item> items_;
    size_t bytes_ = 0;
};

// Source range ends of the two astrocentric sink classes.
void source_ends(const sol_context *c, int &ea, int &eb);

// One FP64 force evaluation (Acceleration::Compute) of the device state
// `st` (6 x NP) at time t into `out` (6 x NP), on the context's stream.
int eval_force(sol_context *c, const double *st, double t, double *out);

// Whether the workgroup-resident driver can run this context (small, no
// gas), and nsteps fixed RK4 steps with it from the state y (6 x NP, updated
// in place; ytmp is scratch of the same size) at t0 with the device step
// sizes h_seq, writing the stage states [nsteps][4][6 NP] to stages when
// it is not null.  One launch; synchronous.
bool resident_rk4_ok(const sol_context *c);
int resident_rk4(sol_context *c, double *y, double *ytmp, double t0, const double *h_seq, int64_t nsteps,
                 double *stages);

// Frees the adjoint's recorded state (adjoint.cpp).
void adjoint_release(sol_context *c);
// Marks the recorded forward pass stale (parameters or force model changed).
void adjoint_invalidate(sol_context *c);

}  // namespace sol
