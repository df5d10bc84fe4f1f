// context.cpp -- the C ABI of include/solaris_amd.h on one MI355X.
//
// A context owns the device mirror of BodyData (structure-of-arrays), the
// stage buffers of the integrators, the pair-sum work plan and one HIP
// stream.  The drivers follow the reference's control flow step for step
// (RungeKuttaFehlberg78::Driver, RungeKutta4::Driver, DormandPrince::Driver)
// with all array work on the device; only the scalar step-size decisions
// run on the host, from one 8-byte error maximum per attempt.
#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "context.h"
#include "stream_pool.h"
#include "tableaux.h"
#include "unit_lease.h"

using namespace sol;

// The tables of tableaux.h packed at the offsets stages.hip reads.
void sol::fill_coefficients(std::vector<double> &c)
{
    c.assign(275, 0.0);
    for (int s = 0; s < 13; ++s)
        for (int l = 0; l < 12; ++l) c[0 + s * 12 + l] = tab::kRkfD[s][l];
    for (int s = 0; s < 4; ++s)
        for (int l = 0; l < 3; ++l) c[156 + s * 3 + l] = tab::kRk4A[s][l];
    for (int k = 0; k < 4; ++k) { c[168 + k] = tab::kRk4B[k]; c[172 + k] = tab::kRk4C[k]; }
    for (int k = 0; k < 9; ++k)
        for (int l = 0; l < 8; ++l) c[176 + k * 8 + l] = tab::kDpA[k][l];
    for (int k = 0; k < 9; ++k) { c[248 + k] = tab::kDpB[k]; c[257 + k] = tab::kDpBdh[k]; c[266 + k] = tab::kDpC[k]; }
}

namespace {

double host_reduction_factor(const sol_gas_component &g, double t)
{   // GasComponent::ReductionFactor, Solaris/GasComponent.cpp:36-61
    switch (g.type) {
    case SOL_GAS_CONSTANT: return 1.0;
    case SOL_GAS_LINEAR:
        if (t <= g.t0) return 1.0;
        if (t > g.t0 && t <= g.t1) return 1.0 - (t - g.t0) / (g.t1 - g.t0);
        return 0.0;
    case SOL_GAS_EXPONENTIAL: return std::exp(-t / g.time_scale);
    default: return 1.0;
    }
}

thread_local std::string g_create_error;

}  // namespace

// Source range ends of the two astrocentric sink classes
// (Solaris/Acceleration.cpp:285-289).
void sol::source_ends(const sol_context *c, int &ea, int &eb)
{
    ea = c->end_massive >= 0 ? c->end_massive : c->n_massive + c->nb.super_planetesimal;
    eb = c->end_other >= 0 ? c->end_other : c->n_massive;
}

namespace {

int n_pl_spl(const sol_nbodies &nb) { return nb.super_planetesimal + nb.planetesimal; }

bool mixed_on(const sol_context *c) { return c->precision == SOL_PRECISION_MIXED && c->J32 != nullptr; }

struct SegSpec { int sb, se, jb, je; };

// Stream-K work plan over sink ranges x source ranges; *pairs receives the
// pair terms one launch evaluates (self pairs excluded).
PairPlan make_plan(const sol_context *c, const SegSpec *segs, int ns, double *pairs)
{
    PairPlan p{};
    int64_t items = 0;
    int tiles = 0;
    p.nseg = 0;
    p.chunk = c->chunk;
    double np = 0.0;
    for (int k = 0; k < ns; ++k) {
        const SegSpec &s = segs[k];
        const int nsink = s.se - s.sb, nsrc = s.je - s.jb;
        if (nsink <= 0 || nsrc <= 0) continue;
        PairSeg &g = p.seg[p.nseg++];
        g.sink_begin = s.sb; g.sink_end = s.se;
        g.src_begin = s.jb; g.src_end = s.je;
        g.ntiles = (nsink + kWave - 1) / kWave;
        g.nchunks = (nsrc + c->chunk - 1) / c->chunk;
        g.tile_begin = tiles;
        g.item_begin = items;
        tiles += g.ntiles;
        items += (int64_t)g.ntiles * g.nchunks;
        const int lo = std::max(s.sb, s.jb), hi = std::min(s.se, s.je);
        np += (double)nsink * (double)nsrc - (hi > lo ? hi - lo : 0);
    }
    p.ntiles = tiles;
    p.total_items = items;
    if (pairs) *pairs = np;
    const int64_t wmax = (int64_t)c->cu_count * 4 * c->waves_per_simd;
    p.nwaves = (int)std::max<int64_t>(1, std::min<int64_t>(wmax, items));
    // slots per wave: the largest number of tiles one wave's range touches
    auto tile_of = [&](int64_t x) {
        int s = 0;
        while (s + 1 < p.nseg && x >= p.seg[s + 1].item_begin) ++s;
        return p.seg[s].tile_begin + (int)((x - p.seg[s].item_begin) / p.seg[s].nchunks);
    };
    int spw = 1;
    if (items > 0) {
        for (int64_t w = 0; w < p.nwaves; ++w) {
            const int64_t lo = (w * items) / p.nwaves, hi = ((w + 1) * items) / p.nwaves;
            if (hi > lo) spw = std::max(spw, tile_of(hi - 1) - tile_of(lo) + 1);
        }
    }
    p.slots_per_wave = spw;
    return p;
}

// Bodies of the mutual block below which the one-directional sum is kept.
constexpr int kSymMinBodies = 2048;

constexpr int kBesideMinBodies = 8192;   // the neighbour search beside the pair sum (pair_sums)

// A call's arrays go through pinned memory that the kernels read and write in
// place, up to this many bodies of six doubles: it saves a copy command, its
// wait and a kernel on each side.  Measured for set_state, get_array and a
// force evaluation of giants and test particles, us, with copies and without:
// 515 bodies 35, 36, 66 and 22, 16, 38; 16,385 50, 61, 117 and 40, 49, 99;
// 40,001 93, 140, 234 and 95, 140, 245 (the host's own copy then costs what
// the copy command does).  The side outputs, half the size and four copies:
// 515 bodies 73 and 19, 16,385 58 and 35, 65,537 117 and 96.
constexpr int kIoBodies = 32768;

// Builds the pair-sum work plans for the context's sink classes: the full
// one-directional plan (every evaluation that tracks nearest neighbours,
// the mixed form, barycentric frames) and, when the self-interacting block
// [1, M) is large, the symmetric plan of that block plus a one-directional
// plan of the remaining (sink, source) ranges.
void build_plan(sol_context *c)
{
    SegSpec segs[kMaxSeg];
    int ns = 0;
    int ea = 0, eb = 0;
    if (c->barycentric) {
        segs[ns++] = {0, c->n_massive, 0, c->n_massive};
        segs[ns++] = {c->n_massive, c->n, 0, c->n_massive};
    } else {
        source_ends(c, ea, eb);
        segs[ns++] = {1, c->n_massive, 1, ea};
        segs[ns++] = {c->n_massive, c->n, 1, eb};
    }
    double pairs = 0.0;
    c->plan = make_plan(c, segs, ns, &pairs);
    c->pair_inter_per_launch = pairs;
    // interactions per evaluation: pair terms plus the Kepler term of every
    // astrocentric sink
    double kepler = 0.0;
    for (int k = 0; k < ns; ++k)
        if (!c->barycentric && segs[k].se > segs[k].sb) kepler += (double)(segs[k].se - segs[k].sb);
    c->interactions_per_eval = pairs + kepler;

    c->sym = SymPlan{};
    c->plan_rest = PairPlan{};
    c->rest_inter_per_launch = 0.0;
    c->sym_inter_per_launch = 0.0;
    if (c->barycentric || c->sym_disabled) return;
    const int nm = c->n_massive;
    // largest M such that every body of [1, M) is a source of every other
    const int M = std::min(ea, eb) > nm ? std::min(std::min(ea, eb), c->n) : std::min(nm, ea);
    if (M - 1 < kSymMinBodies) return;
    // Workgroups of the same number of items k each, at most 26 per CU (of
    // which 3 or 4 run at a time): short ones fill the device evenly to the
    // end, and each adds a record per column it touches to the epilogue's
    // reads.  k = 1, 2, 3, 4, 5: at 32,769 bodies 482, 460, 450, 481 (k = 4)
    // and 509 us for FP64 with 2 or 3 items in a workgroup; at 65,537 1,604
    // (k = 5) to 1,697 (k = 8) and 1,683 (k = 1), the epilogue 54, 49 and 90.
    // Mixed precision, whose pairs take half the time, splits the items of small
    // systems into units: pair sum and epilogue of 3,001 bodies 43 + 14 us with
    // whole items, 25 + 15 with two units and 16 + 18 with four, 5,001 44 + 15,
    // 28 + 17 and 22 + 21, 8,193 54 + 16, 40 + 20 and 34 + 26, 12,001 71 + 19,
    // 57 + 23 and 54 + 32, 16,385 94 + 20, 85 + 27 and 113 + 40; FP64 gains
    // what its epilogue loses (8,193 bodies 48 + 16, 45 + 19).
    // SOLARIS_AMD_SYM_WAVES overrides the count (tests use it to give each
    // workgroup many items).
    const int64_t groups = (M - 1 + kSymGroup - 1) / kSymGroup;
    int64_t items = groups * (groups + 1) / 2;
    const int shift = !mixed_on(c) ? 0 : items <= 400 ? 2 : items <= 1600 ? 1 : 0;
    items <<= shift;
    const int64_t most = (int64_t)c->cu_count * 26;
    const int64_t per = (items + most - 1) / most;
    int64_t waves = (items + per - 1) / per;
    if (const char *e = std::getenv("SOLARIS_AMD_SYM_WAVES")) {
        const long v = std::atol(e);
        if (v > 0) waves = v;
    }
    sym_plan_make(c->sym, M, waves, shift);
    c->sym_inter_per_launch = (double)(M - 1) * (double)(M - 2);
    SegSpec rest[kMaxSeg];
    int nr = 0;
    rest[nr++] = {1, std::min(M, nm), M, ea};                 // mutual sinks of the first class, sources past M
    if (M > nm) rest[nr++] = {nm, M, M, eb};                  // mutual sinks of the second class, sources past M
    if (M < nm) rest[nr++] = {M, nm, 1, ea};                  // first-class sinks outside the block
    rest[nr++] = {std::max(M, nm), c->n, 1, eb};              // second-class sinks outside the block
    c->plan_rest = make_plan(c, rest, nr, &c->rest_inter_per_launch);
}

int ensure_partials(sol_context *c)
{
    if (c->sym.M > 0 && !c->grid.params) {
        // the nearest-neighbour search that goes with the symmetric sum
        NNGrid &g = c->grid;
        const size_t mc = nn_grid_max_cells(c->n), np = (size_t)c->np;
        ArrayBlock b;
        b.add(&g.params, 1); b.add(&g.bbox, kGridBboxBlocks * 6);
        b.add(&g.count, mc + 1); b.add(&g.start, mc + 1);
        b.add(&g.cellof, np); b.add(&g.rank, np); b.add(&g.spos, np);
        b.add(&g.r2, np); b.add(&g.idx, np);
        if (int r = b.make(c)) return r;
        g.max_cells = (int32_t)mc;
    }
    if (c->sym.M > 0 && c->n >= kBesideMinBodies && !c->stream2) {
        // for the search beside the sum (pair_sums)
        HIPCHECK(c, StreamPool::take(c->device, &c->stream2));
        HIPCHECK(c, hipEventCreateWithFlags(&c->ev_fork, hipEventDisableTiming));
        HIPCHECK(c, hipEventCreateWithFlags(&c->ev_join, hipEventDisableTiming));
    }
    if (c->sym.M > 0) {
        const size_t na = (size_t)sym_units(c->sym) * 3 * kSymGroup;
        const size_t nb = (size_t)c->sym.nwaves * c->sym.slots_per_wave * 3 * kSymGroup;
        if (na > c->apart_cap || nb > c->bpart_cap) {
            const size_t ca = std::max(na, c->apart_cap), cb = std::max(nb, c->bpart_cap);
            if (c->apart) (void)hipFree(c->apart);
            c->apart = c->bpart = nullptr;
            c->apart_cap = c->bpart_cap = 0;
            ArrayBlock b;
            b.add(&c->apart, ca);
            b.add(&c->bpart, cb);
            void *q = nullptr;
            HIPCHECK(c, hipMalloc(&q, b.bytes()));
            b.place(q);
            c->apart_cap = ca;
            c->bpart_cap = cb;
        }
    }
    const size_t need = std::max((size_t)c->plan.nwaves * c->plan.slots_per_wave,
                                 (size_t)c->plan_rest.nwaves * c->plan_rest.slots_per_wave);
    if (need <= c->part_slots) return SOL_OK;
    if (c->part) (void)hipFree(c->part);
    c->part = nullptr; c->nnr2 = nullptr; c->nnidx = nullptr;
    c->part_slots = 0;
    ArrayBlock b;
    b.add(&c->part, need * 3 * kWave);
    b.add(&c->nnr2, need * kWave);
    b.add(&c->nnidx, need * kWave);
    void *q = nullptr;
    HIPCHECK(c, hipMalloc(&q, b.bytes()));
    b.place(q);
    c->part_slots = need;
    return SOL_OK;
}

// Event pair around a launch when profiling (kind 0: pair sum, 1: epilogue).
hipEvent_t prof_event(sol_context *c)
{
    if (c->ev_used == c->ev_pool.size()) {
        hipEvent_t e;
        if (hipEventCreate(&e) != hipSuccess) return nullptr;
        c->ev_pool.push_back(e);
    }
    return c->ev_pool[c->ev_used++];
}

// kinds: 0 one-directional pair sum, 1 epilogue, 2 pair sum with the
// nearest-neighbour search, 3 symmetric pair sum
struct ProfScope {
    sol_context *c;
    hipEvent_t a = nullptr;
    int kind;
    double inter;
    ProfScope(sol_context *c_, int kind_, double inter_ = 0.0) : c(c_), kind(kind_), inter(inter_)
    {
        if (c->profiling && (a = prof_event(c))) (void)hipEventRecord(a, c->stream);
    }
    ~ProfScope()
    {
        if (!a) return;
        hipEvent_t b = prof_event(c);
        if (!b) return;
        (void)hipEventRecord(b, c->stream);
        c->timed.push_back({a, b, kind, inter});
    }
};

// Folds finished event pairs into the totals and recycles the events.
void prof_collect(sol_context *c)
{
    if (c->timed.empty()) return;
    (void)hipStreamSynchronize(c->stream);
    for (auto &t : c->timed) {
        float ms = 0.0f;
        (void)hipEventElapsedTime(&ms, t.a, t.b);
        if (t.kind == 0) { c->prof.pair_launches++; c->prof.pair_ms += ms; c->prof.pair_interactions += t.inter; }
        else if (t.kind == 2) { c->prof.pair_nn_launches++; c->prof.pair_nn_ms += ms; }
        else if (t.kind == 3) {
            c->prof.pair_sym_launches++; c->prof.pair_sym_ms += ms; c->prof.pair_sym_interactions += t.inter;
        } else { c->prof.epilogue_launches++; c->prof.epilogue_ms += ms; }
    }
    c->timed.clear();
    c->ev_used = 0;
}

GasDev to_dev(const sol_gas_component &g)
{
    GasDev d{};
    d.alpha = g.alpha; d.mmw = g.mean_molecular_weight; d.particle_diameter = g.particle_diameter;
    d.type = g.type; d.time_scale = g.time_scale; d.t0 = g.t0; d.t1 = g.t1; d.inner_edge = g.inner_edge;
    d.eta_c = g.eta.c; d.eta_i = g.eta.index; d.tau_c = g.tau.c; d.tau_i = g.tau.index;
    d.sh_c = g.scale_height.c; d.sh_i = g.scale_height.index; d.rho_c = g.density.c; d.rho_i = g.density.index;
    d.mfp_c = g.mean_free_path.c; d.mfp_i = g.mean_free_path.index;
    return d;
}

// Epilogue arguments common to all stages.
EpiArgs base_args(sol_context *c)
{
    EpiArgs a{};
    a.plan = c->plan;
    a.part = c->part; a.nnr2 = c->nnr2; a.nnidx = c->nnidx;
    a.n = c->n; a.np = c->np; a.nblk = c->nblk; a.barycentric = c->barycentric;
    a.n_massive = c->n_massive; a.n_central = c->nb.central_body; a.n_giant = c->nb.giant_planet;
    source_ends(c, a.src_end_a, a.src_end_b);
    a.drag_lo = c->n_massive; a.drag_hi = c->n_massive + n_pl_spl(c->nb);
    const bool gas_live = c->has_gas && !c->gas_dead;
    a.gas_on = gas_live ? 1 : 0;
    a.drag_eval = c->eval_drag;
    a.mig_on = gas_live ? 1 : 0;
    a.J = c->J;
    a.J32 = mixed_on(c) ? c->J32 : nullptr;
    a.mixed = mixed_on(c) ? 1 : 0;
    a.mass = c->mass; a.radius = c->radius; a.density = c->density; a.cd = c->cd; a.gs = c->gs; a.ge = c->ge;
    a.migt = c->migt; a.migc = c->migc; a.dragc = c->dragc;
    a.gas = c->gasdev;
    a.rm3_out = c->rm3; a.nni_out = c->nni; a.nnd_out = c->nnd;
    a.y0 = c->y0; a.acc0 = c->acc0; a.fst = c->fst;
    a.yscale = c->yscale; a.y_out = c->y; a.err_out = c->error; a.errblk = c->errblk;
    a.scal = nullptr; a.coef = c->coef;
    return a;
}

double *fslot(sol_context *c, int s) { return c->fst + (size_t)(s - 1) * 6 * c->np; }
double *ind_buf(sol_context *c, int parity) { return c->ind + (size_t)(parity & 1) * c->nblk * 6; }


// The pair sums of one evaluation from the current J (and J32): the
// symmetric sum of the mutual block plus the one-directional sum of the
// rest when the context has a symmetric plan (astrocentric, block of at
// least 2,048 bodies), else the one-directional sum of everything.
//
// With nn (the last stage of an attempt, sol_compute with side outputs) the
// symmetric path adds the grid search for the nearest neighbours (FP64
// positions, O(N)); the forces of every stage then come from the same
// kernel, which in mixed precision also keeps the FP32 rounding of the
// pair sums cancelling in the error estimate's F10 - F12 (RKF78) and
// F7 - F8 (Dormand-Prince).  Sets the epilogue's plan fields.
int pair_sums(sol_context *c, bool nn, EpiArgs &a)
{
    const double eps2 = c->softening * c->softening;
    a.nn_sep = 0;
    if (c->sym.M > 0) {
        // The nearest-neighbour search (six short launches) beside the pair
        // sum, on the second stream, where that is long enough to pay for the
        // events; one after the other and beside, us per force evaluation:
        // 4,001 bodies 109 and 113..122, 6,001 132 and 131..137, 8,193 159 and
        // 149..156, 16,385 281 and 253, 40,001 929 and 885.  (A profiled
        // context times its launches one by one.)
        const bool beside = nn && !c->profiling && c->n >= kBesideMinBodies;
        if (beside) HIPCHECK(c, hipEventRecord(c->ev_fork, c->stream));
        {
            ProfScope ps(c, 3, c->sym_inter_per_launch);
            if (mixed_on(c))
                launch_pairs_sym_mixed(c->stream, c->sym, c->J32, c->J, c->apart, c->bpart, eps2);
            else
                launch_pairs_sym(c->stream, c->sym, c->J, c->apart, c->bpart, eps2);
        }
        if (beside) HIPCHECK(c, hipStreamWaitEvent(c->stream2, c->ev_fork, 0));
        if (nn) {
            ProfScope ps(c, 2, 0.0);
            launch_nn_grid(beside ? c->stream2 : c->stream, c->grid, c->plan, c->J, c->n, c->barycentric != 0);
            a.nnr2 = c->grid.r2;
            a.nnidx = c->grid.idx;
            a.nn_sep = 1;
        }
        if (c->plan_rest.total_items > 0) {
            ProfScope ps(c, 0, c->rest_inter_per_launch);
            launch_pairs(c->stream, c->plan_rest, c->J, c->part, c->nnr2, c->nnidx, false, false, mixed_on(c), eps2,
                         c->J32);
        }
        if (beside) {
            HIPCHECK(c, hipEventRecord(c->ev_join, c->stream2));
            HIPCHECK(c, hipStreamWaitEvent(c->stream, c->ev_join, 0));
        }
        a.plan = c->plan_rest;
        a.sym = c->sym;
        a.use_sym = 1;
        a.apart = c->apart;
        a.bpart = c->bpart;
        return SOL_OK;
    }
    {
        ProfScope ps(c, nn ? 2 : 0, c->pair_inter_per_launch);
        launch_pairs(c->stream, c->plan, c->J, c->part, c->nnr2, c->nnidx, nn, c->barycentric != 0, mixed_on(c),
                     eps2, c->J32);
    }
    a.plan = c->plan;
    a.use_sym = 0;
    return SOL_OK;
}

// One full force evaluation of the state `st` (6 x NP) at time t, the
// reference's Acceleration::Compute, with the derivative in `out`.
// rows: the state in the interface's rows instead, which go to st = cin.
// kind: EPI_COMPUTE, EPI_ROWS or EPI_STAGE0 (the Driver's evaluation at y0; also
// writes yscale for RKF78 with the trial h).
int evaluate_at(sol_context *c, const double *st, double t, double h, double *out, int kind, int integ,
                bool last, bool want_yscale, const double *rows = nullptr)
{
    int ea, eb;
    source_ends(c, ea, eb);
    if (rows)
        launch_prep_rows(c->stream, c->n, c->np, rows, c->cin, c->gm, c->J, mixed_on(c) ? c->J32 : nullptr,
                         ind_buf(c, 0), c->barycentric, ea, eb);
    else
        launch_prep(c->stream, c->n, c->np, st, c->gm, c->J, mixed_on(c) ? c->J32 : nullptr, ind_buf(c, 0),
                    c->barycentric, ea, eb);
    const bool gas_live = c->has_gas && !c->gas_dead;
    if (gas_live && (c->eval_mig1 || c->eval_mig2)) {
        const int do1 = c->eval_mig1 && c->nb.proto_planet > 0;
        const int do2 = c->eval_mig2 && c->nb.giant_planet > 0;
        if (do1 || do2)
            launch_migration(c->stream, c->nb.central_body, c->nb.giant_planet, c->n_massive, c->np, st, c->mass,
                             c->stop, c->migt, c->migc, c->gasdev, c->barycentric, t, do1, do2);
    }
    EpiArgs a = base_args(c);
    a.h = h;
    a.t = t;
    if (int r = pair_sums(c, last, a)) return r;
    a.kind = kind;
    a.integ = integ;
    a.stage = 0;
    a.last = last ? 1 : 0;
    a.want_nn = last ? 1 : 0;
    a.vel = st + 3 * (size_t)c->np;
    a.ind_in = ind_buf(c, 0);
    a.fout = out;
    a.yscale_out = want_yscale ? c->yscale : nullptr;
    {
        ProfScope ps(c, 1);
        launch_epilogue(c->stream, a);
    }
    HIPCHECK(c, hipGetLastError());
    if (c->barycentric && c->has_gas && !c->gas_dead && host_reduction_factor(c->gas, t) < 1.0e-5) {
        // Solaris/Acceleration.cpp:151-160: the gas is gone for good
        c->gas_dead = true;
        c->eval_drag = c->eval_mig1 = c->eval_mig2 = 0;
    }
    return SOL_OK;
}

int integ_kind(int32_t integrator)
{
    switch (integrator) {
    case SOL_RUNGE_KUTTA_FEHLBERG78: return INTEG_RKF78;
    case SOL_RUNGE_KUTTA4: return INTEG_RK4;
    case SOL_DORMAND_PRINCE: return INTEG_DP;
    default: return -1;
    }
}

int n_stages(int ik) { return ik == INTEG_RKF78 ? 12 : ik == INTEG_RK4 ? 3 : 8; }


// Stage evaluations 1..S of one Step from Y0 and ACCEL at (t, h) into Y,
// ERROR and the error maximum (left in c->h_scal[2] after the sync when
// read_err is set).
int run_stages(sol_context *c, int ik, double t, double h, bool read_err, double *errmax_out)
{
    const int S = n_stages(ik);
    EpiArgs a = base_args(c);
    a.h = h;
    a.t = t;
    a.integ = ik;
    // stage 1 state from y0 and f0
    a.stage = 0;
    a.fst_next = fslot(c, 1);
    a.ind_out = ind_buf(c, 1);
    launch_combine_first(c->stream, a);
    for (int s = 1; s <= S; ++s) {
        const bool last = (s == S);
        EpiArgs e = a;
        if (int r = pair_sums(c, last, e)) return r;
        e.stage = s;
        e.kind = last ? EPI_FINAL : EPI_MID;
        e.last = last ? 1 : 0;
        e.want_nn = last ? 1 : 0;
        e.vel = fslot(c, s);
        e.fout = fslot(c, s);
        e.ind_in = ind_buf(c, s);
        e.ind_out = ind_buf(c, s + 1);
        e.fst_next = last ? nullptr : fslot(c, s + 1);
        {
            ProfScope ps(c, 1);
            launch_epilogue(c->stream, e);
        }
    }
    launch_errmax_final(c->stream, c->errblk, c->nblk, c->scal + 2);
    HIPCHECK(c, hipGetLastError());
    if (read_err) {
        HIPCHECK(c, hipMemcpyAsync(c->h_scal + 2, c->scal + 2, sizeof(double), hipMemcpyDeviceToHost, c->stream));
        HIPCHECK(c, hipStreamSynchronize(c->stream));
        if (errmax_out) *errmax_out = c->h_scal[2];
    }
    return SOL_OK;
}

// Small systems run whole Driver loops in one workgroup; with gas only in
// the astrocentric frame (the barycentric frame switches the gas off for
// good during a run, Solaris/Acceleration.cpp:151-160) and not for
// Dormand-Prince (kept on the multi-kernel path with a nebula).
bool use_resident(const sol_context *c, int ik)
{
    if (c->resident_disabled) return false;
    if (c->has_gas && !c->gas_dead && (c->barycentric || ik == INTEG_DP)) return false;
    if (c->precision != SOL_PRECISION_FP64 || c->softening != 0.0) return false;
    if (c->n < 2 || c->n > kResidentMaxBodies || resident_lds_bytes(c->n) > c->lds_limit) return false;
    return true;
}

// Bodies every slice of the grid form holds: the sources of every sink
// and the massive bodies (AC: [0, max(n_massive, end_a, end_b)), BC: the
// massive bodies).
int grid_sources(const sol_context *c)
{
    if (c->barycentric) return std::max(1, c->n_massive);
    int ea, eb;
    source_ends(c, ea, eb);
    return std::max(1, std::max(c->n_massive, std::max(ea, eb)));
}

// Slices of `block` threads the device holds at once.
int grid_capacity_of(sol_context *c, int ik, int block)
{
    const bool gas = c->has_gas && !c->gas_dead;
    const int bi = block == 64 ? 0 : block == 128 ? 1 : 2;
    int &cap = c->grid_capacity[(2 * ik + (gas ? 1 : 0)) * 3 + bi];
    if (cap < 0) cap = resident_grid_capacity(ik, block, block, c->lds_limit, c->cu_count, gas);
    return cap;
}

// The grid form (slices of one system, one workgroup each, one body per
// thread) for systems with few sources: at most a quarter of a slice, at
// least grid_min_bodies bodies, and no more slices than the device keeps
// resident at once.  The slice is the smallest of 64, 128 and 256 threads
// that needs at most 160 slices (every attempt's grid-wide decision costs
// more with more slices; a step's latency is that of one body per thread
// whatever the slice), else 256 (grid_block > 0 fixes it).
bool grid_slices(sol_context *c, int ik, SliceMap *m)
{
    if (c->resident_disabled || c->grid_disabled) return false;
    if (c->has_gas && !c->gas_dead && c->barycentric) return false;
    if (c->precision != SOL_PRECISION_FP64 || c->softening != 0.0) return false;
    const int src = grid_sources(c);
    int block = c->grid_block;
    if (block == 0) {
        block = 256;
        for (int b = 64; b <= 128; b *= 2)
            if (src <= b / 4 && slice_map_make(c->n, c->np, src, b).nslices <= 160) { block = b; break; }
    }
    if (src > block / 4) return false;
    const SliceMap sm = slice_map_make(c->n, c->np, src, block);
    const int cap = grid_capacity_of(c, ik, block);
    if (sm.nslices > cap || sm.nslices > kGridMaxSlices) return false;
    if (m) *m = sm;
    return true;
}

bool use_grid(sol_context *c, int ik, SliceMap *m) { return c->n >= c->grid_min_bodies && grid_slices(c, ik, m); }

// The resident arrays of the context's own (system-layout) buffers.
ResArrays resident_arrays(sol_context *c)
{
    ResArrays A{};
    A.tot = c->np;
    A.y0 = c->y0; A.y = c->y; A.acc0 = c->acc0; A.yscale = c->yscale; A.err = c->error; A.fst = c->fst;
    A.mass = c->mass; A.rm3 = c->rm3; A.nnd = c->nnd; A.nni = c->nni;
    A.radius = c->radius;
    A.density = c->density; A.cd = c->cd; A.gs = c->gs; A.ge = c->ge; A.stop = c->stop; A.migt = c->migt;
    A.migc = c->migc; A.dragc = c->dragc; A.cache_stride = c->np;
    A.gas = c->gasdev;
    A.gas_on = c->has_gas && !c->gas_dead ? 1 : 0;
    // the Driver turns both migration switches on for its first evaluation
    A.mig_do1 = c->nb.proto_planet > 0;
    A.mig_do2 = c->nb.giant_planet > 0;
    return A;
}

// The ResSystem of a whole system at the time line's state.
ResSystem resident_system(const sol_context *c, double eps, const sol_timeline *tl, bool clip, int32_t stop_mask)
{
    ResSystem S{};
    S.n = c->n;
    S.nm = c->n_massive;
    source_ends(c, S.end_a, S.end_b);
    S.base = 0;
    S.barycentric = c->barycentric;
    S.clip = clip ? 1 : 0;
    S.status = RES_RUNNING;
    S.millenium = tl->millenium;
    S.t = tl->time; S.h_next = tl->hNext; S.h_did = tl->hDid; S.eps = eps;
    S.elapsed = tl->elapsedTime; S.last_save = tl->lastSave; S.last_nsteps = tl->lastNSteps;
    S.length = tl->length; S.output = tl->output;
    S.flush_count = tl->flush_count;
    S.stop_mask = stop_mask & (SOL_STOP_OUTPUT | SOL_STOP_EVENT);
    S.e3 = c->ev_e3; S.h3 = c->ev_h3; S.coll = c->ev_factor;
    S.src = c->n; S.shift = 0;
    S.drag_lo = c->n_massive; S.drag_hi = c->n_massive + n_pl_spl(c->nb);
    S.mig_lo = c->nb.central_body;
    S.giant_end = c->nb.central_body + c->nb.giant_planet;
    return S;
}

// Slice-layout buffers for tot slots and the slices' descriptors.
int grid_buffers(sol_context *c, const SliceMap &m)
{
    const int64_t tot = (int64_t)m.nslices * m.stride;
    if (tot > c->gbuf_tot) {
        int r;
        if ((r = dalloc(c, &c->gbuf, 111 * (size_t)tot)) || (r = dalloc(c, &c->gibuf, 2 * (size_t)tot))) return r;
        c->gbuf_tot = tot;
    }
    if (m.nslices > c->grid_sys_cap) {
        int r;
        if ((r = dalloc(c, &c->grid_sys_d, (size_t)m.nslices))) return r;
        c->grid_sys_cap = m.nslices;
    }
    if (!c->gsync) {
        int r;
        if ((r = dalloc(c, &c->gsync, 1))) return r;
    }
    return SOL_OK;
}

// The slice-layout arrays in gbuf / gibuf (component stride tot).
ResArrays grid_arrays(sol_context *c, const SliceMap &m)
{
    const int64_t T = (int64_t)m.nslices * m.stride;
    ResArrays A = resident_arrays(c);
    double *p = c->gbuf;
    auto take = [&](int64_t k) { double *q = p; p += k * T; return q; };
    A.tot = T;
    A.y0 = take(6); A.y = take(6); A.acc0 = take(6); A.yscale = take(6); A.err = take(6); A.fst = take(72);
    A.mass = take(1); A.radius = take(1); A.density = take(1); A.cd = take(1); A.gs = take(1); A.ge = take(1);
    A.stop = take(1); A.rm3 = take(1); A.nnd = take(1);
    A.nni = c->gibuf; A.migt = c->gibuf + T;
    A.sync = c->gsync;
    A.nsync = m.nslices;
    A.sync_ticks = (uint64_t)(c->grid_wait_s * (double)c->rtc_hz);
    return A;
}

SliceArrays system_arrays(sol_context *c)
{
    SliceArrays s{};
    s.y0 = c->y0; s.y = c->y; s.acc0 = c->acc0; s.yscale = c->yscale; s.err = c->error;
    s.rm3 = c->rm3; s.nnd = c->nnd; s.nni = c->nni; s.migt = c->migt;
    s.mass = c->mass; s.radius = c->radius;
    s.density = c->density; s.cd = c->cd; s.gs = c->gs; s.ge = c->ge; s.stop = c->stop;
    return s;
}

// The mesh form (mesh.hip): astrocentric FP64 gravity without gas, sources
// enough to share out, and no more workgroups than the device holds at once.
// From 32 sources on: an RKF78 attempt of 33 bodies takes 48 us on the mesh
// and 58 in one workgroup, of 17 bodies 47 and 35.
constexpr int kMeshMinSources = 32;
// ... and to 23 bodies per workgroup, 5,889 bodies: RKF78 and Dormand-Prince, us
// per attempt in the mesh form and with one launch per stage: 3,501 268 and 460,
// 193 and 334; 5,001 455 and 470, 326 and 344; 5,889 518 and 596, 369 and 434;
// with 31 per workgroup (another session) 6,001 627 and 580, 452 and 426; 7,937
// 801 and 626, 582 and 461.
constexpr int kMeshContextShare = 23;
constexpr int kPathMesh = 100, kPathQuad = 101;     // reported as SOL_PATH_GRID

bool use_mesh(sol_context *c, int ik, int *share_out = nullptr, int *groups_out = nullptr)
{
    if (c->resident_disabled || c->grid_disabled || c->barycentric) return false;
    if (c->has_gas && !c->gas_dead) return false;
    if (c->precision != SOL_PRECISION_FP64) return false;
    // a profiled context (sol_profile) keeps the launches that are timed
    if (c->profiling && !use_resident(c, ik)) return false;
    int ea, eb;
    source_ends(c, ea, eb);
    if (std::max(ea, eb) < kMeshMinSources) return false;
    const int share = mesh_share(c->n, c->n_massive, ea, eb, c->cu_count);
    if (share == 0 || share > kMeshContextShare) return false;
    const int groups = mesh_groups(c->n, c->n_massive, ea, eb, share);
    int &cap = c->mesh_caps[ik][share / 8];
    if (cap < 0) cap = mesh_capacity(ik, c->n, share, c->cu_count);
    if (cap < groups) return false;
    if (share_out) *share_out = share;
    if (groups_out) *groups_out = groups;
    return true;
}

// The quad form (quad.hip) takes the systems of the grid form, and smaller
// ones, that have at most eight sources besides the star and bodies for at
// most a workgroup per CU (14,339 with two planets).  The Sun, two planets and
// test particles, us per RKF78 attempt in one workgroup or in slices, and in
// quads: 4 bodies 15 and 6.0, 515 17.7 and 6.7, 5,001 18.8 and 7.4, 14,338 20.4
// and 8.0.  With live gas: the grid form's slices of 64 and 128 places, us per
// RKF78 attempt: 125 bodies 64 (one workgroup) and 32, 505 51 and 32, 16,389 56
// and 37.
struct QuadShape { int sources, own, groups, places; };   // places: bodies of a workgroup with gas (0: no gas)

bool use_quad(sol_context *c, int ik, QuadShape *out = nullptr)
{
    if (c->resident_disabled || c->grid_disabled || c->barycentric || c->grid_block != 0) return false;
    if (c->precision != SOL_PRECISION_FP64 || c->softening != 0.0 || c->n < c->quad_min_bodies) return false;
    QuadShape q{};
    q.sources = grid_sources(c) - 1;
    if (q.sources < 1 || q.sources > kQuadMaxSources) return false;
    // a profiled context (sol_profile) keeps the launches that are timed
    if (c->profiling && !use_grid(c, ik, nullptr) && !use_resident(c, ik)) return false;
    if (c->has_gas && !c->gas_dead) {
        SliceMap m{};
        if (!grid_slices(c, ik, &m) || m.stride > kQuadGasBodies || m.nslices < 1 ||
            m.nslices > std::min(c->cu_count, kQuadMaxGroups))
            return false;
        q.own = m.per; q.groups = m.nslices; q.places = m.stride;
        int &cap = c->quad_gas_caps[ik][q.sources / 4][q.places / kQuadGasBodies];
        if (cap < 0) cap = quad_gas_capacity(ik, q.sources, q.places, c->cu_count);
        if (cap < q.groups) return false;
    } else {
        q.own = 16 - q.sources;
        q.groups = quad_groups(c->n, q.sources, c->cu_count);
        if (q.groups == 0) return false;
        int &cap = c->quad_caps[ik][q.sources / 4];
        if (cap < 0) cap = quad_capacity(ik, q.sources, c->cu_count);
        if (cap < q.groups) return false;
    }
    if (out) *out = q;
    return true;
}

// The path a Driver call or a caller loop of integrator ik takes: the quad
// and the grid form where they apply (few sources, more bodies than
// grid_min_bodies), the mesh form for many sources, else one workgroup where the system fits,
// else one launch per stage.
int path_of(sol_context *c, int ik, SliceMap *m)
{
    if (use_quad(c, ik)) return kPathQuad;
    if (use_grid(c, ik, m)) return SOL_PATH_GRID;
    if (use_mesh(c, ik)) return kPathMesh;
    return use_resident(c, ik) ? SOL_PATH_RESIDENT : SOL_PATH_MULTI_KERNEL;
}

bool use_resident_any(sol_context *c, int ik) { return path_of(c, ik, nullptr) != SOL_PATH_MULTI_KERNEL; }

// resident_run's return when the grid form could not complete (a slice
// that was not resident): the call is to be made again from the same state
// (on the grid form once more, then on another path).
constexpr int kGridRetry = -1000;

// Time line, counters, switches and status after a run of the resident
// drivers that ended with S.
int resident_finish(sol_context *c, const ResSystem &S, sol_timeline *tl, int64_t max_steps, bool clip,
                    double *body_h, int64_t *steps_out, int64_t *attempts_out, int32_t stop_mask, int32_t *reason)
{
    tl->time = S.t; tl->hNext = S.h_next; tl->hDid = S.h_did;
    tl->elapsedTime = S.elapsed; tl->lastSave = S.last_save; tl->lastNSteps = S.last_nsteps;
    if (clip) tl->flush_count = S.flush_count;
    if (reason) {
        // the last step's reasons (S.reason is written at every clipped step)
        *reason = S.reason & (stop_mask | SOL_STOP_END);
        if (S.status == RES_DONE) *reason |= SOL_STOP_END;
        if (max_steps > 0 && S.steps >= max_steps) *reason |= SOL_STOP_STEPS;
    }
    if (body_h) *body_h = S.body_h;
    if (steps_out) *steps_out += S.steps;
    if (attempts_out) *attempts_out += S.attempts;
    // the Driver leaves the drag switch on and the migration switches off
    c->eval_drag = 1;
    c->eval_mig1 = c->eval_mig2 = 0;
    if (S.status == RES_UNDERFLOW)
        return c->fail(SOL_ERR_UNDERFLOW, "Stepsize-underflow occurred during Runge-Kutta-Fehlberg7(8) step!");
    if (S.status == RES_MAXITER)
        return c->fail(SOL_ERR_MAXITER,
                       "An error occurred during Prince-Dormand driver: iteration number exceeded maxIter!");
    return SOL_OK;
}

int mesh_run(sol_context *c, int path, int ik, double eps, sol_timeline *tl, int64_t max_steps, bool clip,
             double *body_h, int64_t *steps_out, int64_t *attempts_out, int32_t stop_mask, int32_t *reason);

// Runs accepted steps of integrator ik in the resident kernel: exactly one
// Driver call when clip is false and max_steps == 1, or the caller loop
// with DecisionMaking's clipping until the end of the time line (or
// max_steps steps) when clip is true.  Launches are bounded to about 0.2 s
// of work each.  A system that the grid form takes is scattered into its
// slices first and gathered back at the end.
int resident_run(sol_context *c, int ik, double eps, sol_timeline *tl, int64_t max_steps, bool clip, double *body_h,
                 int64_t *steps_out, int64_t *attempts_out, int32_t stop_mask = 0, int32_t *reason = nullptr)
{
    SliceMap m{};
    const int path = path_of(c, ik, &m);
    if (path == kPathMesh || path == kPathQuad)
        return mesh_run(c, path, ik, eps, tl, max_steps, clip, body_h, steps_out, attempts_out, stop_mask, reason);
    const bool grid = path == SOL_PATH_GRID;
    ResSystem S0 = resident_system(c, eps, tl, clip, stop_mask);
    ResArrays A;
    ResSystem *sys_d = c->res_d;
    int nsys = 1;
    if (grid) {
        int r = grid_buffers(c, m);
        if (r) return r;
        A = grid_arrays(c, m);
        S0.src = m.src;
        nsys = m.nslices;
        c->grid_sys_h.assign((size_t)nsys, S0);
        for (int k = 0; k < nsys; ++k) {
            ResSystem &Sk = c->grid_sys_h[(size_t)k];
            Sk.n = slice_count(m, k);
            Sk.base = k * m.stride;
            Sk.shift = k * m.per;
        }
        sys_d = c->grid_sys_d;
        HIPCHECK(c, hipMemcpyAsync(sys_d, c->grid_sys_h.data(), nsys * sizeof(ResSystem), hipMemcpyHostToDevice,
                                   c->stream));
        launch_slice_scatter(c->stream, m, system_arrays(c), A);
        HIPCHECK(c, hipGetLastError());
    } else {
        A = resident_arrays(c);
        *c->res_h = S0;
        HIPCHECK(c, hipMemcpyAsync(sys_d, c->res_h, sizeof(ResSystem), hipMemcpyHostToDevice, c->stream));
    }
    ResSystem &S = grid ? c->grid_sys_h[0] : *c->res_h;
    const int block = grid ? m.stride : resident_block_size(c->n);
    const int nsrc = grid ? m.src : c->n;
    const double per_step = 13.0 * (double)block * (double)nsrc / 4.0e9 + 2.0e-5;
    const int64_t chunk = std::max<int64_t>(1, std::min<int64_t>(20000, (int64_t)(0.2 / per_step)));
    for (;;) {
        const int64_t k = max_steps > 0 ? std::min(chunk, max_steps - S.steps) : chunk;
        std::unique_ptr<UnitLease> lease;
        if (grid) {
            const int per_cu = std::max(1, grid_capacity_of(c, ik, m.stride) / std::max(1, c->cu_count));
            lease.reset(new UnitLease(c->device, (nsys + per_cu - 1) / per_cu, c->cu_count));
            HIPCHECK(c, launch_resident_grid(c->stream, ik, sys_d, nsys, A, (int)k, m.stride, m.stride,
                                             c->lds_limit));
            HIPCHECK(c, hipMemcpyAsync(c->grid_sys_h.data(), sys_d, nsys * sizeof(ResSystem),
                                       hipMemcpyDeviceToHost, c->stream));
        } else {
            launch_resident(c->stream, ik, sys_d, 1, A, (int)k, block, c->n, c->lds_limit);
            HIPCHECK(c, hipGetLastError());
            HIPCHECK(c, hipMemcpyAsync(c->res_h, sys_d, sizeof(ResSystem), hipMemcpyDeviceToHost, c->stream));
        }
        HIPCHECK(c, hipStreamSynchronize(c->stream));
        if (grid) {
            for (int q = 0; q < nsys; ++q)
                if (c->grid_sys_h[(size_t)q].status == RES_SYNC_ERROR) {
                    // a slice was not resident (or waited out the budget):
                    // nothing was gathered and the time line is untouched, so
                    // the call runs again; after the second such run the
                    // context stays off the grid form
                    if (++c->grid_failures >= 2) c->grid_disabled = true;
                    return kGridRetry;
                }
            // every slice takes the same decisions: they must agree
            for (int q = 1; q < nsys; ++q) {
                const ResSystem &Sq = c->grid_sys_h[(size_t)q];
                if (Sq.status != S.status || Sq.steps != S.steps || Sq.t != S.t || Sq.h_next != S.h_next)
                    return c->fail(SOL_ERR_DEVICE, "resident grid: slice %d disagrees with slice 0 (status %d/%d, "
                                   "steps %lld/%lld)", q, Sq.status, S.status, (long long)Sq.steps,
                                   (long long)S.steps);
            }
        }
        if (!std::isfinite(S.t) || !std::isfinite(S.h_next))
            return c->fail(SOL_ERR_DEVICE, "resident driver: non-finite time or step size (t %g, hNext %g)", S.t,
                           S.h_next);
        if (S.status != RES_RUNNING) break;
        if (max_steps > 0 && S.steps >= max_steps) break;
    }
    if (grid) {
        launch_slice_gather(c->stream, m, system_arrays(c), A);
        HIPCHECK(c, hipGetLastError());
        HIPCHECK(c, hipStreamSynchronize(c->stream));
    }
    return resident_finish(c, S, tl, max_steps, clip, body_h, steps_out, attempts_out, stop_mask, reason);
}

// Arrays and exchange words of the mesh and the quad form.
int mesh_buffers(sol_context *c, bool gas)
{
    sol_context::Mesh &m = c->mesh;
    const size_t np = c->np;
    if (!m.pos) {
        ArrayBlock b;
        b.add(&m.y0, 6 * np); b.add(&m.y, 6 * np); b.add(&m.acc0, 6 * np);
        b.add(&m.yscale, 6 * np); b.add(&m.error, 6 * np);
        b.add(&m.rm3, np); b.add(&m.nnd, np); b.add(&m.nni, np);
        b.add(&m.run, 1); b.add(&m.part_of, (size_t)kMeshMaxGroups);
        b.add(&m.pos, 6 * np);
        if (int r = b.make(c)) return r;
    }
    if (gas && !m.dragc) {
        ArrayBlock b;
        b.add(&m.migt, np); b.add(&m.migc, 3 * np);
        b.add(&m.migt_prev, np); b.add(&m.migc_prev, 3 * np);
        b.add(&m.dragc, 3 * np);
        if (int r = b.make(c)) return r;
    }
    return SOL_OK;
}

// resident_run on the mesh or the quad form: accepted steps of integrator ik
// with the system's bodies shared out over workgroups, about 0.2 s of work per
// launch.  The context's arrays are replaced by the run's at its end only.
int mesh_run(sol_context *c, int path, int ik, double eps, sol_timeline *tl, int64_t max_steps, bool clip,
             double *body_h, int64_t *steps_out, int64_t *attempts_out, int32_t stop_mask, int32_t *reason)
{
    const bool quad = path == kPathQuad;
    int share = 0, groups = 0;
    QuadShape shape{};
    if (quad ? !use_quad(c, ik, &shape) : !use_mesh(c, ik, &share, &groups)) return kGridRetry;
    if (quad) groups = shape.groups;
    if (int r = mesh_buffers(c, shape.places != 0)) return r;
    sol_context::Mesh &m = c->mesh;
    MeshRun &to = c->mesh_h[0], &back = c->mesh_h[1];
    ResSystem &S = back.system;
    S = resident_system(c, eps, tl, clip, stop_mask);
    if (!quad) {
        // (the words are zero)
        to.system = S;
        to.part = MeshPart{0, 0, groups, share};
        HIPCHECK(c, hipMemcpyAsync(m.run, &to, offsetof(MeshRun, words) + sizeof(MeshSync), hipMemcpyHostToDevice,
                                   c->stream));
    }
    MeshArgs A{};
    A.systems = &m.run->system;
    A.parts = &m.run->part; A.part_of = m.part_of;
    A.sync = &m.run->words.mesh;
    A.pos = m.pos; A.gm = c->gm;
    A.tot = c->np;
    A.mass = c->mass; A.radius = c->radius;
    A.y0 = m.y0; A.y = m.y; A.acc0 = m.acc0; A.yscale = m.yscale; A.err = m.error;
    A.rm3 = m.rm3; A.nnd = m.nnd; A.nni = m.nni;
    A.eps2 = c->softening * c->softening;
    A.ticks = (uint64_t)(c->grid_wait_s * (double)c->rtc_hz);
    QuadArgs Q{};
    Q.system = &m.run->system;
    Q.sync = &m.run->words.quad;
    Q.sources = shape.sources;
    Q.groups = groups;
    Q.own = shape.own;
    Q.tot = A.tot;
    Q.gm = A.gm; Q.mass = A.mass; Q.radius = A.radius;
    Q.y0 = A.y0; Q.y = A.y; Q.acc0 = A.acc0; Q.yscale = A.yscale; Q.err = A.err;
    Q.rm3 = A.rm3; Q.nnd = A.nnd; Q.nni = A.nni;
    Q.ticks = A.ticks;
    if (shape.places) {
        Q.gas = c->gasdev;
        Q.density = c->density; Q.cd = c->cd; Q.gs = c->gs; Q.ge = c->ge; Q.stop = c->stop;
        Q.migt_in = c->migt; Q.migc_in = c->migc;
        Q.migt = m.migt; Q.migc = m.migc; Q.dragc = m.dragc;
        // the Driver turns both migration switches on for its first evaluation
        Q.mig_do1 = c->nb.proto_planet > 0;
        Q.mig_do2 = c->nb.giant_planet > 0;
    }
    // (a quad step with drag takes about 40 us)
    const int64_t chunk = quad ? 4000 : mesh_chunk(c->n);
    A.y0_in = c->y0;
    for (bool first = true;; first = false) {
        const int64_t k = max_steps > 0 ? std::min(chunk, max_steps - S.steps) : chunk;
        const UnitLease lease(c->device, groups, c->cu_count);
        if (quad) {
            Q.y0_in = A.y0_in;
            Q.system_in = S;
            HIPCHECK(c, shape.places ? launch_quad_gas(c->stream, ik, Q, shape.places, (int)k)
                                     : launch_quad(c->stream, ik, Q, (int)k));
        } else {
            HIPCHECK(c, launch_mesh(c->stream, ik, A, 1, groups, c->n, share, (int)k, first));
        }
        HIPCHECK(c, hipMemcpyAsync(&back, m.run, kMeshRunBack, hipMemcpyDeviceToHost, c->stream));
        HIPCHECK(c, hipStreamSynchronize(c->stream));
        // (without an exchange the quad form leaves its words alone)
        const bool lost = back.words.mesh.error != 0 && (!quad || quad_exchanges(ik, Q));
        if (lost || S.status == RES_SYNC_ERROR) {
            // a workgroup that was not resident: as for the grid form, the
            // call runs again from its unchanged start
            if (++c->grid_failures >= 2) c->grid_disabled = true;
            return kGridRetry;
        }
        if (!std::isfinite(S.t) || !std::isfinite(S.h_next))
            return c->fail(SOL_ERR_DEVICE, "mesh driver: non-finite time or step size (t %g, hNext %g)", S.t,
                           S.h_next);
        if (S.status != RES_RUNNING) break;
        if (max_steps > 0 && S.steps >= max_steps) break;
        A.y0_in = m.y0;
        if (quad) {
            // (its launches do not read what they write; pos is the mesh form's)
            HIPCHECK(c, hipMemcpyAsync(m.pos, m.y0, 6 * (size_t)c->np * sizeof(double), hipMemcpyDeviceToDevice,
                                       c->stream));
            A.y0_in = m.pos;
        }
        if (shape.places) {
            // the next launch reads what this one left; a lost one still leaves the context's
            HIPCHECK(c, hipMemcpyAsync(m.migt_prev, m.migt, c->np * sizeof(int32_t), hipMemcpyDeviceToDevice,
                                       c->stream));
            HIPCHECK(c, hipMemcpyAsync(m.migc_prev, m.migc, 3 * (size_t)c->np * sizeof(double),
                                       hipMemcpyDeviceToDevice, c->stream));
            Q.migt_in = m.migt_prev;
            Q.migc_in = m.migc_prev;
        }
    }
    if (shape.places) {
        std::swap(c->migt, m.migt);
        std::swap(c->migc, m.migc);
        std::swap(c->dragc, m.dragc);
    }
    std::swap(c->y0, m.y0);
    std::swap(c->y, m.y);
    std::swap(c->acc0, m.acc0);
    if (ik == INTEG_RKF78) std::swap(c->yscale, m.yscale);
    if (ik != INTEG_RK4) std::swap(c->error, m.error);
    std::swap(c->rm3, m.rm3);
    std::swap(c->nnd, m.nnd);
    std::swap(c->nni, m.nni);
    return resident_finish(c, S, tl, max_steps, clip, body_h, steps_out, attempts_out, stop_mask, reason);
}

int driver_rkf78(sol_context *c, double eps, sol_timeline *tl, double *body_h, int64_t *attempts)
{
    for (int tries = 0; tries < 3 && use_resident_any(c, INTEG_RKF78); ++tries) {
        const int r = resident_run(c, INTEG_RKF78, eps, tl, 1, false, body_h, nullptr, attempts);
        if (r != kGridRetry) return r;
    }
    const double SAFETY = 0.9, PGROW = -0.2, PSHRNK = -0.25, ERRCON = 1.89e-4;
    const double t0 = tl->time;
    double h = tl->hNext;
    c->eval_drag = c->eval_mig1 = c->eval_mig2 = 1;
    int r = evaluate_at(c, c->y0, t0, h, c->acc0, EPI_STAGE0, INTEG_RKF78, false, true);
    if (r) return r;
    c->eval_mig1 = c->eval_mig2 = 0;
    double errmax = 0.0;
    for (;;) {
        double raw = 0.0;
        r = run_stages(c, INTEG_RKF78, t0, h, true, &raw);
        if (r) return r;
        if (attempts) ++*attempts;
        errmax = raw / eps;
        if (errmax < 1.0) { tl->hDid = h; break; }
        const double htemp = SAFETY * h * std::pow(errmax, PSHRNK);
        h = std::fabs(htemp) > std::fabs(0.1 * h) ? htemp : 0.1 * h;
        if (tl->time + h == tl->time) {
            if (body_h) *body_h = h;
            return c->fail(SOL_ERR_UNDERFLOW, "Stepsize-underflow occurred during Runge-Kutta-Fehlberg7(8) step!");
        }
    }
    tl->time += tl->hDid;
    tl->hNext = errmax > ERRCON ? (SAFETY * h * std::pow(errmax, PGROW)) : (5.0 * h);
    if (body_h) *body_h = tl->hNext;
    std::swap(c->y0, c->y);
    return SOL_OK;
}

int driver_rk4(sol_context *c, sol_timeline *tl, double *body_h, int64_t *attempts)
{
    for (int tries = 0; tries < 3 && use_resident_any(c, INTEG_RK4); ++tries) {
        const int r = resident_run(c, INTEG_RK4, 0.0, tl, 1, false, body_h, nullptr, attempts);
        if (r != kGridRetry) return r;
    }
    const double t0 = tl->time, h = tl->hNext;
    c->eval_drag = c->eval_mig1 = c->eval_mig2 = 1;
    int r = evaluate_at(c, c->y0, t0, h, c->acc0, EPI_STAGE0, INTEG_RK4, false, false);
    if (r) return r;
    c->eval_mig1 = c->eval_mig2 = 0;
    r = run_stages(c, INTEG_RK4, t0, h, false, nullptr);
    if (r) return r;
    if (attempts) ++*attempts;
    tl->hDid = h;
    tl->time += tl->hDid;
    tl->hNext = h;
    if (body_h) *body_h = h;
    std::swap(c->y0, c->y);
    return SOL_OK;
}

int driver_dp(sol_context *c, double eps, sol_timeline *tl, double *body_h, int64_t *attempts)
{
    for (int tries = 0; tries < 3 && use_resident_any(c, INTEG_DP); ++tries) {
        const int r = resident_run(c, INTEG_DP, eps, tl, 1, false, body_h, nullptr, attempts);
        if (r != kGridRetry) return r;
    }
    const int maxIter = 10;
    const double t0 = tl->time;
    c->eval_drag = c->eval_mig1 = c->eval_mig2 = 1;
    int r = evaluate_at(c, c->y0, t0, tl->hNext, c->acc0, EPI_STAGE0, INTEG_DP, false, false);
    if (r) return r;
    c->eval_mig1 = c->eval_mig2 = 0;
    int iter = 0;
    double errmax = 0.0, h = 0.0;
    do {
        iter++;
        h = tl->hNext;
        r = run_stages(c, INTEG_DP, t0, h, true, &errmax);
        if (r) return r;
        if (attempts) ++*attempts;
        tl->hDid = h;
        tl->hNext = errmax < 1.0e-20 ? 2.0 * h : 0.9 * h * std::pow(eps / errmax, 1.0 / 7.0);
    } while (errmax > eps && iter <= maxIter);
    if (body_h) *body_h = h;
    if (iter > maxIter)
        return c->fail(SOL_ERR_MAXITER,
                       "An error occurred during Prince-Dormand driver: iteration number exceeded maxIter!");
    tl->time += tl->hDid;
    std::swap(c->y0, c->y);
    return SOL_OK;
}

int check_ctx(sol_context *c)
{
    if (!c) return SOL_ERR_ARGUMENT;
    return SOL_OK;
}

}  // namespace

int sol::eval_force(sol_context *c, const double *st, double t, double *out)
{
    return evaluate_at(c, st, t, 0.0, out, EPI_COMPUTE, INTEG_RK4, false, false);
}

bool sol::resident_rk4_ok(const sol_context *c) { return use_resident(c, INTEG_RK4); }

int sol::resident_rk4(sol_context *c, double *y, double *ytmp, double t0, const double *h_seq, int64_t nsteps,
                      double *stages)
{
    if (nsteps <= 0) return SOL_OK;
    if (nsteps > INT32_MAX) return c->fail(SOL_ERR_ARGUMENT, "resident RK4: too many steps for one launch");
    ResSystem &S = *c->res_h;
    S = ResSystem{};
    S.n = c->n;
    S.nm = c->n_massive;
    source_ends(c, S.end_a, S.end_b);
    S.base = 0;
    S.barycentric = c->barycentric;
    S.status = RES_RUNNING;
    S.t = t0;
    S.length = 1.0e300;
    HIPCHECK(c, hipMemcpyAsync(c->res_d, c->res_h, sizeof(ResSystem), hipMemcpyHostToDevice, c->stream));
    ResArrays A{};
    A.tot = c->np;
    A.y0 = y; A.y = ytmp; A.acc0 = c->acc0; A.yscale = c->yscale; A.err = c->error; A.fst = c->fst;
    A.mass = c->mass; A.rm3 = c->rm3; A.nnd = c->nnd; A.nni = c->nni;
    A.radius = c->radius;
    A.h_seq = h_seq;
    A.stages_out = stages;
    launch_resident(c->stream, INTEG_RK4, c->res_d, 1, A, (int)nsteps, resident_block_size(c->n), c->n,
                    c->lds_limit);
    HIPCHECK(c, hipGetLastError());
    HIPCHECK(c, hipMemcpyAsync(c->res_h, c->res_d, sizeof(ResSystem), hipMemcpyDeviceToHost, c->stream));
    HIPCHECK(c, hipStreamSynchronize(c->stream));
    if (S.steps != nsteps)
        return c->fail(SOL_ERR_DEVICE, "resident RK4: %lld of %lld steps done", (long long)S.steps,
                       (long long)nsteps);
    return SOL_OK;
}

extern "C" {

const char *sol_version(void) { return "solaris_amd 0.1 (gfx950)"; }

const char *sol_last_error(const sol_context *ctx)
{
    if (!ctx) return g_create_error.c_str();
    return ctx->err.c_str();
}

int sol_create(sol_context **out, const sol_nbodies *nb, int32_t barycentric, int32_t device)
{
    if (!out || !nb) { g_create_error = "null argument"; return SOL_ERR_ARGUMENT; }
    *out = nullptr;
    const int sum = nb->central_body + nb->giant_planet + nb->rocky_planet + nb->proto_planet +
                    nb->super_planetesimal + nb->planetesimal + nb->test_particle;
    if (nb->total <= 0) { g_create_error = "host memory allocation"; return SOL_ERR_ALLOCATION; }
    if (sum != nb->total || nb->central_body != 1) {
        g_create_error = "body counts must add up to total, with exactly one central body";
        return SOL_ERR_ARGUMENT;
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) {
        g_create_error = "no HIP device available";
        return SOL_ERR_DEVICE;
    }
    if (device < 0 || device >= ndev) { g_create_error = "device index out of range"; return SOL_ERR_ARGUMENT; }
    sol_context *c = new sol_context();
    c->device = device;
    c->nb = *nb;
    c->n = nb->total;
    c->np = (c->n + kBlock - 1) / kBlock * kBlock;
    c->nblk = c->np / kBlock;
    c->n_massive = nb->central_body + nb->giant_planet + nb->rocky_planet + nb->proto_planet;
    c->barycentric = barycentric ? 1 : 0;
    int r = SOL_OK;
    auto bail = [&](int code) {
        g_create_error = c->err;
        sol_destroy(c);
        return code;
    };
    if (hipSetDevice(device) != hipSuccess) { c->err = "hipSetDevice failed"; return bail(SOL_ERR_DEVICE); }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess && prop.multiProcessorCount > 0) {
        c->cu_count = prop.multiProcessorCount;
        c->lds_limit = prop.sharedMemPerBlock > 2048 ? prop.sharedMemPerBlock - 2048 : 0;
    }
    if (const char *e = std::getenv("SOLARIS_AMD_NO_RESIDENT")) c->resident_disabled = e[0] == '1';
    if (const char *e = std::getenv("SOLARIS_AMD_NO_GRID")) c->grid_disabled = e[0] == '1';
    if (const char *e = std::getenv("SOLARIS_AMD_GRID_BLOCK")) {
        const int b = std::atoi(e);
        if (b >= 64 && b <= 256 && b % 64 == 0) c->grid_block = b;
    }
    if (const char *e = std::getenv("SOLARIS_AMD_GRID_MIN")) c->grid_min_bodies = c->quad_min_bodies = std::max(2, std::atoi(e));
    if (const char *e = std::getenv("SOLARIS_AMD_GRID_WAIT")) c->grid_wait_s = std::max(0.0, std::atof(e));
    {
        int khz = 0;
        if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device) == hipSuccess && khz > 0)
            c->rtc_hz = (uint64_t)khz * 1000;
    }
    if (const char *e = std::getenv("SOLARIS_AMD_NO_SYM")) c->sym_disabled = e[0] == '1';
    std::fill_n(&c->mesh_caps[0][0], 3 * 4, -1);
    std::fill_n(&c->quad_caps[0][0], 3 * 3, -1);
    std::fill_n(&c->quad_gas_caps[0][0][0], 3 * 3 * 2, -1);
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        c->err = "hipStreamCreate failed";
        return bail(SOL_ERR_DEVICE);
    }
    const size_t np = c->np;
    {
        ArrayBlock b;
        b.add(&c->mass, np); b.add(&c->gm, np); b.add(&c->radius, np); b.add(&c->density, np);
        b.add(&c->cd, np); b.add(&c->gs, np); b.add(&c->ge, np); b.add(&c->stop, np);
        b.add(&c->type, np); b.add(&c->migt, np);
        b.add(&c->y0, 6 * np); b.add(&c->y, 6 * np); b.add(&c->acc0, 6 * np);
        b.add(&c->yscale, 6 * np); b.add(&c->error, 6 * np); b.add(&c->fst, 12 * 6 * np);
        b.add(&c->cin, 6 * np); b.add(&c->aos, 6 * np);
        b.add(&c->J, np); b.add(&c->ind, 2 * (size_t)c->nblk * 6);
        b.add(&c->rm3, np); b.add(&c->nnd, np); b.add(&c->nni, np);
        b.add(&c->migc, 3 * np); b.add(&c->dragc, 3 * np);
        b.add(&c->errblk, (size_t)c->nblk); b.add(&c->scal, 8); b.add(&c->coef, 275);
        b.add(&c->integ, 11 * np); b.add(&c->res_d, 1);
        if ((r = b.make(c))) return bail(r);
    }
    // pinned, in one allocation
    {
        if (c->n <= 2 * kIoBodies) c->io_bytes = 6 * sizeof(double) * (size_t)std::min(c->n, kIoBodies);
        const size_t runs = 2 * sizeof(MeshRun), scal = 8 * sizeof(double);
        const size_t res = (sizeof(ResSystem) + 127) / 128 * 128;
        if (hipHostMalloc((void **)&c->pinned, runs + res + scal + c->io_bytes, hipHostMallocDefault) != hipSuccess) {
            c->pinned = nullptr;
            c->err = "hipHostMalloc failed";
            return bail(SOL_ERR_DEVICE);
        }
        std::memset(c->pinned, 0, runs + res + scal);
        c->mesh_h = reinterpret_cast<MeshRun *>(c->pinned);
        c->res_h = reinterpret_cast<ResSystem *>(c->pinned + runs);
        c->h_scal = reinterpret_cast<double *>(c->pinned + runs + res);
        if (c->io_bytes) c->io_h = reinterpret_cast<double *>(c->pinned + runs + res + scal);
    }
    // the copies below are made on the default stream
    if (hipStreamSynchronize(c->stream) != hipSuccess) {
        c->err = "filling the context's arrays failed";
        return bail(SOL_ERR_DEVICE);
    }
    std::vector<double> coef;
    fill_coefficients(coef);
    if (hipMemcpy(c->coef, coef.data(), coef.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
        c->err = "coefficient upload failed";
        return bail(SOL_ERR_DEVICE);
    }
    // indexOfNN starts at -1 (Solaris/Acceleration.cpp:253, :262)
    std::vector<int32_t> minus1(np, -1);
    if (hipMemcpy(c->nni, minus1.data(), np * sizeof(int32_t), hipMemcpyHostToDevice) != hipSuccess) {
        c->err = "upload failed";
        return bail(SOL_ERR_DEVICE);
    }
    build_plan(c);
    if ((r = ensure_partials(c))) return bail(r);
    *out = c;
    return SOL_OK;
}

int sol_destroy(sol_context *c)
{
    if (!c) return SOL_OK;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    if (c->stream2) StreamPool::give_back(c->device, c->stream2);
    adjoint_release(c);
    for (void *p : c->allocs) (void)hipFree(p);
    if (c->part) (void)hipFree(c->part);
    if (c->apart) (void)hipFree(c->apart);
    if (c->pinned) (void)hipHostFree(c->pinned);
    if (c->integ_h) (void)hipHostFree(c->integ_h);
    for (hipEvent_t e : c->ev_pool) (void)hipEventDestroy(e);
    if (c->ev_fork) (void)hipEventDestroy(c->ev_fork);
    if (c->ev_join) (void)hipEventDestroy(c->ev_join);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return SOL_OK;
}

int sol_set_bodies(sol_context *c, const sol_body_params *p)
{
    if (check_ctx(c) || !p) return SOL_ERR_ARGUMENT;
    adjoint_invalidate(c);
    HIPCHECK(c, hipSetDevice(c->device));
    // the copies below are synchronous on the null stream, which does not
    // order them after kernels still queued on the context's stream
    HIPCHECK(c, hipStreamSynchronize(c->stream));
    const size_t n = c->n;
    std::vector<double> zero(n, 0.0), gm(n);
    std::vector<int32_t> zi(n, 0);
    auto up = [&](double *dst, const double *src) {
        return hipMemcpy(dst, src ? src : zero.data(), n * sizeof(double), hipMemcpyHostToDevice);
    };
    if (p->type) {
        // the interaction ranges assume type-sorted bodies (Solaris/Simulator.cpp:449-495)
        for (size_t i = 1; i < n; ++i)
            if (p->type[i] < p->type[i - 1])
                return c->fail(SOL_ERR_ARGUMENT, "bodies are not sorted by type (body %zu)", i);
    }
    for (size_t i = 0; i < n; ++i) gm[i] = kGauss2 * (p->mass ? p->mass[i] : 0.0);
    HIPCHECK(c, up(c->mass, p->mass));
    HIPCHECK(c, up(c->radius, p->radius));
    HIPCHECK(c, up(c->density, p->density));
    HIPCHECK(c, up(c->cd, p->cd));
    HIPCHECK(c, up(c->gs, p->gamma_stokes));
    HIPCHECK(c, up(c->ge, p->gamma_epstein));
    HIPCHECK(c, up(c->stop, p->mig_stop_at));
    HIPCHECK(c, hipMemcpy(c->gm, gm.data(), n * sizeof(double), hipMemcpyHostToDevice));
    HIPCHECK(c, hipMemcpy(c->type, p->type ? p->type : zi.data(), n * sizeof(int32_t), hipMemcpyHostToDevice));
    HIPCHECK(c, hipMemcpy(c->migt, p->mig_type ? p->mig_type : zi.data(), n * sizeof(int32_t), hipMemcpyHostToDevice));
    return SOL_OK;
}

int sol_set_nebula(sol_context *c, const sol_gas_component *g)
{
    if (check_ctx(c)) return SOL_ERR_ARGUMENT;
    adjoint_invalidate(c);
    HIPCHECK(c, hipSetDevice(c->device));
    c->has_gas = g != nullptr;
    c->gas_dead = false;
    if (g) { c->gas = *g; c->gasdev = to_dev(*g); }
    HIPCHECK(c, hipMemsetAsync(c->migc, 0, 3 * (size_t)c->np * sizeof(double), c->stream));
    HIPCHECK(c, hipMemsetAsync(c->dragc, 0, 3 * (size_t)c->np * sizeof(double), c->stream));
    HIPCHECK(c, hipStreamSynchronize(c->stream));
    return SOL_OK;
}

int sol_set_evaluate(sol_context *c, int32_t d, int32_t m1, int32_t m2)
{
    if (check_ctx(c)) return SOL_ERR_ARGUMENT;
    c->eval_drag = d != 0; c->eval_mig1 = m1 != 0; c->eval_mig2 = m2 != 0;
    return SOL_OK;
}

int sol_get_evaluate(const sol_context *c, int32_t *d, int32_t *m1, int32_t *m2)
{
    if (!c) return SOL_ERR_ARGUMENT;
    if (d) *d = c->eval_drag;
    if (m1) *m1 = c->eval_mig1;
    if (m2) *m2 = c->eval_mig2;
    return SOL_OK;
}

int sol_set_precision(sol_context *c, int32_t precision, double softening)
{
    if (check_ctx(c)) return SOL_ERR_ARGUMENT;
    adjoint_invalidate(c);
    if (precision != SOL_PRECISION_FP64 && precision != SOL_PRECISION_MIXED)
        return c->fail(SOL_ERR_ARGUMENT, "unknown precision %d", precision);
    if (!(softening >= 0.0)) return c->fail(SOL_ERR_ARGUMENT, "softening must be >= 0");
    HIPCHECK(c, hipSetDevice(c->device));
    if (precision == SOL_PRECISION_MIXED && !c->J32) {
        int r = dalloc(c, &c->J32, (size_t)c->np);
        if (r) return r;
    }
    const bool plan = c->precision != precision;
    c->precision = precision;
    c->softening = softening;
    if (plan) {
        HIPCHECK(c, hipStreamSynchronize(c->stream));
        build_plan(c);
        return ensure_partials(c);
    }
    return SOL_OK;
}

int sol_set_side_outputs(sol_context *c, int32_t enable)
{
    if (check_ctx(c)) return SOL_ERR_ARGUMENT;
    c->side_outputs = enable != 0;
    return SOL_OK;
}

int sol_set_source_ranges(sol_context *c, int32_t a, int32_t b)
{
    if (check_ctx(c)) return SOL_ERR_ARGUMENT;
    adjoint_invalidate(c);
    if (a > c->n || b > c->n) return c->fail(SOL_ERR_ARGUMENT, "source range beyond total");
    HIPCHECK(c, hipSetDevice(c->device));
    c->end_massive = a;
    c->end_other = b;
    build_plan(c);
    return ensure_partials(c);
}

// A call's rows of six doubles per body in: where the kernels read them.
static size_t row_bytes(const sol_context *c) { return 6 * (size_t)c->n * sizeof(double); }
static bool rows_pinned(const sol_context *c) { return row_bytes(c) <= c->io_bytes; }
static int rows_in(sol_context *c, const double *host, const double **rows)
{
    if (rows_pinned(c)) {
        std::memcpy(c->io_h, host, row_bytes(c));
        *rows = c->io_h;
        return SOL_OK;
    }
    HIPCHECK(c, hipMemcpyAsync(c->aos, host, row_bytes(c), hipMemcpyHostToDevice, c->stream));
    *rows = c->aos;
    return SOL_OK;
}

// ... and out: where the last kernel writes them, and the end of the call.
// The rows read and the rows written share a buffer: the kernel that reads is
// done before the one that writes starts.
static double *rows_out(sol_context *c) { return rows_pinned(c) ? c->io_h : c->aos; }
static int rows_done(sol_context *c, double *host)
{
    HIPCHECK(c, hipGetLastError());
    if (!rows_pinned(c))
        HIPCHECK(c, hipMemcpyAsync(host, c->aos, row_bytes(c), hipMemcpyDeviceToHost, c->stream));
    HIPCHECK(c, hipStreamSynchronize(c->stream));
    if (rows_pinned(c)) std::memcpy(host, c->io_h, row_bytes(c));
    return SOL_OK;
}

int sol_compute(sol_context *c, double t, const double *yh, double *dydt)
{
    if (check_ctx(c) || !yh || !dydt) return SOL_ERR_ARGUMENT;
    HIPCHECK(c, hipSetDevice(c->device));
    CallEnd end(c);
    const double *rows;
    int r = rows_in(c, yh, &rows);
    if (r) return r;
    r = evaluate_at(c, c->cin, t, 0.0, rows_out(c), EPI_ROWS, INTEG_RKF78, c->side_outputs, false, rows);
    if (r) return r;
    return end(rows_done(c, dydt));
}

int sol_get_side_outputs(sol_context *c, double *rm3, int32_t *nn, double *dist, int32_t *mig)
{
    if (check_ctx(c)) return SOL_ERR_ARGUMENT;
    HIPCHECK(c, hipSetDevice(c->device));
    const size_t n = c->n;
    CallEnd end(c);
    if (24 * n <= c->io_bytes) {
        launch_pack_side(c->stream, c->n, c->rm3, c->nnd, c->nni, c->migt, c->io_h);
        HIPCHECK(c, hipGetLastError());
        HIPCHECK(c, hipStreamSynchronize(c->stream));
        const int32_t *k = reinterpret_cast<const int32_t *>(c->io_h + 2 * n);
        if (rm3) std::memcpy(rm3, c->io_h, n * sizeof(double));
        if (dist) std::memcpy(dist, c->io_h + n, n * sizeof(double));
        if (nn) std::memcpy(nn, k, n * sizeof(int32_t));
        if (mig) std::memcpy(mig, k + n, n * sizeof(int32_t));
        return end(SOL_OK);
    }
    if (rm3) HIPCHECK(c, hipMemcpyAsync(rm3, c->rm3, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    if (nn) HIPCHECK(c, hipMemcpyAsync(nn, c->nni, n * sizeof(int32_t), hipMemcpyDeviceToHost, c->stream));
    if (dist) HIPCHECK(c, hipMemcpyAsync(dist, c->nnd, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    if (mig) HIPCHECK(c, hipMemcpyAsync(mig, c->migt, n * sizeof(int32_t), hipMemcpyDeviceToHost, c->stream));
    HIPCHECK(c, hipStreamSynchronize(c->stream));
    return end(SOL_OK);
}

int sol_set_mig_type(sol_context *c, const int32_t *mig)
{
    if (check_ctx(c) || !mig) return SOL_ERR_ARGUMENT;
    HIPCHECK(c, hipSetDevice(c->device));
    HIPCHECK(c, hipMemcpyAsync(c->migt, mig, c->n * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
    HIPCHECK(c, hipStreamSynchronize(c->stream));
    return SOL_OK;
}

static int upload_soa(sol_context *c, const double *host, double *dst)
{
    HIPCHECK(c, hipSetDevice(c->device));
    CallEnd end(c);
    const double *rows;
    if (int r = rows_in(c, host, &rows)) return r;
    launch_aos_to_soa(c->stream, c->n, c->np, rows, dst);
    HIPCHECK(c, hipStreamSynchronize(c->stream));
    return end(SOL_OK);
}

int sol_set_state(sol_context *c, const double *y0)
{
    if (check_ctx(c) || !y0) return SOL_ERR_ARGUMENT;
    return upload_soa(c, y0, c->y0);
}

int sol_set_accel(sol_context *c, const double *a)
{
    if (check_ctx(c) || !a) return SOL_ERR_ARGUMENT;
    return upload_soa(c, a, c->acc0);
}

int sol_get_array(sol_context *c, int32_t which, double *out)
{
    if (check_ctx(c) || !out) return SOL_ERR_ARGUMENT;
    const double *src = nullptr;
    switch (which) {
    case SOL_ARRAY_Y0: src = c->y0; break;
    case SOL_ARRAY_Y: src = c->y; break;
    case SOL_ARRAY_ACCEL: src = c->acc0; break;
    case SOL_ARRAY_YSCALE: src = c->yscale; break;
    case SOL_ARRAY_ERROR: src = c->error; break;
    default: return c->fail(SOL_ERR_ARGUMENT, "unknown array %d", which);
    }
    HIPCHECK(c, hipSetDevice(c->device));
    CallEnd end(c);
    launch_soa_to_aos(c->stream, c->n, c->np, src, rows_out(c));
    return end(rows_done(c, out));
}

int sol_driver(sol_context *c, int32_t integrator, double eps, sol_timeline *tl, double *body_h)
{
    if (check_ctx(c) || !tl) return SOL_ERR_ARGUMENT;
    HIPCHECK(c, hipSetDevice(c->device));
    CallEnd end(c);
    switch (integrator) {
    case SOL_RUNGE_KUTTA_FEHLBERG78: return end(driver_rkf78(c, eps, tl, body_h, nullptr));
    case SOL_RUNGE_KUTTA4: {
        // the RK4 step reads no error back, so its kernels may still be queued
        const int r = driver_rk4(c, tl, body_h, nullptr);
        if (r) return r;
        HIPCHECK(c, hipStreamSynchronize(c->stream));
        return end(SOL_OK);
    }
    case SOL_DORMAND_PRINCE: return end(driver_dp(c, eps, tl, body_h, nullptr));
    default: return c->fail(SOL_ERR_UNSUPPORTED, "integrator %d is not provided", integrator);
    }
}

int sol_step(sol_context *c, int32_t integrator, double time, double h)
{
    if (check_ctx(c)) return SOL_ERR_ARGUMENT;
    const int ik = integ_kind(integrator);
    if (ik < 0) return c->fail(SOL_ERR_UNSUPPORTED, "integrator %d is not provided", integrator);
    HIPCHECK(c, hipSetDevice(c->device));
    CallEnd end(c);
    int r = run_stages(c, ik, time, h, false, nullptr);
    if (r) return r;
    HIPCHECK(c, hipStreamSynchronize(c->stream));
    return end(SOL_OK);
}

int sol_error_max(sol_context *c, int32_t integrator, double eps, double *out)
{
    if (check_ctx(c) || !out) return SOL_ERR_ARGUMENT;
    const size_t nv = 6 * (size_t)c->n;
    std::vector<double> e(nv), s(nv);
    int r = sol_get_array(c, SOL_ARRAY_ERROR, e.data());
    if (r) return r;
    if (integrator == SOL_DORMAND_PRINCE) {
        double m = 0.0;
        for (double v : e) if (std::fabs(v) > m) m = std::fabs(v);
        *out = m;
        return SOL_OK;
    }
    r = sol_get_array(c, SOL_ARRAY_YSCALE, s.data());
    if (r) return r;
    double m = 0.0;
    for (size_t i = 0; i < nv; ++i) {
        const double v = std::fabs(e[i] / s[i]);
        if (v > m) m = v;
    }
    *out = m / eps;
    return SOL_OK;
}

int sol_integrate(sol_context *c, int32_t integrator, double eps, sol_timeline *tl, int64_t max_steps,
                  sol_run_stats *stats)
{
    int32_t reason = 0;
    return sol_integrate_until(c, integrator, eps, tl, max_steps, 0, &reason, stats);
}

int sol_set_events(sol_context *c, const sol_event_settings *ev)
{
    if (check_ctx(c) || !ev) return SOL_ERR_ARGUMENT;
    if (!(ev->ejection >= 0.0) || !(ev->hit_centrum >= 0.0) || !(ev->collision_factor >= 0.0))
        return c->fail(SOL_ERR_ARGUMENT, "event thresholds must be >= 0 (0 turns a check off)");
    // Simulator::CheckEvent's e3 and h3 (Solaris/Simulator.cpp:628-629)
    c->ev_e3 = ev->ejection > 0.0 ? 1.0 / (ev->ejection * ev->ejection * ev->ejection) : 0.0;
    c->ev_h3 = ev->hit_centrum > 0.0 ? 1.0 / (ev->hit_centrum * ev->hit_centrum * ev->hit_centrum) : 0.0;
    c->ev_factor = ev->collision_factor;
    return SOL_OK;
}

// True when CheckEvent would find an event on the side outputs of the last
// evaluation (device check, one flag read back).
static int events_now(sol_context *c, bool &event)
{
    event = false;
    if (c->ev_e3 == 0.0 && c->ev_h3 == 0.0 && c->ev_factor == 0.0) return SOL_OK;
    if (!c->ev_flag) {
        int r = dalloc(c, &c->ev_flag, 1);
        if (r) return r;
    }
    launch_event_check(c->stream, c->n, c->rm3, c->nni, c->nnd, c->radius, c->ev_e3, c->ev_h3, c->ev_factor,
                       c->ev_flag);
    HIPCHECK(c, hipGetLastError());
    int32_t f = 0;
    HIPCHECK(c, hipMemcpyAsync(&f, c->ev_flag, sizeof f, hipMemcpyDeviceToHost, c->stream));
    HIPCHECK(c, hipStreamSynchronize(c->stream));
    event = f != 0;
    return SOL_OK;
}

int sol_integrate_until(sol_context *c, int32_t integrator, double eps, sol_timeline *tl, int64_t max_steps,
                        int32_t stop_mask, int32_t *reason, sol_run_stats *stats)
{
    if (check_ctx(c) || !tl || !reason) return SOL_ERR_ARGUMENT;
    *reason = 0;
    const int ik = integ_kind(integrator);
    if (ik < 0) return c->fail(SOL_ERR_UNSUPPORTED, "integrator %d is not provided", integrator);
    if (stop_mask & ~(SOL_STOP_OUTPUT | SOL_STOP_EVENT | SOL_STOP_END | SOL_STOP_STEPS))
        return c->fail(SOL_ERR_ARGUMENT, "unknown bits in stop_mask 0x%x", stop_mask);
    if (tl->flush_count < 0 || tl->flush_count >= 100)
        return c->fail(SOL_ERR_ARGUMENT, "timeline flush_count %d is not in [0, 100)", tl->flush_count);
    HIPCHECK(c, hipSetDevice(c->device));
    CallEnd end(c);
    hipEvent_t e0, e1;
    HIPCHECK(c, hipEventCreate(&e0));
    HIPCHECK(c, hipEventCreate(&e1));
    HIPCHECK(c, hipEventRecord(e0, c->stream));
    int64_t steps = 0, attempts = 0;
    int r = SOL_OK;
    SliceMap gm{};
    int path = path_of(c, ik, &gm);
    for (int tries = 0; tries < 3 && path != SOL_PATH_MULTI_KERNEL; ++tries) {
        r = resident_run(c, ik, eps, tl, max_steps, true, nullptr, &steps, &attempts, stop_mask, reason);
        if (r != kGridRetry) break;
        r = SOL_OK;
        path = path_of(c, ik, &gm);
    }
    if (path == SOL_PATH_MULTI_KERNEL) for (;;) {
        double bh = 0.0;
        if (ik == INTEG_RKF78) r = driver_rkf78(c, eps, tl, &bh, &attempts);
        else if (ik == INTEG_RK4) r = driver_rk4(c, tl, &bh, &attempts);
        else r = driver_dp(c, eps, tl, &bh, &attempts);
        if (r) break;
        ++steps;
        if (!std::isfinite(tl->time) || !std::isfinite(tl->hNext)) {
            r = c->fail(SOL_ERR_DEVICE, "non-finite time or step size (t %g, hNext %g)", tl->time, tl->hNext);
            break;
        }
        int32_t why = 0;
        // Simulator::DecisionMaking, Solaris/Simulator.cpp:183-245
        tl->elapsedTime += tl->hDid;
        tl->lastSave += tl->hDid;
        tl->lastNSteps += tl->hDid;
        if (stop_mask & SOL_STOP_EVENT) {     // CheckEvent (:621-735) comes first
            bool ev = false;
            if ((r = events_now(c, ev))) break;
            if (ev) why |= SOL_STOP_EVENT;
        }
        const double actual = 1000.0 * 365.25 * tl->millenium + tl->time;
        bool stop = false;
        if (std::fabs(actual) >= std::fabs(tl->length)) stop = true;
        else if (c->n <= 1) stop = true;
        else {
            if (std::fabs(actual + tl->hNext) > std::fabs(tl->length)) tl->hNext = tl->length - actual;
            if (std::fabs(tl->lastSave) >= std::fabs(tl->output)) {
                tl->lastSave = 0.0;
                why |= SOL_STOP_OUTPUT;
            }
            if (std::fabs(tl->lastSave + tl->hNext) > std::fabs(tl->output)) tl->hNext = tl->output - tl->lastSave;
        }
        // Counter::succededStep % CheckForSM (:154-162)
        tl->flush_count = (tl->flush_count + 1) % 100;
        if (tl->flush_count == 0) launch_flush_small(c->stream, c->n, c->np, c->y, c->y0);
        why &= stop_mask;
        if (stop) why |= SOL_STOP_END;
        if (max_steps > 0 && steps >= max_steps) why |= SOL_STOP_STEPS;
        if (why) { *reason = why; break; }
    }
    (void)hipEventRecord(e1, c->stream);
    (void)hipEventSynchronize(e1);
    float ms = 0.0f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (stats) {
        const int per = n_stages(ik) + 0;
        stats->accepted_steps = steps;
        stats->attempts = attempts;
        stats->force_evaluations = steps + attempts * per;
        stats->interactions = (double)stats->force_evaluations * c->interactions_per_eval;
        stats->device_ms = ms;
        int groups = 0;
        if (path == kPathMesh) (void)use_mesh(c, ik, nullptr, &groups);
        if (path == kPathQuad) {
            QuadShape q{};
            (void)use_quad(c, ik, &q);
            groups = q.groups;
        }
        stats->path = path == kPathMesh || path == kPathQuad ? SOL_PATH_GRID : path;
        stats->slices = path == SOL_PATH_GRID ? gm.nslices : groups;
    }
    return end(r);
}

int sol_integrals(sol_context *c, double *out)
{
    if (check_ctx(c) || !out) return SOL_ERR_ARGUMENT;
    HIPCHECK(c, hipSetDevice(c->device));
    const size_t np = c->np, n = c->n;
    launch_integrals(c->stream, c->n, c->np, c->y0, c->mass, c->integ);
    // the potential's partial sums in the eleventh row, over every body but
    // the test particles (the massless type, last in body order)
    const int nparts = launch_potential(c->stream, c->n - c->nb.test_particle, c->np, c->y0, c->mass,
                                        c->integ + 10 * np, (int)np);
    if (!c->integ_h && hipHostMalloc((void **)&c->integ_h, 12 * np * sizeof(double), hipHostMallocDefault) != hipSuccess) {
        c->integ_h = nullptr;
        return c->fail(SOL_ERR_DEVICE, "hipHostMalloc of %zu bytes failed", 12 * np * sizeof(double));
    }
    const double *h = c->integ_h, *m = c->integ_h + 11 * np;
    HIPCHECK(c, hipMemcpyAsync(c->integ_h, c->integ, 11 * np * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIPCHECK(c, hipMemcpyAsync(c->integ_h + 11 * np, c->mass, n * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIPCHECK(c, hipStreamSynchronize(c->stream));
    // Calculate::Integrals (Solaris/Calculate.cpp:43-63), body order
    double M = 0.0;
    for (int i = 0; i < c->n_massive; ++i) M += m[i];
    out[0] = M;
    for (int k = 0; k < 6; ++k) {
        double s = 0.0;
        for (size_t i = 0; i < n; ++i) s += h[k * np + i];
        out[1 + k] = s / M;
    }
    out[7] = std::sqrt(out[1] * out[1] + out[2] * out[2] + out[3] * out[3]);
    out[8] = std::sqrt(out[4] * out[4] + out[5] * out[5] + out[6] * out[6]);
    double cc[3] = {0, 0, 0};
    for (int k = 0; k < 3; ++k)
        for (size_t i = 0; i < n; ++i) cc[k] += h[(6 + k) * np + i];
    out[9] = cc[0]; out[10] = cc[1]; out[11] = cc[2];
    out[12] = std::sqrt(cc[0] * cc[0] + cc[1] * cc[1] + cc[2] * cc[2]);
    double ke = 0.0, pe = 0.0;
    for (size_t i = 0; i < n; ++i) ke += h[9 * np + i];
    // each pair once: the reference's ordered-pair sum times 1/2
    for (int k = 0; k < nparts; ++k) pe += h[10 * np + k];
    pe *= kGauss2;
    out[13] = ke; out[14] = pe; out[15] = ke - pe;
    return SOL_OK;
}

int sol_profile(sol_context *c, int32_t enable, sol_kernel_profile *out)
{
    if (check_ctx(c)) return SOL_ERR_ARGUMENT;
    HIPCHECK(c, hipSetDevice(c->device));
    prof_collect(c);
    if (out) *out = c->prof;
    if (enable) {
        c->prof = sol_kernel_profile{};
        c->profiling = true;
    } else {
        c->profiling = false;
    }
    return SOL_OK;
}

int sol_interactions_per_evaluation(const sol_context *c, double *count)
{
    if (!c || !count) return SOL_ERR_ARGUMENT;
    *count = c->interactions_per_eval;
    return SOL_OK;
}

}  // extern "C"
