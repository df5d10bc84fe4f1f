/*
 * solaris_amd.h -- C ABI of the MI355X (gfx950) force-evaluation and
 * integration library.
 *
 * Every entry point takes plain pointers and sizes; no C++ or GPU runtime
 * types cross this boundary, and no C++ exception escapes it.  Host arrays
 * use the reference's array-of-structs layout: 6 doubles per body,
 * [x, y, z, vx, vy, vz] for states and [vx, vy, vz, ax, ay, az] for
 * derivatives (Solaris/Acceleration.cpp:258, :274-283).  Inside the context
 * the state is held on the GPU as structure-of-arrays.
 *
 * Return convention: 0 on success, non-zero on failure (the reference
 * returns 1 for every failure, Solaris/Error.cpp:13-20; here the value also
 * names the failure class).  sol_last_error() gives the message.
 *
 * Threading: one context per host thread; each context owns one HIP stream.
 * There are no global mutable objects.
 */
#ifndef SOLARIS_AMD_H_
#define SOLARIS_AMD_H_

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* ---- status codes --------------------------------------------------- */
#define SOL_OK              0
#define SOL_ERROR           1  /* generic failure (reference's "return 1") */
#define SOL_ERR_ARGUMENT    2  /* bad argument, size or ordering */
#define SOL_ERR_DEVICE      3  /* HIP runtime failure */
#define SOL_ERR_UNDERFLOW   4  /* RKF78 step-size underflow, t+h == t
                                  (Solaris/RungeKuttaFehlberg78.cpp:116-122) */
#define SOL_ERR_MAXITER     5  /* Dormand-Prince retries exceeded maxIter
                                  (Solaris/DormandPrince.cpp:158-162) */
#define SOL_ERR_ALLOCATION  6  /* e.g. nBodies.total == 0
                                  (Solaris/BodyData.cpp:68-72) */
#define SOL_ERR_UNSUPPORTED 7  /* integrator or mode not provided
                                  (e.g. RUNGE_KUTTA56, Solaris/RungeKutta56.h) */

/* ---- enumerations: same numeric values as the reference -------------- */
/* BodyType, Solaris/Body.h:14-24 */
enum {
    SOL_UNDEFINED_BODY_TYPE = 0,
    SOL_CENTRAL_BODY        = 1,
    SOL_GIANT_PLANET        = 2,
    SOL_ROCKY_PLANET        = 3,
    SOL_PROTO_PLANET        = 4,
    SOL_SUPER_PLANETESIMAL  = 5,
    SOL_PLANETESIMAL        = 6,
    SOL_TEST_PARTICLE       = 7
};
/* MigrationType, Solaris/Body.h:35-39 */
enum { SOL_MIGRATION_NO = 0, SOL_MIGRATION_TYPE_I = 1, SOL_MIGRATION_TYPE_II = 2 };
/* IntegratorType, Solaris/IntegratorType.h:12-17 */
enum {
    SOL_DORMAND_PRINCE          = 0,
    SOL_RUNGE_KUTTA4            = 1,
    SOL_RUNGE_KUTTA56           = 2,
    SOL_RUNGE_KUTTA_FEHLBERG78  = 3
};
/* GasDecreaseType, Solaris/GasDecreaseType.h */
enum { SOL_GAS_CONSTANT = 0, SOL_GAS_LINEAR = 1, SOL_GAS_EXPONENTIAL = 2 };
/* Arithmetic of the pairwise gravity terms (state update, Kepler term and
 * error norm are FP64 in both modes). */
enum { SOL_PRECISION_FP64 = 0, SOL_PRECISION_MIXED = 1 };
/* Device arrays that sol_get_array() can copy out (BodyData fields,
 * Solaris/BodyData.h:38-43). */
enum { SOL_ARRAY_Y0 = 0, SOL_ARRAY_Y = 1, SOL_ARRAY_ACCEL = 2,
       SOL_ARRAY_YSCALE = 3, SOL_ARRAY_ERROR = 4 };

/* ---- plain-data descriptions ----------------------------------------- */
/* NBodies, Solaris/NBodies.h.  Bodies must be sorted by type in the order
 * central, giant, rocky, proto, super-planetesimal, planetesimal, test
 * particle (Solaris/Simulator.cpp:449-495); the counts define the
 * interaction ranges. */
typedef struct sol_nbodies {
    int32_t central_body;
    int32_t giant_planet;
    int32_t rocky_planet;
    int32_t proto_planet;
    int32_t super_planetesimal;
    int32_t planetesimal;
    int32_t test_particle;
    int32_t total;
} sol_nbodies;

/* PowerLaw: c * x^index, Solaris/PowerLaw.cpp:17-20 */
typedef struct sol_power_law { double c; double index; } sol_power_law;

/* GasComponent fields read by the force model (Solaris/GasComponent.h).
 * mean_free_path must hold what the reference constructor computed
 * (Solaris/GasComponent.cpp:30-32); it is not re-derived from density. */
typedef struct sol_gas_component {
    double        alpha;
    double        mean_molecular_weight;
    double        particle_diameter;
    int32_t       type;          /* SOL_GAS_* */
    int32_t       reserved;
    double        time_scale;
    double        t0;
    double        t1;
    double        inner_edge;
    double        a;
    sol_power_law eta;
    sol_power_law tau;
    sol_power_law scale_height;
    sol_power_law density;
    sol_power_law mean_free_path;
} sol_gas_component;

/* Per-body parameter arrays (host pointers, each of length total). */
typedef struct sol_body_params {
    const double  *mass;
    const double  *radius;
    const double  *density;
    const double  *cd;
    const double  *gamma_stokes;
    const double  *gamma_epstein;
    const double  *mig_stop_at;
    const int32_t *type;
    const int32_t *mig_type;
} sol_body_params;

/* The TimeLine fields the drivers and the caller loop use
 * (Solaris/TimeLine.h:6-44). */
typedef struct sol_timeline {
    double  start;
    double  length;
    double  output;
    double  save;
    double  time;
    double  hNext;
    double  hDid;
    double  elapsedTime;
    double  lastSave;
    double  lastNSteps;
    int32_t millenium;
    /* Accepted steps since the start of the run modulo CheckForSM (100):
     * Counter::succededStep % Constants::CheckForSM of the caller loop
     * (Solaris/Simulator.cpp:154-159, Solaris/Constants.h:16), which times
     * the small-number flush.  Start a run with 0; sol_integrate and
     * sol_integrate_until keep it, so that a run split over many calls
     * flushes at the same steps as one call. */
    int32_t flush_count;
} sol_timeline;

/* Counters filled by sol_integrate(). */
typedef struct sol_run_stats {
    int64_t accepted_steps;   /* Counter::succededStep (Solaris/Simulator.cpp:154) */
    int64_t attempts;         /* accepted + rejected attempts */
    int64_t force_evaluations;
    double  interactions;     /* sum over evaluations of pair + Kepler terms */
    double  device_ms;        /* GPU time of the run, HIP events */
    int32_t path;             /* SOL_PATH_*: how the run was integrated */
    int32_t slices;           /* SOL_PATH_GRID: workgroups the system was split over */
} sol_run_stats;

/* sol_run_stats.path: one launch per stage (gravity, gas and stage-combine
 * kernels); whole Driver loops in one workgroup (small systems); whole
 * Driver loops over several workgroups of one launch, which exchange step
 * decisions (systems with few sources) or also positions (self-gravitating
 * systems of 32 to 5,889 bodies). */
enum { SOL_PATH_MULTI_KERNEL = 0, SOL_PATH_RESIDENT = 1, SOL_PATH_GRID = 2 };

typedef struct sol_context sol_context;

/* ---- context ---------------------------------------------------------- */
/* Replaces the construction of BodyData (Solaris/BodyData.cpp:66-187) and
 * Acceleration (Solaris/Acceleration.cpp:35-50).  barycentric selects
 * ComputeBaryCentric vs ComputeAstroCentric (Solaris/Acceleration.cpp:71-78). */
int sol_create(sol_context **ctx, const sol_nbodies *nbodies,
               int32_t barycentric, int32_t device);
int sol_destroy(sol_context *ctx);
/* Error::_errMsg (Solaris/Error.cpp:13-20); ctx may be NULL for failures of
 * sol_create.  The string stays valid until the next call on ctx. */
const char *sol_last_error(const sol_context *ctx);

/* Per-body parameters (BodyData arrays, Solaris/BodyData.h:12-31). */
int sol_set_bodies(sol_context *ctx, const sol_body_params *params);
/* Acceleration::nebula (Solaris/Acceleration.h:44); NULL removes the gas. */
int sol_set_nebula(sol_context *ctx, const sol_gas_component *gas);
/* Acceleration::evaluateGasDrag / evaluateTypeIMigration /
 * evaluateTypeIIMigration (Solaris/Acceleration.h:54-56). */
int sol_set_evaluate(sol_context *ctx, int32_t gas_drag, int32_t type_i,
                     int32_t type_ii);
int sol_get_evaluate(const sol_context *ctx, int32_t *gas_drag,
                     int32_t *type_i, int32_t *type_ii);
/* Pairwise-gravity arithmetic.  softening (AU) is a Plummer length applied
 * to pair terms only; 0 reproduces the reference. */
int sol_set_precision(sol_context *ctx, int32_t precision, double softening);
/* Source ranges [1, end) of the two astrocentric sink classes (bodies of
 * type <= ProtoPlanet, and all others).  -1 keeps the reference's
 * type-based ranges (Solaris/Acceleration.cpp:285-289).  No counterpart in
 * the reference: it expresses mutually attracting planetesimals. */
int sol_set_source_ranges(sol_context *ctx, int32_t end_massive_sinks,
                          int32_t end_other_sinks);

/* ---- force model ------------------------------------------------------ */
/* Acceleration::Compute(double t, double *y, double *totalAccel)
 * (Solaris/Acceleration.h:19, Solaris/Acceleration.cpp:60-81).
 * y and dydt are host arrays of 6*total doubles. */
int sol_compute(sol_context *ctx, double t, const double *y, double *dydt);
/* Side outputs of the last force evaluation: Acceleration::rm3
 * (Solaris/Acceleration.h:52), BodyData::indexOfNN / distanceOfNN and the
 * mutated BodyData::migType (Solaris/Acceleration.cpp:253-264, :439-443).
 * Any pointer may be NULL. */
int sol_get_side_outputs(sol_context *ctx, double *rm3, int32_t *index_nn,
                         double *distance_nn, int32_t *mig_type);
/* Overwrites the device copy of BodyData::migType. */
int sol_set_mig_type(sol_context *ctx, const int32_t *mig_type);
/* enable = 0: sol_compute skips the nearest-neighbour search and leaves the
 * rm3 / indexOfNN / distanceOfNN side outputs as they were.  1 (the
 * default) writes them as the reference does (with a symmetric block: the
 * grid search, 0.1 ms at 65,537 bodies).  The drivers are not affected:
 * they track nearest neighbours on the last evaluation of each attempt
 * only, as the reference's side outputs require.  No counterpart in the
 * reference. */
int sol_set_side_outputs(sol_context *ctx, int32_t enable);

/* ---- integrators ------------------------------------------------------ */
/* Upload BodyData::y0 (6*total doubles, host). */
int sol_set_state(sol_context *ctx, const double *y0);
/* Copy a device array (SOL_ARRAY_*) of 6*total doubles to the host. */
int sol_get_array(sol_context *ctx, int32_t which, double *out);
/* Upload BodyData::accel (the derivative at y0 that Step() reads as f0). */
int sol_set_accel(sol_context *ctx, const double *accel);

/* One Driver call on the device-resident state:
 *   RungeKuttaFehlberg78::Driver (Solaris/RungeKuttaFehlberg78.cpp:66-140),
 *   RungeKutta4::Driver          (Solaris/RungeKutta4.cpp:20-56),
 *   DormandPrince::Driver        (Solaris/DormandPrince.cpp:126-170).
 * Reads tl->time and tl->hNext; writes tl->hDid, tl->time, tl->hNext.
 * epsilon is the integrator's 10^accuracy.  After success the device Y0
 * holds the new state and Y the previous one (the reference's pointer
 * swap, Solaris/RungeKuttaFehlberg78.cpp:132).  body_h receives
 * BodyData::h after the call. */
int sol_driver(sol_context *ctx, int32_t integrator, double epsilon,
               sol_timeline *tl, double *body_h);
/* One Step call from device Y0 and ACCEL at (time, h) into Y and ERROR:
 *   RungeKuttaFehlberg78::Step (Solaris/RungeKuttaFehlberg78.cpp:147-250),
 *   RungeKutta4::Step          (Solaris/RungeKutta4.cpp:58-130),
 *   DormandPrince::Step2       (Solaris/DormandPrince.cpp:246-491).
 * RungeKutta4 leaves ERROR as it was, as the reference leaves
 * BodyData::error. */
int sol_step(sol_context *ctx, int32_t integrator, double time, double h);
/* RungeKuttaFehlberg78::GetErrorMax (Solaris/RungeKuttaFehlberg78.cpp:252-262)
 * over the device ERROR and YSCALE arrays, divided by epsilon; with
 * integrator == SOL_DORMAND_PRINCE, DormandPrince::GetErrorMax
 * (Solaris/DormandPrince.cpp:493-503) over ERROR alone. */
int sol_error_max(sol_context *ctx, int32_t integrator, double epsilon,
                  double *error_max);

/* The Simulator::Integrate loop (Solaris/Simulator.cpp:121-178) without
 * events and file output: Driver calls, the step clipping of
 * Simulator::DecisionMaking (Solaris/Simulator.cpp:181-248) and the
 * |y| < 1e-50 flush at every 100th accepted step (:159-162), until the end
 * of the time line or max_steps accepted steps (max_steps <= 0: no limit).
 * stats may be NULL.  The same as sol_integrate_until with stop_mask 0. */
int sol_integrate(sol_context *ctx, int32_t integrator, double epsilon,
                  sol_timeline *tl, int64_t max_steps, sol_run_stats *stats);

/* Thresholds of the caller loop's event checks, Simulator::CheckEvent
 * (Solaris/Simulator.cpp:621-735), from the run's Settings (ejection,
 * hitCentrum, collision->factor; :626-629, :688).  0 turns a check off.
 * No counterpart as a call: the reference reads them from its settings. */
typedef struct sol_event_settings {
    double ejection;          /* AU: body i >= 1 with rm3[i] < 1/ejection^3 */
    double hit_centrum;       /* AU: body i >= 1 with rm3[i] > 1/hit_centrum^3 */
    double collision_factor;  /* body i whose nearest neighbour j has
                                 factor * (radius[i] + radius[j]) > distanceOfNN[i] */
} sol_event_settings;
int sol_set_events(sol_context *ctx, const sol_event_settings *events);

/* Reasons sol_integrate_until returns (bits of *reason). */
#define SOL_STOP_END     1  /* the time line's length was reached (DecisionMaking's stop) */
#define SOL_STOP_OUTPUT  2  /* an output is due: DecisionMaking would save the phases and
                               integrals now (Solaris/Simulator.cpp:236-240) */
#define SOL_STOP_EVENT   4  /* CheckEvent would find an ejection, hit-centrum or collision */
#define SOL_STOP_STEPS   8  /* max_steps accepted steps */

/* sol_integrate that returns after the first accepted step at which the
 * caller loop has host work: with SOL_STOP_OUTPUT in stop_mask when an
 * output is due, with SOL_STOP_EVENT when an event threshold set by
 * sol_set_events is crossed (on the last stage's rm3 and nearest-neighbour
 * outputs, as CheckEvent reads them), and always at the end of the time
 * line or after max_steps.  *reason receives every reason that holds for
 * that step.  On return the time line is as DecisionMaking leaves it after
 * the step (clipped hNext, lastSave reset if an output was due), device Y0
 * holds the state to save, and sol_get_side_outputs gives the arrays
 * CheckEvent reads.  A caller that removes or merges bodies creates a
 * context for the new body set and continues with the same time line.
 * No counterpart in the reference, whose loop returns to the host after
 * every step; this lets a run stay on the device between outputs. */
int sol_integrate_until(sol_context *ctx, int32_t integrator, double epsilon,
                        sol_timeline *tl, int64_t max_steps, int32_t stop_mask,
                        int32_t *reason, sol_run_stats *stats);

/* Calculate::Integrals on device Y0 (Solaris/Calculate.cpp:43-63):
 * out[16] = M, barycentre r and v, |r_bc|, |v_bc|, angular momentum and its
 * length, kinetic, potential and total energy. */
int sol_integrals(sol_context *ctx, double *out16);

/* Kernel timing of the context's own stream. */
typedef struct sol_kernel_profile {
    int64_t pair_launches;     /* pair-sum launches without the nearest-neighbour search */
    double  pair_ms;           /* their summed duration (HIP events) */
    double  pair_interactions; /* pair terms they evaluated */
    int64_t epilogue_launches;
    double  epilogue_ms;
    int64_t pair_nn_launches;  /* pair-sum launches that also track the nearest neighbour */
    double  pair_nn_ms;
    int64_t pair_sym_launches; /* symmetric pair sums of the self-interacting block */
    double  pair_sym_ms;
    double  pair_sym_interactions; /* interactions they formed (two per pair) */
} sol_kernel_profile;
/* enable = 1 clears the totals and starts bracketing every pair-sum and
 * epilogue launch with HIP events on the context's stream; enable = 0
 * stops.  out (may be NULL) receives the totals so far (this call waits
 * for the stream).  No counterpart in the reference, which has no
 * profiling; it serves benchmark and roofline reporting. */
int sol_profile(sol_context *ctx, int32_t enable, sol_kernel_profile *out);

/* Interactions per force evaluation under the context's source ranges:
 * sum over sinks i >= 1 of (1 + |S(i) \ {i}|). */
int sol_interactions_per_evaluation(const sol_context *ctx, double *count);

/* ---- batched ensemble ------------------------------------------------- */
/* Many independent systems (each a star plus planets, no gas) integrated
 * together in persistent launches: every workgroup takes the next system
 * from a device-side queue (the systems with the most work expected first)
 * and runs its whole Driver loops with the caller loop's clipping, then
 * takes the next.  The larger systems go to a second queue, launched beside
 * the first, whose workgroups give each body two lanes.  The first queue's
 * launch shape (threads per system) is picked by timing, and each launch
 * is replayed from a captured HIP graph.  No
 * counterpart in the reference, where each system is a separate simulation
 * (Simulator::Integrate, Solaris/Simulator.cpp:121-178); per system the
 * semantics are those of sol_integrate.  A failing system stops with its
 * own status.
 * Once the running systems of at least 48 sources fit the device at several
 * workgroups each, they go on in that form, which sums in another order; the
 * launch shape decides on the order of sums too.  A system's last digits can
 * therefore depend on the other systems of its ensemble (the same ensemble run
 * again has the same bits in the same launch shape), which close encounters
 * amplify (1e-12 to 3e-11 AU over two days).  With SOLARIS_AMD_NO_GRID=1, which keeps
 * all in the queues, and SOLARIS_AMD_ENSEMBLE_BLOCK set to at least the bodies
 * of the first queue's largest system they do not. */
typedef struct sol_ensemble sol_ensemble;
enum { SOL_SYSTEM_RUNNING = 0, SOL_SYSTEM_DONE = 1, SOL_SYSTEM_UNDERFLOW = 2, SOL_SYSTEM_MAXITER = 3 };

int sol_ensemble_create(sol_ensemble **ens, int32_t nsys, const sol_nbodies *nbodies,
                        int32_t device);
int sol_ensemble_destroy(sol_ensemble *ens);
const char *sol_ensemble_last_error(const sol_ensemble *ens);
/* System k: per-body parameters, initial state (6*total doubles, AoS) and
 * its time line (time, hNext, length, output). */
int sol_ensemble_set_system(sol_ensemble *ens, int32_t k, const sol_body_params *params,
                            const double *y0, const sol_timeline *tl);
/* Integrates every running system until it reaches the end of its time
 * line or max_steps accepted steps in this call (max_steps <= 0: no
 * limit).  stats (may be NULL) sums over systems. */
int sol_ensemble_run(sol_ensemble *ens, int32_t integrator, double epsilon, int64_t max_steps,
                     sol_run_stats *stats);
/* Picks the launch shape of sol_ensemble_run (threads per system, and with
 * it bodies per thread) by timing each candidate over probe_steps accepted
 * steps of every running system; the systems' states and time lines are
 * restored afterwards, so a caller can tune before a timed run.
 * sol_ensemble_run tunes by itself (8 steps) when this was not called.
 * SOLARIS_AMD_ENSEMBLE_BLOCK=<threads> in the environment fixes the shape
 * instead. */
int sol_ensemble_tune(sol_ensemble *ens, int32_t integrator, double epsilon, int32_t probe_steps);
/* The launch shape and counters of an ensemble. */
typedef struct sol_ensemble_info {
    int32_t block;              /* threads per system (workgroup size) */
    int32_t bodies_per_thread;  /* 1, 2 or 4 */
    int32_t grid;               /* workgroups of the last launch */
    int32_t tuned;              /* 1 once the shape is chosen */
    int64_t launches;           /* persistent launches of sol_ensemble_run so far */
    int64_t graph_launches;     /* of which replays of the captured graph */
    int32_t candidates;         /* shapes the tuner timed (at most 8) */
    int32_t candidate_block[8];
    double  candidate_ms[8];    /* their probe times */
    /* the wide queue: systems of at least wide_min_bodies bodies, in
     * workgroups of wide_block threads with up to wide_lanes lanes per body
     * splitting the source loop, launched beside the queue above (which
     * block, bodies_per_thread, grid and the candidates describe);
     * wide_block 0: no wide queue */
    int32_t wide_block;
    int32_t wide_lanes;
    int32_t wide_min_bodies;
    int32_t wide_systems;       /* systems in the wide queue */
    int32_t wide_grid;          /* its workgroups in the last launch */
} sol_ensemble_info;
int sol_ensemble_get_info(const sol_ensemble *ens, sol_ensemble_info *info);
/* State (6*total doubles), time line and status (SOL_SYSTEM_*) of system k. */
int sol_ensemble_get_system(sol_ensemble *ens, int32_t k, double *y0, sol_timeline *tl,
                            int32_t *status, int64_t *steps);

/* ---- adjoint of fixed-step RK4 ---------------------------------------- */
/* Forward pass to record: nsteps RungeKutta4::Step calls
 * (Solaris/RungeKutta4.cpp:58-130) chained from the device Y0 at time t0,
 * each step starting with the force evaluation at its own state (as
 * RungeKutta4::Driver does, Solaris/RungeKutta4.cpp:20-56), step i of size
 * h_seq[i] (or h when h_seq is NULL).  The step sequence is frozen and the
 * state is kept on the device every checkpoint_every steps.  Gravity only,
 * astrocentric, FP64, no softening: a context with a nebula, barycentric
 * frame, mixed precision or softening is rejected with
 * SOL_ERR_UNSUPPORTED.  Y0 is left unchanged and Y receives the final
 * state; y_final (may be NULL) gets it too (6*total doubles).  No
 * counterpart in the reference, which has no gradients. */
int sol_adjoint_forward(sol_context *ctx, double t0, double h, const double *h_seq,
                        int64_t nsteps, int32_t checkpoint_every, double *y_final);
/* Reverse pass over the recorded steps: given dL/dy_final (6*total
 * doubles, AoS) returns dL/dy0 (6*total) and dL/dm (total doubles, per
 * body mass in solar masses; the central body's entry included).  Each
 * segment between checkpoints is recomputed forward, then the discrete
 * adjoint of the RK4 stages runs backwards through it with the force
 * vector-Jacobian product evaluated on the device.  Either output may be
 * NULL.  No counterpart in the reference. */
int sol_adjoint_backward(sol_context *ctx, const double *grad_y_final, double *grad_y0,
                         double *grad_mass);

/* ---- a call that allocates nothing ------------------------------------ */
/* Gravity of sol_compute (GravityAC with the reference's type-based source
 * ranges: Kepler term, pair terms, indirect term; the star's derivative
 * zero) for a gas-free astrocentric system whose arrays are already on the
 * current device: y and dydt are device arrays of 6*total doubles (AoS),
 * mass a device array of total doubles.  It allocates no device memory.
 * total is at most 131072 (larger sizes are rejected with
 * SOL_ERR_ARGUMENT).  The kernels are queued on `stream` (a hipStream_t,
 * NULL for the null stream) and the call returns without waiting.  Where y
 * and dydt overlap, y is first copied to a static device array of the
 * library (48 bytes per body), so such calls that overlap on one GPU (on
 * different streams or host threads) race; others do not.  err (may be NULL) receives
 * the message of a failure, at most err_len bytes with the terminating
 * zero.  No counterpart in the reference: it is for callers that cannot
 * allocate device memory, such as code under HIP graph capture and
 * serving loops. */
int sol_compute_gravity_noalloc(const sol_nbodies *nbodies, const double *y, const double *mass,
                                double *dydt, void *stream, char *err, int32_t err_len);

/* Library version string. */
const char *sol_version(void);

#ifdef __cplusplus
}
#endif

#endif /* SOLARIS_AMD_H_ */
