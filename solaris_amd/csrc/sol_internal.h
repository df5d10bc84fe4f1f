// sol_internal.h -- types shared by the HIP kernels and the host context.
//
// Device layout (one context, N bodies, NP = N rounded up to 256):
//   state arrays (Y0, Y, ACCEL, YSCALE, ERROR, stage derivatives F_s) are
//   structure-of-arrays: component c of body i at [c*NP + i], c = 0..5;
//   J[i] = (x, y, z, k^2 m) of the positions being evaluated, one 32-byte
//   record per body, read by the pair kernel as a wave-uniform stream.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "../../include/solaris_amd.h"
#include "sym_plan.h"

namespace sol {

constexpr double kGauss  = 1.720209895e-2;           // Solaris/Constants.h:28
constexpr double kGauss2 = 2.959122082855911025e-4;  // Solaris/Constants.h:29
constexpr int kBlock = 256;   // threads per block of the elementwise kernels
constexpr int kWave = 64;     // CDNA wavefront
constexpr int kMaxSeg = 4;    // sink ranges per pair-sum launch

// One sink class: sinks [sink_begin, sink_end) see sources
// [src_begin, src_end) (minus themselves).  Sinks are cut into tiles of 64
// (one wavefront) and sources into chunks; a work item is one
// (tile, chunk) pair.
struct PairSeg {
    int32_t sink_begin, sink_end;
    int32_t src_begin, src_end;
    int32_t ntiles, nchunks;
    int32_t tile_begin;       // global index of this segment's first tile
    int32_t pad;
    int64_t item_begin;       // global index of this segment's first item
};

// Work plan of one pair-sum launch.  The items are split into nwaves
// contiguous ranges (wave w owns [w*T/W, (w+1)*T/W)), so every wave gets
// the same number of items to within one.  A wave accumulates over
// consecutive items of the same tile and writes one partial per tile it
// touched into its slots; slots_per_wave bounds that count.
struct PairPlan {
    PairSeg seg[kMaxSeg];
    int32_t nseg;
    int32_t chunk;            // sources per item
    int32_t nwaves;
    int32_t slots_per_wave;
    int64_t total_items;
    int32_t ntiles;
    int32_t pad;
};

// Gas disk parameters as the kernels read them (sol_gas_component).
struct GasDev {
    double alpha, mmw, particle_diameter;
    int32_t type, pad;
    double time_scale, t0, t1, inner_edge;
    double eta_c, eta_i, tau_c, tau_i, sh_c, sh_i, rho_c, rho_i, mfp_c, mfp_i;
};

// EPI_ROWS: as EPI_COMPUTE, the derivative in the interface's rows of six
enum EpiKind { EPI_COMPUTE = 0, EPI_STAGE0 = 1, EPI_MID = 2, EPI_FINAL = 3, EPI_ROWS = 4 };
enum IntegKind { INTEG_RKF78 = 0, INTEG_RK4 = 1, INTEG_DP = 2 };

// Arguments of the per-stage epilogue (see stages.hip).
struct EpiArgs {
    PairPlan plan;
    const double *part;       // pair partial sums, [slot][3][64]
    const double *nnr2;       // nearest-neighbour partials, [slot][64]
    const int32_t *nnidx;
    int32_t n, np, nblk, barycentric;
    int32_t n_massive, n_central, n_giant, src_end_a;
    int32_t src_end_b, drag_lo, drag_hi, gas_on;
    int32_t mig_on, kind, integ, stage;
    int32_t last, want_nn, drag_eval, pad1;
    const double4 *J;         // stage positions (and k^2 m); rewritten in place for the next stage
    float4 *J32;              // FP32 copy of J for the mixed-precision pair sum (or null)
    int32_t mixed, pad2;
    const double *vel;        // stage velocities (3 x NP)
    const double *mass, *radius, *density, *cd, *gs, *ge;
    const int32_t *migt;      // BodyData::migType on the device
    const double *migc;       // cached migration accelerations (3 x NP)
    double *dragc;            // cached gas-drag accelerations (3 x NP)
    GasDev gas;
    const double *ind_in;     // indirect-term block partials of this stage, [blk][2][3]
    double *ind_out;          // ... of the next stage
    double *fout;             // derivative of this stage (6 x NP)
    double *rm3_out; int32_t *nni_out; double *nnd_out;
    const double *y0;         // 6 x NP
    const double *acc0;       // f0 (6 x NP)
    const double *fst;        // stage derivatives, stage l >= 1 at fst + (l-1)*6*NP
    double *fst_next;         // derivative slot of stage s+1 (its velocity part is written)
    const double *yscale;
    double *yscale_out, *y_out, *err_out, *errblk;
    double h, t;              // step size and step start time, by value (captured at launch)
    const double *scal;       // device scalars [0] = h, [1] = t when set (steps controlled on
                              // the device); null: h and t above
    const double *coef;       // integrator coefficient tables (context.cpp)
    SymPlan sym;              // symmetric pair sum of the mutual block (used when use_sym)
    int32_t use_sym, pad3;
    const double *apart, *bpart;   // its row-side and column-side records
    int32_t nn_sep, pad4;     // nearest neighbours: 0 in the pair partials, 1 per sink in nnr2/nnidx (grid search)
};

// Arguments of one force vector-Jacobian product (adjoint.hip).  Y is the
// stage state and W the weight (both 6 x NP); the sink pass runs
// tiles_s x nch_s waves (sinks [1, n) in tiles of 64, sources [1, jmax) in
// chunks of ch_s), the source pass tiles_b x nch_b (sources [1, jmax) in
// tiles of 64, sinks [1, n) in chunks of ch_b).
struct VjpArgs {
    int32_t n, np, n_massive, ea;
    int32_t eb, jmax, tiles_s, nch_s;
    int32_t ch_s, tiles_b, nch_b, ch_b;
    const double *Y, *W, *gm;
    double *psink;            // [nch_s][3][NP]
    double *psrc;             // [nch_b][7][NP]
    double *lam;              // adjoint of the step's end state
    double *ybar;             // adjoint of the step's start state, accumulated
    double *wnext;            // next stage weight alpha*lam + beta*G (or null)
    double alpha, beta;
    double *wfirst;           // with wnext null: the step's last product, which
    double cfirst;            // also starts the next step (see k_vjp_combine)
    double *mbar;             // dL/d(k^2 m), accumulated per body
    double *m0blk;            // central-mass term, accumulated per combine block
    int32_t src_few;          // source sums by k_vjp_parts (at most 64 sources)
};

// The adjoint of a system with few sources (adjoint_few.hip): bodies [1, src)
// are sources, at most kFewMaxSources of them.  Steps are counted from the
// recorded pass's first; stages holds the stage states of steps first, ...
constexpr int kFewMaxSources = 32;
struct FewArgs {
    int32_t n, np, nm, ea;
    int32_t eb, src, K, first;
    int32_t s0, s1, t0, t1;       // steps of the sources' chain and of the sinks'
    const double *gm, *h;
    double *y;                    // forward: the state (6 x NP), in place
    double *stages;               // [step - first][4][6][NP], or null (forward)
    double *ckpt;                 // forward: every K-th state, or null
    const double4 *sp_in;         // forward: the sources' stage records of the sinks' chunk
    double4 *sp_out;              // ... and of the sources' chunk, [step][4][src]
    double *lam, *mbar, *m0src;   // backward: adjoint state, mass gradients
    double *u, *sums;
};
void launch_few_forward(hipStream_t st, const FewArgs &a);
void launch_few_backward(hipStream_t st, const FewArgs &a);
void launch_few_sums(hipStream_t st, const FewArgs &a);
void launch_few_mass(hipStream_t st, const FewArgs &a, double *out);

// Integrator coefficient tables packed at the offsets the kernels read
// (275 doubles).
void fill_coefficients(std::vector<double> &c);

// Host-side launchers (pairs.hip / stages.hip).
void launch_pairs(hipStream_t st, const PairPlan &plan, const double4 *J, double *part,
                  double *nnr2, int32_t *nnidx, bool nn, bool barycentric, bool mixed,
                  double eps2, const float4 *J32);
// Grid of the exact nearest-neighbour search (nngrid.hip): cubic cells of
// side h from lo, dim[0] x dim[1] x dim[2] of them (x fastest).
struct GridParams {
    double lo[3];
    double h, slack;
    int32_t dim[3];
    int32_t ncells;
};

// Device buffers of the search: params, bounding-box partials
// [kGridBboxBlocks][6], counts and starts [max_cells + 1], per-source cell
// and rank, the sources sorted by cell ((x, y, z, index) records), and the
// result per sink: squared distance and index (-1: none).
constexpr int kGridBboxBlocks = 256;
struct NNGrid {
    GridParams *params;
    double *bbox;
    int32_t *count, *start, *cellof, *rank;
    double4 *spos;
    double *r2;
    int32_t *idx;
    int32_t max_cells, pad;
};
size_t nn_grid_max_cells(int n);
// Nearest neighbour of every sink of `plan` among its segment's sources
// (itself excluded) from the positions J, into G.r2 / G.idx.
void launch_nn_grid(hipStream_t st, const NNGrid &G, const PairPlan &plan, const double4 *J, int n, bool bc);

// Symmetric pair sum over the mutual block (sym_plan.h): row-side records
// in apart, column-side records in bpart.
void launch_pairs_sym(hipStream_t st, const SymPlan &sp, const double4 *J, double *apart, double *bpart,
                      double eps2);
// Its mixed-precision form (FP32 terms from J32, close pairs in FP64 from J).
void launch_pairs_sym_mixed(hipStream_t st, const SymPlan &sp, const float4 *J32, const double4 *J, double *apart,
                            double *bpart, double eps2);
void launch_prep(hipStream_t st, int n, int np, const double *state, const double *gm,
                 double4 *J, float4 *J32, double *ind_out, int barycentric, int src_end_a,
                 int src_end_b);
// launch_prep from rows of six doubles (device or pinned host memory), which
// also go to `state` as components.
void launch_prep_rows(hipStream_t st, int n, int np, const double *aos, double *state, const double *gm,
                      double4 *J, float4 *J32, double *ind_out, int barycentric, int src_end_a, int src_end_b);
// rm3 and nnd (n doubles each), then nni and migt (n int32 each) into out.
void launch_pack_side(hipStream_t st, int n, const double *rm3, const double *nnd, const int32_t *nni,
                      const int32_t *migt, double *out);
void launch_migration(hipStream_t st, int n_central, int n_giant, int n_massive, int np,
                      const double *state, const double *mass, const double *stop,
                      int32_t *migt, double *migc, const GasDev &gas, int barycentric,
                      double t, int do_type1, int do_type2);
void launch_epilogue(hipStream_t st, const EpiArgs &a);
void launch_combine_first(hipStream_t st, const EpiArgs &a);
void launch_errmax_final(hipStream_t st, const double *errblk, int nblk, double *out);
void launch_aos_to_soa(hipStream_t st, int n, int np, const double *aos, double *soa);
void launch_soa_to_aos(hipStream_t st, int n, int np, const double *soa, double *aos);
void launch_flush_small(hipStream_t st, int n, int np, double *a, double *b);
void launch_event_check(hipStream_t st, int n, const double *rm3, const int32_t *nni, const double *nnd,
                        const double *radius, double e3, double h3, double factor, int32_t *flag);
void launch_integrals(hipStream_t st, int n, int np, const double *y0, const double *mass,
                      double *per_body /* 10 x NP */);
// sum_{i<j<nm} m_i m_j / r_ij as partial sums part[0 .. return value)
// (at most max_parts of them), to be added in order
int launch_potential(hipStream_t st, int nm, int np, const double *y0, const double *mass, double *part,
                     int max_parts);
// adjoint.hip
void launch_vjp(hipStream_t st, const VjpArgs &a);
void launch_adj_stage(hipStream_t st, size_t len, const double *y, const double *k, double a, double h,
                      double *out);
void launch_adj_final(hipStream_t st, size_t len, const double *y, const double *kb, size_t stride, double h,
                      double *out);
void launch_adj_init(hipStream_t st, size_t len, const double *lam, double *ybar, double *w, double c);
void launch_adj_mass(hipStream_t st, int n, const double *mbar, const double *m0blk, int nblk, double *out);

}  // namespace sol
