// stages.hip -- per-body kernels around the pair sum.
//
//  k_prep        state -> J records (x, y, z, k^2 m) and the per-block sums
//                of the indirect term k^2 m_j r_j / r_j^3 over each source
//                range (Solaris/Acceleration.cpp:256-264, :314-316).
//  k_migration   Type I / Type II migration at the Driver's first force
//                evaluation into the per-body cache (Acceleration.cpp:424-528,
//                :645-764), mutating migType on the device.
//  k_epilogue    per body: reduce the pair partials, add the Kepler term and
//                subtract the indirect sum (GravityAC, :268-326), add gas drag
//                (GasDragAC, :331-422) and the cached migration (:190-242);
//                store the stage derivative; then either form the next RK
//                stage's state (the stage-combine loops of
//                RungeKuttaFehlberg78::Step :170-234, RungeKutta4::Step
//                :100-116, DormandPrince::Step2 :274-409) or the final state,
//                error estimate and the per-block error maximum (:236-242,
//                :252-262; DormandPrince.cpp:471-503).
// All arithmetic is FP64.  Reductions use a fixed order, so results are
// reproducible run to run.
#include <float.h>

#include <algorithm>

#include "gasdev.h"
#include "sol_internal.h"
#include "static_for.h"
#include "tableaux.h"

namespace sol {
namespace {

// Coefficient tables (device buffer written by the context, see
// context.cpp): offsets into it.
constexpr int kRkfD = 0;       // [13][12]
constexpr int kRk4A = 156;     // [4][3]
constexpr int kRk4B = 168;     // [4]
constexpr int kRk4C = 172;     // [4]
constexpr int kDpA = 176;      // [9][8]
constexpr int kDpB = 248;      // [9]
constexpr int kDpBdh = 257;    // [9]
constexpr int kDpC = 266;      // [9]

__global__ __launch_bounds__(256) void k_migration(int n_central, int n_giant, int n_massive, int np,
                                                    const double *__restrict__ st, const double *__restrict__ mass,
                                                    const double *__restrict__ stop, int32_t *__restrict__ migt,
                                                    double *__restrict__ migc, GasDev g, int bc, double t,
                                                    int do1, int do2)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_central || i >= n_massive) return;
    const bool is_giant = i < n_central + n_giant;
    if (is_giant ? !do2 : !do1) return;
    const int want = is_giant ? SOL_MIGRATION_TYPE_II : SOL_MIGRATION_TYPE_I;
    if (migt[i] != want) return;
    double ox, oy, oz;
    int32_t mig = migt[i];
    migration_accel(is_giant, st[i], st[np + i], st[2 * np + i], st[3 * np + i], st[4 * np + i], st[5 * np + i],
                    mass[i], mass[0], stop[i], mig, g, bc, t, ox, oy, oz);
    if (mig != migt[i]) migt[i] = mig;
    migc[i] = ox;
    migc[np + i] = oy;
    migc[2 * np + i] = oz;
}

// ---- block reductions with a fixed order ------------------------------
__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}

__device__ __forceinline__ double wave_max(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmax(v, __shfl_xor(v, o, kWave));
    return v;
}

// Sums v[0..5] over the block; result valid in thread 0.
__device__ void block_sum6(double v[6], double (*lds)[6])
{
    const int wid = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
#pragma unroll
    for (int k = 0; k < 6; ++k) v[k] = wave_sum(v[k]);
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < 6; ++k) lds[wid][k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 0; k < 6; ++k) {
            double s = lds[0][k];
            for (int q = 1; q < kBlock / kWave; ++q) s += lds[q][k];
            v[k] = s;
        }
    }
    __syncthreads();
}

// Indirect-term contribution of body i at position p (AC): k^2 m r / r^3,
// split by membership in the two source ranges [1, ea) and [1, eb).
__device__ __forceinline__ void indirect_contrib(int i, int n, double x, double y, double z, double gm,
                                                 int ea, int eb, double v[6])
{
    for (int k = 0; k < 6; ++k) v[k] = 0.0;
    if (i >= 1 && i < n) {
        const double r2 = SQR(x) + SQR(y) + SQR(z);
        const double r = sqrt(r2);
        const double rm3 = 1.0 / (r2 * r);
        const double cx = gm * rm3 * x, cy = gm * rm3 * y, cz = gm * rm3 * z;
        if (i < ea) { v[0] = cx; v[1] = cy; v[2] = cz; }
        if (i < eb) { v[3] = cx; v[4] = cy; v[5] = cz; }
    }
}

__global__ __launch_bounds__(256) void k_prep(int n, int np, const double *__restrict__ st,
                                               const double *__restrict__ gm, double4 *__restrict__ J,
                                               float4 *__restrict__ J32, double *__restrict__ ind_out,
                                               int bc, int ea, int eb)
{
    __shared__ double lds[kBlock / kWave][6];
    const int i = blockIdx.x * kBlock + threadIdx.x;
    double x = 0.0, y = 0.0, z = 0.0, m = 0.0;
    if (i < n) {
        x = st[i]; y = st[np + i]; z = st[2 * np + i]; m = gm[i];
    }
    if (i < np) {
        J[i] = make_double4(x, y, z, m);
        if (J32) J32[i] = make_float4((float)x, (float)y, (float)z, (float)m);
    }
    if (bc) return;
    double v[6];
    indirect_contrib(i, n, x, y, z, m, ea, eb, v);
    block_sum6(v, lds);
    if (threadIdx.x == 0)
        for (int k = 0; k < 6; ++k) ind_out[blockIdx.x * 6 + k] = v[k];
}

// Rows of six doubles (the interface's layout) through LDS, so that both
// sides move whole lines: aos may be pinned host memory, which the kernels
// read and write across the bus without a copy command of its own.
__device__ __forceinline__ void load_rows(const double *__restrict__ aos, int n, double *lds, double v[6])
{
    const int64_t first = (int64_t)blockIdx.x * kBlock * 6;
    const int len = min(6 * kBlock, (int)max((int64_t)0, 6 * (int64_t)n - first));
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const int q = k * kBlock + threadIdx.x;
        lds[q] = q < len ? aos[first + q] : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 6; ++c) v[c] = lds[6 * threadIdx.x + c];
}

__device__ __forceinline__ void store_rows(double *__restrict__ aos, int n, double *lds, const double v[6])
{
    const int64_t first = (int64_t)blockIdx.x * kBlock * 6;
    const int len = min(6 * kBlock, (int)max((int64_t)0, 6 * (int64_t)n - first));
#pragma unroll
    for (int c = 0; c < 6; ++c) lds[6 * threadIdx.x + c] = v[c];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const int q = k * kBlock + threadIdx.x;
        if (q < len) aos[first + q] = lds[q];
    }
}

// k_prep from the interface's rows, which are also laid out as components
// (what k_aos_to_soa would do first).
__global__ __launch_bounds__(256) void k_prep_rows(int n, int np, const double *__restrict__ aos,
                                                    double *__restrict__ st, const double *__restrict__ gm,
                                                    double4 *__restrict__ J, float4 *__restrict__ J32,
                                                    double *__restrict__ ind_out, int bc, int ea, int eb)
{
    __shared__ double rows[6 * kBlock];
    __shared__ double lds[kBlock / kWave][6];
    const int i = blockIdx.x * kBlock + threadIdx.x;
    double s[6];
    const double m = i < n ? gm[i] : 0.0;
    load_rows(aos, n, rows, s);
#pragma unroll
    for (int c = 0; c < 6; ++c) st[c * np + i] = s[c];
    J[i] = make_double4(s[0], s[1], s[2], m);
    if (J32) J32[i] = make_float4((float)s[0], (float)s[1], (float)s[2], (float)m);
    if (bc) return;
    double v[6];
    indirect_contrib(i, n, s[0], s[1], s[2], m, ea, eb, v);
    block_sum6(v, lds);
    if (threadIdx.x == 0)
        for (int k = 0; k < 6; ++k) ind_out[blockIdx.x * 6 + k] = v[k];
}

// ---- pair-partial lookup ------------------------------------------------
__device__ __forceinline__ int64_t wave_lo(const PairPlan &p, int64_t w)
{
    return (w * p.total_items) / p.nwaves;
}

__device__ __forceinline__ int64_t wave_of_item(const PairPlan &p, int64_t x)
{
    int64_t w = ((x + 1) * p.nwaves - 1) / p.total_items;
    return w < p.nwaves - 1 ? w : p.nwaves - 1;
}

__device__ __forceinline__ int tile_of_item(const PairPlan &p, int64_t x)
{
    const int s = (p.nseg > 1 && x >= p.seg[1].item_begin) ? 1 : 0;
    return p.seg[s].tile_begin + (int)((x - p.seg[s].item_begin) / p.seg[s].nchunks);
}

// Sum of the pair partials for sink i; false if i is in no sink class.
__device__ bool gather_pairs(const EpiArgs &a, int i, double &px, double &py, double &pz,
                             double &best, int &bidx)
{
    const PairPlan &p = a.plan;
    px = py = pz = 0.0;
    best = DBL_MAX; bidx = -1;
    bool found = false;
    if (a.want_nn && a.nn_sep && a.nnidx[i] >= 0) { best = a.nnr2[i]; bidx = a.nnidx[i]; }
    if (a.use_sym && i >= 1 && i < a.sym.M) {
        // symmetric sum of the mutual block: the row records of items (g, h),
        // h >= g, then the column records of the waves that cover column g
        const SymPlan &sp = a.sym;
        const int g = (i - 1) / kSymGroup, r = (i - 1) - g * kSymGroup;
        // row records: independent loads, unrolled so that many are in flight
        if (sp.shift == 0) {
            const double *row = a.apart + (sym_col_start(g) + g) * (3 * kSymGroup) + r;
#pragma unroll 8
            for (int h = g; h < sp.ngroups; ++h) {
                px += row[0];
                py += row[kSymGroup];
                pz += row[2 * kSymGroup];
                row += (int64_t)(h + 1) * (3 * kSymGroup);
            }
        } else {
#pragma unroll 8
            for (int k = g << sp.shift; k < sp.ngroups << sp.shift; ++k) {
                const int h = k >> sp.shift, unit = k & ((1 << sp.shift) - 1);
                const double *row = a.apart + (((sym_col_start(h) + g) << sp.shift) + unit) * (3 * kSymGroup) + r;
                px += row[0];
                py += row[kSymGroup];
                pz += row[2 * kSymGroup];
            }
        }
        // column records of the waves w0..w1 that cover column g's units
        // [A, B).  The waves hold contiguous non-empty ranges, so every wave
        // after w0 starts inside the column (its slot 0): only w0's first
        // column is decoded, and the other loads are independent.
        const int64_t A = sym_col_start(g) << sp.shift, B = sym_col_start(g + 1) << sp.shift;
        const int64_t w0 = sym_wave_of(sp, A), w1 = sym_wave_of(sp, B - 1);
        {
            int a0, h0;
            sym_decode(sym_wave_lo(sp, w0) >> sp.shift, a0, h0);
            const double *q = a.bpart + (w0 * sp.slots_per_wave + (g - h0)) * (3 * kSymGroup);
            px += q[r];
            py += q[kSymGroup + r];
            pz += q[2 * kSymGroup + r];
        }
        const double *qb = a.bpart + (size_t)r;
        const int64_t stride = (int64_t)sp.slots_per_wave * (3 * kSymGroup);
#pragma unroll 8
        for (int64_t w = w0 + 1; w <= w1; ++w) {
            const double *qw = qb + w * stride;
            px += qw[0];
            py += qw[kSymGroup];
            pz += qw[2 * kSymGroup];
        }
        found = true;
    }
    for (int s = 0; s < p.nseg; ++s) {
        const PairSeg &sg = p.seg[s];
        if (i < sg.sink_begin || i >= sg.sink_end) continue;
        const int t = (i - sg.sink_begin) / kWave;
        const int lane = (i - sg.sink_begin) - t * kWave;
        const int g = sg.tile_begin + t;
        const int64_t A = sg.item_begin + (int64_t)t * sg.nchunks;
        const int64_t B = A + sg.nchunks;
        const int64_t w0 = wave_of_item(p, A), w1 = wave_of_item(p, B - 1);
        for (int64_t w = w0; w <= w1; ++w) {
            const int64_t lo = wave_lo(p, w), hi = wave_lo(p, w + 1);
            if (lo >= hi || hi <= A || lo >= B) continue;
            const int k = g - tile_of_item(p, lo);
            const int64_t slot = w * p.slots_per_wave + k;
            const double *q = a.part + slot * (3 * kWave);
            px += q[lane];
            py += q[kWave + lane];
            pz += q[2 * kWave + lane];
            if (a.want_nn && !a.nn_sep) {
                const double r2 = a.nnr2[slot * kWave + lane];
                const int j = a.nnidx[slot * kWave + lane];
                if (j >= 0) {
                    const bool take = a.barycentric ? (r2 < best || (r2 == best && j > bidx))
                                                    : (r2 < best || (r2 == best && (bidx < 0 || j < bidx)));
                    if (take) { best = r2; bidx = j; }
                }
            }
        }
        return true;
    }
    return found;
}

// Stage derivative component c of stage l for body i.
__device__ __forceinline__ double fetch_f(const EpiArgs &a, int l, int c, int i, int s_reg, const double f[6])
{
    if (l == s_reg) return f[c];
    if (l == 0) return a.acc0[c * a.np + i];
    return a.fst[(int64_t)(l - 1) * 6 * a.np + c * a.np + i];
}

// State of stage SN (the reference's yTemp before the SN-th evaluation)
// with the tableau compiled in (tableaux.h), so each stage is straight-line
// code over its nonzero coefficients and every derivative load can be
// issued before the first use.  A runtime loop over the packed table put
// one coefficient read and one derivative load behind each term.
// RKF78 and RK4: acc = the first nonzero d_l F_l, then acc + d_l F_l over
// the others in ascending l, out = y0 + h acc (RungeKuttaFehlberg78.cpp:
// 100-116, RungeKutta4.cpp:74-110).  Dormand-Prince (DormandPrince.cpp:
// 274-409): var = a_0 F_0 + the nonzero a_l F_l in ascending l over the
// acceleration halves; positions y0 + c h v0 + h^2 var, velocities
// v0 + h var.  FREG: stage SN - 1's derivative is f (registers), else
// every derivative comes from memory.
template <int INTEG, int SN, bool FREG>
__device__ __forceinline__ void combine_ct(const EpiArgs &a, int i, const double f[6], double h, double out[6])
{
    const int np = a.np;
    constexpr int s_reg = FREG ? SN - 1 : -1;
    if constexpr (INTEG == INTEG_DP) {
        constexpr double cc = tab::kDpC[SN];
        const double h2 = h * h;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            double var = tab::kDpA[SN][0] * fetch_f(a, 0, j + 3, i, s_reg, f);
            static_for<1, SN>([&](auto L) {
                constexpr double d = tab::kDpA[SN][L];
                if constexpr (d != 0.0) var += d * fetch_f(a, L, j + 3, i, s_reg, f);
            });
            const double p0 = a.y0[j * np + i], v0 = a.y0[(j + 3) * np + i];
            out[j] = p0 + cc * h * v0 + h2 * (var);
            out[j + 3] = v0 + h * (var);
        }
    } else {
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            double acc = 0.0;
            bool first = true;
            static_for<0, SN>([&](auto L) {
                constexpr double d = INTEG == INTEG_RKF78 ? tab::kRkfD[SN][L] : tab::kRk4A[SN][L];
                if constexpr (d != 0.0) {
                    const double v = d * fetch_f(a, L, c, i, s_reg, f);
                    acc = first ? v : acc + v;
                    first = false;
                }
            });
            out[c] = a.y0[c * np + i] + h * acc;
        }
    }
}

// combine_ct for the run-time stage sn; s_reg is sn - 1 (that stage's
// derivative in f) or, for the first stage of an attempt, -1.
template <int INTEG, int NS>
__device__ __forceinline__ void combine_dispatch(const EpiArgs &a, int sn, int i, int s_reg, const double f[6],
                                                 double h, double out[6])
{
    static_for<1, NS + 1>([&](auto S) {
        if (sn == S) {
            if constexpr (S == 1) {
                if (s_reg < 0) {
                    combine_ct<INTEG, 1, false>(a, i, f, h, out);
                    return;
                }
            }
            combine_ct<INTEG, S, true>(a, i, f, h, out);
        }
    });
}

__device__ void combine_stage(const EpiArgs &a, int sn, int i, int s_reg, const double f[6], double h,
                              double out[6])
{
    if (a.integ == INTEG_RKF78) combine_dispatch<INTEG_RKF78, 12>(a, sn, i, s_reg, f, h, out);
    else if (a.integ == INTEG_RK4) combine_dispatch<INTEG_RK4, 3>(a, sn, i, s_reg, f, h, out);
    else combine_dispatch<INTEG_DP, 8>(a, sn, i, s_reg, f, h, out);
}

// Writes the next stage's state for body i: J record (positions and k^2 m),
// velocity part of the next derivative slot, and returns the indirect-term
// contribution in v.
__device__ void emit_next(const EpiArgs &a, int i, const double y[6], double v[6])
{
    const double gm = kGauss2 * a.mass[i];
    double4 *J = const_cast<double4 *>(a.J);
    J[i] = make_double4(y[0], y[1], y[2], gm);
    if (a.J32) a.J32[i] = make_float4((float)y[0], (float)y[1], (float)y[2], (float)gm);
    a.fst_next[i] = y[3];
    a.fst_next[a.np + i] = y[4];
    a.fst_next[2 * a.np + i] = y[5];
    if (!a.barycentric) indirect_contrib(i, a.n, y[0], y[1], y[2], gm, a.src_end_a, a.src_end_b, v);
}

__global__ __launch_bounds__(256) void k_epilogue(EpiArgs a)
{
    const double *__restrict__ coef = a.coef;
    __shared__ double ind_sum[6];
    __shared__ double lds[kBlock / kWave][6];
    __shared__ double red[kBlock / kWave];
    __shared__ double rows[6 * kBlock];
    const int i = blockIdx.x * kBlock + threadIdx.x;
    const int np = a.np;
    const double h = a.scal ? a.scal[0] : a.h, t = a.scal ? a.scal[1] : a.t;

    // sum of the indirect-term block partials of this stage (AC only)
    if (!a.barycentric && threadIdx.x < kWave) {
        double v[6] = {0, 0, 0, 0, 0, 0};
        for (int b = threadIdx.x; b < a.nblk; b += kWave)
            for (int k = 0; k < 6; ++k) v[k] += a.ind_in[b * 6 + k];
        for (int k = 0; k < 6; ++k) v[k] = wave_sum(v[k]);
        if (threadIdx.x == 0)
            for (int k = 0; k < 6; ++k) ind_sum[k] = v[k];
    }
    __syncthreads();

    const bool valid = i < a.n;
    double f[6] = {0, 0, 0, 0, 0, 0};
    if (valid) {
        const double4 p = a.J[i];
        const double vx = a.vel[i], vy = a.vel[np + i], vz = a.vel[2 * np + i];
        double px, py, pz, best;
        int bidx;
        const bool sink = gather_pairs(a, i, px, py, pz, best, bidx);
        double ax = 0.0, ay = 0.0, az = 0.0, rm3 = 0.0;
        const bool star_ac = !a.barycentric && i == 0;
        if (!star_ac) {
            if (!a.barycentric) {
                const double r2 = SQR(p.x) + SQR(p.y) + SQR(p.z);
                const double r = sqrt(r2);
                rm3 = 1.0 / (r2 * r);
                const double mu = kGauss2 * (a.mass[0] + a.mass[i]);
                const int end = (i < a.n_massive) ? a.src_end_a : a.src_end_b;
                const int sgi = (i < a.n_massive) ? 0 : 3;
                double ix = ind_sum[sgi], iy = ind_sum[sgi + 1], iz = ind_sum[sgi + 2];
                if (i < end) {            // the sink is one of its own sources: drop j == i
                    const double gm = kGauss2 * a.mass[i];
                    ix -= gm * rm3 * p.x; iy -= gm * rm3 * p.y; iz -= gm * rm3 * p.z;
                }
                ax = -mu * rm3 * p.x;     // Kepler term first, pair sum added last
                ay = -mu * rm3 * p.y;
                az = -mu * rm3 * p.z;
                if (sink) { ax += px - ix; ay += py - iy; az += pz - iz; }
            } else if (sink) {
                ax = px; ay = py; az = pz;
            }
            if (a.gas_on && i >= a.drag_lo && i < a.drag_hi) {
                double dx, dy, dz;
                if (a.drag_eval) {
                    const double tt = (a.integ == INTEG_RK4) ? t + coef[kRk4C + a.stage] * h
                                    : (a.integ == INTEG_DP) ? t + coef[kDpC + a.stage] * h : t;
                    const double factor = reduction_factor(a.gas, tt);
                    gas_drag(a.gas, factor, kGauss2 * a.mass[0], a.mass[0], p.x, p.y, p.z, vx, vy, vz,
                             a.radius[i], a.density[i], a.cd[i], a.gs[i], a.ge[i], dx, dy, dz);
                    a.dragc[i] = dx; a.dragc[np + i] = dy; a.dragc[2 * np + i] = dz;
                } else {   // evaluateGasDrag off: the cached array is re-added (:182-198)
                    dx = a.dragc[i]; dy = a.dragc[np + i]; dz = a.dragc[2 * np + i];
                }
                ax += dx; ay += dy; az += dz;
            }
            if (a.mig_on && i >= a.n_central && i < a.n_massive && a.migt[i] != SOL_MIGRATION_NO) {
                ax += a.migc[i]; ay += a.migc[np + i]; az += a.migc[2 * np + i];
            }
            f[0] = vx; f[1] = vy; f[2] = vz; f[3] = ax; f[4] = ay; f[5] = az;
        }
        if (a.kind == EPI_COMPUTE || a.kind == EPI_STAGE0) {
            for (int c = 0; c < 6; ++c) a.fout[c * np + i] = f[c];
        } else if (a.kind != EPI_ROWS) {
            for (int c = 3; c < 6; ++c) a.fout[c * np + i] = f[c];
        }
        if (a.last) {
            if (!a.barycentric) a.rm3_out[i] = rm3;
            a.nni_out[i] = (a.want_nn && bidx >= 0) ? bidx : -1;
            double dnn = 0.0;
            if (a.want_nn && bidx >= 0) {
                if (a.mixed) {   // the FP32 search picked the index; the distance is FP64
                    const double4 q = a.J[bidx];
                    const double dx = q.x - p.x, dy = q.y - p.y, dz = q.z - p.z;
                    dnn = sqrt(dx * dx + dy * dy + dz * dz);
                } else {
                    dnn = sqrt(best);
                }
            }
            a.nnd_out[i] = dnn;
        }
    }

    if (a.kind == EPI_ROWS) {
        store_rows(a.fout, a.n, rows, f);
    } else if (a.kind == EPI_STAGE0) {
        // yscale = |y0| + |h f0| + TINY (RungeKuttaFehlberg78.cpp:87-89)
        if (valid && a.yscale_out)
            for (int c = 0; c < 6; ++c)
                a.yscale_out[c * np + i] = fabs(a.y0[c * np + i]) + fabs(h * f[c]) + 1.0e-30;
    } else if (a.kind == EPI_MID) {
        double v[6] = {0, 0, 0, 0, 0, 0};
        if (valid) {
            double y[6];
            combine_stage(a, a.stage + 1, i, a.stage, f, h, y);
            emit_next(a, i, y, v);
        }
        if (!a.barycentric) {
            block_sum6(v, lds);
            if (threadIdx.x == 0)
                for (int k = 0; k < 6; ++k) a.ind_out[blockIdx.x * 6 + k] = v[k];
        }
    } else if (a.kind == EPI_FINAL) {
        double ratio = 0.0;
        if (valid) {
            const int s = a.stage;
            double y[6], e[6];
            if (a.integ == INTEG_RKF78) {
                // RungeKuttaFehlberg78.cpp:236-242
                const double b0 = 41.0 / 840.0, b5 = 34.0 / 105.0, b6 = 9.0 / 35.0, b8 = 9.0 / 280.0,
                             b10 = 41.0 / 840.0;
                for (int c = 0; c < 6; ++c) {
                    const double F0 = fetch_f(a, 0, c, i, s, f), F5 = fetch_f(a, 5, c, i, s, f);
                    const double F6 = fetch_f(a, 6, c, i, s, f), F7 = fetch_f(a, 7, c, i, s, f);
                    const double F8 = fetch_f(a, 8, c, i, s, f), F9 = fetch_f(a, 9, c, i, s, f);
                    const double F10 = fetch_f(a, 10, c, i, s, f), F11 = fetch_f(a, 11, c, i, s, f);
                    const double F12 = fetch_f(a, 12, c, i, s, f);
                    y[c] = a.y0[c * np + i] + h * (b0 * F0 + b5 * F5 + b6 * (F6 + F7) + b8 * (F8 + F9) + b10 * F10);
                    e[c] = h * fabs(F0 + F10 - F11 - F12) * 41.0 / 840.0;
                    ratio = fmax(ratio, fabs(e[c] / a.yscale[c * np + i]));
                }
            } else if (a.integ == INTEG_RK4) {
                // RungeKutta4.cpp:119-121; the step leaves BodyData::error as it was
                const double *B = coef + kRk4B;
                for (int c = 0; c < 6; ++c) {
                    y[c] = a.y0[c * np + i] + h * (B[0] * fetch_f(a, 0, c, i, s, f) + B[1] * fetch_f(a, 1, c, i, s, f) +
                                                   B[2] * fetch_f(a, 2, c, i, s, f) + B[3] * fetch_f(a, 3, c, i, s, f));
                    e[c] = 0.0;
                }
            } else {
                // DormandPrince.cpp:471-483
                const double *B = coef + kDpB, *Bd = coef + kDpBdh;
                const double h2 = h * h;
                for (int j = 0; j < 3; ++j) {
                    const double F0 = fetch_f(a, 0, j + 3, i, s, f), F4 = fetch_f(a, 4, j + 3, i, s, f);
                    const double F5 = fetch_f(a, 5, j + 3, i, s, f), F6 = fetch_f(a, 6, j + 3, i, s, f);
                    const double F7 = fetch_f(a, 7, j + 3, i, s, f), F8 = fetch_f(a, 8, j + 3, i, s, f);
                    const double p0 = a.y0[j * np + i], v0 = a.y0[(j + 3) * np + i];
                    y[j] = p0 + h * v0 + h2 * (B[0] * F0 + B[4] * F4 + B[5] * F5 + B[6] * F6 + B[7] * F7 + B[8] * F8);
                    e[j] = h2 * fabs(F7 - F8) / 20.0;
                    y[j + 3] = v0 + h * (Bd[0] * F0 + Bd[4] * F4 + Bd[5] * F5 + Bd[6] * F6 + Bd[7] * F7);
                    e[j + 3] = 0.0;
                    ratio = fmax(ratio, e[j]);
                }
            }
            for (int c = 0; c < 6; ++c) {
                a.y_out[c * np + i] = y[c];
                if (a.integ != INTEG_RK4) a.err_out[c * np + i] = e[c];
            }
        }
        ratio = wave_max(ratio);
        const int wid = threadIdx.x / kWave;
        if ((threadIdx.x & (kWave - 1)) == 0) red[wid] = ratio;
        __syncthreads();
        if (threadIdx.x == 0) {
            double m = red[0];
            for (int q = 1; q < kBlock / kWave; ++q) m = fmax(m, red[q]);
            a.errblk[blockIdx.x] = m;
        }
    }
}

// First stage state of an attempt, from y0 and f0 (all in memory).
__global__ __launch_bounds__(256) void k_combine_first(EpiArgs a)
{
    const double *__restrict__ coef = a.coef;
    __shared__ double lds[kBlock / kWave][6];
    const int i = blockIdx.x * kBlock + threadIdx.x;
    const double h = a.scal ? a.scal[0] : a.h;
    double v[6] = {0, 0, 0, 0, 0, 0};
    if (i < a.n) {
        double y[6];
        const double dummy[6] = {0, 0, 0, 0, 0, 0};
        combine_stage(a, 1, i, -1, dummy, h, y);
        emit_next(a, i, y, v);
    }
    if (!a.barycentric) {
        block_sum6(v, lds);
        if (threadIdx.x == 0)
            for (int k = 0; k < 6; ++k) a.ind_out[blockIdx.x * 6 + k] = v[k];
    }
}

__global__ void k_errmax_final(const double *__restrict__ blk, int nblk, double *__restrict__ out)
{
    double m = 0.0;
    for (int b = threadIdx.x; b < nblk; b += kWave) m = fmax(m, blk[b]);
    m = wave_max(m);
    if (threadIdx.x == 0) *out = m;
}

__global__ __launch_bounds__(256) void k_aos_to_soa(int n, int np, const double *__restrict__ aos,
                                                     double *__restrict__ soa)
{
    __shared__ double rows[6 * kBlock];
    const int i = blockIdx.x * kBlock + threadIdx.x;
    double v[6];
    load_rows(aos, n, rows, v);
#pragma unroll
    for (int c = 0; c < 6; ++c) soa[c * np + i] = v[c];
}

__global__ __launch_bounds__(256) void k_soa_to_aos(int n, int np, const double *__restrict__ soa,
                                                     double *__restrict__ aos)
{
    __shared__ double rows[6 * kBlock];
    const int i = blockIdx.x * kBlock + threadIdx.x;
    double v[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) v[c] = soa[c * np + i];
    store_rows(aos, n, rows, v);
}

// The side outputs one after another: rm3, nnd, then nni and migType.
__global__ __launch_bounds__(256) void k_pack_side(int n, const double *__restrict__ rm3,
                                                    const double *__restrict__ nnd, const int32_t *__restrict__ nni,
                                                    const int32_t *__restrict__ migt, double *__restrict__ out)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    out[i] = rm3[i];
    out[(int64_t)n + i] = nnd[i];
    int32_t *k = reinterpret_cast<int32_t *>(out + 2 * (int64_t)n);
    k[i] = nni[i];
    k[(int64_t)n + i] = migt[i];
}

// Tools::CheckAgainstSmallestNumber on two state arrays (Solaris/Tools.cpp:39-46).
__global__ void k_flush_small(int n, int np, double *__restrict__ a, double *__restrict__ b)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    for (int c = 0; c < 6; ++c) {
        if (fabs(a[c * np + i]) < 1.0e-50) a[c * np + i] = 0.0;
        if (fabs(b[c * np + i]) < 1.0e-50) b[c * np + i] = 0.0;
    }
}

// Simulator::CheckEvent's thresholds (Solaris/Simulator.cpp:631-644,
// :688-695) over the side outputs of the last evaluation: one block, a
// grid-stride loop over the bodies, and one flag (any body crosses a set
// threshold) written by thread 0.  e3 = 1/ejection^3, h3 = 1/hitCentrum^3
// and factor are 0 when their check is off.
__global__ __launch_bounds__(256) void k_event_check(int n, const double *__restrict__ rm3,
                                                     const int32_t *__restrict__ nni, const double *__restrict__ nnd,
                                                     const double *__restrict__ radius, double e3, double h3,
                                                     double factor, int32_t *__restrict__ flag)
{
    int ev = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        if (i >= 1 && e3 > 0.0 && rm3[i] < e3) ev = 1;
        if (i >= 1 && h3 > 0.0 && rm3[i] > h3) ev = 1;
        const int j = nni[i];
        if (factor > 0.0 && j >= 0 && j < n && factor * (radius[i] + radius[j]) > nnd[i]) ev = 1;
    }
    ev = __syncthreads_or(ev);
    if (threadIdx.x == 0) *flag = ev;
}

// Per-body terms of Calculate::Integrals (Solaris/Calculate.cpp:74-172):
// rows 0-5 m*y, 6-8 m (r x v), 9 kinetic 0.5 m v^2, 10 sum_j m_i m_j / r_ij.
__global__ __launch_bounds__(256) void k_integrals(int n, int np, const double *__restrict__ y,
                                                    const double *__restrict__ mass, double *__restrict__ out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double m = mass[i];
    const double x = y[i], yy = y[np + i], z = y[2 * np + i];
    const double vx = y[3 * np + i], vy = y[4 * np + i], vz = y[5 * np + i];
    for (int c = 0; c < 6; ++c) out[c * np + i] = m * y[c * np + i];
    out[6 * np + i] = m * (yy * vz - z * vy);
    out[7 * np + i] = m * (z * vx - x * vz);
    out[8 * np + i] = m * (x * vy - yy * vx);
    out[9 * np + i] = 0.5 * m * (vx * vx + vy * vy + vz * vz);
}

// Potential energy sum S = sum_{i<j} m_i m_j / r_ij over the bodies that
// can carry mass (i, j < nm: all but the test particles, which come last;
// the reference's loop over all ordered pairs, Solaris/Calculate.cpp:
// 150-172, is 2 S, and its test-particle terms are zero).
// Each pair once: the bodies in tiles of 256, one item per tile pair
// (a <= b), a workgroup of 128 threads per item with tile b's (x, y, z, m)
// in LDS and two sinks of tile a per thread (t and t + 128), so that each
// source read serves two sinks; on the diagonal only j > i.  1 / r is the
// hardware reciprocal square root with one second-order correction,
// (1 - e)^(-1/2) ~ 1 + e/2 + 3/8 e^2 for e = 1 - r^2 y^2, in place of the
// reference's IEEE square root and division.  Places past the end hold
// sources far away with no mass and sinks far away on the other side
// (finite terms, weighted by 0).  Workgroups take items a grid's stride
// apart and write one partial sum each (a fixed-order tree within the
// workgroup), summed on the host in order, so the result does not depend
// on timing.
__device__ __forceinline__ double inv_r(double r2)
{
    const double y0 = __builtin_amdgcn_rsq(r2);
    const double e = __builtin_fma(-r2, y0 * y0, 1.0);
    return __builtin_fma(y0, e * __builtin_fma(0.375, e, 0.5), y0);
}

__global__ __launch_bounds__(128) void k_potential(int nm, int np, int ntile, int64_t nitems,
                                                   const double *__restrict__ y, const double *__restrict__ mass,
                                                   double *__restrict__ part)
{
    __shared__ double4 src[256];
    __shared__ double red[128 / kWave];
    const int t = threadIdx.x;
    double acc = 0.0;
    for (int64_t it = blockIdx.x; it < nitems; it += gridDim.x) {
        // item -> (a, b), a <= b: rows of the upper triangle in order
        int a = (int)((2.0 * ntile + 1.0 - sqrt((2.0 * ntile + 1.0) * (2.0 * ntile + 1.0) - 8.0 * (double)it)) / 2.0);
        a = a < 0 ? 0 : a >= ntile ? ntile - 1 : a;
        while (a > 0 && (int64_t)a * (2 * ntile - a + 1) / 2 > it) --a;
        while ((int64_t)(a + 1) * (2 * ntile - a) / 2 <= it) ++a;
        const int b = a + (int)(it - (int64_t)a * (2 * ntile - a + 1) / 2);
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int j = b * 256 + h * 128 + t;
            src[h * 128 + t] = j < nm ? make_double4(y[j], y[np + j], y[2 * np + j], mass[j])
                                      : make_double4(1.0e18, 1.0e18, 1.0e18, 0.0);
        }
        __syncthreads();
        const int i0 = a * 256 + t, i1 = i0 + 128;
        const bool v0 = i0 < nm, v1 = i1 < nm;
        if (!v0) continue;   // so is i1
        const double ux = y[i0], uy = y[np + i0], uz = y[2 * np + i0];
        const double vx = v1 ? y[i1] : -1.0e18, vy = v1 ? y[np + i1] : -1.0e18, vz = v1 ? y[2 * np + i1] : -1.0e18;
        double s0 = 0.0, s1 = 0.0;
        if (a != b) {
            for (int k = 0; k < 256; ++k) {
                const double4 q = src[k];
                const double ax = q.x - ux, ay = q.y - uy, az = q.z - uz;
                const double bx = q.x - vx, by = q.y - vy, bz = q.z - vz;
                s0 = __builtin_fma(q.w, inv_r(ax * ax + ay * ay + az * az), s0);
                s1 = __builtin_fma(q.w, inv_r(bx * bx + by * by + bz * bz), s1);
            }
        } else {
            for (int k = 0; k < 256; ++k) {
                const double4 q = src[k];
                const bool t0 = k > t, t1 = k > t + 128;
                const double ax = q.x - ux, ay = q.y - uy, az = q.z - uz;
                const double bx = q.x - vx, by = q.y - vy, bz = q.z - vz;
                const double r0 = t0 ? ax * ax + ay * ay + az * az : 1.0;
                const double r1 = t1 ? bx * bx + by * by + bz * bz : 1.0;
                s0 = __builtin_fma(t0 ? q.w : 0.0, inv_r(r0), s0);
                s1 = __builtin_fma(t1 ? q.w : 0.0, inv_r(r1), s1);
            }
        }
        acc = __builtin_fma(mass[i0], s0, acc);
        if (v1) acc = __builtin_fma(mass[i1], s1, acc);
    }
    // fixed-order sum over the workgroup
#pragma unroll
    for (int o = kWave / 2; o >= 1; o >>= 1) acc += __shfl_xor(acc, o, kWave);
    if ((t & (kWave - 1)) == 0) red[t / kWave] = acc;
    __syncthreads();
    if (t == 0) {
        double u = 0.0;
        for (int w = 0; w < 128 / kWave; ++w) u += red[w];
        part[blockIdx.x] = u;
    }
}

inline int nblocks(int n) { return (n + kBlock - 1) / kBlock; }

}  // namespace

void launch_prep(hipStream_t st, int n, int np, const double *state, const double *gm, double4 *J,
                 float4 *J32, double *ind_out, int bc, int ea, int eb)
{
    hipLaunchKernelGGL(k_prep, dim3(np / kBlock), dim3(kBlock), 0, st, n, np, state, gm, J, J32, ind_out, bc,
                       ea, eb);
}

void launch_prep_rows(hipStream_t st, int n, int np, const double *aos, double *state, const double *gm, double4 *J,
                      float4 *J32, double *ind_out, int bc, int ea, int eb)
{
    hipLaunchKernelGGL(k_prep_rows, dim3(np / kBlock), dim3(kBlock), 0, st, n, np, aos, state, gm, J, J32, ind_out,
                       bc, ea, eb);
}

void launch_pack_side(hipStream_t st, int n, const double *rm3, const double *nnd, const int32_t *nni,
                      const int32_t *migt, double *out)
{
    hipLaunchKernelGGL(k_pack_side, dim3(nblocks(n)), dim3(kBlock), 0, st, n, rm3, nnd, nni, migt, out);
}

void launch_migration(hipStream_t st, int n_central, int n_giant, int n_massive, int np, const double *state,
                      const double *mass, const double *stop, int32_t *migt, double *migc, const GasDev &gas,
                      int bc, double t, int do1, int do2)
{
    if (n_massive <= 0) return;
    hipLaunchKernelGGL(k_migration, dim3(nblocks(n_massive)), dim3(kBlock), 0, st, n_central, n_giant, n_massive,
                       np, state, mass, stop, migt, migc, gas, bc, t, do1, do2);
}

void launch_epilogue(hipStream_t st, const EpiArgs &a)
{
    hipLaunchKernelGGL(k_epilogue, dim3(a.nblk), dim3(kBlock), 0, st, a);
}

void launch_combine_first(hipStream_t st, const EpiArgs &a)
{
    hipLaunchKernelGGL(k_combine_first, dim3(a.nblk), dim3(kBlock), 0, st, a);
}

void launch_errmax_final(hipStream_t st, const double *errblk, int nblk, double *out)
{
    hipLaunchKernelGGL(k_errmax_final, dim3(1), dim3(kWave), 0, st, errblk, nblk, out);
}

void launch_aos_to_soa(hipStream_t st, int n, int np, const double *aos, double *soa)
{
    hipLaunchKernelGGL(k_aos_to_soa, dim3(nblocks(np)), dim3(kBlock), 0, st, n, np, aos, soa);
}

void launch_soa_to_aos(hipStream_t st, int n, int np, const double *soa, double *aos)
{
    hipLaunchKernelGGL(k_soa_to_aos, dim3(nblocks(n)), dim3(kBlock), 0, st, n, np, soa, aos);
}

void launch_flush_small(hipStream_t st, int n, int np, double *a, double *b)
{
    hipLaunchKernelGGL(k_flush_small, dim3(nblocks(n)), dim3(kBlock), 0, st, n, np, a, b);
}

void launch_event_check(hipStream_t st, int n, const double *rm3, const int32_t *nni, const double *nnd,
                        const double *radius, double e3, double h3, double factor, int32_t *flag)
{
    hipLaunchKernelGGL(k_event_check, dim3(1), dim3(kBlock), 0, st, n, rm3, nni, nnd, radius, e3, h3, factor, flag);
}

void launch_integrals(hipStream_t st, int n, int np, const double *y0, const double *mass, double *out)
{
    hipLaunchKernelGGL(k_integrals, dim3(nblocks(n)), dim3(kBlock), 0, st, n, np, y0, mass, out);
}

int launch_potential(hipStream_t st, int nm, int np, const double *y0, const double *mass, double *part,
                     int max_parts)
{
    if (nm < 2) return 0;
    const int ntile = (nm + 255) / 256;
    const int64_t nitems = (int64_t)ntile * (ntile + 1) / 2;
    const int grid = (int)std::min<int64_t>(nitems, std::min(8192, max_parts));
    hipLaunchKernelGGL(k_potential, dim3(grid), dim3(128), 0, st, nm, np, ntile, nitems, y0, mass, part);
    return grid;
}

}  // namespace sol
