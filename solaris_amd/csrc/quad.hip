// quad.hip -- whole Driver loops of systems with few sources, four lanes per
// body.
//
// Two to nine bodies that pull (the star and up to eight planets) and any
// number that only follow: an evaluation is a chain of about 60 dependent FP64
// operations per body and nothing else, and a launch of one body per lane
// (the slices of resident.hip) leaves three of four SIMDs without a second
// wave, where a wave issues an FP64 operation every 8 cycles: 515 bodies took
// 17 us per RKF78 attempt for 1.3 us per stage.  What bounds it is thus the
// number of operations in one lane, and here four lanes share a body:
//
//   pulls       lane l takes the pulls of sources l, l + 4, ..., each with its
//               indirect term, and lane 0 the body's own 1 / r^3; lane c
//               (c < 3) gathers and adds component c;
//   state       lane c keeps component c of position and velocity and of all
//               stage derivatives in registers (the stages are unrolled) and
//               forms only that component of the next state.
//
// A wave holds 16 bodies: all sources first, advanced identically in every
// wave, then its own.  The sources' positions pass through the wave's LDS
// records, so no stage has a barrier.  Once per attempt the workgroups
// exchange their error maxima (not at all in RK4 without events): each polls
// the others' words, while it already evaluates the state the step would be
// accepted with.
//
// Per attempt, before (slices of resident.hip, below 129 bodies one workgroup)
// and after, us: RKF78 of 4 bodies 15.2 and 6.0, 515 17.7 and 6.7, 5,001 18.8
// and 7.4, 14,338 20.4 and 8.0; Dormand-Prince of 515 13.7 and 5.3; RK4 of 515
// 4.4 and 1.5.  An evaluation of about 120 instructions takes 0.38 us, the
// exchange 1.9 us.  With gas, RKF78 of 125 bodies 63.7 and 31.7, 505 51.3 and
// 31.9, 16,389 55.9 and 37.
#include <float.h>

#include <algorithm>
#include <type_traits>

#include "gasdev.h"
#include "lane_pairs.h"
#include "quad.h"
#include "quad_stages.h"
#include "static_for.h"
#include "tableaux.h"

namespace sol {
namespace {

#define QUAD_SCOPE __HIP_MEMORY_SCOPE_SYSTEM

constexpr int kQuadWaves = kQuadThreads / kWave;
constexpr int kQuads = kWave / 4;

template <int INTEG>
constexpr int q_stages() { return INTEG == INTEG_RKF78 ? 12 : INTEG == INTEG_RK4 ? 3 : 8; }
// rows of stage derivatives: the step's first evaluation and its stages
template <int INTEG>
constexpr int q_rows() { return q_stages<INTEG>() + 1; }

// Whether a run stops at events of the side outputs.
__host__ __device__ __forceinline__ bool quad_events(const ResSystem &S)
{
    return S.clip && (S.stop_mask & SOL_STOP_EVENT) && (S.e3 > 0.0 || S.h3 > 0.0 || S.coll > 0.0);
}

// A call rather than inlined code: its registers would be held through the stages.
__device__ __attribute__((noinline)) double quad_pow(double x, double y) { return pow(x, y); }

__device__ __forceinline__ double quad_wmax(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmax(v, __shfl_xor(v, o, kWave));
    return v;
}

// What a lane needs for the pulls on its body.
template <int NA>
struct QPulls {
    double mu;                 // k^2 (m0 + mi)
    double w[4 * NA];          // k^2 m of source a (0: not a source of this body)
    int slot[NA];              // the records of this lane's sources l, l + 4, ...
    bool near[NA];             // a candidate for the nearest neighbour
};

// |d|^-3 from r2 = |d|^2: the hardware's reciprocal square root and its
// second-order correction, as pair_range in resident.hip.  Its cap is above
// 1 / |d| of any two distinct bodies, so that a body's own record (d = 0, weight
// 0) comes out finite.
__device__ __forceinline__ double quad_rm3(double r2)
{
    const double y = fmin(__builtin_amdgcn_rsq(r2), 1.0e50);
    const double tt = y * y;
    const double e = __builtin_fma(-r2, tt, 1.0);
    const double y3 = tt * y;
    return __builtin_fma(y3, e * __builtin_fma(1.875, e, 1.5), y3);
}

// x^2 + y^2 + z^2, the first or the second square rounded first.
template <bool SECOND>
__device__ __forceinline__ double quad_sq(double x, double y, double z)
{
    return __builtin_fma(z, z, SECOND ? __builtin_fma(x, x, y * y) : __builtin_fma(y, y, x * x));
}

// The value of lane LANE of the quad in all four.
template <int LANE>
__device__ __forceinline__ double quad_from(double v) { return dpp_mov<LANE * 0x55>(v); }

// Side outputs of a body: 1 / |r|^3, distance squared and index of the nearest
// source.
struct QSide {
    double rm3, best;
    int idx;
};

// The nearest of the quad's four lanes, the smaller index of equals.
__device__ __forceinline__ void quad_nearest(QSide &side)
{
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const double ob = s == 0 ? dpp_mov<0xB1>(side.best) : dpp_mov<0x4E>(side.best);
        const int oi = s == 0 ? __builtin_amdgcn_mov_dpp(side.idx, 0xB1, 0xF, 0xF, false)
                              : __builtin_amdgcn_mov_dpp(side.idx, 0x4E, 0xF, 0xF, false);
        const bool take = ob < side.best || (ob == side.best && oi < side.idx);
        side.best = take ? ob : side.best;
        side.idx = take ? oi : side.idx;
    }
}

// Acceleration component of this lane for the position whose component it
// holds.  tab: the wave's source records (x, y, z), [0] the origin.
//
// Lane l forms d_a / |d_a|^3 - r_a / |r_a|^3 of its sources a and lane 0 the
// body's own 1 / |r|^3; lane c gathers component c of all and adds the weighted
// terms in the sources' order.  Every operation is that of resident.hip on the
// same operands, fused as the compiler fuses it there (FIRST: a step's first
// evaluation, which it fuses in another order than the stages'), so a run has
// the same bits in quads, in slices and in one workgroup.  (Weights in the
// lanes and a reduction over the quad take 85 instead of 120 operations, 5.6
// instead of 7.0 us per RKF78 attempt of 515 bodies, but round otherwise, and a
// particle's encounters over some years grow that to 1e-7.)
template <int NA, bool SIDE, bool FIRST>
__device__ __forceinline__ double quad_force(const QPulls<NA> &P, double (*tab)[4], int ns, int src, int l, double pos,
                                             QSide &side)
{
    if (src > 0) tab[src][l] = pos;
    const double x = quad_from<0>(pos), y = quad_from<1>(pos), z = quad_from<2>(pos);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (SIDE) { side.best = DBL_MAX; side.idx = 0x7fffffff; }
    double rm3 = 0.0, sum = 0.0;
    static_for<0, NA>([&](auto T) {
        constexpr int t = T;
        const double *rec = tab[P.slot[t]];
        double rx = rec[0], ry = rec[1], rz = rec[2];
        const double dx = rx - x, dy = ry - y, dz = rz - z;
        const double d2 = quad_sq<true>(dx, dy, dz);
        const double wd = quad_rm3(d2);
        if (t == 0) {                          // lane 0: the body itself
            rx = l == 0 ? x : rx;
            ry = l == 0 ? y : ry;
            rz = l == 0 ? z : rz;
        }
        const double r2 = quad_sq<FIRST>(rx, ry, rz);
        const double r = sqrt(r2);
        const double m3 = 1.0 / (r2 * r);
        if (t == 0) rm3 = quad_from<0>(m3);
        const double gx = __builtin_fma(dx, wd, -(rx * m3)), gy = __builtin_fma(dy, wd, -(ry * m3)),
                     gz = __builtin_fma(dz, wd, -(rz * m3));
        if (SIDE && P.near[t] && d2 < side.best) { side.best = d2; side.idx = P.slot[t]; }
        static_for<(t == 0 ? 1 : 0), 4>([&](auto L) {
            constexpr int a = 4 * t + L;
            if (a <= ns) {
                const double u = quad_from<L>(gx), v = quad_from<L>(gy), w = quad_from<L>(gz);
                sum = __builtin_fma(P.w[a], l == 0 ? u : l == 1 ? v : w, sum);
            }
        });
    });
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (SIDE) {
        side.rm3 = rm3;
        quad_nearest(side);
    }
    return __builtin_fma(-P.mu * rm3, pos, sum);
}

// The same with gas, in two halves: the sources' quads publish r_a and r_a /
// |r_a|^3, and after a barrier every quad forms its pulls, so that a quad takes
// one root and one division for its own |r|^-3 and none per record.  The lanes
// share that root and division with the drag's: base is the cylindrical radius
// rc (lane 2: the spherical one), over_rc3 mu / rc^3.  tab: the workgroup's
// records (x, y, z, -, and those times |r|^-3), two sets in turn, so that one
// barrier between writing and reading suffices.
//
// The operations are those of quad_force, so what differs from resident.hip is
// the drag's last bits alone, which rarely reach an acceleration some 1e7 times
// as large.  (Weights in the lanes and sums over the quad took 39.8 us per RKF78
// attempt of 16,389 bodies, this 38.5, and rounded otherwise: over 100 days a
// planetesimal's encounters grew that to 1e-8.)
struct QGasPlace {
    double x, y, z, base, rm3, over_rc3;
};

template <bool FIRST>
__device__ __forceinline__ QGasPlace quad_publish(double (*tab)[8], int src, int l, double pos, double mu)
{
    QGasPlace W;
    W.x = quad_from<0>(pos);
    W.y = quad_from<1>(pos);
    W.z = quad_from<2>(pos);
    const double r2 = quad_sq<FIRST>(W.x, W.y, W.z), q = SQR(W.x) + SQR(W.y);
    W.base = sqrt(l == 2 ? r2 : q);
    const double rc = quad_from<0>(W.base), r = quad_from<2>(W.base);
    const double part = (l < 2 ? 1.0 : mu) / (l < 2 ? r2 * r : q * rc);
    W.rm3 = quad_from<0>(part);
    W.over_rc3 = quad_from<2>(part);
    if (src > 0) {
        tab[src][l] = pos;
        tab[src][4 + l] = pos * W.rm3;
    }
    return W;
}

// Acceleration component of this lane; last: the nearest source too.
template <int NA>
__device__ __forceinline__ double quad_force_gas(const QPulls<NA> &P, double (*tab)[8], int ns, int l, double pos,
                                                 const QGasPlace &W, bool last, QSide &side)
{
    side.rm3 = W.rm3;
    side.best = DBL_MAX;
    side.idx = 0x7fffffff;
    double sum = 0.0;
    static_for<0, NA>([&](auto T) {
        constexpr int t = T;
        const double *rec = tab[P.slot[t]];
        const double dx = rec[0] - W.x, dy = rec[1] - W.y, dz = rec[2] - W.z;
        const double d2 = quad_sq<true>(dx, dy, dz);
        const double wd = quad_rm3(d2);
        const double gx = __builtin_fma(dx, wd, -rec[4]), gy = __builtin_fma(dy, wd, -rec[5]),
                     gz = __builtin_fma(dz, wd, -rec[6]);
        if (P.near[t] && d2 < side.best) { side.best = d2; side.idx = P.slot[t]; }
        static_for<(t == 0 ? 1 : 0), 4>([&](auto L) {
            constexpr int a = 4 * t + L;
            if (a <= ns) {
                const double u = quad_from<L>(gx), v = quad_from<L>(gy), w = quad_from<L>(gz);
                sum = __builtin_fma(P.w[a], l == 0 ? u : l == 1 ? v : w, sum);
            }
        });
    });
    if (last) quad_nearest(side);
    return __builtin_fma(-P.mu * W.rm3, pos, sum);
}

// One component of a body: state, previous state, stage derivatives, scale
// and error.
template <int INTEG, bool LDS>
struct QBody {
    double p, v, po, vo;
    QStages<q_rows<INTEG>(), LDS> d;
    double sp, sv, ep, ev;
};

// Coefficient L of stage S, and the first two stages l with a nonzero one (S
// if there is none).
template <int INTEG, int S>
constexpr double q_coef(int l)
{
    return INTEG == INTEG_RKF78 ? tab::kRkfD[S][l] : INTEG == INTEG_RK4 ? tab::kRk4A[S][l] : tab::kDpA[S][l];
}
template <int INTEG, int S>
constexpr int q_nonzero(int from)
{
    for (int l = from; l < S; ++l)
        if (q_coef<INTEG, S>(l) != 0.0) return l;
    return S;
}

// c0 f0 + c1 f1, the first or the second product rounded first.
template <bool SECOND>
__device__ __forceinline__ double quad_two(double c0, double f0, double c1, double f1)
{
    return SECOND ? __builtin_fma(c0, f0, c1 * f1) : __builtin_fma(c1, f1, c0 * f0);
}

// The sum of coefficient times derivative over the nonzero coefficients of
// stage S in tableau order, fused as the compiler fuses it in resident.hip.
template <int INTEG, int S, typename Get>
__device__ __forceinline__ double quad_sum(Get f)
{
    constexpr int l0 = q_nonzero<INTEG, S>(0), l1 = q_nonzero<INTEG, S>(l0 + 1);
    if constexpr (l1 >= S) {
        return q_coef<INTEG, S>(l0) * f(l0);
    } else {
        constexpr double c0 = q_coef<INTEG, S>(l0), c1 = q_coef<INTEG, S>(l1);
        double acc = quad_two<!(l1 == S - 1 || (c0 < 0.0 && c1 > 0.0))>(c0, f(l0), c1, f(l1));
        static_for<l1 + 1, S>([&](auto L) {
            if constexpr (q_coef<INTEG, S>(L) != 0.0) acc = __builtin_fma(q_coef<INTEG, S>(L), f(L), acc);
        });
        return acc;
    }
}

// State of stage S, as resident.hip's stage_state.
template <int INTEG, int S, bool LDS>
__device__ __forceinline__ void quad_stage(const QBody<INTEG, LDS> &B, double h, double &pos, double &vel)
{
    const double av = quad_sum<INTEG, S>([&](int l) { return B.d.F(l); });
    if constexpr (INTEG == INTEG_DP)
        pos = __builtin_fma(h * h, av, __builtin_fma(tab::kDpC[S] * h, B.v, B.p));
    else
        pos = __builtin_fma(h, quad_sum<INTEG, S>([&](int l) { return B.d.V(l); }), B.p);
    vel = __builtin_fma(h, av, B.v);
}

// Final state and error estimate (kept in B); returns this lane's part of the
// error maximum.
template <int INTEG, bool LDS>
__device__ __forceinline__ double quad_final(QBody<INTEG, LDS> &B, double h, double &pos, double &vel)
{
    auto V = [&](int l) { return B.d.V(l); };
    auto F = [&](int l) { return B.d.F(l); };
    if constexpr (INTEG == INTEG_RKF78) {
        constexpr double b0 = 41.0 / 840.0, b5 = 34.0 / 105.0, b6 = 9.0 / 35.0, b8 = 9.0 / 280.0, b10 = 41.0 / 840.0;
        auto sum = [&](auto f) {
            double s = quad_two<true>(b0, f(0), b5, f(5));
            s = __builtin_fma(b6, f(6) + f(7), s);
            s = __builtin_fma(b8, f(8) + f(9), s);
            return __builtin_fma(b10, f(10), s);
        };
        pos = __builtin_fma(h, sum(V), B.p);
        vel = __builtin_fma(h, sum(F), B.v);
        B.ep = h * fabs(V(0) + V(10) - V(11) - V(12)) * 41.0 / 840.0;
        B.ev = h * fabs(F(0) + F(10) - F(11) - F(12)) * 41.0 / 840.0;
        return fmax(fabs(B.ep / B.sp), fabs(B.ev / B.sv));
    } else if constexpr (INTEG == INTEG_RK4) {
        constexpr const double *b = tab::kRk4B;
        auto sum = [&](auto f) {
            return __builtin_fma(b[3], f(3), __builtin_fma(b[2], f(2), quad_two<true>(b[0], f(0), b[1], f(1))));
        };
        pos = __builtin_fma(h, sum(V), B.p);
        vel = __builtin_fma(h, sum(F), B.v);
        return 0.0;
    } else {
        constexpr const double *b = tab::kDpB, *d = tab::kDpBdh;
        const double h2 = h * h;
        double s = quad_two<false>(b[0], F(0), b[4], F(4)), u = quad_two<false>(d[0], F(0), d[4], F(4));
        s = __builtin_fma(b[5], F(5), s);
        u = __builtin_fma(d[5], F(5), u);
        s = __builtin_fma(b[6], F(6), s);
        u = __builtin_fma(d[6], F(6), u);
        s = __builtin_fma(b[7], F(7), s);
        u = __builtin_fma(d[7], F(7), u);
        s = __builtin_fma(b[8], F(8), s);
        pos = __builtin_fma(h2, s, __builtin_fma(h, B.v, B.p));
        vel = __builtin_fma(h, u, B.v);
        B.ep = h2 * fabs(F(7) - F(8)) / 20.0;
        B.ev = 0.0;
        return B.ep;
    }
}

// ---- gas -------------------------------------------------------------------

// What the drag reads, in LDS: the nebula, derived constants (edge =
// rho_c inner_edge^(rho_i - 4); thermal: the factor of sqrt(r) in the mean
// thermal speed), the exponent each lane of a quad takes, and the parameters
// of the bodies.
struct QGas {
    GasDev g;
    double edge, thermal, idx[4];
    int32_t quarters[4], by_quarters;      // 4 idx, where all four are whole and at most 16
    double R[kQuadGasBodies], rho_b[kQuadGasBodies], cd[kQuadGasBodies], gs[kQuadGasBodies], ge[kQuadGasBodies];
};

// x^(k / 4), |k| <= 16, from square roots and products (r1 = sqrt(x)): a third
// of the operations of pow.
__device__ __forceinline__ double quad_quarters(double x, double r1, int k)
{
    const int a = k < 0 ? -k : k, n = a >> 2;
    const double r2 = sqrt(r1), x2 = x * x;
    double p = (a & 1 ? r2 : 1.0) * (a & 2 ? r1 : 1.0);
    p *= (n & 1 ? x : 1.0) * (n & 2 ? x2 : 1.0);
    p = n & 4 ? p * (x2 * x2) : p;
    return k < 0 ? 1.0 / p : p;
}

// GasDragAC (gas_drag in gasdev.h, with the same branches), component of this
// lane of the drag at (x, y, z, vx, vy, vz).  What bounds an evaluation with gas
// is this function's operations: a pow costs some 250 and a body needs three to
// five, one division or root 12 to 25.  So the lanes of a quad take one power
// each, of the cylindrical radius for the scale height, the density and eta and
// of the spherical one for the mean free path; exponents in quarters go without
// pow; and the circular velocity is (-y, x) sqrt(mu / rc^3).  The relative error
// of the drag against 80 bits over 0.5 to 3 AU, most of it cancellation in the
// velocity against the gas, is 1.6e-14 rms (before: 1.8e-14).  A call rather
// than inlined code, whose constants would be held through the loop.
__device__ __attribute__((noinline)) double quad_drag(const QUAD_LDS QGas *c, double factor, double base, double over_rc3,
                                                      double x, double y, double z, double vx, double vy, double vz)
{
    const int l = threadIdx.x & 3, place = threadIdx.x >> 2;
    const double idx = c->idx[l], R = c->R[place];
    const double rc = dpp_mov<0x00>(base), r = dpp_mov<0xAA>(base);
    const double r1 = sqrt(base);
    // as pl() in gasdev.h: the exponents 1 and 1/2 (and here all quarters) without pow
    double p = idx == 1.0 ? base : r1;
    if (c->by_quarters) p = quad_quarters(base, r1, c->quarters[l]);
    else if (idx != 1.0 && idx != 0.5) p = pow(base, idx);
    const double h = c->g.sh_c * dpp_mov<0x00>(p), rho_p = dpp_mov<0x55>(p);
    const double lambda = c->g.mfp_c * dpp_mov<0xAA>(p), eta = c->g.eta_c * dpp_mov<0xFF>(p);
    const double s = (rc > 0.0 ? sqrt(over_rc3) : 0.0) * sqrt(1.0 - 2.0 * eta);
    const double ux = vx + y * s, uy = vy - x * s, uz = vz;
    const double w = exp(-SQR(z / h));
    const double rho = factor * (c->g.inner_edge < rc ? c->g.rho_c * rho_p * w : c->edge * SQR(SQR(rc)) * w);
    double C;
    if (R <= 0.1 * lambda) {                                  // Epstein
        C = c->ge[place] * (c->thermal * sqrt(r)) * rho;
    } else if (R >= 10.0 * lambda) {                          // Stokes
        C = c->gs[place] * sqrt(ux * ux + uy * uy + uz * uz) * rho;
    } else {                                                    // transition
        const double l1 = 0.1 * lambda, l2 = 10.0 * lambda;
        const double ge = 1.0 / (c->rho_b[place] * l1);
        const double gsk = 3.0 / 8.0 * c->cd[place] / (c->rho_b[place] * l2);
        const double vth = c->thermal * sqrt(r);
        const double K = gsk * sqrt(ux * ux + uy * uy + uz * uz) / (ge * vth);
        // one logarithm and one power per lane again
        const double lg = log10(l & 1 ? l2 / l1 : K);
        const double kappa = dpp_mov<0x00>(lg) / dpp_mov<0x55>(lg);
        const double pk = l & 1 ? pow(R, kappa) : pow(l1, -kappa);
        C = ge * vth * dpp_mov<0x00>(pk) * dpp_mov<0x55>(pk) * rho;
    }
    return -C * (l == 0 ? ux : l == 1 ? uy : uz);
}

__device__ __attribute__((noinline)) void quad_migration(const GasDev &g, bool giant, double x, double y, double z,
                                                         double vx, double vy, double vz, double m, double mc,
                                                         double stop, int32_t &type, double t, double (&o)[3])
{
    migration_accel(giant, x, y, z, vx, vy, vz, m, mc, stop, type, g, 0, t, o[0], o[1], o[2]);
}

// The Driver loop.  Without gas a wave is on its own but for the exchange
// (its sources, its 16 - sources bodies, its records); with gas the workgroup
// is: the sources once, `own` bodies, a barrier per evaluation, and the stages
// in a loop with their derivatives in LDS, as the drag is too long to unroll.
template <int INTEG, int NA, bool GAS>
__device__ __forceinline__ void quad_run(const QuadArgs &A, int max_steps, double *columns, QGas *gas)
{
    constexpr int kWaves = GAS ? 4 * kQuadGasBodies / kWave : kQuadWaves;
    __shared__ __attribute__((aligned(16))) double records[GAS ? 2 : kQuadWaves][4 * NA][GAS ? 8 : 4];
    __shared__ double sh_max[2][kWaves], sh_val;
    __shared__ int sh_any[2][kWaves], sh_ev, sh_ok;
    constexpr int nst = q_stages<INTEG>();
    const int nwaves = GAS ? (int)blockDim.x / kWave : kQuadWaves;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = uniform(tid / kWave);
    const int quad = (GAS ? tid : lane) >> 2, l = lane & 3, comp = l < 3 ? l : 2;
    const int ns = A.sources;
    const int unit = GAS ? (int)blockIdx.x : (int)blockIdx.x * kQuadWaves + wave;   // that has the sources once
    ResSystem S = A.system_in;
    const int n = S.n;
    int i = quad < ns ? 1 + quad : 1 + ns + unit * A.own + (quad - ns);
    const bool valid = i < n && quad - ns < A.own;
    if (!valid) i = 1;         // the first source once more; nothing of it is kept
    const bool keeps = valid && (quad >= ns || unit == 0);
    const int src = quad < ns && l < 3 ? 1 + quad : 0;
    double (*tab)[GAS ? 8 : 4] = records[GAS ? 0 : wave];
    if (GAS) {
        for (int k = tid; k < 2 * 4 * NA * 8; k += (int)blockDim.x) (&records[0][0][0])[k] = 0.0;
        __syncthreads();
    } else {
        tab[quad < 4 * NA ? quad : 0][l] = 0.0;     // 16 quads, at most 12 records
    }

    QPulls<NA> P;
    {
        const int end = i < S.nm ? S.end_a : S.end_b;
        P.mu = kGauss2 * (A.mass[0] + A.mass[i]);
#pragma unroll
        for (int a = 0; a < 4 * NA; ++a) P.w[a] = a >= 1 && a <= ns && a < end && a != i ? A.gm[a] : 0.0;
#pragma unroll
        for (int t = 0; t < NA; ++t) {
            const int a = l + 4 * t;
            P.slot[t] = a <= ns ? a : 0;
            P.near[t] = a >= 1 && a <= ns && a < end && a != i;
        }
    }
    QBody<INTEG, GAS> B;
    if constexpr (GAS) { B.d.col = (QUAD_LDS double *)columns + tid; B.d.stride = (int)blockDim.x; }
    B.p = B.po = A.y0_in[comp * A.tot + i];
    B.v = B.vo = A.y0_in[(3 + comp) * A.tot + i];
    B.sp = B.sv = B.ep = B.ev = 0.0;
    B.d.clear();
    QSide side{0.0, 0.0, 0}, none;
    const bool events = quad_events(S);
    const bool combine = INTEG != INTEG_RK4 || events;
    bool flushed = false;      // small numbers were flushed in this launch
    int x = 0;                 // exchanges

    // Gas: the drag body's parameters, the migration of a massive one (types
    // and accelerations are this thread's until the end).
    bool drags = false;
    double mig = 0.0, mig_next = 0.0, drag = 0.0, migc = 0.0;
    int32_t mt = 0, mt_next = 0;
    bool migrates = false, giant = false, fresh = false, fresh_next = false;
    const double m0 = A.mass[0];
    if constexpr (GAS) {
        drags = i >= S.drag_lo && i < S.drag_hi;
        const GasDev &g = A.gas;
        if (tid == 0) {
            // MeanThermalSpeed_CMU and Temperature_CMU, as gas_drag in gasdev.h
            const double kb = 1.3806488e-23 * ((1.0 / 1.98911e30) * SQR(1.0 / 1.495978707e11)) / SQR(1.0 / 86400.0);
            const double mp = 1.672621777e-27 * (1.0 / 1.98911e30);
            const double cvth = sqrt((8.0 * kb) / (3.14159265358979323846 * g.mmw * mp));
            const double ctp = kGauss2 * (1.0 / (kb / mp));
            gas->g = g;
            gas->edge = g.rho_c * pow(g.inner_edge, g.rho_i - 4.0);
            gas->thermal = cvth * sqrt(SQR(g.sh_c) * g.mmw * ctp * pow(m0, 2.0 * g.sh_i - 3.0));
            gas->idx[0] = g.sh_i; gas->idx[1] = g.rho_i; gas->idx[2] = g.mfp_i; gas->idx[3] = g.eta_i;
            gas->by_quarters = 1;
            for (int k = 0; k < 4; ++k) {
                const double v = 4.0 * gas->idx[k];
                const bool whole = fabs(v) <= 16.0 && v == trunc(v);
                gas->quarters[k] = whole ? (int)v : 0;
                if (!whole) gas->by_quarters = 0;
            }
        }
        if (l == 0) {
            gas->R[quad] = A.radius[i]; gas->rho_b[quad] = A.density[i]; gas->cd[quad] = A.cd[i];
            gas->gs[quad] = A.gs[i]; gas->ge[quad] = A.ge[i];
        }
        __syncthreads();
        mt = A.migt_in[i];
        migc = A.migc_in[comp * A.tot + i];
        giant = i < S.giant_end;
        migrates = i >= S.mig_lo && i < S.nm && (giant ? A.mig_do2 : A.mig_do1) != 0;
    }
    // Migration of the Driver's first evaluation at (pos, vel, t) for this
    // thread's component; type: the body's, which it may end.
    auto migration = [&](double t, double pos, double vel, int32_t &type, bool &is) -> double {
        is = migrates && type == (giant ? SOL_MIGRATION_TYPE_II : SOL_MIGRATION_TYPE_I);
        double o[3] = {0.0, 0.0, 0.0};
        if (is)
            quad_migration(gas->g, giant, dpp_mov<0x00>(pos), dpp_mov<0x55>(pos), dpp_mov<0xAA>(pos), dpp_mov<0x00>(vel),
                           dpp_mov<0x55>(vel), dpp_mov<0xAA>(vel), A.mass[i], m0, A.stop[i], type, t, o);
        return l == 0 ? o[0] : l == 1 ? o[1] : o[2];
    };
    // Acceleration at (pos, vel) with the gas's factor and the migration m.
    // first: a step's first evaluation (as in quad_force), last: its last.
    auto accelerate = [&](auto first, bool last, double pos, double vel, double factor, double m, QSide &sd) -> double {
        if constexpr (GAS) {
            const QGasPlace W = quad_publish<decltype(first)::value>(tab, src, l, pos, kGauss2 * m0);
            auto resist = [&] {
                if (drags)
                    drag = quad_drag((const QUAD_LDS QGas *)gas, factor, W.base, W.over_rc3, W.x, W.y, W.z,
                                     dpp_mov<0x00>(vel), dpp_mov<0x55>(vel), dpp_mov<0xAA>(vel));
            };
            // the drag before the barrier hides its wait (505 bodies, us per attempt: Dormand-Prince 24.7 and
            // 23.7, RK4 11.7 and 11.0); in RKF78 its call would hold too much (16,389 bodies 38.5 and 41.1)
            if constexpr (INTEG != INTEG_RKF78) resist();
            __syncthreads();
            const double f = quad_force_gas<NA>(P, tab, ns, l, pos, W, last, sd);
            if constexpr (INTEG == INTEG_RKF78) resist();
            tab = tab == records[0] ? records[1] : records[0];
            return (drags ? f + drag : f) + m;
        }
        return 0.0;
    };

    // f0 of the next step: the acceleration at (p, v)
    double f0 = 0.0;
    bool again = GAS;          // with gas f0 is formed at the step's start: the first one, and after a flush
    if constexpr (!GAS) f0 = quad_force<NA, false, true>(P, tab, ns, src, l, B.p, none);

    for (int step = 0; step < max_steps; ++step) {
        const double t0 = S.t;
        double h = S.h_next, errmax = 0.0;
        int iter = 0, outcome = 0;             // outcome: 0 accept, 2 underflow, 3 maxiter
        bool event = false;
        if constexpr (GAS) {
            if (again) {
                mt_next = mt;
                mig_next = migration(t0, B.p, B.v, mt_next, fresh_next);
                f0 = accelerate(std::true_type(), false, B.p, B.v, reduction_factor(A.gas, t0), mig_next, none);
                again = false;
            }
            mig = mig_next;
            mt = mt_next;
            fresh = fresh_next;
            if (fresh) migc = mig;
        }
        B.d.put(0, B.v, f0);
        if (INTEG == INTEG_RKF78) {
            B.sp = fabs(B.p) + fabs(h * B.v) + 1.0e-30;
            B.sv = fabs(B.v) + fabs(h * f0) + 1.0e-30;
        }
        double pos, vel;
        for (;;) {
            ++iter;
            double last_drag = 0.0;
            if constexpr (GAS) {
                for (int q = 1; q <= nst; ++q) {
                    static_for<1, nst + 1>([&](auto T) {
                        if (q == T) quad_stage<INTEG, T>(B, h, pos, vel);
                    });
                    // RK4 and Dormand-Prince pass t + c h, RKF78 passes t to every stage
                    double ts = t0;
                    if (INTEG != INTEG_RKF78)
                        static_for<1, nst + 1>([&](auto T) {
                            if (q == T) ts = t0 + (INTEG == INTEG_RK4 ? tab::kRk4C[T < 4 ? T : 0] : tab::kDpC[T < 9 ? T : 0]) * h;
                        });
                    const double f = accelerate(std::false_type(), q == nst, pos, vel, reduction_factor(A.gas, ts), mig, side);
                    B.d.put(q, vel, f);
                }
                last_drag = drag;
            } else {
                static_for<1, nst + 1>([&](auto T) {
                    quad_stage<INTEG, T>(B, h, pos, vel);
                    if constexpr (T < nst) B.d.put(T, vel, quad_force<NA, false, false>(P, tab, ns, src, l, pos, none));
                    else B.d.put(T, vel, quad_force<NA, true, false>(P, tab, ns, src, l, pos, side));
                });
            }
            const double ratio = quad_final<INTEG>(B, h, pos, vel);
            double raw = 0.0;
            // f0 of the next step, should this one be accepted
            auto next_f0 = [&]() {
                if constexpr (GAS) {
                    const double tn = t0 + h;
                    mt_next = mt;
                    mig_next = migration(tn, pos, vel, mt_next, fresh_next);
                    f0 = accelerate(std::true_type(), false, pos, vel, reduction_factor(A.gas, tn), mig_next, none);
                    drag = last_drag;
                } else {
                    f0 = quad_force<NA, false, true>(P, tab, ns, src, l, pos, none);
                }
            };
            if (combine) {
                ++x;
                // the side outputs' events and the workgroup's error maximum
                int ev = 0;
                if (events && valid && l == 0) {
                    if (S.e3 > 0.0 && side.rm3 < S.e3) ev = 1;
                    if (S.h3 > 0.0 && side.rm3 > S.h3) ev = 1;
                    if (S.coll > 0.0 && side.best < DBL_MAX &&
                        S.coll * (A.radius[i] + A.radius[side.idx]) > sqrt(side.best))
                        ev = 1;
                }
                const double m = quad_wmax(valid ? ratio : 0.0);
                ev = __any(ev) ? 1 : 0;
                const int par = x & 1;
                if (lane == 0) { sh_max[par][wave] = m; sh_any[par][wave] = ev; }
                __syncthreads();
                double g = sh_max[par][0];
                int any = sh_any[par][0];
                for (int w = 1; w < nwaves; ++w) { g = fmax(g, sh_max[par][w]); any |= sh_any[par][w]; }
                unsigned long long *mw = A.sync->words[x & 1][0], *lw = A.sync->words[x & 1][1];
                if (tid == 0 && A.groups > 1) {
                    // a NaN has its sign bit cleared and is passed over below
                    const unsigned long long e = (unsigned long long)__double_as_longlong(fabs(g));
                    const unsigned long long tag = (unsigned long long)((uint32_t)x | (any ? 0x80000000u : 0u)) << 32;
                    __hip_atomic_store(mw + blockIdx.x, tag | (e >> 32), __ATOMIC_RELAXED, QUAD_SCOPE);
                    __hip_atomic_store(lw + blockIdx.x, tag | (e & 0xffffffffull), __ATOMIC_RELAXED, QUAD_SCOPE);
                }
                next_f0();             // meanwhile
                if (A.groups > 1 && wave == 0) {
                    constexpr int kPolls = kQuadMaxGroups / kWave;
                    const uint64_t c0 = __builtin_amdgcn_s_memrealtime();
                    bool ok = true;
                    unsigned long long a[kPolls], b[kPolls];
                    for (int it = 0;; ++it) {
                        bool here = true;
#pragma unroll
                        for (int k = 0; k < kPolls; ++k)
                            if (k * kWave < A.groups) {
                                a[k] = __hip_atomic_load(mw + k * kWave + lane, __ATOMIC_RELAXED, QUAD_SCOPE);
                                b[k] = __hip_atomic_load(lw + k * kWave + lane, __ATOMIC_RELAXED, QUAD_SCOPE);
                            }
#pragma unroll
                        for (int k = 0; k < kPolls; ++k)
                            if (k * kWave < A.groups)
                                here &= k * kWave + lane >= A.groups ||
                                        ((uint32_t)(a[k] >> 32 & 0x7fffffff) == (uint32_t)x &&
                                         (uint32_t)(b[k] >> 32 & 0x7fffffff) == (uint32_t)x);
                        if (__all(here) && A.ticks != 0) break;       // (no budget: never)
                        if ((it & 7) == 7 || A.ticks == 0) {
                            if (__hip_atomic_load(&A.sync->error, __ATOMIC_RELAXED, QUAD_SCOPE) != 0) { ok = false; break; }
                            if (__builtin_amdgcn_s_memrealtime() - c0 >= A.ticks) {
                                __hip_atomic_store(&A.sync->error, 1u, __ATOMIC_RELAXED, QUAD_SCOPE);
                                ok = false;
                                break;
                            }
                        }
                    }
                    g = 0.0;
                    any = 0;
#pragma unroll
                    for (int k = 0; k < kPolls; ++k)
                        if (k * kWave + lane < A.groups) {
                            g = fmax(g, __longlong_as_double((long long)(a[k] << 32 | (b[k] & 0xffffffffull))));
                            any |= (int)(a[k] >> 63);
                        }
                    g = quad_wmax(g);
                    any = __any(any) ? 1 : 0;
                    if (lane == 0) { sh_val = g; sh_ev = any; sh_ok = ok ? 1 : 0; }
                }
                if (A.groups > 1) {
                    __syncthreads();
                    if (uniform(sh_ok) == 0) {
                        if (tid == 0 && blockIdx.x == 0) A.system->status = RES_SYNC_ERROR;
                        return;
                    }
                    g = sh_val;
                    any = sh_ev;
                }
                raw = uniform(fabs(g));
                event = uniform(any) != 0;
            } else {
                next_f0();
            }
            S.attempts += 1;
            B.po = pos;                       // the attempt's final state, as the Driver's second array
            B.vo = vel;
            if (INTEG == INTEG_RKF78) {
                errmax = raw / S.eps;
                if (errmax < 1.0) { outcome = 0; break; }
                const double htemp = 0.9 * h * quad_pow(errmax, -0.25);
                h = fabs(htemp) > fabs(0.1 * h) ? htemp : 0.1 * h;
                if (t0 + h == t0) { outcome = 2; break; }
            } else if (INTEG == INTEG_RK4) {
                outcome = 0;
                break;
            } else {
                errmax = raw;
                const double hn = errmax < 1.0e-20 ? 2.0 * h : 0.9 * h * quad_pow(S.eps / errmax, 1.0 / 7.0);
                S.h_did = h;
                S.h_next = hn;
                if (!(errmax > S.eps && iter <= 10)) { outcome = iter > 10 ? 3 : 0; break; }
                h = hn;
            }
            // again with the new h; a non-finite derivative of this attempt
            // meets no coefficient, the zero ones are left out
        }
        if (outcome != 0) {
            S.status = outcome == 2 ? RES_UNDERFLOW : RES_MAXITER;
            S.body_h = h;
            break;
        }
        double h_next;
        if (INTEG == INTEG_RKF78) {
            h_next = errmax > 1.89e-4 ? (0.9 * h * quad_pow(errmax, -0.2)) : (5.0 * h);
        } else if (INTEG == INTEG_RK4) {
            h_next = h;
        } else {
            h_next = S.h_next;
            h = S.h_did;
        }
        // the Driver's pointer swap
        B.po = B.p;
        B.vo = B.v;
        B.p = pos;
        B.v = vel;
        bool stop = false, flush = false;
        int reason = 0;
        S.h_did = h;
        S.t = t0 + h;
        S.h_next = h_next;
        S.body_h = INTEG == INTEG_DP ? h : h_next;
        S.steps += 1;
        if (S.clip) {
            // Simulator::DecisionMaking, Solaris/Simulator.cpp:183-245
            S.elapsed += h;
            S.last_save += h;
            S.last_nsteps += h;
            if (event) reason |= SOL_STOP_EVENT;
            const double actual = 1000.0 * 365.25 * S.millenium + S.t;
            if (fabs(actual) >= fabs(S.length)) {
                stop = true;
            } else {
                if (fabs(actual + S.h_next) > fabs(S.length)) S.h_next = S.length - actual;
                if (fabs(S.last_save) >= fabs(S.output)) {
                    S.last_save = 0.0;
                    reason |= SOL_STOP_OUTPUT;
                }
                if (fabs(S.last_save + S.h_next) > fabs(S.output)) S.h_next = S.output - S.last_save;
            }
            S.flush_count = (S.flush_count + 1) % 100;
            flush = S.flush_count == 0;
            S.reason = reason | (stop ? SOL_STOP_END : 0);
            reason &= S.stop_mask;
        }
        if (stop || reason) S.status = stop ? RES_DONE : RES_STOPPED;
        if (flush) {
            flushed = true;
            if (fabs(B.p) < 1.0e-50) B.p = 0.0;
            if (fabs(B.v) < 1.0e-50) B.v = 0.0;
            if (fabs(B.po) < 1.0e-50) B.po = 0.0;
            if (fabs(B.vo) < 1.0e-50) B.vo = 0.0;
            if constexpr (GAS) again = true;
            else f0 = quad_force<NA, false, true>(P, tab, ns, src, l, B.p, none);
        }
        if (S.status != RES_RUNNING) break;
    }

    if (keeps && l < 3) {
        const int64_t p = comp * A.tot + i, v = p + 3 * A.tot;
        A.y0[p] = B.p;
        A.y0[v] = B.v;
        A.y[p] = B.po;
        A.y[v] = B.vo;
        A.acc0[p] = B.d.V(0);
        A.acc0[v] = B.d.F(0);
        if constexpr (GAS) {
            A.migc[p] = migc;
            A.dragc[p] = drag;
        }
        if (INTEG == INTEG_RKF78) { A.yscale[p] = B.sp; A.yscale[v] = B.sv; }
        if (INTEG != INTEG_RK4) { A.err[p] = B.ep; A.err[v] = B.ev; }
    }
    if (keeps && l == 0) {
        if constexpr (GAS) A.migt[i] = mt;
        const bool has = side.best < DBL_MAX;
        A.rm3[i] = side.rm3;
        A.nnd[i] = has ? sqrt(side.best) : 0.0;
        A.nni[i] = has ? side.idx : -1;
    }
    if (blockIdx.x == 0) {
        // the star is not integrated: no derivative, no error, no neighbour
        if (tid < 6) {
            const int64_t o = tid * A.tot;
            const double v = A.y0_in[o], w = flushed && fabs(v) < 1.0e-50 ? 0.0 : v;
            A.y0[o] = w;
            A.y[o] = w;
            A.acc0[o] = 0.0;
            if (INTEG == INTEG_RKF78) A.yscale[o] = fabs(v) + 1.0e-30;
            if (INTEG != INTEG_RK4) A.err[o] = 0.0;
        }
        if (tid == 0) {
            if constexpr (GAS) A.migt[0] = A.migt_in[0];
            A.rm3[0] = 0.0;
            A.nnd[0] = 0.0;
            A.nni[0] = -1;
            *A.system = S;
        }
    }
}

template <int INTEG, int NA>
__global__ __launch_bounds__(kQuadThreads) void k_quad(QuadArgs A, int max_steps)
{
    quad_run<INTEG, NA, false>(A, max_steps, nullptr, nullptr);
}

template <int INTEG, int NA>
__global__ __launch_bounds__(4 * kQuadGasBodies) void k_quad_gas(QuadArgs A, int max_steps)
{
    extern __shared__ __attribute__((aligned(16))) double quad_columns[];
    __shared__ QGas gas;
    quad_run<INTEG, NA, true>(A, max_steps, quad_columns, &gas);
}

__global__ __launch_bounds__(kQuadMaxGroups) void k_quad_zero(QuadSync *s)
{
    if (threadIdx.x == 0) s->error = 0;
    s->words[0][0][threadIdx.x] = s->words[0][1][threadIdx.x] = 0ull;
    s->words[1][0][threadIdx.x] = s->words[1][1][threadIdx.x] = 0ull;
}

template <int INTEG>
const void *quad_kernel_of(int sources)
{
    return sources <= 3   ? (const void *)k_quad<INTEG, 1>
           : sources <= 7 ? (const void *)k_quad<INTEG, 2>
                          : (const void *)k_quad<INTEG, 3>;
}

template <int INTEG>
const void *quad_gas_kernel_of(int sources)
{
    return sources <= 3   ? (const void *)k_quad_gas<INTEG, 1>
           : sources <= 7 ? (const void *)k_quad_gas<INTEG, 2>
                          : (const void *)k_quad_gas<INTEG, 3>;
}

const void *quad_kernel(int integ, int sources, bool gas)
{
    return integ == INTEG_RKF78 ? (gas ? quad_gas_kernel_of<INTEG_RKF78>(sources) : quad_kernel_of<INTEG_RKF78>(sources))
         : integ == INTEG_RK4   ? (gas ? quad_gas_kernel_of<INTEG_RK4>(sources) : quad_kernel_of<INTEG_RK4>(sources))
                                : (gas ? quad_gas_kernel_of<INTEG_DP>(sources) : quad_kernel_of<INTEG_DP>(sources));
}

size_t column_bytes(int integ, int places)
{
    const int rows = integ == INTEG_RKF78 ? q_rows<INTEG_RKF78>()
                   : integ == INTEG_RK4   ? q_rows<INTEG_RK4>() : q_rows<INTEG_DP>();
    return quad_column_bytes(rows, 4 * places);
}

}  // namespace

int quad_groups(int n, int sources, int cus)
{
    if (sources < 1 || sources > kQuadMaxSources) return 0;
    const int own = kQuads - sources;
    const int waves = std::max(1, (n - 1 - sources + own - 1) / own);
    const int groups = (waves + kQuadWaves - 1) / kQuadWaves;
    return groups <= std::min(cus, kQuadMaxGroups) ? groups : 0;
}

int quad_capacity(int integ, int sources, int cu_count)
{
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, quad_kernel(integ, sources, false), kQuadThreads, 0) !=
        hipSuccess)
        return 0;
    return per_cu * cu_count;
}

int quad_gas_capacity(int integ, int sources, int places, int cu_count)
{
    const void *f = quad_kernel(integ, sources, true);
    int per_cu = 0;
    // (the attribute for the most places, so that it holds for every launch)
    if (sources < 1 || sources > kQuadMaxSources || places <= sources || places > kQuadGasBodies ||
        hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)column_bytes(integ, kQuadGasBodies)) !=
            hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, 4 * places, column_bytes(integ, places)) != hipSuccess)
        return 0;
    return per_cu * cu_count;
}

bool quad_exchanges(int integ, const QuadArgs &a)
{
    return a.groups > 1 && (integ != INTEG_RK4 || quad_events(a.system_in));
}

hipError_t launch_quad(hipStream_t st, int integ, const QuadArgs &a, int max_steps)
{
    if (a.groups < 1 || a.groups > kQuadMaxGroups || a.sources < 1 || a.sources > kQuadMaxSources ||
        a.own != kQuads - a.sources)
        return hipErrorInvalidValue;
    if (quad_exchanges(integ, a))
        hipLaunchKernelGGL(k_quad_zero, dim3(1), dim3(kQuadMaxGroups), 0, st, a.sync);
    QuadArgs args = a;
    void *kargs[] = {&args, &max_steps};
    return hipLaunchKernel(quad_kernel(integ, a.sources, false), dim3(a.groups), dim3(kQuadThreads), kargs, 0, st);
}

hipError_t launch_quad_gas(hipStream_t st, int integ, const QuadArgs &a, int places, int max_steps)
{
    if (a.groups < 1 || a.groups > kQuadMaxGroups || a.sources < 1 || a.sources > kQuadMaxSources || a.own < 1 ||
        a.sources + a.own > places || places > kQuadGasBodies || places % kQuads != 0)
        return hipErrorInvalidValue;
    if (quad_exchanges(integ, a))
        hipLaunchKernelGGL(k_quad_zero, dim3(1), dim3(kQuadMaxGroups), 0, st, a.sync);
    QuadArgs args = a;
    void *kargs[] = {&args, &max_steps};
    return hipLaunchKernel(quad_kernel(integ, a.sources, true), dim3(a.groups), dim3(4 * places), kargs,
                           column_bytes(integ, places), st);
}

}  // namespace sol
