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
//   pulls       lane l takes the pulls of bodies l, l + 4, ... (the star, body
//               0, as a source at the origin with weight k^2 (m0 + mi)), and
//               each source's indirect term with its direct one; the sums are
//               reduced over the quad so that lane c (c < 3) has component c;
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
// and after, us: RKF78 of 4 bodies 15.2 and 5.4, 515 17.6 and 5.6, 5,001 18.6
// and 6.1, 14,338 20.4 and 6.9; Dormand-Prince of 515 13.9 and 4.9; RK4 of 515
// 4.4 and 1.2.  An evaluation of 85 to 100 instructions takes 0.28 us, the
// exchange 1.9 us.
#include <float.h>

#include <algorithm>

#include "lane_pairs.h"
#include "quad.h"
#include "static_for.h"
#include "tableaux.h"

namespace sol {
namespace {

#define QUAD_SCOPE __HIP_MEMORY_SCOPE_SYSTEM

constexpr int kQuadWaves = kQuadThreads / kWave;
constexpr int kQuads = kWave / 4;

template <int INTEG>
constexpr int q_stages() { return INTEG == INTEG_RKF78 ? 12 : INTEG == INTEG_RK4 ? 3 : 8; }

// A call rather than inlined code: its registers would be held through the stages.
__device__ __attribute__((noinline)) double quad_pow(double x, double y) { return pow(x, y); }

__device__ __forceinline__ double quad_wmax(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmax(v, __shfl_xor(v, o, kWave));
    return v;
}

// What a lane needs for the pulls on its body: NA of them, l, l + 4, ...
template <int NA>
struct QPulls {
    double w[NA], u[NA];       // weights of the direct and the indirect term (0: not a source of this body)
    int slot[NA];              // the source's record
    bool near[NA];             // a candidate for the nearest neighbour
};

// |d|^-3 from r2 = |d|^2: the hardware's reciprocal square root and its
// second-order correction.  Its cap is above 1 / |d| of any two distinct
// bodies, so that a body's own record and the star's indirect term (d = 0)
// come out as exactly 0.
__device__ __forceinline__ double quad_rm3(double r2, double c15, double c1875)
{
    const double y = fmin(__builtin_amdgcn_rsq(r2), 1.0e50);
    const double tt = y * y;
    const double e = __builtin_fma(-r2, tt, 1.0);
    const double y3 = tt * y;
    return __builtin_fma(y3, e * __builtin_fma(c1875, e, c15), y3);
}

// Side outputs of a body: 1 / |r|^3 (lane 0), distance squared and index of
// the nearest source.
struct QSide {
    double rm3, best;
    int idx;
};

// Acceleration component of this lane for the position whose component it
// holds.  tab: the wave's source records (x, y, z), [0] the origin.
template <int NA, bool SIDE>
__device__ __forceinline__ double quad_force(const QPulls<NA> &P, double (*tab)[4], int src, int l, double pos,
                                             QSide &side)
{
    if (src > 0) tab[src][l] = pos;
    const double x = dpp_mov<0x00>(pos), y = dpp_mov<0x55>(pos), z = dpp_mov<0xAA>(pos);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const double c15 = 1.5, c1875 = 1.875;
    double f[3] = {0.0, 0.0, 0.0};
    if (SIDE) { side.best = DBL_MAX; side.idx = 0x7fffffff; }
#pragma unroll
    for (int t = 0; t < NA; ++t) {
        const double *r = tab[P.slot[t]];
        const double rx = r[0], ry = r[1], rz = r[2];
        const double dx = rx - x, dy = ry - y, dz = rz - z;
        const double d2 = dx * dx + dy * dy + dz * dz;
        const double s2 = rx * rx + ry * ry + rz * rz;
        const double wd = quad_rm3(d2, c15, c1875), ws = quad_rm3(s2, c15, c1875);
        const double g = P.w[t] * wd, k = P.u[t] * ws;
        f[0] += g * dx - k * rx;
        f[1] += g * dy - k * ry;
        f[2] += g * dz - k * rz;
        if (SIDE) {
            if (t == 0) side.rm3 = wd;          // lane 0: the star
            if (P.near[t] && d2 < side.best) { side.best = d2; side.idx = P.slot[t]; }
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // lanes 0, 1 keep components 0, 1 and lanes 2, 3 component 2
    const bool hi = l >= 2;
    const double a = (hi ? f[2] : f[0]) + dpp_mov<0x4E>(hi ? f[0] : f[2]);
    const double b = f[1] + dpp_mov<0x4E>(f[1]);
    const double keep = l == 1 ? b : a, send = l == 0 ? b : a;
    if (SIDE) {
        // the smaller index of equals
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
    return keep + dpp_mov<0xB1>(send);
}

// One component of a body: state, previous state, stage derivatives
// (velocities V, accelerations F), scale and error.
struct QBody {
    double p, v, po, vo;
    double V[13], F[13];
    double sp, sv, ep, ev;
};

// State of stage S in tableau order, as resident.hip's stage_state.
template <int INTEG, int S>
__device__ __forceinline__ void quad_stage(const QBody &B, double h, double &pos, double &vel)
{
    if constexpr (INTEG == INTEG_DP) {
        double var = tab::kDpA[S][0] * B.F[0];
        static_for<1, S>([&](auto L) {
            if constexpr (tab::kDpA[S][L] != 0.0) var += tab::kDpA[S][L] * B.F[L];
        });
        pos = B.p + tab::kDpC[S] * h * B.v + h * h * (var);
        vel = B.v + h * (var);
    } else {
        double ap = 0.0, av = 0.0;
        bool first = true;
        static_for<0, S>([&](auto L) {
            constexpr double d = INTEG == INTEG_RKF78 ? tab::kRkfD[S][L] : tab::kRk4A[S][L];
            if constexpr (d != 0.0) {
                const double x = d * B.V[L], y = d * B.F[L];
                ap = first ? x : ap + x;
                av = first ? y : av + y;
                first = false;
            }
        });
        pos = B.p + h * ap;
        vel = B.v + h * av;
    }
}

// Final state and error estimate (kept in B); returns this lane's part of the
// error maximum.
template <int INTEG>
__device__ __forceinline__ double quad_final(QBody &B, double h, double &pos, double &vel)
{
    if constexpr (INTEG == INTEG_RKF78) {
        constexpr double b0 = 41.0 / 840.0, b5 = 34.0 / 105.0, b6 = 9.0 / 35.0, b8 = 9.0 / 280.0, b10 = 41.0 / 840.0;
        auto sum = [&](const double *F) {
            return b0 * F[0] + b5 * F[5] + b6 * (F[6] + F[7]) + b8 * (F[8] + F[9]) + b10 * F[10];
        };
        pos = B.p + h * sum(B.V);
        vel = B.v + h * sum(B.F);
        B.ep = h * fabs(B.V[0] + B.V[10] - B.V[11] - B.V[12]) * 41.0 / 840.0;
        B.ev = h * fabs(B.F[0] + B.F[10] - B.F[11] - B.F[12]) * 41.0 / 840.0;
        return fmax(fabs(B.ep / B.sp), fabs(B.ev / B.sv));
    } else if constexpr (INTEG == INTEG_RK4) {
        auto sum = [&](const double *F) {
            return tab::kRk4B[0] * F[0] + tab::kRk4B[1] * F[1] + tab::kRk4B[2] * F[2] + tab::kRk4B[3] * F[3];
        };
        pos = B.p + h * sum(B.V);
        vel = B.v + h * sum(B.F);
        return 0.0;
    } else {
        constexpr const double *b = tab::kDpB, *d = tab::kDpBdh;
        const double *F = B.F;
        const double h2 = h * h;
        pos = B.p + h * B.v + h2 * (b[0] * F[0] + b[4] * F[4] + b[5] * F[5] + b[6] * F[6] + b[7] * F[7] + b[8] * F[8]);
        vel = B.v + h * (d[0] * F[0] + d[4] * F[4] + d[5] * F[5] + d[6] * F[6] + d[7] * F[7]);
        B.ep = h2 * fabs(F[7] - F[8]) / 20.0;
        B.ev = 0.0;
        return B.ep;
    }
}

template <int INTEG, int NA>
__global__ __launch_bounds__(kQuadThreads) void k_quad(QuadArgs A, int max_steps)
{
    __shared__ __attribute__((aligned(16))) double records[kQuadWaves][4 * NA][4];
    __shared__ double sh_max[2][kQuadWaves], sh_val;
    __shared__ int sh_any[2][kQuadWaves], sh_ev, sh_ok;
    constexpr int nst = q_stages<INTEG>();
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = uniform(tid / kWave);
    const int quad = lane >> 2, l = lane & 3, comp = l < 3 ? l : 2;
    const int ns = A.sources, mine = kQuads - ns;
    const int gw = (int)blockIdx.x * kQuadWaves + wave;
    ResSystem S = *A.system_in;
    if (S.status != RES_RUNNING) return;      // the same in every workgroup

    const int n = S.n;
    int i = quad < ns ? 1 + quad : 1 + ns + gw * mine + (quad - ns);
    const bool valid = i < n;
    if (!valid) i = 1;         // the first source once more; nothing of it is kept
    const bool keeps = valid && (quad >= ns || gw == 0);
    const int src = quad < ns && l < 3 ? 1 + quad : 0;
    double (*tab)[4] = records[wave];
    tab[lane >> 2 < 4 * NA ? lane >> 2 : 0][l] = 0.0;     // 16 quads, at most 12 records

    QPulls<NA> P;
    {
        const int end = i < S.nm ? S.end_a : S.end_b;
#pragma unroll
        for (int t = 0; t < NA; ++t) {
            const int a = l + 4 * t;
            const bool is = a >= 1 && a <= ns && a < end && a != i;
            P.slot[t] = a <= ns ? a : 0;
            P.u[t] = is ? A.gm[a] : 0.0;
            P.w[t] = a == 0 ? kGauss2 * (A.mass[0] + A.mass[i]) : P.u[t];
            P.near[t] = is;
        }
    }
    QBody B;
    B.p = B.po = A.y0_in[comp * A.tot + i];
    B.v = B.vo = A.y0_in[(3 + comp) * A.tot + i];
    B.sp = B.sv = B.ep = B.ev = 0.0;
    static_for<0, 13>([&](auto L) { B.V[L] = B.F[L] = 0.0; });
    QSide side{0.0, 0.0, 0}, none;
    const bool events = S.clip && (S.stop_mask & SOL_STOP_EVENT) && (S.e3 > 0.0 || S.h3 > 0.0 || S.coll > 0.0);
    const bool combine = INTEG != INTEG_RK4 || events;
    bool flushed = false;      // small numbers were flushed in this launch
    int x = 0;                 // exchanges
    // f0 of the next step: the acceleration at (p, v)
    double f0 = quad_force<NA, false>(P, tab, src, l, B.p, none);

    for (int step = 0; step < max_steps; ++step) {
        const double t0 = S.t;
        double h = S.h_next, errmax = 0.0;
        int iter = 0, outcome = 0;             // outcome: 0 accept, 2 underflow, 3 maxiter
        bool event = false;
        B.V[0] = B.v;
        B.F[0] = f0;
        if (INTEG == INTEG_RKF78) {
            B.sp = fabs(B.p) + fabs(h * B.V[0]) + 1.0e-30;
            B.sv = fabs(B.v) + fabs(h * B.F[0]) + 1.0e-30;
        }
        double pos, vel;
        for (;;) {
            ++iter;
            static_for<1, nst + 1>([&](auto T) {
                quad_stage<INTEG, T>(B, h, pos, vel);
                B.V[T] = vel;
                if constexpr (T < nst) B.F[T] = quad_force<NA, false>(P, tab, src, l, pos, none);
                else B.F[T] = quad_force<NA, true>(P, tab, src, l, pos, side);
            });
            const double ratio = quad_final<INTEG>(B, h, pos, vel);
            double raw = 0.0;
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
                for (int w = 1; w < kQuadWaves; ++w) { g = fmax(g, sh_max[par][w]); any |= sh_any[par][w]; }
                unsigned long long *mw = A.sync->words[x & 1][0], *lw = A.sync->words[x & 1][1];
                if (tid == 0 && A.groups > 1) {
                    // a NaN has its sign bit cleared and is passed over below
                    const unsigned long long e = (unsigned long long)__double_as_longlong(fabs(g));
                    const unsigned long long tag = (unsigned long long)((uint32_t)x | (any ? 0x80000000u : 0u)) << 32;
                    __hip_atomic_store(mw + blockIdx.x, tag | (e >> 32), __ATOMIC_RELAXED, QUAD_SCOPE);
                    __hip_atomic_store(lw + blockIdx.x, tag | (e & 0xffffffffull), __ATOMIC_RELAXED, QUAD_SCOPE);
                }
                // meanwhile f0 of the next step, should this one be accepted
                f0 = quad_force<NA, false>(P, tab, src, l, pos, none);
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
                f0 = quad_force<NA, false>(P, tab, src, l, pos, none);
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
            f0 = quad_force<NA, false>(P, tab, src, l, B.p, none);
        }
        if (S.status != RES_RUNNING) break;
    }

    if (keeps && l < 3) {
        const int64_t p = comp * A.tot + i, v = p + 3 * A.tot;
        A.y0[p] = B.p;
        A.y0[v] = B.v;
        A.y[p] = B.po;
        A.y[v] = B.vo;
        A.acc0[p] = B.V[0];
        A.acc0[v] = B.F[0];
        if (INTEG == INTEG_RKF78) { A.yscale[p] = B.sp; A.yscale[v] = B.sv; }
        if (INTEG != INTEG_RK4) { A.err[p] = B.ep; A.err[v] = B.ev; }
    }
    if (keeps && l == 0) {
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
            A.rm3[0] = 0.0;
            A.nnd[0] = 0.0;
            A.nni[0] = -1;
            *A.system = S;
        }
    }
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

const void *quad_kernel(int integ, int sources)
{
    return integ == INTEG_RKF78 ? quad_kernel_of<INTEG_RKF78>(sources)
         : integ == INTEG_RK4   ? quad_kernel_of<INTEG_RK4>(sources)
                                : quad_kernel_of<INTEG_DP>(sources);
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
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, quad_kernel(integ, sources), kQuadThreads, 0) !=
        hipSuccess)
        return 0;
    return per_cu * cu_count;
}

hipError_t launch_quad(hipStream_t st, int integ, const QuadArgs &a, int max_steps)
{
    if (a.groups < 1 || a.groups > kQuadMaxGroups || a.sources < 1 || a.sources > kQuadMaxSources)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_quad_zero, dim3(1), dim3(kQuadMaxGroups), 0, st, a.sync);
    QuadArgs args = a;
    void *kargs[] = {&args, &max_steps};
    return hipLaunchKernel(quad_kernel(integ, a.sources), dim3(a.groups), dim3(kQuadThreads), kargs, 0, st);
}

}  // namespace sol
