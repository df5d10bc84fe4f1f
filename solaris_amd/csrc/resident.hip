// resident.hip -- whole Driver loops of small systems inside one workgroup.
//
// One workgroup integrates one system (n <= kResidentMaxBodies bodies):
// the RKF78 / RK4 / Dormand-Prince Driver (Solaris/RungeKuttaFehlberg78.cpp:
// 66-140, Solaris/RungeKutta4.cpp:20-56, Solaris/DormandPrince.cpp:126-170),
// including the retry loop and the step-size arithmetic, and - when asked -
// the caller loop's step clipping and small-number flush
// (Simulator::DecisionMaking, Solaris/Simulator.cpp:159-245), all on the
// device.  A launch runs at most max_steps accepted steps per system and
// returns; the host relaunches until every system is done.  Systems are
// independent: a failing system (step-size underflow, too many retries)
// stops with its own status and the others go on.
//
// Within a system each thread owns bodies i = tid, tid + blockDim, ...
// (one, two or four of them).  The positions of the stage being evaluated
// are staged in LDS as (x, y, z, k^2 m) records, with r_j rm3_j records for
// the indirect term's sources; every sink reads them as a broadcast stream.
// Stage derivatives live in global memory ([stage][6][TOT] over all
// systems' bodies, TOT = sum of per-system padded counts) and are read
// back only by the thread that wrote them; y0 and the previous stage stay
// in registers, and for a single RKF78 system four derivatives stay in LDS
// too.  With a nebula (astrocentric), the drag of the drag bodies is added
// at every stage and the migration of the massive bodies is computed at
// the Driver's first evaluation and reused by its stages, as the
// multi-kernel path does (kernels instantiated with GAS).
//
// Grid form (k_resident_grid): a system with few sources and many sinks is
// split into slices, one workgroup each.  Every slice holds the sources
// ([0, src): the bodies every sink and every source reads) and its share of
// the sinks; the slices advance the sources with identical arithmetic, so
// they stay identical, and each attempt's error maximum and event flag are
// combined over the grid (GridSync) so that every slice takes the same
// decisions.  The launch holds no more slices than the device keeps
// resident at once; a wait that times out stops every slice with an error
// (the host then runs the call another way from its unchanged start).
#include <float.h>
#include <stdlib.h>

#include <type_traits>

#include "gasdev.h"
#include "sol_internal.h"
#include "resident.h"
#include "static_for.h"
#include "tableaux.h"

namespace sol {
namespace {

__device__ __forceinline__ double wmax(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmax(v, __shfl_xor(v, o, kWave));
    return v;
}

__device__ double block_max_all(double v, double *red, double *out)
{
    const int wid = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    const int nw = blockDim.x / kWave;
    v = wmax(v);
    if (lane == 0) red[wid] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = red[0];
        for (int q = 1; q < nw; ++q) m = fmax(m, red[q]);
        *out = m;
    }
    __syncthreads();
    return *out;
}

// pow of the step-size control, once per attempt.  Out of line: inlined,
// its polynomial constants are hoisted out of the step loop and spilled.
__device__ __attribute__((noinline)) double step_pow(double x, double y) { return pow(x, y); }

// Per-launch constants of the block's system, held in registers (the
// ResSystem fields would otherwise be re-read from memory after every
// barrier).
struct Ctx {
    const ResArrays *A;
    int n, base, nm, end_a, end_b, end_max;
    bool bc;
    int64_t tot;
    double4 *sJ;        // LDS: positions + k^2 m of the stage
    double4 *sT;        // LDS: r_j rm3_j of the indirect-term sources
    // gas: the system's body index of local body i is i (i < src) or
    // i + shift; drag on [drag_lo, drag_hi), Type II on [1, giant_end)
    int src, shift, drag_lo, drag_hi, giant_end;
    double m0;          // the central body's mass
    double tstage, factor;   // time of the stage being evaluated and the gas reduction factor there
    // body slot of this thread and slots per workgroup; lanes per body
    // 1 << lsh, this thread's lane among them `sub` (the lanes of a body
    // share its source loop and hold identical results after it)
    int me, nth, lsh, sub;
    // SPLIT with two lanes per body and every body a source of every other
    // (AC): the paired sum (pair_range2)
    bool pair2;
    // SPLIT: per-wave partial sums of the indirect term, [wave][6]: the
    // sources [1, end_a) in 0..2, [1, end_b) in 3..5
    double *part;
};

// the whole system's index of local body i
__device__ __forceinline__ int sys_index(const Ctx &c, int i) { return i < c.src ? i : i + c.shift; }

__device__ __forceinline__ double &at(double *p, const Ctx &c, int comp, int i) { return p[comp * c.tot + c.base + i]; }
__device__ __forceinline__ double cat(const double *p, const Ctx &c, int comp, int i) { return p[comp * c.tot + c.base + i]; }

// The own bodies' accesses go through a block-uniform array pointer plus a
// 32-bit per-lane byte offset, vb = 8 (k tot + base + i) for component k of
// body i, which the global load/store instructions add themselves: no
// per-lane 64-bit address has to be formed or kept for each array and
// stage.
__device__ __forceinline__ double ld(const double *p, uint32_t vb) { return *(const double *)((const char *)p + vb); }
__device__ __forceinline__ void st(double *p, uint32_t vb, double v) { *(double *)((char *)p + vb) = v; }

// Derivatives of stage l (0 = f0 in ACC0).
__device__ __forceinline__ double *stage(const Ctx &c, int l)
{
    return l == 0 ? c.A->acc0 : c.A->fst + (l - 1) * 6 * c.tot;
}

// Byte offsets of the six components of own body i.  The empty asm makes i
// opaque, so the offsets are formed here, next to their loads and stores,
// and not hoisted out of the step loop as one live 64-bit address per
// array, stage and component (which the 128 registers of a 1024-thread
// block cannot hold).
__device__ __forceinline__ void offsets(const Ctx &c, int i, uint32_t vb[6])
{
    asm volatile("" : "+v"(i));
#pragma unroll
    for (int k = 0; k < 6; ++k) vb[k] = (uint32_t)((k * c.tot + c.base + i) * 8);
}

template <int INTEG>
constexpr int n_stages() { return INTEG == INTEG_RKF78 ? 12 : INTEG == INTEG_RK4 ? 3 : 8; }

// Entry l of stage s of the first-order tableaux (RKF78 D, RK4 a).
template <int INTEG>
constexpr double dcoef(int s, int l) { return INTEG == INTEG_RKF78 ? tab::kRkfD[s][l] : tab::kRk4A[s][l]; }

// Own bodies of this thread: i = me + q * nth, q < BPT (me = threadIdx.x
// and nth = blockDim.x, or with L lanes per body threadIdx.x / L and
// blockDim.x / L).
__device__ __forceinline__ int own(const Ctx &c, int q) { return c.me + q * c.nth; }

// With one body per thread the state y0 and the previous stage's
// derivative stay in registers (Reg); with more, both are read back from
// memory.
//
// LF (one body per thread, where the LDS allows it): stage derivatives
// kept in LDS, each thread's in its own row of lds_stride<LF>() doubles, so
// that every slot and component is a fixed offset from one address.  The
// stride is odd, so a wave's 8-byte reads take the two LDS passes they need
// and no more.  LF = 4: the four most-read RKF78 derivatives, F0, F3, F4
// and F5 (32 of the 53 reads per component of an attempt); LF = 12: every
// derivative but the last stage's, which stays in registers (prev).
template <int BPT, int LF = 0>
struct Reg {
    static constexpr bool on = BPT == 1;
    static constexpr int lds_f = LF;
    double y0[BPT][6], prev[BPT][6];
    double *sF;   // LF: this thread's LDS row
};

template <int LF>
__host__ __device__ constexpr int lds_stride() { return 6 * LF + 1; }
// LDS slot of stage derivative L (-1: memory only)
template <int LF>
__host__ __device__ constexpr int lds_slot(int L)
{
    if constexpr (LF == 4) return L == 0 ? 0 : L == 3 ? 1 : L == 4 ? 2 : L == 5 ? 3 : -1;
    else if constexpr (LF == 12) return L < 12 ? L : -1;
    else return -1;
}

// v plus lane l's value moved by the DPP control CTRL (rows RM; lanes the
// move leaves out add 0), on the two halves of a double.
template <int CTRL, int RM>
__device__ __forceinline__ double dpp_add(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, RM, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, RM, 0xF, false);
    return v + __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Sum over the wave, in lane 63: quads (quad_perm 1,0,3,2 and 2,3,0,1),
// half rows (row_half_mirror), rows (row_mirror), then row 0 into row 1
// and row 2 into row 3 (row_bcast:15), rows 0-1 into rows 2-3
// (row_bcast:31).  Moves between lanes, no LDS.
__device__ __forceinline__ double wave_sum_to_63(double v)
{
    v = dpp_add<0xB1, 0xF>(v);
    v = dpp_add<0x4E, 0xF>(v);
    v = dpp_add<0x141, 0xF>(v);
    v = dpp_add<0x140, 0xF>(v);
    v = dpp_add<0x142, 0xA>(v);
    v = dpp_add<0x143, 0xC>(v);
    return v;
}

// Publishes the stage positions of the own bodies to LDS: sJ[i] = (x, y, z,
// k^2 m_i), and for the bodies that are sources of the indirect term (AC,
// 1 <= i < end_max) sT[i] = r_i rm3_i.  rm3 = 1 / |r_i|^3 of the own bodies
// (0 for the star and in BC) is returned for the Kepler term.  The barrier
// makes both arrays visible to every sink.
//
// SPLIT: no sT; instead each wave's partial sums of k^2 m_i r_i rm3_i over
// its bodies in [1, end_a) and in [1, end_b) go to c.part (one lane per
// body adds), so that the sinks take the indirect term as a whole sum
// rather than pair by pair.  That halves the LDS bytes a sink reads per
// source and takes three operations out of each pair term.
template <int BPT, bool SPLIT>
__device__ void publish(const Ctx &c, const double (&pos)[BPT][3], const double (&gm)[BPT], double (&rm3)[BPT])
{
    double ta[3] = {0.0, 0.0, 0.0}, tb[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
        const int i = own(c, q);
        rm3[q] = 0.0;
        if (i >= c.n) break;
        const double x = pos[q][0], y = pos[q][1], z = pos[q][2];
        c.sJ[i] = make_double4(x, y, z, gm[q]);
        if (!c.bc && i >= 1) {
            // Solaris/Acceleration.cpp:257-263
            const double r2 = x * x + y * y + z * z;
            const double r = sqrt(r2);
            rm3[q] = 1.0 / (r2 * r);
            const double tx = x * rm3[q], ty = y * rm3[q], tz = z * rm3[q];
            if constexpr (SPLIT) {
                if (c.sub == 0 && i < c.end_a) { ta[0] += gm[q] * tx; ta[1] += gm[q] * ty; ta[2] += gm[q] * tz; }
                if (c.sub == 0 && i < c.end_b) { tb[0] += gm[q] * tx; tb[1] += gm[q] * ty; tb[2] += gm[q] * tz; }
            } else {
                if (i < c.end_max) c.sT[i] = make_double4(tx, ty, tz, 0.0);
            }
        }
    }
    if constexpr (SPLIT) {
        if (!c.bc) {
            // one source range for both classes (every body a source of
            // every other, as in the ensemble): one sum serves both
            const bool one = c.end_a == c.end_b;
#pragma unroll
            for (int k = 0; k < 3; ++k) ta[k] = wave_sum_to_63(ta[k]);
            if (!one) {
#pragma unroll
                for (int k = 0; k < 3; ++k) tb[k] = wave_sum_to_63(tb[k]);
            }
            if ((threadIdx.x & (kWave - 1)) == kWave - 1) {
                double *w = c.part + 6 * (threadIdx.x / kWave);
#pragma unroll
                for (int k = 0; k < 3; ++k) { w[k] = ta[k]; w[3 + k] = one ? ta[k] : tb[k]; }
            }
        }
    }
    __syncthreads();
}

// The pair term of sink p and source q with weight w = k^2 m_j:
// px += w rijm3 dx (and the same for y, z), rijm3 = 1 / r^3 from the
// hardware reciprocal square root and its second-order correction.  The
// sink's own record gives dx = dy = dz = 0 and r^2 = 0, whose reciprocal
// square root (infinite) is capped at kRsqCap, above 1 / r of any two
// distinct bodies (more than 1e-50 AU apart), so its term is exactly
// w rijm3 * 0 = 0 and needs no mask.  c15 = 1.5 and c1875 = 1.875, held in
// registers by the caller (with a constant operand the addend would be
// copied for every pair).
constexpr double kRsqCap = 1.0e50;

__device__ __forceinline__ void pair_term(const double4 &p, const double4 &q, double c15, double c1875, double &px,
                                          double &py, double &pz)
{
    const double dx = q.x - p.x, dy = q.y - p.y, dz = q.z - p.z;
    const double r2 = dx * dx + dy * dy + dz * dz;
    const double y0 = fmin(__builtin_amdgcn_rsq(r2), kRsqCap);
    const double tt = y0 * y0;
    const double e = __builtin_fma(-r2, tt, 1.0);
    const double y3 = tt * y0;
    const double rijm3 = __builtin_fma(y3, e * __builtin_fma(c1875, e, c15), y3);
    const double f = q.w * rijm3;
    px = __builtin_fma(f, dx, px);
    py = __builtin_fma(f, dy, py);
    pz = __builtin_fma(f, dz, pz);
}

// Pair sums of sink i (position p) over the sources j in [j0, j1), the
// sink itself left out.  AC (GravityAC, Solaris/Acceleration.cpp:294-317):
// over the sources in order, k^2 m_j (d_ij / r_ij^3 - r_j rm3_j), the
// indirect term taken pair by pair as the reference does.  BC (GravityBC,
// :530-634): k^2 m_j d_ij / r_ij^3.  1 / r_ij^3 is the hardware reciprocal
// square root cubed with one second-order correction,
// (1 - e)^(-3/2) ~ 1 + 3/2 e + 15/8 e^2 for e = 1 - r^2 y^2.  NN: the
// nearest source (BC: the last of equals, AC: the first).
//
// SPLIT (the indirect term as a block sum, up to 1 << lsh lanes per sink,
// no nearest neighbour): pair_term, four sources per trip with their LDS
// records read first, the rest one at a time; the lanes of a sink take
// every (1 << lsh)-th source from j0 + sub.
//
// Otherwise one source at a time with the sink's own term masked (zero
// weight, r^2 replaced by 1, so it adds exactly +-0; AC: it also carries
// -r_i rm3_i): one loop over the whole range rather than two
// self-excluding ones, which would diverge from lane to lane.
template <bool BC, bool NN, bool SPLIT>
__device__ __forceinline__ void pair_range(const Ctx &c, const double4 &p, int i, int j0, int j1, double &px,
                                           double &py, double &pz, double &best, int &bidx)
{
    constexpr int U = 4;
    if constexpr (SPLIT) {
        const int stride = 1 << c.lsh;
        j0 += c.sub;
        double c15 = 1.5, c1875 = 1.875;
        asm volatile("" : "+v"(c15), "+v"(c1875));
        int j = j0;
        for (; j + (U - 1) * stride < j1; j += U * stride) {
            double4 q[U];
#pragma unroll
            for (int u = 0; u < U; ++u) q[u] = c.sJ[j + u * stride];
#pragma unroll
            for (int u = 0; u < U; ++u) pair_term(p, q[u], c15, c1875, px, py, pz);
        }
        for (; j < j1; j += stride) pair_term(p, c.sJ[j], c15, c1875, px, py, pz);
    } else {
#pragma unroll 2
        for (int j = j0; j < j1; ++j) {
            const double4 q = c.sJ[j];
            double4 t;
            if constexpr (!BC) t = c.sT[j];
            const bool self = j == i;
            const double dx = q.x - p.x, dy = q.y - p.y, dz = q.z - p.z;
            const double r2 = self ? 1.0 : dx * dx + dy * dy + dz * dz;
            const double w = self ? 0.0 : q.w;
            const double y0 = __builtin_amdgcn_rsq(r2);
            const double tt = y0 * y0;
            const double e = __builtin_fma(-r2, tt, 1.0);
            const double y3 = tt * y0;
            const double rijm3 = __builtin_fma(y3, e * __builtin_fma(1.875, e, 1.5), y3);
            if constexpr (BC) {
                const double f = w * rijm3;
                px = __builtin_fma(f, dx, px);
                py = __builtin_fma(f, dy, py);
                pz = __builtin_fma(f, dz, pz);
            } else {
                px = __builtin_fma(w, __builtin_fma(dx, rijm3, -t.x), px);
                py = __builtin_fma(w, __builtin_fma(dy, rijm3, -t.y), py);
                pz = __builtin_fma(w, __builtin_fma(dz, rijm3, -t.z), pz);
            }
            if constexpr (NN) {
                if (!self && (BC ? (r2 <= best) : (r2 < best))) { best = r2; bidx = j; }
            }
        }
    }
}

// The paired split sum (c.pair2: two lanes per body, every body a source
// of every other).  The four lanes of bodies b0 = 2g and b1 = 2g + 1 each
// take every fourth source from j0 + (lane & 3) for both bodies, so that a
// source record read from LDS serves two sinks (half the LDS reads of one
// sink per lane pair, for the same arithmetic).  A butterfly over the four
// lanes (DPP quad permutations) leaves both sums in all of them, the same
// in each; each lane keeps its own body's.  All four lanes of a pair must
// call it together (the DPP moves read the other lanes of the quad): the
// caller runs it for every pair with b0 < n before lanes part by body, so
// a lane whose own body is past the system's end still takes its share of
// its partner's sources (and discards its own sums).
__device__ __forceinline__ void pair_range2(const Ctx &c, int i, int j0, int j1, double &px, double &py,
                                            double &pz)
{
    const int b0 = i & ~1;
    const double4 p0 = c.sJ[b0], p1 = c.sJ[b0 + 1];
    double c15 = 1.5, c1875 = 1.875;
    asm volatile("" : "+v"(c15), "+v"(c1875));
    double x0 = 0.0, y0 = 0.0, z0 = 0.0, x1 = 0.0, y1 = 0.0, z1 = 0.0;
    int j = j0 + (int)(threadIdx.x & 3);
    for (; j + 4 < j1; j += 8) {
        const double4 qa = c.sJ[j], qb = c.sJ[j + 4];
        pair_term(p0, qa, c15, c1875, x0, y0, z0);
        pair_term(p1, qa, c15, c1875, x1, y1, z1);
        pair_term(p0, qb, c15, c1875, x0, y0, z0);
        pair_term(p1, qb, c15, c1875, x1, y1, z1);
    }
    if (j < j1) {
        const double4 q = c.sJ[j];
        pair_term(p0, q, c15, c1875, x0, y0, z0);
        pair_term(p1, q, c15, c1875, x1, y1, z1);
    }
    x0 = dpp_add<0x4E, 0xF>(dpp_add<0xB1, 0xF>(x0));
    y0 = dpp_add<0x4E, 0xF>(dpp_add<0xB1, 0xF>(y0));
    z0 = dpp_add<0x4E, 0xF>(dpp_add<0xB1, 0xF>(z0));
    x1 = dpp_add<0x4E, 0xF>(dpp_add<0xB1, 0xF>(x1));
    y1 = dpp_add<0x4E, 0xF>(dpp_add<0xB1, 0xF>(y1));
    z1 = dpp_add<0x4E, 0xF>(dpp_add<0xB1, 0xF>(z1));
    const bool second = (i & 1) != 0;
    px = second ? x1 : x0;
    py = second ? y1 : y0;
    pz = second ? z1 : z0;
}

// Acceleration of body i from the LDS positions; mu = k^2 (m_0 + m_i),
// rm3 = 1 / |r_i|^3.  AC: the Kepler term -mu rm3 r_i plus the pair sum
// over the sources 1 <= j < end (end by the sink's class,
// Solaris/Acceleration.cpp:285-289); the star gets zero.  BC: the pair sum
// over the massive bodies.
//
// SPLIT (the ensemble's queues, which have no side outputs and no
// events, so no nearest neighbour): each lane of the sink sums its share
// of the sources, and the shares are added over the lanes by a butterfly,
// which leaves the same sums in every lane (a + b = b + a at every level).
template <bool BC, bool NN, bool SPLIT>
__device__ void gravity_one(const Ctx &c, int i, double mu, double rm3, double &ax, double &ay, double &az,
                            int &nni, double &nnd, const double *pre)
{
    const double4 p = c.sJ[i];
    double best = DBL_MAX;
    int bidx = -1;
    double px = 0.0, py = 0.0, pz = 0.0;
    const int jb = BC ? 0 : 1;
    int je = BC ? c.nm : (i < c.nm) ? c.end_a : c.end_b;
    if (!BC && i == 0) je = jb;   // the star is not integrated (AC)
    static_assert(!(SPLIT && NN), "the split sum keeps no nearest neighbour");
    if (SPLIT && !BC && c.pair2) {
        // the paired sum, formed by the caller over [1, n) (the star's sums
        // are not used)
        px = pre[0]; py = pre[1]; pz = pre[2];
    } else {
        pair_range<BC, NN, SPLIT>(c, p, i, jb, je, px, py, pz, best, bidx);
        if constexpr (SPLIT) {
            for (int o = 1; o < (1 << c.lsh); o <<= 1) {
                px += __shfl_xor(px, o, kWave);
                py += __shfl_xor(py, o, kWave);
                pz += __shfl_xor(pz, o, kWave);
            }
        }
    }
    if constexpr (SPLIT) {
        if (!BC && i != 0) {
            // the indirect term: the sum over the sink's source range less
            // the sink's own term, -sum_{j != i} k^2 m_j r_j rm3_j
            const int cls = i < c.nm ? 0 : 3;
            const int nw = blockDim.x / kWave;
            double t[3] = {0.0, 0.0, 0.0};
            for (int w = 0; w < nw; ++w) {
#pragma unroll
                for (int k = 0; k < 3; ++k) t[k] += c.part[6 * w + cls + k];
            }
            if (i < (cls ? c.end_b : c.end_a)) {
                t[0] -= p.w * (p.x * rm3);
                t[1] -= p.w * (p.y * rm3);
                t[2] -= p.w * (p.z * rm3);
            }
            px -= t[0];
            py -= t[1];
            pz -= t[2];
        }
    }
    if (BC) {
        ax = px; ay = py; az = pz;
    } else if (i == 0) {
        ax = ay = az = 0.0;
    } else {
        ax = -mu * rm3 * p.x + px;
        ay = -mu * rm3 * p.y + py;
        az = -mu * rm3 * p.z + pz;
    }
    nni = bidx;
    nnd = bidx >= 0 ? sqrt(best) : 0.0;
}

// Evaluates the own bodies into stage slot l and into f (velocity half from
// vel, zero for the astrocentric star; acceleration half from gravity); the
// last stage also writes the side outputs.  Ends with the barrier after
// which sJ and sT may be overwritten.
template <int BPT, bool BC, bool LAST, int LF, bool GAS, bool SPLIT>
__device__ void evaluate_t(const Ctx &c, const Reg<BPT, LF> &R, int l, const double (&vel)[BPT][3],
                           const double (&mu)[BPT], const double (&rm3)[BPT], const double (&mig)[BPT][3],
                           double (&f)[BPT][6])
{
    // the paired split sum, by whole pairs before lanes part by body
    double pre[3] = {0.0, 0.0, 0.0};
    if constexpr (SPLIT && !BC) {
        if (c.pair2 && (own(c, 0) & ~1) < c.n) pair_range2(c, own(c, 0), 1, c.n, pre[0], pre[1], pre[2]);
    }
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
        const int i = own(c, q);
        if (i >= c.n) break;
        double ax, ay, az, nnd;
        int nni;
        gravity_one<BC, LAST && !SPLIT, SPLIT>(c, i, mu[q], rm3[q], ax, ay, az, nni, nnd, pre);
        if constexpr (GAS) {
            // GasDragAC every stage on the drag bodies (Solaris/Acceleration.cpp:190-198, :331-422), then
            // the migration cached at the Driver's first evaluation (:200-242)
            const int si = sys_index(c, i);
            if (si >= c.drag_lo && si < c.drag_hi) {
                const double4 p = c.sJ[i];
                const int b = c.base + i;
                double dx, dy, dz;
                gas_drag(c.A->gas, c.factor, kGauss2 * c.m0, c.m0, p.x, p.y, p.z, vel[q][0], vel[q][1], vel[q][2],
                         c.A->radius[b], c.A->density[b], c.A->cd[b], c.A->gs[b], c.A->ge[b], dx, dy, dz);
                ax += dx; ay += dy; az += dz;
                if (LAST && c.A->dragc && (i >= c.src || c.shift == 0)) {
                    double *d = c.A->dragc + si;
                    d[0] = dx; d[c.A->cache_stride] = dy; d[2 * c.A->cache_stride] = dz;
                }
            }
            if (i >= 1 && i < c.nm) { ax += mig[q][0]; ay += mig[q][1]; az += mig[q][2]; }
        }
        const bool star_ac = !BC && i == 0;
        f[q][0] = star_ac ? 0.0 : vel[q][0];
        f[q][1] = star_ac ? 0.0 : vel[q][1];
        f[q][2] = star_ac ? 0.0 : vel[q][2];
        f[q][3] = ax; f[q][4] = ay; f[q][5] = az;
        // LF: the LDS-held derivatives live only there, except F0, which the
        // host reads as ACCEL
        const int sl = LF ? lds_slot<LF>(l) : -1;
        if (sl >= 0) {
#pragma unroll
            for (int k = 0; k < 6; ++k) R.sF[sl * 6 + k] = f[q][k];
        }
        if (sl < 0 || l == 0) {
            uint32_t vb[6];
            offsets(c, i, vb);
            double *fs = stage(c, l);
#pragma unroll
            for (int k = 0; k < 6; ++k) st(fs, vb[k], f[q][k]);
        }
        if (LAST) {
            if (!BC) c.A->rm3[c.base + i] = rm3[q];
            if constexpr (!SPLIT) {
                c.A->nni[c.base + i] = nni;
                c.A->nnd[c.base + i] = nnd;
            }
        }
    }
    __syncthreads();
}

template <bool GAS, bool SPLIT, int BPT, int LF>
__device__ __forceinline__ void evaluate(const Ctx &c, const Reg<BPT, LF> &R, int l, bool last,
                                         const double (&vel)[BPT][3], const double (&mu)[BPT],
                                         const double (&rm3)[BPT], const double (&mig)[BPT][3],
                                         double (&f)[BPT][6])
{
    if (c.bc) {
        if (last) evaluate_t<BPT, true, true, LF, GAS, SPLIT>(c, R, l, vel, mu, rm3, mig, f);
        else evaluate_t<BPT, true, false, LF, GAS, SPLIT>(c, R, l, vel, mu, rm3, mig, f);
    } else {
        if (last) evaluate_t<BPT, false, true, LF, GAS, SPLIT>(c, R, l, vel, mu, rm3, mig, f);
        else evaluate_t<BPT, false, false, LF, GAS, SPLIT>(c, R, l, vel, mu, rm3, mig, f);
    }
}

// ---- grid-wide decisions of a system split into slices ----------------
// The GridSync words are touched only by system-scope atomics (coherent
// across the chiplets' L2 caches), never by plain loads or stores, and no
// other data passes between the workgroups; the waits poll without cache
// maintenance, and the readers of the published entries take one acquire
// fence after the barrier.
#define SOL_SYS __HIP_MEMORY_SCOPE_SYSTEM

// Barrier over the workgroups of a cooperative launch (thread 0 of each).
// `dep` is 0, computed from the values this workgroup just published: the
// arrival waits for them, so they are in place before anyone passes.
// false when it did not complete (error set by a workgroup that waited too
// long, or seen here).
__device__ bool grid_barrier(GridSync *s, uint32_t nblocks, uint32_t dep, uint64_t ticks)
{
    const uint32_t g = __hip_atomic_load(&s->gen, __ATOMIC_RELAXED, SOL_SYS);
    // gen < 2^31 within a launch: (g >> 31) == 0 orders the arrival after the read of g
    const uint32_t arrived = __hip_atomic_fetch_add(&s->count, 1u + dep + (g >> 31), __ATOMIC_RELAXED, SOL_SYS);
    if (arrived == nblocks - 1) {
        const uint32_t all = __hip_atomic_exchange(&s->count, 0u, __ATOMIC_RELAXED, SOL_SYS);
        __hip_atomic_fetch_add(&s->gen, 1u + (all >> 31), __ATOMIC_RELAXED, SOL_SYS);
        return true;
    }
    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    for (;;) {
        if (__hip_atomic_load(&s->gen, __ATOMIC_RELAXED, SOL_SYS) != g) return true;
        if (__hip_atomic_load(&s->error, __ATOMIC_RELAXED, SOL_SYS)) return false;
        if (__builtin_amdgcn_s_memrealtime() - t0 >= ticks) {
            __hip_atomic_store(&s->error, 1u, __ATOMIC_RELAXED, SOL_SYS);
            return false;
        }
        __builtin_amdgcn_s_sleep(2);
    }
}

// The maximum of v (>= 0) and the OR of flag over all workgroups of the
// launch (k: this launch's combine count, the same in every workgroup).
// Entries of parity k & 1 are written by combine k and read after its
// barrier; combine k + 2 rewrites them only after the barrier of k + 1,
// which every reader of combine k has passed.  false: the barrier failed.
//
// Each flag word carries the combine's tag, (k + 1) << 1 | flag, written
// after the value (its operand waits for the value's exchange); a reader
// takes an entry's value only once its tag is this combine's (re-reading
// a stale copy until then, within the wait budget), and reads the value
// after the tag (the address waits for the tag's load).
__device__ bool grid_combine(const ResArrays &A, double *sh, double v, int flag, double &vout, int &fout, int &k)
{
    __shared__ int ok_s, flag_s, stale_s;
    GridSync *s = A.sync;
    const int par = k & 1, nb = A.nsync;
    const uint32_t tag = ((uint32_t)k + 1u) & 0x3FFFFFFFu;
    if (threadIdx.x == 0) {
        stale_s = 0;
        // |v|: a maximum >= 0, or a NaN with its sign bit cleared (which
        // the maximum over the entries passes over, as fmax does)
        const unsigned long long ov = __hip_atomic_exchange(&s->vals[par][blockIdx.x],
                                                            (unsigned long long)__double_as_longlong(fabs(v)),
                                                            __ATOMIC_RELAXED, SOL_SYS);
        // the entries are zeroed at each launch (k_zero_sync) and hold only
        // such values and tagged flag words below 2^31 after, so the sign
        // bits added here are 0: they only order the flag word after the
        // value and the arrival after both
        const uint32_t of = __hip_atomic_exchange(&s->flags[par][blockIdx.x],
                                                  (tag << 1 | (flag ? 1u : 0u)) + (uint32_t)(ov >> 63),
                                                  __ATOMIC_RELAXED, SOL_SYS);
        ok_s = grid_barrier(s, (uint32_t)nb, of >> 31, A.sync_ticks) ? 1 : 0;
    }
    __syncthreads();
    if (ok_s != 0 && threadIdx.x < kWave) {
        // once per combine: no copy of the entries read below may predate
        // the barrier
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        double m = 0.0;
        uint32_t fl = 0;
        bool stale = false;
        const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
        for (int b = threadIdx.x; b < nb; b += kWave) {
            uint32_t w = __hip_atomic_load(&s->flags[par][b], __ATOMIC_RELAXED, SOL_SYS);
            while ((w >> 1) != tag) {
                if (__builtin_amdgcn_s_memrealtime() - t0 >= A.sync_ticks) { stale = true; break; }
                __builtin_amdgcn_s_sleep(1);
                w = __hip_atomic_load(&s->flags[par][b], __ATOMIC_RELAXED, SOL_SYS);
            }
            m = fmax(m, __longlong_as_double((long long)__hip_atomic_load(&s->vals[par][b + (int)(w >> 31)],
                                                                          __ATOMIC_RELAXED, SOL_SYS)));
            fl |= w & 1u;
        }
        m = wmax(m);
        const double f = wmax((double)fl);
        const double st = wmax(stale ? 1.0 : 0.0);
        if (threadIdx.x == 0) {
            sh[3] = m;
            flag_s = f != 0.0 ? 1 : 0;
            if (st != 0.0) {
                stale_s = 1;
                __hip_atomic_store(&s->error, 1u, __ATOMIC_RELAXED, SOL_SYS);
            }
        }
    }
    __syncthreads();
    const bool ok = ok_s != 0 && stale_s == 0;
    vout = sh[3];
    fout = flag_s;
    __syncthreads();
    ++k;
    return ok;
}

// Stage derivative L of own body q, component k (at byte offset o).
template <int L, int S, int BPT, int LF>
__device__ __forceinline__ double fget(const Ctx &c, const Reg<BPT, LF> &R, int q, int k, uint32_t o)
{
    if constexpr (Reg<BPT, LF>::on && L == S - 1 && L > 0) return R.prev[q][k];
    else if constexpr (LF > 0 && lds_slot<LF>(L) >= 0) return R.sF[lds_slot<LF>(L) * 6 + k];
    else return ld(stage(c, L), o);
}

// State of stage S (the reference's yTemp before the S-th evaluation) for
// the own bodies: positions into pos, velocities into vel.  The stage
// derivatives with nonzero coefficients and y0 are read first, three
// components at a time, so that their latencies overlap.
//
// First-order tableaux (RKF78, RK4): y0 + h * sum, the sum over the nonzero
// coefficients in the tableau's order, as the reference's hand-written
// stage sums (RungeKuttaFehlberg78.cpp:147-240, RungeKutta4.cpp:58-130).
// Dormand-Prince RKN (DormandPrince.cpp:246-491): positions
// p0 + c_S h v0 + h^2 var and velocities v0 + h var, var = sum_l a_{S,l} F_l
// over the acceleration halves.
template <int INTEG, int S, int BPT, int LF>
__device__ __forceinline__ void stage_state(const Ctx &c, const Reg<BPT, LF> &R, double h, double (&pos)[BPT][3],
                                            double (&vel)[BPT][3])
{
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
        const int i = own(c, q);
        if (i >= c.n) break;
        uint32_t vb[6];
        offsets(c, i, vb);
        auto y0 = [&](int k) { return Reg<BPT>::on ? R.y0[q][k] : ld(c.A->y0, vb[k]); };
        if constexpr (INTEG == INTEG_DP) {
            double p0[3], v0[3], f[3][S];
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                p0[j] = y0(j);
                v0[j] = y0(j + 3);
                static_for<0, S>([&](auto L) {
                    if constexpr (L == 0 || tab::kDpA[S][L] != 0.0) f[j][L] = fget<L, S>(c, R, q, j + 3, vb[j + 3]);
                });
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                double var = tab::kDpA[S][0] * f[j][0];
                static_for<1, S>([&](auto L) {
                    if constexpr (tab::kDpA[S][L] != 0.0) var += tab::kDpA[S][L] * f[j][L];
                });
                pos[q][j] = p0[j] + tab::kDpC[S] * h * v0[j] + h * h * (var);
                vel[q][j] = v0[j] + h * (var);
            }
        } else {
            // positions, then velocities: three components' loads at a time
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                double yv[3], f[3][S];
#pragma unroll
                for (int kk = 0; kk < 3; ++kk) {
                    const int k = 3 * half + kk;
                    yv[kk] = y0(k);
                    static_for<0, S>([&](auto L) {
                        if constexpr (dcoef<INTEG>(S, L) != 0.0) f[kk][L] = fget<L, S>(c, R, q, k, vb[k]);
                    });
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int kk = 0; kk < 3; ++kk) {
                    double acc = 0.0;
                    bool first = true;
                    static_for<0, S>([&](auto L) {
                        constexpr double d = dcoef<INTEG>(S, L);
                        if constexpr (d != 0.0) {
                            const double v = d * f[kk][L];
                            acc = first ? v : acc + v;
                            first = false;
                        }
                    });
                    const double out = yv[kk] + h * acc;
                    if (half == 0) pos[q][kk] = out;
                    else vel[q][kk] = out;
                }
            }
        }
    }
}

// stage_state for the run-time stage number s (1 <= s <= n_stages).
template <int INTEG, int BPT, int LF, int S = 1>
__device__ __forceinline__ void stage_state_at(int s, const Ctx &c, const Reg<BPT, LF> &R, double h,
                                               double (&pos)[BPT][3], double (&vel)[BPT][3])
{
    if constexpr (S <= n_stages<INTEG>()) {
        if (s == S) stage_state<INTEG, S, BPT>(c, R, h, pos, vel);
        else stage_state_at<INTEG, BPT, LF, S + 1>(s, c, R, h, pos, vel);
    }
}

// Final state into Y (and into ynew) and the error estimate into ERR for
// the own bodies; returns this thread's contribution to the error maximum
// (RKF78: max |err / yscale|, Dormand-Prince: max position error).
template <int INTEG, int BPT, int LF>
__device__ double final_state(const Ctx &c, const Reg<BPT, LF> &R, double h, double (&ynew)[BPT][6])
{
    constexpr int NS = n_stages<INTEG>() + 1;
    double ratio = 0.0;
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
        const int i = own(c, q);
        if (i >= c.n) break;
        uint32_t vb[6];
        offsets(c, i, vb);
        auto y0 = [&](int k) { return Reg<BPT>::on ? R.y0[q][k] : ld(c.A->y0, vb[k]); };
        if constexpr (INTEG == INTEG_RKF78) {
            // RungeKuttaFehlberg78.cpp:231-248
            constexpr double b0 = 41.0 / 840.0, b5 = 34.0 / 105.0, b6 = 9.0 / 35.0, b8 = 9.0 / 280.0,
                             b10 = 41.0 / 840.0;
            double e[6];
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                double f[3][13], yv[3], sc[3];
#pragma unroll
                for (int kk = 0; kk < 3; ++kk) {
                    const int k = 3 * half + kk;
                    const uint32_t o = vb[k];
                    f[kk][0] = fget<0, NS>(c, R, q, k, o);
                    static_for<5, 13>([&](auto L) { f[kk][L] = fget<L, NS>(c, R, q, k, o); });
                    yv[kk] = y0(k);
                    sc[kk] = ld(c.A->yscale, o);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int kk = 0; kk < 3; ++kk) {
                    const int k = 3 * half + kk;
                    const double *F = f[kk];
                    ynew[q][k] = yv[kk] + h * (b0 * F[0] + b5 * F[5] + b6 * (F[6] + F[7]) + b8 * (F[8] + F[9]) +
                                               b10 * F[10]);
                    e[k] = h * fabs(F[0] + F[10] - F[11] - F[12]) * 41.0 / 840.0;
                    ratio = fmax(ratio, fabs(e[k] / sc[kk]));
                }
            }
#pragma unroll
            for (int k = 0; k < 6; ++k) { st(c.A->y, vb[k], ynew[q][k]); st(c.A->err, vb[k], e[k]); }
        } else if constexpr (INTEG == INTEG_RK4) {
            double f[6][4];
#pragma unroll
            for (int k = 0; k < 6; ++k)
                static_for<0, 4>([&](auto L) { f[k][L] = fget<L, NS>(c, R, q, k, vb[k]); });
#pragma unroll
            for (int k = 0; k < 6; ++k) {
                ynew[q][k] = y0(k) + h * (tab::kRk4B[0] * f[k][0] + tab::kRk4B[1] * f[k][1] +
                                          tab::kRk4B[2] * f[k][2] + tab::kRk4B[3] * f[k][3]);
                st(c.A->y, vb[k], ynew[q][k]);
            }
        } else {
            // DormandPrince.cpp:455-491
            constexpr const double *B = tab::kDpB, *Bd = tab::kDpBdh;
            const double h2 = h * h;
            double e[3];
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const uint32_t o = vb[j + 3];
                double F[9];
                F[0] = fget<0, NS>(c, R, q, j + 3, o);
                static_for<4, 9>([&](auto L) { F[L] = fget<L, NS>(c, R, q, j + 3, o); });
                const double p0 = y0(j), v0 = y0(j + 3);
                ynew[q][j] = p0 + h * v0 + h2 * (B[0] * F[0] + B[4] * F[4] + B[5] * F[5] + B[6] * F[6] +
                                                 B[7] * F[7] + B[8] * F[8]);
                e[j] = h2 * fabs(F[7] - F[8]) / 20.0;
                ynew[q][j + 3] = v0 + h * (Bd[0] * F[0] + Bd[4] * F[4] + Bd[5] * F[5] + Bd[6] * F[6] + Bd[7] * F[7]);
                ratio = fmax(ratio, e[j]);
            }
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                st(c.A->y, vb[j], ynew[q][j]);
                st(c.A->err, vb[j], e[j]);
                st(c.A->y, vb[j + 3], ynew[q][j + 3]);
                st(c.A->err, vb[j + 3], 0.0);
            }
        }
    }
    return ratio;
}

// CheckEvent's thresholds on the last stage's side outputs of the
// workgroup's bodies (Solaris/Simulator.cpp:631-644, :688-695): this
// thread's part.
__device__ int event_here(const ResSystem &S, const Ctx &c, const ResArrays &A)
{
    int event = 0;
    for (int i = threadIdx.x; i < c.n; i += blockDim.x) {
        const double r3 = A.rm3[c.base + i];
        if (i >= 1 && S.e3 > 0.0 && r3 < S.e3) event = 1;
        if (i >= 1 && S.h3 > 0.0 && r3 > S.h3) event = 1;
        const int j = A.nni[c.base + i];
        if (S.coll > 0.0 && j >= 0 && j < c.n &&
            S.coll * (A.radius[c.base + i] + A.radius[c.base + j]) > A.nnd[c.base + i])
            event = 1;
    }
    return event;
}

// One workgroup per system; BPT bodies per thread at most
// (n <= BPT * blockDim.x).  Blocks have at most 640 threads with one body
// per thread (168 registers) and 512 with more (256 registers).
// Dynamic LDS: sJ and sT, nmax records each, and with LF the rows of the
// LDS-held stage derivatives (nmax x kLdsStride doubles).
//
// SPLIT (one body per thread slot): L = 1 << lsh lanes per body, the
// largest L <= 1 << max_lsh with n L <= blockDim.x that leaves every lane
// at least kSplitMinSources sources; the L lanes of a body split its source
// loop and otherwise repeat the same arithmetic on the same values, so
// their stores agree.
constexpr int kSplitMinSources = 24;

template <int INTEG, int BPT, int LF, bool GRID, bool GAS, bool SPLIT = false>
__device__ __forceinline__ void run_system(ResSystem &S, const ResArrays &A, int max_steps, int nmax, double4 *lds,
                                           double *red, double *sh, int max_lsh = 0, double *part = nullptr)
{
    static_assert(!SPLIT || (BPT == 1 && !GRID), "lanes per body: one body per slot");
    if (S.status != RES_RUNNING) return;
    Ctx c;
    if constexpr (SPLIT) {
        int lsh = 0;
        while (lsh < max_lsh && (S.n << (lsh + 1)) <= (int)blockDim.x && (S.n >> (lsh + 1)) >= kSplitMinSources)
            ++lsh;
        c.lsh = lsh;
        c.me = threadIdx.x >> lsh;
        c.nth = blockDim.x >> lsh;
        c.sub = threadIdx.x & ((1 << lsh) - 1);
        c.pair2 = lsh == 1 && S.barycentric == 0 && S.end_a == S.n && S.end_b == S.n;
    } else {
        c.pair2 = false;
        c.lsh = 0;
        c.me = threadIdx.x;
        c.nth = blockDim.x;
        c.sub = 0;
    }
    c.part = part;
    c.A = &A; c.n = S.n; c.base = S.base; c.nm = S.nm; c.end_a = S.end_a; c.end_b = S.end_b;
    c.end_max = c.end_a > c.end_b ? c.end_a : c.end_b;
    c.bc = S.barycentric != 0;
    c.tot = A.tot; c.sJ = lds; c.sT = lds + nmax;
    c.src = S.src; c.shift = S.shift; c.drag_lo = S.drag_lo; c.drag_hi = S.drag_hi; c.giant_end = S.giant_end;
    c.m0 = A.mass[c.base];
    c.factor = 1.0;
    constexpr int nst = n_stages<INTEG>();
    constexpr bool kReg = Reg<BPT>::on;
    const bool events = S.clip && (S.stop_mask & SOL_STOP_EVENT) && (S.e3 > 0.0 || S.h3 > 0.0 || S.coll > 0.0);
    int ncomb = 0;   // grid-wide combines done in this launch

    // k^2 m_i and k^2 (m_0 + m_i) of the own bodies, for the whole launch
    double gm[BPT], mu[BPT];
#pragma unroll
    for (int q = 0; q < BPT; ++q) {
        const int i = own(c, q) < c.n ? own(c, q) : 0;
        gm[q] = kGauss2 * A.mass[c.base + i];
        mu[q] = kGauss2 * (A.mass[c.base] + A.mass[c.base + i]);
    }
    Reg<BPT, LF> R;
    R.sF = LF ? reinterpret_cast<double *>(lds + 2 * nmax) + own(c, 0) * lds_stride<LF>() : nullptr;
    if constexpr (kReg) {
#pragma unroll
        for (int q = 0; q < BPT; ++q) {
            uint32_t vb[6];
            offsets(c, own(c, q) < c.n ? own(c, q) : 0, vb);
#pragma unroll
            for (int k = 0; k < 6; ++k) R.y0[q][k] = ld(A.y0, vb[k]);
        }
    }

    double mig[BPT][3];   // migration of the own massive bodies, this Driver call
#pragma unroll
    for (int q = 0; q < BPT; ++q) mig[q][0] = mig[q][1] = mig[q][2] = 0.0;

    for (int step = 0; step < max_steps; ++step) {
        const double t0 = S.t;
        double h = S.h_next;
        if constexpr (INTEG == INTEG_RK4) {
            if (A.h_seq) h = A.h_seq[step];
        }
        // f0 at y0 (the Driver's first evaluation), and yscale
        {
            double y0[BPT][6], pos[BPT][3], vel[BPT][3], rm3[BPT], f[BPT][6];
#pragma unroll
            for (int q = 0; q < BPT; ++q) {
                if constexpr (kReg) {
#pragma unroll
                    for (int k = 0; k < 6; ++k) y0[q][k] = R.y0[q][k];
                } else {
                    uint32_t vb[6];
                    offsets(c, own(c, q) < c.n ? own(c, q) : 0, vb);
#pragma unroll
                    for (int k = 0; k < 6; ++k) y0[q][k] = ld(A.y0, vb[k]);
                }
#pragma unroll
                for (int k = 0; k < 3; ++k) { pos[q][k] = y0[q][k]; vel[q][k] = y0[q][k + 3]; }
                if constexpr (INTEG == INTEG_RK4) {
                    if (A.stages_out && own(c, q) < c.n) {
                        uint32_t vb[6];
                        offsets(c, own(c, q), vb);
                        double *Y = A.stages_out + (size_t)(step * 4) * 6 * c.tot;
#pragma unroll
                        for (int k = 0; k < 6; ++k) st(Y, vb[k], y0[q][k]);
                    }
                }
            }
            if constexpr (GAS) {
                // the Driver's first evaluation computes the migration of the
                // massive bodies once (Solaris/Acceleration.cpp:200-242); the
                // stages reuse it
                c.factor = reduction_factor(A.gas, t0);
#pragma unroll
                for (int q = 0; q < BPT; ++q) {
                    const int i = own(c, q);
                    mig[q][0] = mig[q][1] = mig[q][2] = 0.0;
                    if (i < S.mig_lo || i >= c.nm) continue;
                    const bool giant = i < c.giant_end;
                    if (!(giant ? A.mig_do2 : A.mig_do1)) continue;
                    const int b = c.base + i;
                    int32_t mt = A.migt[b];
                    if (mt != (giant ? SOL_MIGRATION_TYPE_II : SOL_MIGRATION_TYPE_I)) continue;
                    const int32_t before = mt;
                    migration_accel(giant, pos[q][0], pos[q][1], pos[q][2], vel[q][0], vel[q][1], vel[q][2],
                                    A.mass[b], c.m0, A.stop[b], mt, A.gas, c.bc, t0, mig[q][0], mig[q][1],
                                    mig[q][2]);
                    if (mt != before) A.migt[b] = mt;
                    if (A.migc && c.shift == 0) {
                        double *d = A.migc + i;
                        d[0] = mig[q][0]; d[A.cache_stride] = mig[q][1]; d[2 * A.cache_stride] = mig[q][2];
                    }
                }
            }
            publish<BPT, SPLIT>(c, pos, gm, rm3);
            evaluate<GAS, SPLIT>(c, R, 0, false, vel, mu, rm3, mig, f);
            if (INTEG == INTEG_RKF78) {
#pragma unroll
                for (int q = 0; q < BPT; ++q) {
                    const int i = own(c, q);
                    if (i >= c.n) break;
                    uint32_t vb[6];
                    offsets(c, i, vb);
#pragma unroll
                    for (int k = 0; k < 6; ++k) st(A.yscale, vb[k], fabs(y0[q][k]) + fabs(h * f[q][k]) + 1.0e-30);
                }
            }
        }
        int iter = 0;
        double errmax = 0.0;
        int outcome = 0;   // 0 accept, 1 retry, 2 underflow, 3 maxiter
        int event_att = 0; // GRID: the system's event flag of the last attempt
        double ynew[BPT][6];
        for (;;) {
            ++iter;
            if (INTEG == INTEG_DP) h = S.h_next;
            for (int s = 1; s <= nst; ++s) {
                double pos[BPT][3], vel[BPT][3], rm3[BPT], f[BPT][6];
                stage_state_at<INTEG, BPT>(s, c, R, h, pos, vel);
                if constexpr (INTEG == INTEG_RK4) {
                    if (A.stages_out) {
#pragma unroll
                        for (int q = 0; q < BPT; ++q) {
                            if (own(c, q) >= c.n) break;
                            uint32_t vb[6];
                            offsets(c, own(c, q), vb);
                            double *Y = A.stages_out + (size_t)(step * 4 + s) * 6 * c.tot;
#pragma unroll
                            for (int k = 0; k < 3; ++k) { st(Y, vb[k], pos[q][k]); st(Y, vb[k + 3], vel[q][k]); }
                        }
                    }
                }
                if constexpr (GAS) {
                    // drag at the stage's time: RK4 and Dormand-Prince pass
                    // t + c_s h, RKF78 passes t to every stage
                    const double ts = INTEG == INTEG_RK4 ? t0 + tab::kRk4C[s] * h
                                    : INTEG == INTEG_DP  ? t0 + tab::kDpC[s] * h : t0;
                    c.factor = reduction_factor(A.gas, ts);
                }
                publish<BPT, SPLIT>(c, pos, gm, rm3);
                evaluate<GAS, SPLIT>(c, R, s, s == nst, vel, mu, rm3, mig, f);
                if constexpr (kReg) {
#pragma unroll
                    for (int q = 0; q < BPT; ++q)
#pragma unroll
                        for (int k = 0; k < 6; ++k) R.prev[q][k] = f[q][k];
                }
            }
            const double ratio = final_state<INTEG, BPT>(c, R, h, ynew);
            double raw = block_max_all(ratio, red, &sh[0]);
            if constexpr (GRID) {
                // every slice takes the same decision from the system-wide
                // error maximum, and the events of the attempt with it
                if (INTEG != INTEG_RK4 || events) {
                    const int ev = events ? __syncthreads_or(event_here(S, c, A)) : 0;
                    int evg = 0;
                    if (!grid_combine(A, sh, raw, ev, raw, evg, ncomb)) {
                        if (threadIdx.x == 0) S.status = RES_SYNC_ERROR;
                        return;
                    }
                    event_att = evg;
                }
            }
            if (threadIdx.x == 0) S.attempts += 1;
            // the step decision (identical in every thread)
            if (INTEG == INTEG_RKF78) {
                errmax = raw / S.eps;
                if (errmax < 1.0) { outcome = 0; break; }
                const double htemp = 0.9 * h * step_pow(errmax, -0.25);
                h = fabs(htemp) > fabs(0.1 * h) ? htemp : 0.1 * h;
                if (t0 + h == t0) { outcome = 2; break; }
            } else if (INTEG == INTEG_RK4) {
                outcome = 0;
                break;
            } else {
                errmax = raw;
                const double hn = errmax < 1.0e-20 ? 2.0 * h : 0.9 * h * step_pow(S.eps / errmax, 1.0 / 7.0);
                if (threadIdx.x == 0) { S.h_did = h; S.h_next = hn; }
                __syncthreads();
                if (!(errmax > S.eps && iter <= 10)) { outcome = iter > 10 ? 3 : 0; break; }
            }
        }
        __syncthreads();
        if (outcome == 2 || outcome == 3) {
            if (threadIdx.x == 0) {
                S.status = outcome == 2 ? RES_UNDERFLOW : RES_MAXITER;
                S.body_h = h;
            }
            return;
        }
        // accept: time, hDid, hNext (RungeKuttaFehlberg78.cpp:124-133 and the others)
        double h_next;
        if (INTEG == INTEG_RKF78) {
            h_next = errmax > 1.89e-4 ? (0.9 * h * step_pow(errmax, -0.2)) : (5.0 * h);
        } else if (INTEG == INTEG_RK4) {
            h_next = h;
        } else {
            h_next = S.h_next;
            h = S.h_did;
        }
        // swap y0 and y (the Driver's pointer swap), own bodies
#pragma unroll
        for (int q = 0; q < BPT; ++q) {
            const int i = own(c, q);
            if (i >= c.n) break;
            uint32_t vb[6];
            offsets(c, i, vb);
            double old[6];
#pragma unroll
            for (int k = 0; k < 6; ++k) old[k] = kReg ? R.y0[q][k] : ld(A.y0, vb[k]);
#pragma unroll
            for (int k = 0; k < 6; ++k) { st(A.y0, vb[k], ynew[q][k]); st(A.y, vb[k], old[k]); }
            if constexpr (kReg) {
#pragma unroll
                for (int k = 0; k < 6; ++k) R.y0[q][k] = ynew[q][k];
            }
        }
        __syncthreads();
        // CheckEvent's thresholds on the last stage's side outputs
        // (Solaris/Simulator.cpp:631-644, :688-695), when asked for
        int event;
        if constexpr (GRID) event = event_att;
        else event = __syncthreads_or(events ? event_here(S, c, A) : 0);
        if (threadIdx.x == 0) {
            bool stop = false;
            int reason = 0, flush = 0;
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
                // Counter::succededStep % CheckForSM (:154-159)
                S.flush_count = (S.flush_count + 1) % 100;
                flush = S.flush_count == 0;
                S.reason = reason | (stop ? SOL_STOP_END : 0);
                reason &= S.stop_mask;
            }
            sh[1] = stop ? 1.0 : reason ? 2.0 : 0.0;
            sh[2] = flush ? 1.0 : 0.0;
        }
        __syncthreads();
        const double next = sh[1];
        if (sh[2] != 0.0) {
            for (int i = threadIdx.x; i < c.n; i += blockDim.x)
                for (int k = 0; k < 6; ++k) {
                    if (fabs(cat(A.y0, c, k, i)) < 1.0e-50) at(A.y0, c, k, i) = 0.0;
                    if (fabs(cat(A.y, c, k, i)) < 1.0e-50) at(A.y, c, k, i) = 0.0;
                }
            if constexpr (kReg) {
#pragma unroll
                for (int q = 0; q < BPT; ++q)
#pragma unroll
                    for (int k = 0; k < 6; ++k)
                        if (fabs(R.y0[q][k]) < 1.0e-50) R.y0[q][k] = 0.0;
            }
        }
        __syncthreads();
        if (next != 0.0) {
            if (threadIdx.x == 0) S.status = next == 1.0 ? RES_DONE : RES_STOPPED;
            return;
        }
    }
}

template <int INTEG, int BPT, int LF, bool GAS>
__global__ __launch_bounds__(BPT == 1 ? 640 : 512) void k_resident(ResSystem *systems, ResArrays A, int max_steps,
                                                                     int nmax)
{
    extern __shared__ double4 lds[];
    __shared__ double red[16];
    __shared__ double sh[4];
    run_system<INTEG, BPT, LF, false, GAS>(systems[blockIdx.x], A, max_steps, nmax, lds, red, sh);
}

// RK4 at two bodies per thread in up to 640 threads (1,025 to 1,280
// bodies), where the 512-thread bound would leave four bodies per thread.
// Each body's sums run in one thread in the same order at any bodies per
// thread, so the results are the same (SOLARIS_AMD_RK4_W2=0 keeps four).
template <bool GAS>
__global__ __launch_bounds__(640) void k_resident_rk4_w2(ResSystem *systems, ResArrays A, int max_steps, int nmax)
{
    extern __shared__ double4 lds[];
    __shared__ double red[16];
    __shared__ double sh[4];
    run_system<INTEG_RK4, 2, 0, false, GAS>(systems[blockIdx.x], A, max_steps, nmax, lds, red, sh);
}

// One system as slices (GridSync): workgroup b runs slice b, every slice
// advancing the system's sources identically and its own sinks, with the
// step decisions combined over the grid.  The grid is no larger than what
// the device holds at once; should a workgroup not be resident anyway
// (another process on the device), the grid-wide wait times out and the
// slices stop with RES_SYNC_ERROR.
template <int INTEG, int LF, bool GAS>
__global__ __launch_bounds__(256) void k_resident_grid(ResSystem *systems, ResArrays A, int max_steps, int nmax)
{
    extern __shared__ double4 lds[];
    __shared__ double red[16];
    __shared__ double sh[4];
    run_system<INTEG, 1, LF, true, GAS>(systems[blockIdx.x], A, max_steps, nmax, lds, red, sh);
}

// Persistent form for many systems: every workgroup takes the next entry of
// `order` from a device-side queue (head, an atomic counter the host zeroes
// before the launch), runs that system's Driver loop for up to max_steps
// accepted steps, and takes the next, until the queue is empty.  Systems of
// every size share the launch (n <= BPT * blockDim.x), so the long ones
// placed first in `order` overlap the many short ones.
//
// One body per thread (BPT = 1): the indirect term as a block sum and up to
// 1 << max_lsh lanes per body (run_system's SPLIT), in blocks of up to
// BOUND threads (640 or 768, 168 registers; at 1024 the 128 registers left
// spill, and four lanes per body there measured slower than two at 512).
//
// LF (RKF78, one body per thread): its four most-read stage derivatives in
// LDS rows (the lanes of a body share its row and write the same values).
template <int INTEG, int BPT, int BOUND, int LF = 0>
__global__ __launch_bounds__(BOUND) void k_resident_queue(ResSystem *systems, const int32_t *__restrict__ order,
                                                          QueueWords *q, ResArrays A, int nmax, int max_lsh)
{
    extern __shared__ double4 lds[];
    __shared__ double red[16];
    __shared__ double sh[4];
    __shared__ double part[6 * (BOUND / kWave)];
    __shared__ int32_t slot;
    const int nsys = __builtin_amdgcn_readfirstlane(q->nsys), max_steps = __builtin_amdgcn_readfirstlane(q->max_steps);
    for (;;) {
        if (threadIdx.x == 0) slot = atomicAdd(&q->head, 1);
        __syncthreads();
        const int32_t k = slot;
        __syncthreads();   // every thread has read slot before it is taken again
        if (k >= nsys) return;
        run_system<INTEG, BPT, LF, false, false, BPT == 1>(systems[order[k]], A, max_steps, nmax, lds, red, sh,
                                                          max_lsh, part);
        __syncthreads();
    }
}

__global__ void k_zero_i32(int32_t *p) { *p = 0; }

// Zeroes a GridSync: count, gen, error and every published entry.  The
// entries must start at 0 too: each combine adds the sign bit of the entry
// its exchange replaces to its arrival (an ordering dependency that is 0
// for any value a combine publishes), and memory left by earlier
// allocations can hold any bits there, which would count one workgroup
// twice and release the barrier one arrival early.
__global__ void k_zero_sync(GridSync *s)
{
    if (threadIdx.x == 0) {
        s->count = 0;
        s->gen = 0;
        s->error = 0;
    }
    for (int i = threadIdx.x; i < 2 * kGridMaxSlices; i += blockDim.x) {
        (&s->vals[0][0])[i] = 0ull;
        (&s->flags[0][0])[i] = 0u;
    }
}

// System layout (component stride np) -> slice layout (stride tot): the
// state and the per-body parameters of every slice's bodies.
__global__ __launch_bounds__(256) void k_slice_scatter(SliceMap m, SliceArrays sys, ResArrays A)
{
    const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= (int64_t)m.nslices * m.stride) return;
    const int k = (int)(x / m.stride), l = (int)(x % m.stride);
    if (l >= slice_count(m, k)) return;
    const int b = slice_body(m, k, l);
    for (int comp = 0; comp < 6; ++comp) A.y0[comp * A.tot + x] = sys.y0[comp * (int64_t)m.np + b];
    A.mass[x] = sys.mass[b];
    const_cast<double *>(A.radius)[x] = sys.radius[b];
    if (sys.density) {
        const_cast<double *>(A.density)[x] = sys.density[b];
        const_cast<double *>(A.cd)[x] = sys.cd[b];
        const_cast<double *>(A.gs)[x] = sys.gs[b];
        const_cast<double *>(A.ge)[x] = sys.ge[b];
        const_cast<double *>(A.stop)[x] = sys.stop[b];
        A.migt[x] = sys.migt[b];
    }
}

// Slice layout -> system layout: the state, the Driver's arrays and the
// side outputs, each body from its slice (the sources from slice 0).
__global__ __launch_bounds__(256) void k_slice_gather(SliceMap m, SliceArrays sys, ResArrays A)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= m.n) return;
    const int64_t x = slice_place(m, b);
    for (int comp = 0; comp < 6; ++comp) {
        const int64_t o = comp * (int64_t)m.np + b, xo = comp * A.tot + x;
        sys.y0[o] = A.y0[xo];
        sys.y[o] = A.y[xo];
        sys.acc0[o] = A.acc0[xo];
        sys.yscale[o] = A.yscale[xo];
        sys.err[o] = A.err[xo];
    }
    sys.rm3[b] = A.rm3[x];
    sys.nnd[b] = A.nnd[x];
    // nearest neighbours are sources (local index = system index)
    sys.nni[b] = A.nni[x];
    if (sys.density) sys.migt[b] = A.migt[x];
}

}  // namespace

int resident_block_size(int n)
{
    if (n > 640) { const int bpt = n <= 1024 ? 2 : 4; n = (n + bpt - 1) / bpt; }
    int b = ((n + kWave - 1) / kWave) * kWave;
    if (b < kWave) b = kWave;
    if (b > 1024) b = 1024;
    return b;
}

size_t resident_lds_bytes(int nmax) { return 2 * (size_t)nmax * sizeof(double4); }

namespace {

size_t lds_f_bytes(int nmax, int lf) { return lf ? (size_t)nmax * (6 * lf + 1) * sizeof(double) : 0; }

template <int INTEG, bool GAS>
void launch_bpt(hipStream_t st, ResSystem *systems, int nsys, const ResArrays &A, int max_steps, int block,
                int bpt, int nmax, size_t lds, int lf)
{
    if (bpt == 1 && lf == 12) {
        hipLaunchKernelGGL((k_resident<INTEG, 1, 12, GAS>), dim3(nsys), dim3(block), lds + lds_f_bytes(nmax, 12),
                           st, systems, A, max_steps, nmax);
        return;
    }
    if constexpr (INTEG == INTEG_RKF78) {
        if (bpt == 1 && lf == 4) {
            hipLaunchKernelGGL((k_resident<INTEG, 1, 4, GAS>), dim3(nsys), dim3(block), lds + lds_f_bytes(nmax, 4),
                               st, systems, A, max_steps, nmax);
            return;
        }
    }
    switch (bpt) {
    case 1:
        hipLaunchKernelGGL((k_resident<INTEG, 1, 0, GAS>), dim3(nsys), dim3(block), lds, st, systems, A,
                           max_steps, nmax);
        break;
    case 2:
        if constexpr (INTEG == INTEG_RK4) {
            if (block > 512) {
                hipLaunchKernelGGL((k_resident_rk4_w2<GAS>), dim3(nsys), dim3(block), lds, st, systems, A,
                                   max_steps, nmax);
                break;
            }
        }
        hipLaunchKernelGGL((k_resident<INTEG, 2, 0, GAS>), dim3(nsys), dim3(block), lds, st, systems, A,
                           max_steps, nmax);
        break;
    default:
        hipLaunchKernelGGL((k_resident<INTEG, 4, 0, GAS>), dim3(nsys), dim3(block), lds, st, systems, A,
                           max_steps, nmax);
        break;
    }
}

template <int INTEG>
void launch_integ(hipStream_t st, ResSystem *systems, int nsys, const ResArrays &A, int max_steps, int block,
                  int bpt, int nmax, size_t lds, int lf)
{
    if (A.gas_on) launch_bpt<INTEG, true>(st, systems, nsys, A, max_steps, block, bpt, nmax, lds, lf);
    else launch_bpt<INTEG, false>(st, systems, nsys, A, max_steps, block, bpt, nmax, lds, lf);
}

template <int INTEG>
void launch_queue_bpt(hipStream_t st, ResSystem *systems, const int32_t *order, QueueWords *q, const ResArrays &A,
                      int grid, int block, int bpt, int nmax, size_t lds, int max_lsh, int lf)
{
    if constexpr (INTEG == INTEG_RKF78) {
        if (bpt == 1 && lf == 4 && block <= 640) {
            hipLaunchKernelGGL((k_resident_queue<INTEG, 1, 640, 4>), dim3(grid), dim3(block),
                               lds + lds_f_bytes(nmax, 4), st, systems, order, q, A, nmax, max_lsh);
            return;
        }
    }
    switch (bpt) {
    case 1:
        if (block > 640)
            hipLaunchKernelGGL((k_resident_queue<INTEG, 1, 768>), dim3(grid), dim3(block), lds, st, systems, order,
                               q, A, nmax, max_lsh);
        else
            hipLaunchKernelGGL((k_resident_queue<INTEG, 1, 640>), dim3(grid), dim3(block), lds, st, systems, order,
                               q, A, nmax, max_lsh);
        break;
    case 2:
        hipLaunchKernelGGL((k_resident_queue<INTEG, 2, 512>), dim3(grid), dim3(block), lds, st, systems, order,
                           q, A, nmax, 0);
        break;
    default:
        hipLaunchKernelGGL((k_resident_queue<INTEG, 4, 512>), dim3(grid), dim3(block), lds, st, systems, order,
                           q, A, nmax, 0);
        break;
    }
}

template <int INTEG>
const void *queue_kernel(int bpt, int block, int lf)
{
    if constexpr (INTEG == INTEG_RKF78)
        if (bpt == 1 && lf == 4 && block <= 640) return (const void *)k_resident_queue<INTEG, 1, 640, 4>;
    return bpt == 1 ? (block > 640 ? (const void *)k_resident_queue<INTEG, 1, 768>
                                   : (const void *)k_resident_queue<INTEG, 1, 640>)
         : bpt == 2 ? (const void *)k_resident_queue<INTEG, 2, 512>
                    : (const void *)k_resident_queue<INTEG, 4, 512>;
}

}  // namespace

int resident_queue_bpt(int block, int nmax) { return nmax <= block ? 1 : nmax <= 2 * block ? 2 : 4; }

void launch_resident_queue(hipStream_t st, int integ, ResSystem *systems, const int32_t *order, QueueWords *q,
                           const ResArrays &A, int grid, int block, int nmax, int max_lsh, int lf)
{
    const size_t lds = resident_lds_bytes(nmax);
    const int bpt = resident_queue_bpt(block, nmax);
    hipLaunchKernelGGL(k_zero_i32, dim3(1), dim3(1), 0, st, &q->head);
    switch (integ) {
    case INTEG_RKF78:
        launch_queue_bpt<INTEG_RKF78>(st, systems, order, q, A, grid, block, bpt, nmax, lds,
                                      max_lsh, lf);
        break;
    case INTEG_RK4:
        launch_queue_bpt<INTEG_RK4>(st, systems, order, q, A, grid, block, bpt, nmax, lds,
                                    max_lsh, 0);
        break;
    default:
        launch_queue_bpt<INTEG_DP>(st, systems, order, q, A, grid, block, bpt, nmax, lds,
                                   max_lsh, 0);
        break;
    }
}

size_t resident_queue_lds_f(int nmax) { return lds_f_bytes(nmax, 4); }

int resident_queue_occupancy(int integ, int block, int nmax, int lf)
{
    const int bpt = resident_queue_bpt(block, nmax);
    if (integ != INTEG_RKF78 || bpt != 1 || block > 640) lf = 0;
    const size_t lds = resident_lds_bytes(nmax) + lds_f_bytes(nmax, lf == 4 ? 4 : 0);
    const void *f = integ == INTEG_RKF78 ? queue_kernel<INTEG_RKF78>(bpt, block, lf)
                  : integ == INTEG_RK4   ? queue_kernel<INTEG_RK4>(bpt, block, 0)
                                         : queue_kernel<INTEG_DP>(bpt, block, 0);
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, block, lds) != hipSuccess || per_cu < 1) per_cu = 1;
    return per_cu;
}

// LDS-held stage derivatives for nmax bodies at one body per thread within
// lds_limit bytes: all but the last stage's (12), else RKF78's four
// most-read (4), else none (0).
static int pick_lds_slots(int integ, int nmax, size_t lds_limit)
{
    const size_t base = resident_lds_bytes(nmax);
    if (lds_limit == 0) return 0;
    if (base + lds_f_bytes(nmax, 12) <= lds_limit) return 12;
    if (integ == INTEG_RKF78 && base + lds_f_bytes(nmax, 4) <= lds_limit) return 4;
    return 0;
}

// Bodies per thread: the smallest of 1, 2, 4 that covers nmax.  A block of
// more than 640 threads, or of more than 512 that does not cover nmax, is
// narrowed to 512; one too small for 4 per thread is widened to the
// smallest that is not.  With lds_limit > 0 (a single system), one body
// per thread keeps stage derivatives in LDS when they fit in lds_limit
// bytes.
void launch_resident(hipStream_t st, int integ, ResSystem *systems, int nsys, const ResArrays &A, int max_steps,
                     int block, int nmax, size_t lds_limit)
{
    const size_t lds = resident_lds_bytes(nmax);
    if (block > 640 || (block > 512 && nmax > block)) block = 512;
    if (block * 4 < nmax) block = ((nmax + 3) / 4 + kWave - 1) / kWave * kWave;
    int bpt = nmax <= block ? 1 : nmax <= 2 * block ? 2 : 4;
    const char *w2 = getenv("SOLARIS_AMD_RK4_W2");
    if (integ == INTEG_RK4 && bpt == 4 && nmax <= 1280 && !(w2 && w2[0] == '0')) {
        // two bodies per thread in k_resident_rk4_w2 (up to 640 threads):
        // at four, the stage arrays spill (103 VGPRs against 26)
        block = ((nmax + 1) / 2 + kWave - 1) / kWave * kWave;
        bpt = 2;
    }
    const int lf = bpt == 1 ? pick_lds_slots(integ, nmax, lds_limit) : 0;
    switch (integ) {
    case INTEG_RKF78: launch_integ<INTEG_RKF78>(st, systems, nsys, A, max_steps, block, bpt, nmax, lds, lf); break;
    case INTEG_RK4: launch_integ<INTEG_RK4>(st, systems, nsys, A, max_steps, block, bpt, nmax, lds, lf); break;
    default: launch_integ<INTEG_DP>(st, systems, nsys, A, max_steps, block, bpt, nmax, lds, lf); break;
    }
}

namespace {

template <int INTEG, int LF, bool GAS>
hipError_t grid_launch(hipStream_t st, ResSystem *systems, int nslices, const ResArrays &A, int max_steps,
                       int block, int nmax, size_t lds)
{
    const void *f = (const void *)k_resident_grid<INTEG, LF, GAS>;
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_resident_grid<INTEG, LF, GAS>), dim3(nslices), dim3(block), lds, st, systems, A,
                       max_steps, nmax);
    return hipGetLastError();
}

template <int INTEG, bool GAS>
const void *grid_kernel_lf(int lf)
{
    if (lf == 12) return (const void *)k_resident_grid<INTEG, 12, GAS>;
    if constexpr (INTEG == INTEG_RKF78) {
        if (lf == 4) return (const void *)k_resident_grid<INTEG, 4, GAS>;
    }
    return (const void *)k_resident_grid<INTEG, 0, GAS>;
}

// The grid kernel of an integrator, LDS slot count and gas choice.
const void *grid_kernel(int integ, int lf, bool gas)
{
    switch (integ) {
    case INTEG_RKF78: return gas ? grid_kernel_lf<INTEG_RKF78, true>(lf) : grid_kernel_lf<INTEG_RKF78, false>(lf);
    case INTEG_RK4: return gas ? grid_kernel_lf<INTEG_RK4, true>(lf) : grid_kernel_lf<INTEG_RK4, false>(lf);
    default: return gas ? grid_kernel_lf<INTEG_DP, true>(lf) : grid_kernel_lf<INTEG_DP, false>(lf);
    }
}

template <int INTEG, bool GAS>
hipError_t grid_launch_lf(hipStream_t st, ResSystem *systems, int nslices, const ResArrays &A, int max_steps,
                          int block, int nmax, size_t lds, int lf)
{
    if (lf == 12) return grid_launch<INTEG, 12, GAS>(st, systems, nslices, A, max_steps, block, nmax, lds);
    if constexpr (INTEG == INTEG_RKF78) {
        if (lf == 4) return grid_launch<INTEG, 4, GAS>(st, systems, nslices, A, max_steps, block, nmax, lds);
    }
    return grid_launch<INTEG, 0, GAS>(st, systems, nslices, A, max_steps, block, nmax, lds);
}

}  // namespace

static size_t resident_grid_lds(int integ, int nmax, size_t lds_limit, int *lf)
{
    const int l = pick_lds_slots(integ, nmax, lds_limit);
    if (lf) *lf = l;
    return resident_lds_bytes(nmax) + lds_f_bytes(nmax, l);
}

hipError_t launch_resident_grid(hipStream_t st, int integ, ResSystem *systems, int nslices, const ResArrays &A,
                                int max_steps, int block, int nmax, size_t lds_limit)
{
    if (block > 256 || nmax > block || A.sync == nullptr || A.nsync != nslices || nslices > kGridMaxSlices)
        return hipErrorInvalidValue;
    int lf = 0;
    const size_t lds = resident_grid_lds(integ, nmax, lds_limit, &lf);
    hipLaunchKernelGGL(k_zero_sync, dim3(1), dim3(256), 0, st, A.sync);
    const bool gas = A.gas_on != 0;
    switch (integ) {
    case INTEG_RKF78:
        return gas ? grid_launch_lf<INTEG_RKF78, true>(st, systems, nslices, A, max_steps, block, nmax, lds, lf)
                   : grid_launch_lf<INTEG_RKF78, false>(st, systems, nslices, A, max_steps, block, nmax, lds, lf);
    case INTEG_RK4:
        return gas ? grid_launch_lf<INTEG_RK4, true>(st, systems, nslices, A, max_steps, block, nmax, lds, lf)
                   : grid_launch_lf<INTEG_RK4, false>(st, systems, nslices, A, max_steps, block, nmax, lds, lf);
    default:
        return gas ? grid_launch_lf<INTEG_DP, true>(st, systems, nslices, A, max_steps, block, nmax, lds, lf)
                   : grid_launch_lf<INTEG_DP, false>(st, systems, nslices, A, max_steps, block, nmax, lds, lf);
    }
}

int resident_grid_capacity(int integ, int block, int nmax, size_t lds_limit, int cu_count, bool gas)
{
    int lf = 0;
    const size_t lds = resident_grid_lds(integ, nmax, lds_limit, &lf);
    const void *f = grid_kernel(integ, lf, gas);
    if (lds > 65536 && hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return 0;
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, block, lds) != hipSuccess) return 0;
    return per_cu * cu_count;
}

void launch_slice_scatter(hipStream_t st, const SliceMap &m, const SliceArrays &sys, const ResArrays &A)
{
    const int64_t total = (int64_t)m.nslices * m.stride;
    hipLaunchKernelGGL(k_slice_scatter, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, m, sys, A);
}

void launch_slice_gather(hipStream_t st, const SliceMap &m, const SliceArrays &sys, const ResArrays &A)
{
    hipLaunchKernelGGL(k_slice_gather, dim3((unsigned)((m.n + 255) / 256)), dim3(256), 0, st, m, sys, A);
}

}  // namespace sol
