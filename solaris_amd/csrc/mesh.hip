// mesh.hip -- whole Driver loops of self-gravitating systems over several
// workgroups.
//
// A system whose bodies all pull on each other has n^2 pair terms per
// evaluation: in one workgroup (resident.hip) that is one of 256 CUs, and
// over one launch per stage (context.cpp) a system of a few thousand bodies
// spends its time in launches.  Here one launch runs the Driver loops of
// RKF78, RK4 or Dormand-Prince with the caller loop's clipping (the control
// flow of run_system in resident.hip) with every workgroup owning `share`
// bodies: it evaluates their accelerations from all sources, keeps their
// state and stage derivatives in LDS, and per stage publishes their next
// positions to the other workgroups.
//
// What bounds it: up to about 500 bodies the latency of an exchange (a store
// to memory, a flag, a poll and the loads of the others' positions, some
// 3,500 of 9,500 cycles per stage) and of the chain around it; above, the
// FP64 pair terms, at two waves per SIMD, where an operation takes 5.9 cycles
// and not the 4.9 of four.  RKF78 per attempt (13 evaluations): 257 bodies 58 us
// (one workgroup 459, one launch per stage 609), 1,501 bodies 117 us (11,900
// and 643), 5,001 bodies 455 us (one launch per stage 470).
//
// Exchange.  A workgroup writes its bodies' (x, y, z) to one of two global
// buffers with system-scope stores, waits until they are in place, and raises
// its own flag word to the exchange's number; a wait polls all flags, and the
// positions are read with system-scope loads.  (Plain loads behind an acquire
// fence measured slower: 11.0 against 9.4 us per stage at 1,501 bodies, as
// each of 27 workgroups per chiplet empties the L2 that the others are
// filling.)  One buffer is rewritten only two exchanges later, when every
// reader has raised the flag in between.  The final state of an attempt is
// published with the workgroup's error maximum, so that an accepted step's
// first evaluation needs no exchange of its own.  Waits are bounded (ticks):
// a workgroup that is not resident ends the launch with RES_SYNC_ERROR, and
// nothing the host keeps has been written.
//
// Pair sums.  The eight waves are four groups of the workgroup's bodies
// (SB each) by two halves of the sources (chunks of 64, alternately).  A
// thread holds one source and meets its wave's bodies, whose positions are
// wave-uniform (scalar registers): no LDS in the loop.  A wave's sums are
// reduced over its lanes by a reduce-scatter (lane swaps that halve the
// values at each level), and the two halves are added through LDS.  The
// indirect term's sum over the sources is the pair sum of a body at the
// origin, which takes the last place of the workgroup's SB x 4.
#include <float.h>

#include <algorithm>
#include <type_traits>

#include "lane_pairs.h"
#include "mesh.h"
#include "static_for.h"
#include "tableaux.h"

namespace sol {
namespace {

#define MESH_SCOPE __HIP_MEMORY_SCOPE_SYSTEM

constexpr int kMeshWaves = kMeshThreads / kWave;
constexpr int kMeshTile = 2048;                           // source records in LDS at a time
constexpr int kMeshHalves = 2;                            // of the sources
constexpr int kMeshSinkGroups = kMeshWaves / kMeshHalves; // of the workgroup's bodies

template <int INTEG>
constexpr int m_stages() { return INTEG == INTEG_RKF78 ? 12 : INTEG == INTEG_RK4 ? 3 : 8; }

__device__ __attribute__((noinline)) double mesh_pow(double x, double y) { return pow(x, y); }

// Per-launch constants of a workgroup.
struct MCtx {
    int i0, nb;                // own bodies i0 + b, b < nb
    int end;                   // their sources are [1, end)
    int base;
    double eps2;
};

// LDS of a workgroup of up to ST - 1 bodies: component k of own body b at
// [k][b].  Fixed rows, so that every access is one address plus a constant.
template <int ST>
struct MLds {
    double y[2][6][ST];            // the state y0 and the Driver's other array, by parity
    double f[13][6][ST];           // stage derivatives
    double ysc[6][ST], er[6][ST];
    double pos[3][ST], vel[3][ST]; // of the stage published last
    double gm[ST], mu[ST], rm3[ST];
    double part[kMeshHalves][3][ST];   // place ST - 1: the body at the origin
    double nnr[ST];
    double tab[13][12], tabc[13];  // the integrator's tableau and stage times
    int nni[ST];
};
#define MESH_LDS __attribute__((address_space(3)))
typedef double double2_t __attribute__((ext_vector_type(2)));

// One of the two position buffers of a system: component k of body slot j at
// p[k * stride + j].  Other workgroups write it during the launch, so it is
// read with device-coherent loads, which pass the caches by; by component, so
// that a wave's load is 512 contiguous bytes.
struct MPos {
    double *p;
    int64_t stride;
    __device__ __forceinline__ double get(int k, int j) const
    {
        return __longlong_as_double((long long)__hip_atomic_load((const unsigned long long *)(p + k * stride) + j,
                                                                 __ATOMIC_RELAXED, MESH_SCOPE));
    }
    __device__ __forceinline__ void put(int k, int j, double v) const
    {
        __hip_atomic_store((unsigned long long *)(p + k * stride) + j, (unsigned long long)__double_as_longlong(v),
                           __ATOMIC_RELAXED, MESH_SCOPE);
    }
};

// The records of up to kMeshTile sources in LDS, as two halves of 16 bytes (a
// wave's reads of either are contiguous).
struct MTile {
    MESH_LDS double2_t *xy, *zw;
    __device__ __forceinline__ double4 at(int j) const
    {
        const double2_t a = xy[j], b = zw[j];
        return make_double4(a.x, a.y, b.x, b.y);
    }
};

// Pair sums of the own bodies over the positions J (and gm = k^2 m) into
// s.part.  The sources go through LDS: every wave reads its share of a tile from memory at once,
// and the loads' latency is paid once per tile.
template <int ST>
__device__ __forceinline__ void mesh_pairs(const MCtx &c, MESH_LDS MLds<ST> &s, const MTile &tile, const MPos &J,
                                           const double *__restrict__ gm)
{
    constexpr int SB = ST / kMeshSinkGroups;         // sinks of a wave
    constexpr int NT = SB == 6 ? 3 : 4;              // pair terms at a time
    constexpr int KC = SB == 2 ? 2 : 1;              // of so many chunks
    constexpr int KW = kMeshTile / kMeshThreads;     // records of a tile a thread reads
    // opaque, so that the addresses below are formed here and not kept over
    // the step loop
    int lane = threadIdx.x & (kWave - 1);
    asm volatile("" : "+v"(lane));
    const int wave = uniform((int)threadIdx.x / kWave);
    const int half = wave % kMeshHalves, b0 = wave / kMeshHalves * SB;
    double4 q[KW];
    auto read = [&](int t0) {
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            const int j = t0 + k * kMeshThreads + wave * kWave;
            if (j < c.end) {
                const int i = min(j + lane, c.end - 1);
                q[k].x = J.get(0, i);
                q[k].y = J.get(1, i);
                q[k].z = J.get(2, i);
                q[k].w = gm[i];
            }
        }
    };
    read(1);
    double sx[SB], sy[SB], sz[SB], eps2[SB], ax[SB], ay[SB], az[SB];
    int own[SB];
#pragma unroll
    for (int b = 0; b < SB; ++b) {
        const int i = min(b0 + b, c.nb - 1);
        const bool origin = b0 + b == ST - 1;
        sx[b] = uniform(origin ? 0.0 : s.pos[0][i]);
        sy[b] = uniform(origin ? 0.0 : s.pos[1][i]);
        sz[b] = uniform(origin ? 0.0 : s.pos[2][i]);
        eps2[b] = origin ? 0.0 : c.eps2;
        own[b] = origin ? -1 : c.i0 + i;
        ax[b] = ay[b] = az[b] = 0.0;
    }
    double c15 = 1.5, c1875 = 1.875;
    asm volatile("" : "+v"(c15), "+v"(c1875));
    const int ib = c.i0 + min(b0, c.nb - 1), il = c.i0 + min(b0 + SB, c.nb) - 1;
    constexpr int step = kMeshHalves * kWave;        // from a wave's chunk to its next
    for (int t0 = 1; t0 < c.end; t0 += kMeshTile) {
        if (t0 > 1) __syncthreads();                        // the tile before is read
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            const int j = k * kMeshThreads + wave * kWave;
            if (t0 + j >= c.end) break;
            const bool on = t0 + j + lane < c.end;      // past the end: a far source of no mass
            tile.xy[j + lane] = double2_t{on ? q[k].x : kFar, on ? q[k].y : kFar};
            tile.zw[j + lane] = double2_t{on ? q[k].z : kFar, on ? q[k].w : 0.0};
        }
        __syncthreads();
        if (t0 + kMeshTile < c.end) read(t0 + kMeshTile);
        const int t1 = min(c.end - t0, kMeshTile);
        for (int jk = half * kWave; jk < t1; jk += KC * step) {
            double4 p[KC];
            int j[KC];
#pragma unroll
            for (int u = 0; u < KC; ++u) {
                j[u] = t0 + jk + u * step + lane;
                p[u] = make_double4(kFar, kFar, kFar, 0.0);
                if (jk + u * step < t1) p[u] = tile.at(jk + u * step + lane);
            }
            const bool apart = t0 + jk + (KC - 1) * step + kWave <= ib || t0 + jk > il;
            auto sets = [&](auto own_c) {
#pragma unroll
                for (int b = 0; b < SB; b += NT / KC)
                    pair_terms<decltype(own_c)::value, NT, KC, SB>(b, p, j, sx, sy, sz, eps2, own, c15, c1875, ax, ay, az);
            };
            if (apart) sets(std::false_type{});
            else sets(std::true_type{});
        }
    }
    double r[3];
    pair_reduce<SB>(ax, ay, az, lane, r);
    constexpr int G = pair_lanes<SB>();
    const int m = lane / G, k = lane % G;
    if (k < 3 && m < SB) s.part[half][k][b0 + m] = k == 0 ? r[0] : k == 1 ? r[1] : r[2];
}

// Nearest source of each own body (the first of equals) into s.nnr (its
// squared distance) and s.nni (-1: none).  A wave takes every eighth body,
// U of them at a time.
template <int U, int ST, typename Get>
__device__ __forceinline__ void mesh_nearest(const MCtx &c, MESH_LDS MLds<ST> &s, Get &&record)
{
    int lane = threadIdx.x & (kWave - 1);
    asm volatile("" : "+v"(lane));
    const int wave = uniform((int)threadIdx.x / kWave);
    double sx[U], sy[U], sz[U], best[U];
    int bidx[U], me[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int b = min(wave + u * kMeshWaves, c.nb - 1);
        sx[u] = uniform(s.pos[0][b]); sy[u] = uniform(s.pos[1][b]); sz[u] = uniform(s.pos[2][b]);
        best[u] = DBL_MAX; bidx[u] = -1;
        me[u] = c.i0 + b;
    }
    for (int j0 = 1; j0 < c.end; j0 += 4 * kWave) {
        double4 q[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) q[k] = record(min(j0 + k * kWave + lane, c.end - 1));
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int j = j0 + k * kWave + lane;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const double dx = q[k].x - sx[u], dy = q[k].y - sy[u], dz = q[k].z - sz[u];
                const double r2 = dx * dx + dy * dy + dz * dz;
                if (j < c.end && j != me[u] && r2 < best[u]) { best[u] = r2; bidx[u] = j; }
            }
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        double d = best[u];
        int id = bidx[u];
        for (int o = 32; o >= 1; o >>= 1) {
            const double d2 = __shfl_xor(d, o, kWave);
            const int i2 = __shfl_xor(id, o, kWave);
            if (i2 >= 0 && (id < 0 || d2 < d || (d2 == d && i2 < id))) { d = d2; id = i2; }
        }
        const int b = wave + u * kMeshWaves;
        if (lane == 0 && b < c.nb) { s.nnr[b] = d; s.nni[b] = id; }
    }
}

template <int ST>
__device__ __forceinline__ void mesh_evaluate(const MCtx &c, MESH_LDS MLds<ST> &s, const MTile &tile,
                                              const MPos &J, const double *gm, bool nearest)
{
    mesh_pairs<ST>(c, s, tile, J, gm);
    if (nearest) {
        constexpr int U = (ST + kMeshWaves - 1) / kMeshWaves;
        if (c.end - 1 <= kMeshTile) mesh_nearest<U, ST>(c, s, [&](int j) { return tile.at(j - 1); });
        else mesh_nearest<U, ST>(c, s, [&](int j) { return make_double4(J.get(0, j), J.get(1, j), J.get(2, j), 0.0); });
    }
    __syncthreads();
}

typedef MESH_LDS double lds_d;

// Tableau rows in LDS: a row's entries past its stage are 0.
template <int INTEG>
constexpr int m_terms() { return INTEG == INTEG_RKF78 ? 12 : INTEG == INTEG_RK4 ? 3 : 8; }
template <int INTEG>
__device__ __forceinline__ double m_entry(int s, int l)
{
    return INTEG == INTEG_RKF78 ? tab::kRkfD[s][l] : INTEG == INTEG_RK4 ? tab::kRk4A[s][l] : tab::kDpA[s][l];
}

// State of the stage whose tableau row is d: position and velocity of one
// component of one body, its state at y0 (velocity three rows on) and its
// derivatives at F.  All terms, so that the reads overlap: derivatives of
// later stages are finite and have coefficient 0.
template <int INTEG, int st>
__device__ __forceinline__ void mesh_stage(const lds_d *y0, const lds_d *F, const lds_d *d, double cs, double h,
                                           double &pos, double &vel)
{
    constexpr int NT = m_terms<INTEG>();
    const double p0 = y0[0], v0 = y0[3 * st];
    double fp[NT], fv[NT], k[NT];
#pragma unroll
    for (int l = 0; l < NT; ++l) {
        k[l] = d[l];
        if (INTEG != INTEG_DP) fp[l] = F[l * 6 * st];
        fv[l] = F[(l * 6 + 3) * st];
    }
    __builtin_amdgcn_sched_barrier(0);
    double ap = 0.0, av = 0.0;
#pragma unroll
    for (int l = 0; l < NT; ++l) {
        if (INTEG != INTEG_DP) ap += k[l] * fp[l];
        av += k[l] * fv[l];
    }
    if (INTEG == INTEG_DP) {
        pos = p0 + cs * h * v0 + h * h * (av);
        vel = v0 + h * (av);
    } else {
        pos = p0 + h * ap;
        vel = v0 + h * av;
    }
}

// Final state and error estimate (into er); the error ratio (RKF78: max
// |err / yscale| of the two components, Dormand-Prince: the position error).
template <int INTEG, int st>
__device__ __forceinline__ double mesh_final(const lds_d *y0, const lds_d *F, const lds_d *ysc, lds_d *er, double h,
                                             double &pos, double &vel)
{
    const double p0 = y0[0], v0 = y0[3 * st];
    double ratio = 0.0;
    if constexpr (INTEG == INTEG_RKF78) {
        // RungeKuttaFehlberg78.cpp:231-248
        constexpr double b0 = 41.0 / 840.0, b5 = 34.0 / 105.0, b6 = 9.0 / 35.0, b8 = 9.0 / 280.0, b10 = 41.0 / 840.0;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const lds_d *G = F + 3 * half * st;
            auto f = [&](int l) { return G[l * 6 * st]; };
            const double y = (half ? v0 : p0) +
                             h * (b0 * f(0) + b5 * f(5) + b6 * (f(6) + f(7)) + b8 * (f(8) + f(9)) + b10 * f(10));
            const double e = h * fabs(f(0) + f(10) - f(11) - f(12)) * 41.0 / 840.0;
            er[3 * half * st] = e;
            ratio = fmax(ratio, fabs(e / ysc[3 * half * st]));
            if (half) vel = y; else pos = y;
        }
    } else if constexpr (INTEG == INTEG_RK4) {
        auto f = [&](int l, int half) { return F[(l * 6 + 3 * half) * st]; };
        pos = p0 + h * (tab::kRk4B[0] * f(0, 0) + tab::kRk4B[1] * f(1, 0) + tab::kRk4B[2] * f(2, 0) +
                        tab::kRk4B[3] * f(3, 0));
        vel = v0 + h * (tab::kRk4B[0] * f(0, 1) + tab::kRk4B[1] * f(1, 1) + tab::kRk4B[2] * f(2, 1) +
                        tab::kRk4B[3] * f(3, 1));
    } else {
        // DormandPrince.cpp:455-491
        constexpr const double *B = tab::kDpB, *Bd = tab::kDpBdh;
        const double h2 = h * h;
        auto f = [&](int l) { return F[(l * 6 + 3) * st]; };
        pos = p0 + h * v0 + h2 * (B[0] * f(0) + B[4] * f(4) + B[5] * f(5) + B[6] * f(6) + B[7] * f(7) + B[8] * f(8));
        vel = v0 + h * (Bd[0] * f(0) + Bd[4] * f(4) + Bd[5] * f(5) + Bd[6] * f(6) + Bd[7] * f(7));
        ratio = h2 * fabs(f(7) - f(8)) / 20.0;
        er[0] = ratio;
        er[3 * st] = 0.0;
    }
    return ratio;
}

__device__ __forceinline__ double mesh_wmax(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmax(v, __shfl_xor(v, o, kWave));
    return v;
}

template <int INTEG, int ST>
__global__ __launch_bounds__(kMeshThreads) void k_mesh(MeshArgs A, int max_steps, int tile_records)
{
    __shared__ MLds<ST> lds;
    MESH_LDS MLds<ST> &s = *(MESH_LDS MLds<ST> *)&lds;
    extern __shared__ __attribute__((aligned(16))) unsigned char tile_lds[];
    MTile tile;
    tile.xy = (MESH_LDS double2_t *)(MESH_LDS unsigned char *)tile_lds;
    tile.zw = tile.xy + tile_records;
    __shared__ ResSystem S;
    __shared__ double sh_red[kMeshWaves];
    __shared__ double sh_val[2];
    __shared__ int sh_ok, sh_ev;
    constexpr int nst = m_stages<INTEG>();
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int pi = uniform(A.part_of[blockIdx.x]);
    const int pgroups = uniform(A.parts[pi].groups), psys = uniform(A.parts[pi].system);
    const int rank = (int)blockIdx.x - uniform(A.parts[pi].first), share = uniform(A.parts[pi].share);
    MeshSync *sy = A.sync + pi;
    if (tid == 0) S = A.systems[psys];
    __syncthreads();
    if (S.status != RES_RUNNING) return;      // the same in every workgroup of the system

    MCtx c;
    {
        // the workgroups of the first sink class, then those of the second;
        // one source range for both: one class
        const int n = uniform(S.n), ea = uniform(min(S.end_a, S.n)), eb = uniform(min(S.end_b, S.n));
        const int last = ea == eb ? n : uniform(S.nm);
        const int ga = (last - 1 + share - 1) / share;
        const bool first = rank < ga;
        c.end = first ? ea : eb;
        c.i0 = first ? 1 + rank * share : last + (rank - ga) * share;
        c.nb = min(share, (first ? last : n) - c.i0);
        c.base = uniform(S.base);
    }
    c.eps2 = A.eps2;
    // this thread's body and component (combine threads), and body (b1)
    const bool mine = tid < 3 * c.nb;
    int cj = mine ? tid / c.nb : 0, cb = mine ? tid - cj * c.nb : 0;
    const bool one_wave = 3 * c.nb <= kWave;
    int cur = 0;               // parity of y0 in s.y
    bool flushed = false;      // small numbers were flushed in this launch
    const MPos J0{A.pos + c.base, A.tot}, J1{A.pos + 3 * A.tot + c.base, A.tot};
    const double *const gm = A.gm + c.base;

    for (int q = tid; q < 6 * c.nb; q += kMeshThreads) {
        const int k = q / c.nb, b = q - k * c.nb;
        const double v = A.y0_in[k * A.tot + c.base + c.i0 + b];
        s.y[0][k][b] = v;
        s.y[1][k][b] = v;
        s.ysc[k][b] = 0.0;
        s.er[k][b] = 0.0;
        if (k < 3) s.pos[k][b] = v;
        else s.vel[k - 3][b] = v;
    }
    for (int q = tid; q < 13 * 6 * ST; q += kMeshThreads) (&s.f[0][0][0])[q] = 0.0;
    if (tid < 13 * 12) {
        const int r = tid / 12, l = tid - 12 * r;
        s.tab[r][l] = r <= nst && l < m_terms<INTEG>() ? m_entry<INTEG>(r, l) : 0.0;
        if (l == 0) s.tabc[r] = INTEG == INTEG_DP && r <= nst ? tab::kDpC[r] : 0.0;
    }
    if (tid < c.nb) {
        const double m = A.mass[c.base + c.i0 + tid];
        s.gm[tid] = kGauss2 * m;
        s.mu[tid] = kGauss2 * (A.mass[c.base] + m);
    }
    __syncthreads();

    uint32_t x = 0;            // exchanges published
    // Publishes the own bodies' positions s.pos as exchange x + 1, and val
    // with the event flag ev (thread 0's) when `with` is set.  Called by
    // every thread; s.pos was written by the combine threads themselves.
    auto publish = [&](double px, bool with, double val, int ev) {
        ++x;
        if (mine) ((x & 1) ? J1 : J0).put(cj, c.i0 + cb, px);
        if (with && tid == 0) {
            const unsigned long long e = (unsigned long long)__double_as_longlong(fabs(val)) |
                                         (ev ? 0x8000000000000000ull : 0ull);
            __hip_atomic_store(&sy->vals[x & 1][rank], e, __ATOMIC_RELAXED, MESH_SCOPE);
        }
        // the stores are in place before the flag goes up
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(0);
        if (!one_wave || x == 1) __syncthreads();
        if (tid == 0) __hip_atomic_store(&sy->flags[rank], x, __ATOMIC_RELAXED, MESH_SCOPE);
    };
    // Waits until every workgroup of the system has published exchange x.
    auto wait = [&]() -> bool {
        if (wave == 0) {
            bool ok = true;
            const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
            for (int it = 0;; ++it) {
                bool here = true;
                uint32_t v[kMeshMaxGroups / kWave];
#pragma unroll
                for (int k = 0; k < kMeshMaxGroups / kWave; ++k)
                    if (k * kWave < pgroups)
                        v[k] = __hip_atomic_load(&sy->flags[k * kWave + lane], __ATOMIC_RELAXED, MESH_SCOPE);
#pragma unroll
                for (int k = 0; k < kMeshMaxGroups / kWave; ++k)
                    if (k * kWave < pgroups) here &= k * kWave + lane >= pgroups || (int32_t)(v[k] - x) >= 0;
                if (__all(here) && A.ticks != 0) break;       // (no budget: never)
                if ((it & 7) == 7 || A.ticks == 0) {
                    if (__hip_atomic_load(&sy->error, __ATOMIC_RELAXED, MESH_SCOPE) != 0) { ok = false; break; }
                    if (__builtin_amdgcn_s_memrealtime() - t0 >= A.ticks) {
                        __hip_atomic_store(&sy->error, 1u, __ATOMIC_RELAXED, MESH_SCOPE);
                        ok = false;
                        break;
                    }
                }
            }
            if (lane == 0) sh_ok = ok ? 1 : 0;
        }
        __syncthreads();
        return sh_ok != 0;
    };
    auto leave = [&]() { if (tid == 0 && rank == 0) A.systems[psys].status = RES_SYNC_ERROR; };
    // 1 / |r|^3 of the own bodies at s.pos, for the Kepler term, by the
    // threads after the combine threads of the first wave
    auto kepler = [&]() {
        const int b = tid - (kMeshThreads - kWave);
        if (b >= 0 && b < c.nb) {
            const double px = s.pos[0][b], py = s.pos[1][b], pz = s.pos[2][b];
            const double r2 = px * px + py * py + pz * pz;
            const double r = sqrt(r2);
            s.rm3[b] = 1.0 / (r2 * r);
        }
    };
    // Stage derivative l of this thread's component from the pair sums.
    auto derivative = [&](int l) {
        if (!mine) return;
        asm volatile("" : "+v"(cj), "+v"(cb));     // addresses formed here, not kept
        const double p = s.pos[cj][cb], rm3 = s.rm3[cb];
        double t = s.part[0][cj][ST - 1] + s.part[1][cj][ST - 1];
        if (c.i0 + cb < c.end) t -= s.gm[cb] * (p * rm3);
        const double a = (s.part[0][cj][cb] + s.part[1][cj][cb]) - t;
        s.f[l][cj][cb] = s.vel[cj][cb];
        s.f[l][3 + cj][cb] = -s.mu[cb] * rm3 * p + a;
    };

    const bool events = S.clip && (S.stop_mask & SOL_STOP_EVENT) && (S.e3 > 0.0 || S.h3 > 0.0 || S.coll > 0.0);
    double px = 0.0, pv = 0.0;
    publish(mine ? s.pos[cj][cb] : 0.0, false, 0.0, 0);
    kepler();
    if (!wait()) { leave(); return; }

    // State of stage q (q <= nst) or the final state with its error maximum
    // and events, published; waits for the others'.
    auto next_state = [&](int q, double h) -> bool {
        double ratio = 0.0;
        if (mine) {
            const lds_d *y0 = &s.y[cur][cj][cb], *F = &s.f[0][cj][cb];
            if (q <= nst) {
                mesh_stage<INTEG, ST>(y0, F, &s.tab[q][0], s.tabc[q], h, px, pv);
            } else {
                ratio = mesh_final<INTEG, ST>(y0, F, &s.ysc[cj][cb], &s.er[cj][cb], h, px, pv);
                s.y[1 - cur][cj][cb] = px;
                s.y[1 - cur][3 + cj][cb] = pv;
            }
        }
        int ev = 0;
        if (q > nst) {
            // the side outputs' events and the workgroup's error maximum
            if (events) {
                if (tid < c.nb) {
                    const int i = c.i0 + tid;
                    const double r3 = s.rm3[tid];
                    if (S.e3 > 0.0 && r3 < S.e3) ev = 1;
                    if (S.h3 > 0.0 && r3 > S.h3) ev = 1;
                    const int k = s.nni[tid];
                    if (S.coll > 0.0 && k >= 0 &&
                        S.coll * (A.radius[c.base + i] + A.radius[c.base + k]) > s.nnr[tid])
                        ev = 1;
                }
                ev = __syncthreads_or(ev);
            }
            ratio = mesh_wmax(ratio);
            if (!one_wave) {
                if (lane == 0) sh_red[wave] = ratio;
                __syncthreads();
                ratio = sh_red[0];
                for (int w = 1; w < kMeshWaves; ++w) ratio = fmax(ratio, sh_red[w]);
            }
        }
        if (mine) {
            s.pos[cj][cb] = px;
            s.vel[cj][cb] = pv;
        }
        publish(px, q > nst, ratio, ev);
        __syncthreads();          // s.pos, s.vel
        kepler();
        return wait();
    };

    for (int step = 0; step < max_steps; ++step) {
        const double t0 = uniform(S.t);
        double h = uniform(S.h_next);
        int iter = 0, outcome = 0, event = 0;   // outcome: 0 accept, 2 underflow, 3 maxiter
        double errmax = 0.0;
        int q = 0;       // the stage whose positions are published: f0 at y0 first
        for (;;) {
            ++iter;
            for (;;) {
                mesh_evaluate(c, s, tile, (x & 1) ? J1 : J0, gm, q == nst);
                if (q == nst && tid < c.nb) {
                    const int id = s.nni[tid];
                    s.nnr[tid] = id >= 0 ? sqrt(s.nnr[tid]) : 0.0;
                    A.rm3[c.base + c.i0 + tid] = s.rm3[tid];
                    A.nnd[c.base + c.i0 + tid] = s.nnr[tid];
                    A.nni[c.base + c.i0 + tid] = id;
                }
                derivative(q);
                if (INTEG == INTEG_RKF78 && q == 0 && mine) {
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                        const int k = 3 * half + cj;
                        s.ysc[k][cb] = fabs(s.y[cur][k][cb]) + fabs(h * s.f[0][k][cb]) + 1.0e-30;
                    }
                }
                ++q;
                if (!next_state(q, h)) { leave(); return; }
                if (q > nst) break;
            }
            // the system's error maximum and events
            if (wave == 0) {
                double m = 0.0;
                int fl = 0;
                for (int w = lane; w < pgroups; w += kWave) {
                    const unsigned long long e = __hip_atomic_load(&sy->vals[x & 1][w], __ATOMIC_RELAXED, MESH_SCOPE);
                    m = fmax(m, __longlong_as_double((long long)(e & 0x7FFFFFFFFFFFFFFFull)));
                    fl |= (int)(e >> 63);
                }
                m = mesh_wmax(m);
                fl = __any(fl) ? 1 : 0;
                if (lane == 0) { sh_val[0] = m; sh_ev = fl; }
            }
            if (tid == 0) S.attempts += 1;
            __syncthreads();
            const double raw = uniform(sh_val[0]);
            event = uniform(sh_ev);
            if (INTEG == INTEG_RKF78) {
                errmax = raw / S.eps;
                if (errmax < 1.0) { outcome = 0; break; }
                const double htemp = 0.9 * h * mesh_pow(errmax, -0.25);
                h = uniform(fabs(htemp) > fabs(0.1 * h) ? htemp : 0.1 * h);
                if (t0 + h == t0) { outcome = 2; break; }
            } else if (INTEG == INTEG_RK4) {
                outcome = 0;
                break;
            } else {
                errmax = raw;
                const double hn = errmax < 1.0e-20 ? 2.0 * h : 0.9 * h * mesh_pow(S.eps / errmax, 1.0 / 7.0);
                __syncthreads();
                if (tid == 0) { S.h_did = h; S.h_next = hn; }
                __syncthreads();
                if (!(errmax > S.eps && iter <= 10)) { outcome = iter > 10 ? 3 : 0; break; }
                h = uniform(S.h_next);
            }
            // again, from the first stage with the new h; a non-finite
            // derivative of this attempt must not meet a coefficient 0
            if (mine) {
#pragma unroll
                for (int l = 1; l <= nst; ++l) s.f[l][cj][cb] = s.f[l][3 + cj][cb] = 0.0;
            }
            q = 1;
            if (!next_state(q, h)) { leave(); return; }
        }
        __syncthreads();
        if (outcome != 0) {
            if (tid == 0) {
                S.status = outcome == 2 ? RES_UNDERFLOW : RES_MAXITER;
                S.body_h = h;
            }
            __syncthreads();
            break;
        }
        double h_next;
        if (INTEG == INTEG_RKF78) {
            h_next = errmax > 1.89e-4 ? (0.9 * h * mesh_pow(errmax, -0.2)) : (5.0 * h);
        } else if (INTEG == INTEG_RK4) {
            h_next = h;
        } else {
            h_next = S.h_next;
            h = S.h_did;
        }
        cur = 1 - cur;     // the Driver's pointer swap
        __syncthreads();
        if (tid == 0) {
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
                S.flush_count = (S.flush_count + 1) % 100;
                flush = S.flush_count == 0;
                S.reason = reason | (stop ? SOL_STOP_END : 0);
                reason &= S.stop_mask;
            }
            if (stop || reason) S.status = stop ? RES_DONE : RES_STOPPED;
            sh_ev = flush;
        }
        __syncthreads();
        const bool flush = sh_ev != 0, end = S.status != RES_RUNNING;
        if (flush) {
            flushed = true;
            for (int q = tid; q < 6 * c.nb; q += kMeshThreads) {
                const int k = q / c.nb, b = q - k * c.nb;
                if (fabs(s.y[0][k][b]) < 1.0e-50) s.y[0][k][b] = 0.0;
                if (fabs(s.y[1][k][b]) < 1.0e-50) s.y[1][k][b] = 0.0;
            }
            __syncthreads();
            if (!end && step + 1 < max_steps) {
                // the flushed positions, published anew
                if (mine) {
                    px = s.y[cur][cj][cb];
                    s.pos[cj][cb] = px;
                    s.vel[cj][cb] = s.y[cur][3 + cj][cb];
                }
                publish(px, false, 0.0, 0);
                __syncthreads();
                kepler();
                if (!wait()) { leave(); return; }
            }
        }
        if (end) break;
    }
    __syncthreads();
    for (int q = tid; q < 6 * c.nb; q += kMeshThreads) {
        const int k = q / c.nb, b = q - k * c.nb;
        const int64_t o = k * A.tot + c.base + c.i0 + b;
        A.y0[o] = s.y[cur][k][b];
        A.y[o] = s.y[1 - cur][k][b];
        A.acc0[o] = s.f[0][k][b];
        if (INTEG == INTEG_RKF78) A.yscale[o] = s.ysc[k][b];
        if (INTEG != INTEG_RK4) A.err[o] = s.er[k][b];
    }
    if (rank == 0) {
        // the star is not integrated: no derivative, no error, no neighbour
        if (tid < 6) {
            const int64_t o = tid * A.tot + c.base;
            const double v = A.y0_in[o], w = flushed && fabs(v) < 1.0e-50 ? 0.0 : v;
            A.y0[o] = w;
            A.y[o] = w;
            A.acc0[o] = 0.0;
            if (INTEG == INTEG_RKF78) A.yscale[o] = fabs(v) + 1.0e-30;
            if (INTEG != INTEG_RK4) A.err[o] = 0.0;
        }
        if (tid == 0) {
            A.rm3[c.base] = 0.0;
            A.nnd[c.base] = 0.0;
            A.nni[c.base] = -1;
            A.systems[psys] = S;
        }
    }
}

__global__ __launch_bounds__(256) void k_mesh_zero(MeshSync *s)
{
    MeshSync *q = s + blockIdx.x;
    if (threadIdx.x == 0) q->error = 0;
    for (int i = threadIdx.x; i < kMeshMaxGroups; i += blockDim.x) {
        q->flags[i] = 0;
        q->vals[0][i] = q->vals[1][i] = 0ull;
    }
}

__global__ __launch_bounds__(256) void k_mesh_commit(MeshArgs A, ResSystem *systems, double *y0)
{
    const int psys = A.parts[blockIdx.x].system;
    const ResSystem &S = A.systems[psys];
    if (A.sync[blockIdx.x].error != 0 || S.status == RES_SYNC_ERROR) return;
    const int n = S.n;
    for (int q = threadIdx.x; q < 6 * n; q += blockDim.x) {
        const int64_t o = q / n * A.tot + S.base + q % n;
        y0[o] = A.y0[o];
    }
    if (threadIdx.x == 0) systems[psys] = S;
}

// The smallest of 8, 16, 24 and 32 places that holds `share` bodies and the
// one at the origin.
template <int INTEG>
const void *mesh_kernel_of(int share)
{
    return share <= 7    ? (const void *)k_mesh<INTEG, 8>
           : share <= 15 ? (const void *)k_mesh<INTEG, 16>
           : share <= 23 ? (const void *)k_mesh<INTEG, 24>
                         : (const void *)k_mesh<INTEG, 32>;
}

const void *mesh_kernel(int integ, int share)
{
    return integ == INTEG_RKF78 ? mesh_kernel_of<INTEG_RKF78>(share)
         : integ == INTEG_RK4   ? mesh_kernel_of<INTEG_RK4>(share)
                                : mesh_kernel_of<INTEG_DP>(share);
}

}  // namespace

int mesh_groups(int n, int nm, int end_a, int end_b, int share)
{
    const int last = std::min(end_a, n) == std::min(end_b, n) ? n : nm;
    return (last - 1 + share - 1) / share + (n - last + share - 1) / share;
}

// Full workgroups of 7, 15, 23 or 31 bodies (with the body at the origin the
// places of a kernel), the smallest that fit: at 2,049 bodies 137 groups of 15
// take 14.1 us per stage and 256 of 8 in the same kernel 16.0.
int mesh_share(int n, int nm, int end_a, int end_b, int cus)
{
    const int most = std::min(cus, kMeshMaxGroups);
    for (int share = 7; share <= kMeshMaxShare; share += 8)
        if (mesh_groups(n, nm, end_a, end_b, share) <= most) return share;
    return 0;
}

// LDS bytes of a tile for systems of up to n bodies.
static size_t mesh_tile_bytes(int n, int *records)
{
    const int r = std::min(kMeshTile, (n - 1 + kMeshThreads - 1) / kMeshThreads * kMeshThreads);
    if (records) *records = r;
    return (size_t)r * 32;
}

int mesh_capacity(int integ, int n, int share, int cu_count)
{
    const void *f = mesh_kernel(integ, share);
    const size_t lds = mesh_tile_bytes(n, nullptr);
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kMeshTile * 32) != hipSuccess) return 0;
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, kMeshThreads, lds) != hipSuccess) return 0;
    return per_cu * cu_count;
}

hipError_t launch_mesh(hipStream_t st, int integ, const MeshArgs &a, int nparts, int ngroups, int max_n,
                       int max_share, int max_steps, bool zeroed)
{
    if (nparts < 1 || ngroups < 1 || max_share < 1 || max_share > kMeshMaxShare) return hipErrorInvalidValue;
    if (!zeroed) hipLaunchKernelGGL(k_mesh_zero, dim3(nparts), dim3(256), 0, st, a.sync);
    MeshArgs args = a;
    int records = 0;
    const size_t lds = mesh_tile_bytes(max_n, &records);
    void *kargs[] = {&args, &max_steps, &records};
    return hipLaunchKernel(mesh_kernel(integ, max_share), dim3(ngroups), dim3(kMeshThreads), kargs, lds, st);
}

hipError_t launch_mesh_commit(hipStream_t st, const MeshArgs &a, int nparts, ResSystem *systems, double *y0)
{
    if (nparts < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_mesh_commit, dim3(nparts), dim3(256), 0, st, a, systems, y0);
    return hipGetLastError();
}

}  // namespace sol
