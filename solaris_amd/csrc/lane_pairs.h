// lane_pairs.h -- pair sums with the sources over the lanes of a wave.
//
// A lane holds a source and meets a few sinks whose positions are
// wave-uniform (scalar registers); the wave's sums are reduced over its lanes
// by a reduce-scatter.  This fills the chip for a few thousand sinks, where a
// sink per lane would leave most of it idle.  Used by mesh.hip and
// noalloc.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

namespace sol {

__device__ __forceinline__ double uniform(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// a summed over the two halves of the wave in the lower lanes, b in the
// upper ones (v_permlane32_swap: a's upper half against b's lower half).
__device__ __forceinline__ double fold32(double a, double b)
{
    const long long ab = __double_as_longlong(a), bb = __double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)ab, (unsigned)bb, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(ab >> 32), (unsigned)(bb >> 32), false, false);
    const double p = __longlong_as_double(((long long)hi[0] << 32) | lo[0]);
    const double q = __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
    return p + q;
}

// a summed over pairs of rows of 16 lanes in the even rows, b in the odd ones.
__device__ __forceinline__ double fold16(double a, double b)
{
    const long long ab = __double_as_longlong(a), bb = __double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)ab, (unsigned)bb, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(ab >> 32), (unsigned)(bb >> 32), false, false);
    const double p = __longlong_as_double(((long long)hi[0] << 32) | lo[0]);
    const double q = __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
    return p + q;
}

// a summed over the halves of each row of 16 in the lanes 0-7 of the row, b
// in the lanes 8-15 (row_ror:8).
__device__ __forceinline__ double fold8(double a, double b, bool upper)
{
    const double keep = upper ? b : a, send = upper ? a : b;
    return keep + dpp_mov<0x128>(send);
}

// Sums over each group of eight lanes, in all of them.
__device__ __forceinline__ void sum8(double (&v)[3])
{
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] += dpp_mov<0xB1>(v[k]);
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] += dpp_mov<0x4E>(v[k]);
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] += dpp_mov<0x141>(v[k]);
}

__device__ __forceinline__ double sum8(double v)
{
    v += dpp_mov<0xB1>(v);
    v += dpp_mov<0x4E>(v);
    v += dpp_mov<0x141>(v);
    return v;
}

// Sums over each group of sixteen lanes, in all of them.
__device__ __forceinline__ void sum16(double (&v)[3])
{
    sum8(v);
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] += dpp_mov<0x140>(v[k]);
}

constexpr double kFar = 1.0e30;    // AU: where a lane without a source has one of no mass

// NT pair terms, of sources p[m % KC] with sinks b0 + m / KC (at (sx, sy,
// sz)[b], squared softening eps2[b]), added to (ax, ay, az)[b].  OWN: leaves
// out the term of a source j[u] with itself (own[b]).  Step by step over the
// NT, with the order kept: left to itself the compiler forms them one after
// the other, each a chain of dependent operations (5.6 instead of 2.9 us of
// pair terms per stage at 1,501 bodies).
template <bool OWN, int NT, int KC, int SB>
__device__ __forceinline__ void pair_terms(int b0, const double4 (&p)[KC], const int (&j)[KC], const double (&sx)[SB],
                                           const double (&sy)[SB], const double (&sz)[SB], const double (&eps2)[SB],
                                           const int (&own)[SB], double c15, double c1875, double (&ax)[SB],
                                           double (&ay)[SB], double (&az)[SB])
{
#define PAIR_STEP(...)                                                                                                 \
    do {                                                                                                               \
        _Pragma("unroll") for (int m = 0; m < NT; ++m) {                                                               \
            const int b = b0 + m / KC, u = m % KC;                                                                     \
            (void)b; (void)u;                                                                                          \
            __VA_ARGS__;                                                                                               \
        }                                                                                                              \
        __builtin_amdgcn_sched_barrier(0);                                                                             \
    } while (0)
    double dx[NT], dy[NT], dz[NT], r[NT], y[NT], t[NT], e[NT], f[NT];
    PAIR_STEP(dx[m] = p[u].x - sx[b]; dy[m] = p[u].y - sy[b]; dz[m] = p[u].z - sz[b]);
    PAIR_STEP(r[m] = __builtin_fma(dx[m], dx[m], eps2[b]));
    PAIR_STEP(r[m] = __builtin_fma(dy[m], dy[m], r[m]));
    PAIR_STEP(r[m] = __builtin_fma(dz[m], dz[m], r[m]); if (OWN) r[m] = j[u] == own[b] ? 1.0 : r[m]);
    PAIR_STEP(y[m] = __builtin_amdgcn_rsq(r[m]));
    PAIR_STEP(t[m] = y[m] * y[m]);
    PAIR_STEP(e[m] = __builtin_fma(-r[m], t[m], 1.0); y[m] = t[m] * y[m]);
    PAIR_STEP(t[m] = __builtin_fma(c1875, e[m], c15); f[m] = p[u].w * y[m];
              if (OWN) f[m] = j[u] == own[b] ? 0.0 : f[m]);
    PAIR_STEP(t[m] = e[m] * t[m]);
    PAIR_STEP(f[m] = __builtin_fma(f[m], t[m], f[m]));
    PAIR_STEP(ax[b] = __builtin_fma(f[m], dx[m], ax[b]); ay[b] = __builtin_fma(f[m], dy[m], ay[b]);
              az[b] = __builtin_fma(f[m], dz[m], az[b]));
#undef PAIR_STEP
}

// Lanes that hold one sink's sums after pair_reduce<SB>.
template <int SB>
constexpr int pair_lanes() { return SB == 2 ? 32 : SB == 4 ? 16 : 8; }

// The sums of SB sinks over the wave: lane l gets those of sink l /
// pair_lanes<SB>() (of none past SB) in r.  Lane swaps that halve the values
// at each level, then sums over the lanes of a sink.
template <int SB>
__device__ __forceinline__ void pair_reduce(const double (&ax)[SB], const double (&ay)[SB], const double (&az)[SB],
                                            int lane, double (&r)[3])
{
    constexpr int G = pair_lanes<SB>();
    double v[3][8];
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        v[0][b] = v[1][b] = v[2][b] = 0.0;
        if (b < SB) {
            v[0][b] = ax[b]; v[1][b] = ay[b]; v[2][b] = az[b];
        }
    }
    if constexpr (G == 32) {
#pragma unroll
        for (int k = 0; k < 3; ++k) r[k] = fold32(v[k][0], v[k][1]);
#pragma unroll
        for (int k = 0; k < 3; ++k) r[k] = fold16(r[k], r[k]);
        sum16(r);
    } else if constexpr (G == 16) {
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int m = 0; m < 2; ++m) v[k][m] = fold32(v[k][m], v[k][m + 2]);
#pragma unroll
        for (int k = 0; k < 3; ++k) r[k] = fold16(v[k][0], v[k][1]);
        sum16(r);
    } else {
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int m = 0; m < 4; ++m) v[k][m] = fold32(v[k][m], v[k][m + 4]);
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int m = 0; m < 2; ++m) v[k][m] = fold16(v[k][m], v[k][m + 2]);
#pragma unroll
        for (int k = 0; k < 3; ++k) r[k] = fold8(v[k][0], v[k][1], (lane & 8) != 0);
        sum8(r);
    }
}

}  // namespace sol
