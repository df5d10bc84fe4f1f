// quad.h -- whole Driver loops of systems with few sources, four lanes per
// body (quad.hip).
#pragma once

#include "resident.h"

namespace sol {

// Limits of the quad form: workgroups, and the bodies besides the star that
// are a source of some other (every wave integrates all of them).
constexpr int kQuadMaxGroups = 256;
constexpr int kQuadMaxSources = 8;
constexpr int kQuadThreads = 256;
constexpr int kQuadGasBodies = 128;     // places of a workgroup with gas, at most: four threads each

// Exchange words of one system's workgroups.  words[p][k][w] is half k of
// workgroup w's error maximum of exchange x (p = x & 1), x | event << 31 in
// its upper half, so that a reader needs no flag of its own.  System-scope
// atomics only.
struct QuadSync {
    uint32_t error, pad[31];
    unsigned long long words[2][2][kQuadMaxGroups];
};

struct QuadArgs {
    // the descriptor, by value, and where it goes at the end
    ResSystem system_in;
    ResSystem *system;
    QuadSync *sync;
    int32_t sources;           // bodies [1, 1 + sources) are integrated by every wave (with gas: workgroup)
    int32_t groups;
    int32_t own;               // bodies of its own a wave (with gas: a workgroup) has
    // read: state, k^2 m and masses; written at the end (component stride tot),
    // none of them read by the launch: the state, the previous state, the Driver's arrays and the side outputs
    int64_t tot;
    const double *y0_in, *gm, *mass, *radius;
    double *y0, *y, *acc0, *yscale, *err, *rm3, *nnd;
    int32_t *nni;
    uint64_t ticks;            // real-time-counter ticks a wait lasts before it gives up
    // gas: the drag bodies' parameters, and migration (read, written at the
    // end): types, and the caches of the Driver's first evaluation and of the
    // last evaluation's drag
    GasDev gas;
    const double *density, *cd, *gs, *ge, *stop, *migc_in;
    const int32_t *migt_in;
    int32_t *migt;
    double *migc, *dragc;
    int32_t mig_do1, mig_do2;
};

// Workgroups for n bodies (0: the system does not fit).
int quad_groups(int n, int sources, int cus);

// Whether the workgroups of that launch exchange words: several of them, and
// decisions to combine (RK4 has events only).  Only then are the words zeroed
// and A.sync->error has a meaning.
bool quad_exchanges(int integ, const QuadArgs &a);
// Zeroes the exchange words and runs max_steps accepted steps of integrator
// `integ`.  The a.groups workgroups have to be resident at once, and
// quad_capacity (quad_gas_capacity) asked for this device before.
hipError_t launch_quad(hipStream_t st, int integ, const QuadArgs &a, int max_steps);
// The same with gas: workgroups of `places` bodies (the sources and a.own).
hipError_t launch_quad_gas(hipStream_t st, int integ, const QuadArgs &a, int places, int max_steps);
// Workgroups of these launches the device holds at once.
int quad_capacity(int integ, int sources, int cu_count);
int quad_gas_capacity(int integ, int sources, int places, int cu_count);

}  // namespace sol
