// mesh.h -- whole Driver loops of self-gravitating systems over several
// workgroups (mesh.hip).
#pragma once

#include <algorithm>

#include "resident.h"

namespace sol {

// Limits of the mesh form: workgroups per system and bodies per workgroup
// (a body's LDS rows take about 1.1 KB).
constexpr int kMeshMaxGroups = 256;
constexpr int kMeshMaxShare = 31;
constexpr int kMeshThreads = 512;

// Exchange words of one system's workgroups.  flags[w] counts the exchanges
// workgroup w has published (it only grows during a launch); vals holds the
// error maxima (the sign bit: an event), double-buffered by the parity of the
// exchange.  All accesses are system-scope atomics.
struct MeshSync {
    uint32_t error, pad[31];
    uint32_t flags[kMeshMaxGroups];
    unsigned long long vals[2][kMeshMaxGroups];
};

// One system of a mesh launch: workgroups [first, first + groups) of the
// grid, `share` bodies each (the last one the rest), in the ResSystem
// `system`.
struct MeshPart {
    int32_t system, first, groups, share;
};

struct MeshArgs {
    ResSystem *systems;
    const MeshPart *parts;     // of the launch
    const int32_t *part_of;    // workgroup -> part
    MeshSync *sync;            // one per part
    double *pos;               // two buffers of positions (3 x tot each), by body slot
    const double *gm;          // k^2 m, by body slot
    // read: state and masses; written at the end (component stride tot): the
    // state, the previous state, the Driver's arrays and the side outputs
    int64_t tot;
    const double *y0_in, *mass, *radius;
    double *y0, *y, *acc0, *yscale, *err, *rm3, *nnd;
    int32_t *nni;
    double eps2;               // Plummer softening squared
    uint64_t ticks;            // real-time-counter ticks a wait lasts before it gives up
};

// Accepted steps of a launch for systems of up to n bodies: about 0.2 s at
// RKF78's 13 evaluations and one attempt each.
inline int mesh_chunk(int n)
{
    const double per_step = 13.0 * (5.0e-6 + (double)n * (double)n * 1.0e-12);
    return std::max(1, (int)std::min(20000.0, 0.2 / per_step));
}

// Bodies per workgroup for n bodies, nm of them massive, with source ranges
// [1, end_a) (massive) and [1, end_b) (the others) on at most `cus`
// workgroups (0: the system does not fit), and the workgroups that takes.  A
// workgroup's bodies have one source range.
int mesh_share(int n, int nm, int end_a, int end_b, int cus);
int mesh_groups(int n, int nm, int end_a, int end_b, int share);

// Zeroes the parts' exchange words (unless they are `zeroed`) and runs
// max_steps accepted steps of integrator `integ` for every part.  The grid is
// the sum of the parts' groups and has to be resident at once; mesh_capacity has
// to have been asked for this device.
hipError_t launch_mesh(hipStream_t st, int integ, const MeshArgs &a, int nparts, int ngroups, int max_n,
                       int max_share, int max_steps, bool zeroed = false);
// After that launch: the state of every part that ran to its end (no wait
// timed out) into y0 (component stride tot) and its descriptor into systems.
// The mesh launch itself may have written some workgroups' rows of a part
// that did not, so y0 is another array than a.y0, and systems than a.systems.
hipError_t launch_mesh_commit(hipStream_t st, const MeshArgs &a, int nparts, ResSystem *systems, double *y0);
// Workgroups of that launch the device holds at once.
int mesh_capacity(int integ, int n, int share, int cu_count);

}  // namespace sol
