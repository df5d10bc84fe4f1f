// noalloc.hip -- sol_compute_gravity_noalloc: the gravity of sol_compute
// for arrays already on the device, with no device memory allocated by the
// call (for callers that cannot allocate: code under HIP graph capture,
// serving loops, harnesses that forbid hipMalloc).
//
// One launch, which reads the caller's arrays and writes dydt.  Only when y and
// dydt overlap is y first copied to the file-scope array `scratch` (6 MiB on
// every GPU the library runs on, its address taken once per device with
// hipGetSymbolAddress): such calls that overlap on one GPU race.
//
// The force is GravityAC (Solaris/Acceleration.cpp:248-329) with the
// reference's type-based source ranges, as sol_compute evaluates it for a
// gas-free astrocentric system: the Kepler term, the pair terms
// k^2 m_j d_ij / r_ij^3 over the sink's sources, itself left out, and the
// indirect term, the sum of k^2 m_j r_j / r_j^3 over the sources less the
// sink's own; the star's derivative is zero.
#include <algorithm>
#include <cstdio>
#include <mutex>

#include "lane_pairs.h"
#include "sol_internal.h"

namespace sol {
namespace {

// the sizes the call accepts
constexpr int kNoallocMaxBodies = 131072;
// at most so many sources go to k_na_few
constexpr int kNoallocFewSources = 64;
constexpr int kNoallocThreads = 512;
constexpr int kNoallocHalves = 2;                                           // of the sources
constexpr int kNoallocSinkGroups = kNoallocThreads / kWave / kNoallocHalves;
constexpr int kNoallocTile = 1024;                                          // sources in LDS at a time

static __device__ __align__(256) double scratch[6 * kNoallocMaxBodies];

constexpr int kMaxDevices = 64;
double *g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_mu;

__global__ __launch_bounds__(256) void k_na_copy(int len, const double *__restrict__ y, double *__restrict__ out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < len) out[i] = y[i];
}

typedef double double2_t __attribute__((ext_vector_type(2)));

// Sink i's derivative from its pair sum (px, py, pz) less the indirect sum
// (tx, ty, tz) over its sources, itself among them when `own`.
__device__ __forceinline__ void na_store(const double *__restrict__ y, const double *__restrict__ mass, int i, int own,
                                         double px, double py, double pz, double tx, double ty, double tz,
                                         double *__restrict__ dydt)
{
    const double *s = y + 6 * (size_t)i;
    double *o = dydt + 6 * (size_t)i;
    const double x = s[0], yy = s[1], z = s[2];
    const double r2 = x * x + yy * yy + z * z;
    const double r = sqrt(r2);
    const double rm3 = 1.0 / (r2 * r);
    const double mu = kGauss2 * (mass[0] + mass[i]);
    const double w = own ? kGauss2 * mass[i] : 0.0;
    o[0] = s[3]; o[1] = s[4]; o[2] = s[5];
    o[3] = -mu * rm3 * x + (px - (tx - w * (x * rm3)));
    o[4] = -mu * rm3 * yy + (py - (ty - w * (yy * rm3)));
    o[5] = -mu * rm3 * z + (pz - (tz - w * (z * rm3)));
}

// Few sources: a thread per sink; the sources in LDS with their indirect
// terms.  Bound by the latency of its loop, about 0.1 us per source, and for
// many sinks by one pass over the state.
__global__ __launch_bounds__(128) void k_na_few(int n, int nm, int end_a, int end_b, const double *__restrict__ y,
                                                const double *__restrict__ mass, double *__restrict__ dydt)
{
    __shared__ double4 sJ[kNoallocFewSources], sT[kNoallocFewSources];
    const int last = max(end_a, end_b);
    for (int j = 1 + threadIdx.x; j < last; j += blockDim.x) {
        const double *s = y + 6 * (size_t)j;
        const double g = kGauss2 * mass[j];
        const double r2 = s[0] * s[0] + s[1] * s[1] + s[2] * s[2];
        const double r = sqrt(r2);
        const double w = g * (1.0 / (r2 * r));
        sJ[j] = make_double4(s[0], s[1], s[2], g);
        sT[j] = make_double4(w * s[0], w * s[1], w * s[2], 0.0);
    }
    __syncthreads();
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (i == 0) {
        for (int c = 0; c < 6; ++c) dydt[c] = 0.0;
        return;
    }
    const int end = i < nm ? end_a : end_b;
    const double x = y[6 * (size_t)i], yy = y[6 * (size_t)i + 1], z = y[6 * (size_t)i + 2];
    double px = 0.0, py = 0.0, pz = 0.0;
    for (int j = 1; j < end; ++j) {
        if (j == i) continue;
        const double4 q = sJ[j], t = sT[j];
        const double dx = q.x - x, dy = q.y - yy, dz = q.z - z;
        const double r2 = dx * dx + dy * dy + dz * dz;
        const double v = __builtin_amdgcn_rsq(r2);
        const double tt = v * v;
        const double e = __builtin_fma(-r2, tt, 1.0);
        const double y3 = tt * v;
        const double f = q.w * __builtin_fma(y3, e * __builtin_fma(1.875, e, 1.5), y3);
        px += f * dx - t.x;
        py += f * dy - t.y;
        pz += f * dz - t.z;
    }
    na_store(y, mass, i, 0, px, py, pz, 0.0, 0.0, 0.0, dydt);
}

// Many sources: the sources over the lanes, SB sinks per wave, four groups of
// sinks by two halves of the sources in a workgroup (lane_pairs.h).  The
// workgroups take the sinks [1, last) with source range [1, end_a) first,
// then [last, n) with [1, end_b), 4 SB - 1 each; the last place is a body at
// the origin, whose pair sum is the indirect term's sum.  The sources pass
// through LDS in tiles, each read once per workgroup, the next one while the
// last is summed.
//
// Bound by the FP64 pair terms from about 2,000 bodies on, below by its
// launch: 515 mutually attracting bodies 4.1 us, 4,097 bodies 24 us (with a
// sink per thread, 65 waves for 1,024 SIMDs and a square root and a division
// per pair, 744 us), 16,385 bodies 270 us.
template <int SB>
__global__ __launch_bounds__(kNoallocThreads) void k_na_many(int n, int last, int end_a, int end_b,
                                                             const double *__restrict__ y,
                                                             const double *__restrict__ mass,
                                                             double *__restrict__ dydt)
{
    constexpr int ST = SB * kNoallocSinkGroups;
    constexpr int share = ST - 1;
    constexpr int NT = SB == 6 ? 3 : 4;              // pair terms at a time
    constexpr int KC = SB == 2 ? 2 : 1;              // of so many chunks of 64 sources
    constexpr int KW = kNoallocTile / kNoallocThreads;
    __shared__ double2_t xy[kNoallocTile], zw[kNoallocTile];
    __shared__ double part[kNoallocHalves][3][ST];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int ga = (last - 1 + share - 1) / share;
    const bool first = (int)blockIdx.x < ga;
    const int end = first ? end_a : end_b;
    const int i0 = first ? 1 + (int)blockIdx.x * share : last + ((int)blockIdx.x - ga) * share;
    const int nb = min(share, (first ? last : n) - i0);

    double4 q[KW];
    auto read = [&](int t0) {
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            const int j = min(t0 + k * kNoallocThreads + tid, end - 1);
            const double *s = y + 6 * (size_t)j;
            q[k] = make_double4(s[0], s[1], s[2], mass[j]);
        }
    };
    read(1);
    const int half = wave % kNoallocHalves, b0 = wave / kNoallocHalves * SB;
    double sx[SB], sy[SB], sz[SB], eps2[SB], ax[SB], ay[SB], az[SB];
    int own[SB];
#pragma unroll
    for (int b = 0; b < SB; ++b) {
        const int i = i0 + min(b0 + b, nb - 1);
        const bool origin = b0 + b == ST - 1;
        sx[b] = uniform(origin ? 0.0 : y[6 * (size_t)i]);
        sy[b] = uniform(origin ? 0.0 : y[6 * (size_t)i + 1]);
        sz[b] = uniform(origin ? 0.0 : y[6 * (size_t)i + 2]);
        own[b] = origin ? -1 : i;
        eps2[b] = 0.0;
        ax[b] = ay[b] = az[b] = 0.0;
    }
    double c15 = 1.5, c1875 = 1.875;
    asm volatile("" : "+v"(c15), "+v"(c1875));
    const int ib = i0 + min(b0, nb - 1), il = i0 + min(b0 + SB, nb) - 1;
    constexpr int step = kNoallocHalves * kWave;     // from a wave's chunk to its next
    for (int t0 = 1; t0 < end; t0 += kNoallocTile) {
        if (t0 > 1) __syncthreads();                 // the tile before is read
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            const int j = k * kNoallocThreads + tid;
            const bool on = t0 + j < end;            // past the end: a far source of no mass
            xy[j] = double2_t{on ? q[k].x : kFar, on ? q[k].y : kFar};
            zw[j] = double2_t{on ? q[k].z : kFar, on ? kGauss2 * q[k].w : 0.0};
        }
        __syncthreads();
        if (t0 + kNoallocTile < end) read(t0 + kNoallocTile);
        const int t1 = min(end - t0, kNoallocTile);
        for (int jk = half * kWave; jk < t1; jk += KC * step) {
            double4 p[KC];
            int j[KC];
#pragma unroll
            for (int u = 0; u < KC; ++u) {
                j[u] = t0 + jk + u * step + lane;
                p[u] = make_double4(kFar, kFar, kFar, 0.0);
                if (jk + u * step < t1) {
                    const double2_t a = xy[jk + u * step + lane], b = zw[jk + u * step + lane];
                    p[u] = make_double4(a.x, a.y, b.x, b.y);
                }
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
    if (k < 3 && m < SB) part[half][k][b0 + m] = k == 0 ? r[0] : k == 1 ? r[1] : r[2];
    __syncthreads();
    if (tid < nb) {
        double s[3], t[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            s[c] = part[0][c][tid] + part[1][c][tid];
            t[c] = part[0][c][ST - 1] + part[1][c][ST - 1];
        }
        na_store(y, mass, i0 + tid, i0 + tid < end ? 1 : 0, s[0], s[1], s[2], t[0], t[1], t[2], dydt);
    }
    if (blockIdx.x == 0 && tid >= kWave && tid < kWave + 6) dydt[tid - kWave] = 0.0;   // the star
}

template <int SB>
void launch_many(hipStream_t st, int blocks, int n, int last, int ea, int eb, const double *y, const double *mass,
                 double *dydt)
{
    hipLaunchKernelGGL(k_na_many<SB>, dim3(blocks), dim3(kNoallocThreads), 0, st, n, last, ea, eb, y, mass, dydt);
}

int say(char *err, int32_t len, int code, const char *msg)
{
    if (err && len > 0) snprintf(err, (size_t)len, "%s", msg);
    return code;
}

}  // namespace
}  // namespace sol

using namespace sol;

extern "C" int sol_compute_gravity_noalloc(const sol_nbodies *nb, const double *y, const double *mass, double *dydt,
                                           void *stream, char *err, int32_t err_len)
{
    if (err && err_len > 0) err[0] = '\0';
    if (!nb || !y || !mass || !dydt) return say(err, err_len, SOL_ERR_ARGUMENT, "null argument");
    const int n = nb->total;
    const int sum = nb->central_body + nb->giant_planet + nb->rocky_planet + nb->proto_planet +
                    nb->super_planetesimal + nb->planetesimal + nb->test_particle;
    if (n < 1 || sum != n || nb->central_body != 1)
        return say(err, err_len, SOL_ERR_ARGUMENT, "body counts must add up to total, with exactly one central body");
    if (n > kNoallocMaxBodies)
        return say(err, err_len, SOL_ERR_ARGUMENT, "sol_compute_gravity_noalloc: more than 131072 bodies");
    const int nm = nb->central_body + nb->giant_planet + nb->rocky_planet + nb->proto_planet;
    const int end_a = nm + nb->super_planetesimal, end_b = nm;
    hipStream_t st = static_cast<hipStream_t>(stream);
    double *copy = nullptr;
    if (y < dydt + 6 * (size_t)n && dydt < y + 6 * (size_t)n) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
            return say(err, err_len, SOL_ERR_DEVICE, "hipGetDevice failed");
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        if (!g_scratch_ptr[dev]) {
            void *ptr = nullptr;
            if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr)
                return say(err, err_len, SOL_ERR_DEVICE, "hipGetSymbolAddress of the scratch array failed");
            g_scratch_ptr[dev] = static_cast<double *>(ptr);
        }
        copy = g_scratch_ptr[dev];
    }
    (void)hipGetLastError();   // so that a failure below is this call's own
    if (copy) {
        hipLaunchKernelGGL(k_na_copy, dim3((6 * n + 255) / 256), dim3(256), 0, st, 6 * n, y, copy);
        y = copy;
    }
    // a sink per thread where the sources are few and the sinks many: with 62
    // sources 9.5 us against 3.7 at 500 sinks and 11.8 against 18.8 at 40,000,
    // with two 3.5 against 3.7 and 4.9 against 18.7
    const int nsrc = std::max(end_a, end_b);
    if (nsrc <= kNoallocFewSources && (nsrc <= 8 || n > 256 * nsrc)) {
        hipLaunchKernelGGL(k_na_few, dim3((n + 127) / 128), dim3(128), 0, st, n, nm, end_a, end_b, y, mass, dydt);
    } else {
        // one source range for both sink classes: one class.  The sinks per
        // workgroup (4 SB - 1) that load a CU least: places times the
        // workgroups of the fullest CU; of equals the larger, which reads
        // the sources less often.
        constexpr int kUnits = 256;
        const int last = end_a == end_b ? n : nm;
        auto groups = [&](int share) { return (last - 1 + share - 1) / share + (n - last + share - 1) / share; };
        int sb = 0, best = 0;
        for (int s : {2, 4, 6, 8}) {
            const int cost = 4 * s * ((groups(4 * s - 1) + kUnits - 1) / kUnits);
            if (sb == 0 || cost <= best) { sb = s; best = cost; }
        }
        const int blocks = groups(4 * sb - 1);
        switch (sb) {
        case 2: launch_many<2>(st, blocks, n, last, end_a, end_b, y, mass, dydt); break;
        case 4: launch_many<4>(st, blocks, n, last, end_a, end_b, y, mass, dydt); break;
        case 6: launch_many<6>(st, blocks, n, last, end_a, end_b, y, mass, dydt); break;
        default: launch_many<8>(st, blocks, n, last, end_a, end_b, y, mass, dydt); break;
        }
    }
    if (hipGetLastError() != hipSuccess) return say(err, err_len, SOL_ERR_DEVICE, "kernel launch failed");
    return SOL_OK;
}
