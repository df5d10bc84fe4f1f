// adjoint_few.hip -- the RK4 adjoint of systems with few sources: a handful
// of planets and any number of bodies that feel only them.
//
// The other kernels of the adjoint (adjoint.hip) work launch by launch: a step
// back is four vector-Jacobian products of two launches each, and the forward
// pass of a system that fits one workgroup runs in one.  Here the order of
// the work follows the couplings instead.
//   * The sources do not feel the sinks: their forward pass is a chain of its
//     own, and the sinks follow with the sources' stage positions given.
//   * The sinks' adjoints do not depend on the sources' adjoints: they too
//     are independent chains, given the recorded positions.
//   * The sources' adjoints need, per product, sums over all sinks (A, B, U of
//     adjoint.hip).  Once the sinks' weights of a chunk of steps are known,
//     the sums of all its products are formed side by side.
// So a chunk of steps is one launch in which the sinks' chains run beside the
// sources' chain of the chunk next to it, and backwards one more for the sums.
// Eight lanes share a body and split its sources; they hold the same state.
//
// What bounds it: the instructions of one wave's chain, 0.48 us per stage
// forward and 0.78 us per product backward (eight planets and 1,024 test
// particles over 500 steps: forward 15.6 -> 1.1 ms, backward 21.2 -> 1.9 ms).
//
// The formulas are those at the head of adjoint.hip; all arithmetic is FP64
// and every sum has a fixed order.
#include "lane_pairs.h"
#include "sol_internal.h"

namespace sol {
namespace {

constexpr int kFewLanes = 8;                                   // lanes per body
constexpr int kFewPer = (kFewMaxSources + kFewLanes - 1) / kFewLanes;   // sources per lane

// A source's stage record: x, y, z, |r|^-3.
typedef double few_rec __attribute__((ext_vector_type(4)));

// 1 / sqrt(r2) to the last digit or two: the hardware's and a second-order
// correction.
__device__ __forceinline__ double few_rsqrt(double r2)
{
    const double y = __builtin_amdgcn_rsq(r2);
    const double e = __builtin_fma(-r2 * y, y, 1.0);
    return __builtin_fma(y, e * __builtin_fma(0.375, e, 0.5), y);
}

// r2^(-3/2) for the forward pass: the hardware's reciprocal square root cubed,
// corrected once, as the pair sums form it (resident.hip).  Errors over r2 of
// 1e-2 to 1e2 in units of 2^-53, rms and largest: 0.64 and 2.4, where 1 / (r2
// sqrt(r2)) has 0.74 and 2.4 and the cube of few_rsqrt 1.55 and 5.4.
__device__ __forceinline__ double few_rm3(double r2)
{
    const double y = __builtin_amdgcn_rsq(r2);
    const double t = y * y;
    const double e = __builtin_fma(-r2, t, 1.0);
    const double y3 = t * y;
    return __builtin_fma(y3, e * __builtin_fma(1.875, e, 1.5), y3);
}

// This thread's body and its share of the sources.
struct Few {
    int i, sub, end;        // body; lane among its eight; its sources are [1, end)
    bool live;
    double gm, mu;
    double gj[kFewPer];     // k^2 m of sources 1 + sub + 8 q (0: not a source of this body)
};

__device__ __forceinline__ Few few_body(const FewArgs &a, bool sources)
{
    Few f;
    const int b = (int)threadIdx.x / kFewLanes;
    f.sub = (int)threadIdx.x % kFewLanes;
    const int i = sources ? 1 + b : a.src + ((int)blockIdx.x - 1) * ((int)blockDim.x / kFewLanes) + b;
    f.live = i < (sources ? a.src : a.n);
    f.i = f.live ? i : (sources ? 1 : a.n - 1);
    f.end = min(f.i < a.nm ? a.ea : a.eb, a.src);
    f.gm = a.gm[f.i];
    f.mu = a.gm[0] + f.gm;
#pragma unroll
    for (int q = 0; q < kFewPer; ++q) {
        const int j = 1 + f.sub + kFewLanes * q;
        f.gj[q] = j < f.end && j != f.i ? a.gm[j] : 0.0;
    }
    return f;
}

// Acceleration at p with the sources' records s.  Eight lanes together, each
// with the whole result.
__device__ __forceinline__ void few_accel(const Few &f, int src, const few_rec *s, const double (&p)[3], double (&a)[3])
{
    double t[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < kFewPer; ++q) {
        const int j = 1 + f.sub + kFewLanes * q;
        if (kFewLanes * q + 1 < src) {
            const few_rec r = s[min(j, src - 1)];
            const double dx = r.x - p[0], dy = r.y - p[1], dz = r.z - p[2];
            double r2 = dx * dx + dy * dy + dz * dz;
            if (j == f.i || j >= f.end) r2 = 1.0;
            const double w = few_rm3(r2);
            t[0] += f.gj[q] * (dx * w - r.x * r.w);
            t[1] += f.gj[q] * (dy * w - r.y * r.w);
            t[2] += f.gj[q] * (dz * w - r.z * r.w);
        }
    }
    const double c = -f.mu * few_rm3(p[0] * p[0] + p[1] * p[1] + p[2] * p[2]);
    sum8(t);
#pragma unroll
    for (int k = 0; k < 3; ++k) a[k] = c * p[k] + t[k];
}

// Forward pass.  Block 0: the sources' chunk [s0, s1) of the steps; the other
// blocks: the sinks' chunk [t0, t1), whose source positions the launch before
// wrote.  Each chain starts from and ends in a.y.
__global__ __launch_bounds__(256) void k_few_forward(FewArgs a)
{
    __shared__ few_rec sp[2][4][kFewMaxSources + 1];
    const bool sources = blockIdx.x == 0;
    const int n0 = sources ? a.s0 : a.t0, n1 = sources ? a.s1 : a.t1;
    if (n0 >= n1) return;
    const int np = a.np, tid = (int)threadIdx.x;
    const Few f = few_body(a, sources);
    const bool mine = f.live && f.sub == 0;
    double x[3], v[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        x[k] = a.y[k * np + f.i];
        v[k] = a.y[(3 + k) * np + f.i];
    }
    const int words = 4 * a.src;             // records of a step
    few_rec nxt[2];
    auto read = [&](int step) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int w = tid + q * (int)blockDim.x;
            if (w < words) nxt[q] = reinterpret_cast<const few_rec *>(a.sp_in)[(size_t)(step - n0) * words + w];
        }
    };
    if (!sources) read(n0);
    for (int step = n0; step < n1; ++step) {
        const double h = a.h[step];
        few_rec(*s)[kFewMaxSources + 1] = sp[step & 1];
        if (!sources) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int w = tid + q * (int)blockDim.x;
                if (w < words) s[w / a.src][w % a.src] = nxt[q];
            }
            __syncthreads();
            if (step + 1 < n1) read(step + 1);
        }
        if (a.ckpt && step % a.K == 0 && mine) {
            double *c = a.ckpt + (size_t)(step / a.K) * 6 * np;
#pragma unroll
            for (int k = 0; k < 3; ++k) { c[k * np + f.i] = x[k]; c[(3 + k) * np + f.i] = v[k]; }
        }
        double kv[3] = {0.0, 0.0, 0.0}, ka[3] = {0.0, 0.0, 0.0};       // sums of b_s k_s
        double p[3] = {x[0], x[1], x[2]}, w[3] = {v[0], v[1], v[2]};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (mine && a.stages) {
                double *c = a.stages + (size_t)((step - a.first) * 4 + q) * 6 * np;
#pragma unroll
                for (int k = 0; k < 3; ++k) { c[k * np + f.i] = p[k]; c[(3 + k) * np + f.i] = w[k]; }
            }
            if (sources) {
                // |r|^-3 by the body's own lanes: left to the readers, who could
                // form it beside their distances, the chain is 15% slower (it
                // is bound by the instructions of one wave)
                if (mine) {
                    const few_rec rec = {p[0], p[1], p[2], few_rm3(p[0] * p[0] + p[1] * p[1] + p[2] * p[2])};
                    s[q][f.i] = rec;
                    reinterpret_cast<few_rec *>(a.sp_out)[((size_t)(step - n0) * 4 + q) * a.src + f.i] = rec;
                }
                __syncthreads();
            }
            double acc[3];
            few_accel(f, a.src, s[q], p, acc);
            const double b = q == 0 || q == 3 ? 1.0 / 6.0 : 1.0 / 3.0;
            const double c = q == 2 ? 1.0 : 0.5;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                kv[k] += b * w[k];
                ka[k] += b * acc[k];
                if (q < 3) {
                    const double pk = x[k] + h * (c * w[k]);
                    w[k] = v[k] + h * (c * acc[k]);
                    p[k] = pk;
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            x[k] += h * kv[k];
            v[k] += h * ka[k];
        }
    }
    if (mine) {
#pragma unroll
        for (int k = 0; k < 3; ++k) { a.y[k * np + f.i] = x[k]; a.y[(3 + k) * np + f.i] = v[k]; }
    }
    if (sources && tid < 6) {
        // the star stays where it is: its rows of the record and checkpoints
        const double s = a.y[tid * np];
        for (int step = n0; step < n1; ++step) {
            if (a.stages)
                for (int q = 0; q < 4; ++q) a.stages[(size_t)((step - a.first) * 4 + q) * 6 * np + tid * np] = s;
            if (a.ckpt && step % a.K == 0) a.ckpt[(size_t)(step / a.K) * 6 * np + tid * np] = s;
        }
    }
}

// Backward pass, one chunk of steps [t0, t1) downwards.  Blocks >= 1: the
// sinks' adjoints (a.lam), with the weight on the acceleration of every
// product to a.u ([step - t0][stage][3][np]).  Block 0: the sources' adjoints
// over the chunk before, [s0, s1), with its sums over the sinks in a.sums
// ([step - s0][stage][source][7]).
__global__ __launch_bounds__(256) void k_few_backward(FewArgs a)
{
    __shared__ double sp[2][4][kFewMaxSources + 1][3];
    __shared__ double su[kFewMaxSources + 1][3];
    const bool sources = blockIdx.x == 0;
    const int n0 = sources ? a.s0 : a.t0, n1 = sources ? a.s1 : a.t1;
    if (n0 >= n1) return;
    const int np = a.np, tid = (int)threadIdx.x, src = a.src;
    const Few f = few_body(a, sources);
    const bool mine = f.live && f.sub == 0;
    double lam[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) lam[c] = a.lam[c * np + f.i];
    double mb = a.mbar[f.i], m0 = sources ? a.m0src[f.i] : 0.0;
    const int words = 12 * src;              // source coordinates of a step
    double nxt[2], own[4][3], sum_nxt[4] = {0.0, 0.0, 0.0, 0.0};
    auto read = [&](int step) {
        const double *Y = a.stages + (size_t)(step - a.first) * 24 * np;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int w = tid + q * (int)blockDim.x;
            // row w / src is stage row / 3, component row % 3
            const int row = w / src;
            if (w < words) nxt[q] = Y[(size_t)((row / 3) * 6 + row % 3) * np + w % src];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int c = 0; c < 3; ++c) own[q][c] = Y[(size_t)(q * 6 + c) * np + f.i];
        if (sources && f.sub < 7) {
            // the sums over the sinks: lane 0-2 A, 3 B, 4-6 U
#pragma unroll
            for (int q = 0; q < 4; ++q)
                sum_nxt[q] = a.sums[((size_t)((step - n0) * 4 + q) * src + f.i) * 7 + f.sub];
        }
    };
    read(n1 - 1);
    for (int step = n1 - 1; step >= n0; --step) {
        const double h = a.h[step];
        double(*s)[kFewMaxSources + 1][3] = sp[step & 1];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int w = tid + q * (int)blockDim.x;
            const int row = w / src;
            if (w < words) s[row / 3][w % src][row % 3] = nxt[q];
        }
        double pos[4][3], sum[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int c = 0; c < 3; ++c) pos[q][c] = own[q][c];
            sum[q] = sum_nxt[q];
        }
        __syncthreads();
        if (step > n0) read(step - 1);
        double yb[6], w[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) { yb[c] = lam[c]; w[c] = h / 6.0 * lam[c]; }
#pragma unroll
        for (int q = 3; q >= 0; --q) {
            const double *p = pos[q];
            const double u0 = w[3], u1 = w[4], u2 = w[5];
            if (sources) {
                if (mine) { su[f.i][0] = u0; su[f.i][1] = u1; su[f.i][2] = u2; }
                __syncthreads();
            } else if (mine) {
                double *o = a.u + (size_t)((step - n0) * 4 + q) * 3 * np + f.i;
                o[0] = u0; o[np] = u1; o[2 * np] = u2;
            }
            // t: sum of -gm_j T(d) u_i, and for a source + gm_i T(d) u_j
            double t[3] = {0.0, 0.0, 0.0}, U[3] = {0.0, 0.0, 0.0}, B = 0.0;
#pragma unroll
            for (int m = 0; m < kFewPer; ++m) {
                const int j = 1 + f.sub + kFewLanes * m;
                if (kFewLanes * m + 1 < src) {
                    const int jc = min(j, src - 1);
                    const double dx = p[0] - s[q][jc][0], dy = p[1] - s[q][jc][1], dz = p[2] - s[q][jc][2];
                    // j as a source of this body, and as a sink that sees it
                    const bool self = j == f.i || j >= src;
                    const bool sees = sources && !self && f.i < (j < a.nm ? a.ea : a.eb);
                    double r2 = dx * dx + dy * dy + dz * dz;
                    if (self || (!sees && j >= f.end)) r2 = 1.0;
                    const double v = few_rsqrt(r2);
                    const double v2 = v * v, v3 = v2 * v;
                    const double c1 = 3.0 * v3 * v2;
                    const double di = dx * u0 + dy * u1 + dz * u2;
                    const double g = f.gj[m];
                    double a1 = -g * v3, a2 = g * c1 * di;
                    t[0] += a1 * u0 + a2 * dx;
                    t[1] += a1 * u1 + a2 * dy;
                    t[2] += a1 * u2 + a2 * dz;
                    if (sources) {
                        const double e0 = sees ? su[jc][0] : 0.0, e1 = sees ? su[jc][1] : 0.0,
                                     e2 = sees ? su[jc][2] : 0.0;
                        const double dj = dx * e0 + dy * e1 + dz * e2;
                        a1 = f.gm * v3;
                        a2 = -f.gm * c1 * dj;
                        t[0] += a1 * e0 + a2 * dx;
                        t[1] += a1 * e1 + a2 * dy;
                        t[2] += a1 * e2 + a2 * dz;
                        B += dj * v3;
                        U[0] += e0; U[1] += e1; U[2] += e2;
                    }
                }
            }
            const double v = few_rsqrt(p[0] * p[0] + p[1] * p[1] + p[2] * p[2]);
            const double v2 = v * v, v3 = v2 * v;
            const double c5 = 3.0 * v3 * v2;
            const double ru = p[0] * u0 + p[1] * u1 + p[2] * u2;
            const double ck = c5 * ru;
            if (sources) {
                const double z = sum[q], g = f.gm * z;
                if (f.sub == 0) t[0] += g;
                if (f.sub == 1) t[1] += g;
                if (f.sub == 2) t[2] += g;
                if (f.sub == 3) B += z;
                if (f.sub == 4) U[0] += z;
                if (f.sub == 5) U[1] += z;
                if (f.sub == 6) U[2] += z;
            }
            sum8(t);
            double G[6];
            G[0] = -f.mu * (v3 * u0 - ck * p[0]) + t[0];
            G[1] = -f.mu * (v3 * u1 - ck * p[1]) + t[1];
            G[2] = -f.mu * (v3 * u2 - ck * p[2]) + t[2];
            double mg = -v3 * ru;
            if (sources) {
                m0 += mg;
                sum8(U);
                B = sum8(B);
                const double rU = p[0] * U[0] + p[1] * U[1] + p[2] * U[2];
                const double cU = c5 * rU;
                G[0] -= f.gm * (v3 * U[0] - cU * p[0]);
                G[1] -= f.gm * (v3 * U[1] - cU * p[1]);
                G[2] -= f.gm * (v3 * U[2] - cU * p[2]);
                mg += B - v3 * rU;
                if (q > 0) __syncthreads();          // su is read
            }
            mb += mg;
            G[3] = w[0]; G[4] = w[1]; G[5] = w[2];
            const double alpha = q == 3 || q == 2 ? h / 3.0 : h / 6.0, beta = q == 3 ? h : 0.5 * h;
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                yb[c] += G[c];
                w[c] = alpha * lam[c] + beta * G[c];
            }
        }
#pragma unroll
        for (int c = 0; c < 6; ++c) lam[c] = yb[c];
        if (sources) __syncthreads();
    }
    if (mine) {
#pragma unroll
        for (int c = 0; c < 6; ++c) a.lam[c * np + f.i] = lam[c];
        a.mbar[f.i] = mb;
        if (sources) a.m0src[f.i] = m0;
    }
}

// The sums over the sinks [src, n) of every product of the chunk [t0, t1): a
// wave per product and source, lanes over the sinks.
__global__ __launch_bounds__(256) void k_few_sums(FewArgs a)
{
    const int np = a.np, lane = (int)threadIdx.x % kWave;
    const int w = (int)blockIdx.x * (256 / kWave) + (int)threadIdx.x / kWave;
    const int per = a.src - 1, prod = w / per, k = 1 + w % per;
    if (prod >= (a.t1 - a.t0) * 4) return;
    const double *Y = a.stages + (size_t)((a.t0 - a.first) * 4 + prod) * 6 * np;
    const double *u = a.u + (size_t)prod * 3 * np;
    const double xk = Y[k], yk = Y[np + k], zk = Y[2 * np + k];
    double A[3] = {0.0, 0.0, 0.0}, U[3] = {0.0, 0.0, 0.0}, B[3] = {0.0, 0.0, 0.0};
    for (int i = a.src + lane; i < a.n; i += kWave) {
        const bool sees = k < (i < a.nm ? a.ea : a.eb);
        const double u0 = sees ? u[i] : 0.0, u1 = sees ? u[np + i] : 0.0, u2 = sees ? u[2 * np + i] : 0.0;
        const double dx = xk - Y[i], dy = yk - Y[np + i], dz = zk - Y[2 * np + i];
        const double r2 = sees ? dx * dx + dy * dy + dz * dz : 1.0;
        const double v = few_rsqrt(r2);
        const double v2 = v * v, v3 = v2 * v;
        const double s = dx * u0 + dy * u1 + dz * u2;
        const double c = 3.0 * v3 * v2 * s;
        A[0] += v3 * u0 - c * dx;
        A[1] += v3 * u1 - c * dy;
        A[2] += v3 * u2 - c * dz;
        B[0] += s * v3;
        U[0] += u0; U[1] += u1; U[2] += u2;
    }
    auto wave = [&](double (&x)[3]) {
        sum16(x);
#pragma unroll
        for (int c = 0; c < 3; ++c) { x[c] = fold16(x[c], x[c]); x[c] = fold32(x[c], x[c]); }
    };
    wave(A);
    wave(U);
    wave(B);
    if (lane < 7) {
        const double r = lane < 3 ? (lane == 0 ? A[0] : lane == 1 ? A[1] : A[2]) : lane == 3 ? B[0]
                       : lane == 4 ? U[0] : lane == 5 ? U[1] : U[2];
        a.sums[((size_t)prod * a.src + k) * 7 + lane] = r;
    }
}

// dL/dm from dL/dgm, the central body's the sum over all bodies of their
// own-mu terms (a sink's whole mbar), in a fixed order.  One block.
__global__ __launch_bounds__(256) void k_few_mass(FewArgs a, double *out)
{
    __shared__ double red[256];
    const int tid = (int)threadIdx.x;
    double s = 0.0;
    for (int i = 1 + tid; i < a.n; i += 256) {
        const double m = a.mbar[i];
        out[i] = kGauss2 * m;
        s += i < a.src ? a.m0src[i] : m;
    }
    red[tid] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) red[tid] += red[tid + o];
        __syncthreads();
    }
    if (tid == 0) out[0] = kGauss2 * red[0];
}

int few_block(int src) { return ((src - 1) * kFewLanes + kWave - 1) / kWave * kWave; }
int few_blocks(const FewArgs &a)
{
    const int per = few_block(a.src) / kFewLanes;
    return 1 + (a.t1 > a.t0 ? (a.n - a.src + per - 1) / per : 0);
}

}  // namespace

void launch_few_forward(hipStream_t st, const FewArgs &a)
{
    hipLaunchKernelGGL(k_few_forward, dim3(few_blocks(a)), dim3(few_block(a.src)), 0, st, a);
}

void launch_few_backward(hipStream_t st, const FewArgs &a)
{
    hipLaunchKernelGGL(k_few_backward, dim3(few_blocks(a)), dim3(few_block(a.src)), 0, st, a);
}

void launch_few_sums(hipStream_t st, const FewArgs &a)
{
    const int waves = (a.t1 - a.t0) * 4 * (a.src - 1);
    hipLaunchKernelGGL(k_few_sums, dim3((waves + 3) / 4), dim3(256), 0, st, a);
}

void launch_few_mass(hipStream_t st, const FewArgs &a, double *out)
{
    hipLaunchKernelGGL(k_few_mass, dim3(1), dim3(256), 0, st, a, out);
}

}  // namespace sol
