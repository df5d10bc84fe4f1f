// quad_stages.h -- where the quad form (quad.hip) keeps the stage derivatives
// of one component of a body.
//
// ROWS is the number of evaluations of an attempt: the step's first and one
// per stage.  Shared by the kernels and the host, which sizes the LDS columns
// (and, in the tests, checks that nothing passes them).
#pragma once

#include <stddef.h>

#if defined(__HIPCC__)
#define SOL_QUAD_HD __host__ __device__ __forceinline__
#else
#define SOL_QUAD_HD inline
#endif
#if defined(__HIP_DEVICE_COMPILE__)
#define QUAD_LDS __attribute__((address_space(3)))
#else
#define QUAD_LDS
#endif

namespace sol {

// Velocities V and accelerations F, in registers, or (LDS) in columns of the
// workgroup's LDS, column = thread: quad_column_bytes(ROWS, threads) in all.
template <int ROWS, bool LDS>
struct QStages {
    double V_[ROWS], F_[ROWS];
    SOL_QUAD_HD double V(int l) const { return V_[l]; }
    SOL_QUAD_HD double F(int l) const { return F_[l]; }
    SOL_QUAD_HD void put(int l, double v, double f) { V_[l] = v; F_[l] = f; }
    SOL_QUAD_HD void clear()
    {
#pragma unroll
        for (int l = 0; l < ROWS; ++l) put(l, 0.0, 0.0);
    }
};
template <int ROWS>
struct QStages<ROWS, true> {
    QUAD_LDS double *col;      // this thread's column
    int stride;                // threads
    SOL_QUAD_HD double V(int l) const { return col[2 * l * stride]; }
    SOL_QUAD_HD double F(int l) const { return col[(2 * l + 1) * stride]; }
    SOL_QUAD_HD void put(int l, double v, double f)
    {
        col[2 * l * stride] = v;
        col[(2 * l + 1) * stride] = f;
    }
    SOL_QUAD_HD void clear()
    {
#pragma unroll
        for (int l = 0; l < ROWS; ++l) put(l, 0.0, 0.0);
    }
};

SOL_QUAD_HD constexpr size_t quad_column_bytes(int rows, int threads)
{
    return (size_t)(2 * rows) * threads * sizeof(double);
}

}  // namespace sol
