// Static contact projection, in FP64 without FMA contraction.
#pragma once
#include <hip/hip_runtime.h>

namespace xpbd {

// Static contact projection in FP64 (alpha = 0, inequality):
// ConstraintProjector.hpp:111-172, StaticDeformableCollisionConstraint.cpp:20-55
__device__ __forceinline__ bool contact_dx(const double* const x[3], const float* w, const double* cp,
                                           const double* cn, const double* cb, double* lam, double* dx)
{
#pragma clang fp contract(off)
    double a[3];
#pragma unroll
    for (int k = 0; k < 3; k++) a[k] = cb[0] * x[0][k] + cb[1] * x[1][k] + cb[2] * x[2][k];
    const double C = cn[0] * (a[0] - cp[0]) + cn[1] * (a[1] - cp[1]) + cn[2] * (a[2] - cp[2]);
    if (C > 0) return false;
    double L = 0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const double gx = cb[i] * cn[0], gy = cb[i] * cn[1], gz = cb[i] * cn[2];
        L += (double)w[i] * (gx * gx + gy * gy + gz * gz);
    }
    const double dl = -C / L;
    *lam += dl;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int k = 0; k < 3; k++) dx[3 * i + k] = (double)w[i] * (cb[i] * cn[k]) * dl;
    return true;
}

}  // namespace xpbd
