// The rotation of jacobi_rotation.h in the form the device kernels take: the
// FP64 square roots and the division of the tangent, several hundred cycles of
// dependent instructions, sat in the serial chain of every Jacobi step (55
// cores of 40-110 rows in LDS: 2.39 -> 1.98 ms; 820 of 20-40: 0.68 -> 0.55).
#pragma once

#include <hip/hip_runtime.h>
#include "jacobi_rotation.h"

// True when the pair is far enough from orthogonal to rotate: jr_rotates()
// without its square roots where the squares are in range.
__device__ inline bool jr_rotates_fast(double al, double be, double ga,
        double ctol)
{
    if(fmin(al, be) > 1e-130)
        return ga*ga > (ctol*ctol)*(al*be);
    return jr_rotates(al, be, ga, ctol);
}

// A rotation by the angle of jacobi_rotation() to single precision: the
// tangent comes from the fast FP32 square root and reciprocal, c = 1/sqrt(1 +
// t^2) and s = c t are FP64, so the rotation is orthogonal to rounding and
// leaves 1e-7 of the pair's inner product, which the quadratic convergence
// does not notice.
__device__ inline void jacobi_rotation_fast(double al, double be, double ga,
        double &c, double &s)
{
    const double d = be-al, h = 2.0*ga;
    const int e = __builtin_amdgcn_frexp_exp(fmax(fabs(d), fabs(h)));
    const float df = (float)ldexp(d, -e), hf = (float)ldexp(h, -e);
    if(fabsf(hf) < 1e-30f || !(fabsf(hf)+fabsf(df) < 4.0f))
    {
        jacobi_rotation(al, be, ga, c, s);
        return;
    }
    const float r = __builtin_amdgcn_sqrtf(df*df+hf*hf);
    const float tf = hf*__builtin_amdgcn_rcpf(fabsf(df)+r);
    const double t = (double)(df >= 0.0f ? tf : -tf);
    // 1/sqrt(x), x in [1, 2]: the hardware's approximation and one step of
    // third order
    const double x = fma(t, t, 1.0);
    const double y = __builtin_amdgcn_rsq(x);
    const double g = fma(-x*y, y, 1.0);
    c = fma(y*g, fma(0.375, g, 0.5), y);
    s = c*t;
}
