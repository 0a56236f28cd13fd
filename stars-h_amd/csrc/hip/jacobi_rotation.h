// Plane rotation of one-sided (Hestenes) Jacobi, shared by the device
// kernels (core.hip, core_block.hip) and by a host unit test, which compiles
// this header with a plain C++ compiler.
//
// Two columns with squared norms al, be and inner product ga are made
// orthogonal by (a, b) <- (c a - s b, s a + c b) with t = s/c the smaller
// root of t^2 + 2 zeta t - 1 = 0, zeta = (be - al)/(2 ga) (Rutishauser,
// "The Jacobi method for real symmetric matrices", Numer. Math. 9, 1966).
// With d = be - al and h = 2 ga that root is
//   t = sign(d) h / (|d| + sqrt(d^2 + h^2)),
// and c = 1/sqrt(1 + t^2), s = c t.  d and h are scaled by the power of two
// that brings the larger one into [1/2, 1), which is exact and keeps the
// squares in range.  h is never 0 here: jr_rotates() requires |ga| > 0.
//
// The division and the square roots sit in the serial chain of every Jacobi
// step.  They start from the hardware's approximations (relative error below
// 2^-24 for arguments in [1/4, 4], measured) and take one step of third order
// each, which leaves rounding, a few units of 2^-53; the library's division
// and square roots took several hundred cycles a step (55 cores of 40-110
// rows in LDS: 2.39 -> 2.02 ms; an angle to single precision only, 1.99).
#ifndef STARSH_JACOBI_ROTATION_H
#define STARSH_JACOBI_ROTATION_H

#include <math.h>

#ifdef __HIPCC__
#define JR_FN __host__ __device__ inline
#else
#define JR_FN static inline
#endif

// Approximations of 1/sqrt(x) and 1/x; on the host rounded to single
// precision, which is no better than the hardware's.
JR_FN double jr_rsq_approx(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsq(x);
#else
    return 1.0f/sqrtf((float)x);
#endif
}

JR_FN double jr_rcp_approx(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcp(x);
#else
    return 1.0f/(float)x;
#endif
}

// Exponent e of x = m 2^e, 1/2 <= |m| < 1.
JR_FN int jr_exponent(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_frexp_exp(x);
#else
    int e = 0;
    (void)frexp(x, &e);
    return e;
#endif
}

// 1/sqrt(x) for x in [1/4, 2]: with g = 1 - x y^2, 1/sqrt(1 - g) = 1 + g/2 +
// 3 g^2/8 + O(g^3).
JR_FN double jr_rsqrt(double x)
{
    const double y = jr_rsq_approx(x);
    const double g = fma(-x*y, y, 1.0);
    return fma(y*g, fma(0.375, g, 0.5), y);
}

// 1/x for x in [1/2, 3]: with g = 1 - x y, 1/(1 - g) = 1 + g + g^2 + O(g^3).
JR_FN double jr_rcp(double x)
{
    const double y = jr_rcp_approx(x);
    const double g = fma(-x, y, 1.0);
    return fma(y*g, 1.0+g, y);
}

// True when the pair is far enough from orthogonal to rotate:
// |ga| > ctol |a| |b|, by the squares where they are in range.  Else the
// norms are taken one at a time, so that the test holds for squared norms
// near the bottom of the FP64 range, where al*be would underflow to 0.
JR_FN bool jr_rotates(double al, double be, double ga, double ctol)
{
    if(fmin(al, be) > 1e-130 && fmax(al, be) < 1e130)
        return ga*ga > (ctol*ctol)*(al*be);
    return al > 0.0 && be > 0.0 && fabs(ga) > ctol*(sqrt(al)*sqrt(be));
}

JR_FN void jacobi_rotation(double al, double be, double ga, double &c,
        double &s)
{
    const double d = be-al, h = 2.0*ga;
    const int e = jr_exponent(fmax(fabs(d), fabs(h)));
    const double ds = ldexp(d, -e), hs = ldexp(h, -e);
    const double q = fma(ds, ds, hs*hs);            // [1/4, 2]
    const double z = jr_rcp(fabs(ds)+q*jr_rsqrt(q));    // of [1/2, 3]
    const double t = (ds >= 0.0 ? hs : -hs)*z;
    c = jr_rsqrt(fma(t, t, 1.0));
    s = c*t;
}

#endif
