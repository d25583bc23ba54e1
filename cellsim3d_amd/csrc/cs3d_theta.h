// cs3d_theta.h - the angle force's float angle without the double division, square
// root and branches of the general acos.
//
// GetAngleForce (propagate.cu:32-36) stores acos(idk / (den + 1e-3)) into a float.
// cs3d_theta computes the angle to within 2^-37 of cs3d_acos of the correctly
// rounded quotient, and returns whether that fixes the float: where
// theta - 2^-37 and theta + 2^-37 round to the same float, every value between
// them does (rounding is monotone), so (float)cs3d_acos(...) is that float.  The
// callers take the general path otherwise, which one angle in 2^13 needs below 2 rad and
// one in 2^14 above (the boundaries lie 2^-23 and 2^-22 apart).
//
// Method.  t = x + 0.425 with x = idk * y, y = 1/(den + 1e-3) from a float
// reciprocal estimate and one Newton step in double (relative error below 2^-43: the
// estimate is within 2^-21.5, and the step squares it).
//   |t| <= 0.275 (angles of 98.6 to 134.4 degrees; the mesh's are 107 to 123 at
//   rest): acos(t - 0.425) as its degree-15 Chebyshev interpolant, computed by
//   gen_theta_coeffs.py: absolute error 2^-37.68, with the quotient's (2^-43 over
//   sin 134.4 deg) and the rounding of the evaluation less than 2^-37.
//   else, to |x| = 0.998: the reductions of cs3d_acos with its f(z) as a degree-8
//   interpolant (gen_acos_coeffs.py 8: relative error 2^-37.5, 2^-42 in the angle)
//   and the square root from a float estimate and one Newton step (2^-43); the
//   quotient's error over sin(acos 0.998) = 2^-4 dominates, 2^-39.
// Beyond 0.998, and for NaN, it returns false.
// In a relaxed or growing tissue no angle leaves the first range; in a colony that
// divides, some lane of 30 % of the waves does.
#pragma once

#include <math.h>

#include "cs3d_acos.h"

#if defined(__HIP_DEVICE_COMPILE__)
#define CS3D_RCP_EST(v) __builtin_amdgcn_rcpf(v)
#define CS3D_RSQ_EST(v) __builtin_amdgcn_rsqf(v)
// A branch hardly ever taken, which the wave takes as one: what it guards is placed
// behind the kernel's common path.  Every launch starts with an empty instruction
// cache, which is filled ahead of straight code only, so each jump over code in place
// is a miss (2000 cells: 42.0 us a step with these out of line, 42.6 in place; the
// division kernel with its events in place took 5.9 us instead of 4.8).
#define CS3D_SELDOM(c) __builtin_expect(__ballot(c) != 0, 0)
#else
#define CS3D_SELDOM(c) (c)
#endif
#if !defined(__HIP_DEVICE_COMPILE__) && !defined(CS3D_RCP_EST)  // a host test may put its own estimates here
#define CS3D_RCP_EST(v) (1.0f / (v))
#define CS3D_RSQ_EST(v) (1.0f / sqrtf(v))
#endif

// The coefficients, constant term first.  The kernels read them from device memory
// with scalar loads (the constant address space): as literals, which a
// double fma cannot take, each took a vector register pair, spilled, or two moves.
constexpr int kThetaCoeffs = 16, kAsinCoeffs = 9;
struct ThetaCoeffs {
    double a[kThetaCoeffs];  // acos(t - 0.425) on |t| <= 0.275
    double f[kAsinCoeffs];   // (asin(sqrt z)/sqrt z - 1)/z on [0, 1/4]
};
constexpr ThetaCoeffs kTheta = {{
    0x1.013fc1d19137cp+1, -0x1.1ad0006c3f28ap+0, 0x1.2562075db2a95p-2, -0x1.7e47498970436p-2,
    0x1.6f3486c6f7662p-2, -0x1.dc98c979d2978p-2, 0x1.30f9b7c2d69d5p-1, -0x1.a5be23a16b627p-1,
    0x1.27b551af3a5fbp+0, -0x1.ad9042f227fbep+0, 0x1.5529ebaa3a12dp+1, -0x1.01829230f9247p+2,
    0x1.a0d7d5213a545p+1, -0x1.37be56487c95fp+2, 0x1.ee6a87627ab84p+4, -0x1.872015f91ed66p+5,
}, {
    0x1.555555555ba9ep-3, 0x1.333333133277ep-4, 0x1.6db6f5e9d0b98p-5, 0x1.f1beb9c867b18p-6,
    0x1.6f347e4a44c5dp-6, 0x1.14eefea06d8d9p-6, 0x1.144d1f0d0554dp-6, 0x1.17d722d86d4bep-10,
    0x1.d06eddee004bep-6,
}};

// C: ThetaCoeffs in any address space
template <class C> CS3D_ACOS_FN bool cs3d_theta(float idk, float den, const C* c, float* theta) {
    const double d = (double)den + 1e-3;
    const double y0 = (double)CS3D_RCP_EST(den + 1e-3f);
    const double y = fma(fma(-d, y0, 1.0), y0, y0);
    const double t = fma((double)idk, y, 0.425);
    // even and odd powers apart: two chains half as long as Horner's
    const double u = t * t;
    double e = c->a[14], o = c->a[15];
#pragma unroll
    for (int i = 12; i >= 0; i -= 2) {
        e = fma(e, u, c->a[i]);
        o = fma(o, u, c->a[i + 1]);
    }
    double a = fma(o, t, e);
    bool in = fabs(t) <= 0.275;
    if (CS3D_SELDOM(!in) && !in) {
        const double x = t - 0.425, ax = fabs(x);
        in = ax <= 0.998;
        const bool big = ax > 0.5;
        const double z = big ? fma(-0.5, ax, 0.5) : x * x;
        const double r0 = (double)CS3D_RSQ_EST((float)z), s0 = z * r0;
        const double s = big ? fma(0.5 * r0, fma(-s0, s0, z), s0) : x;
        double f = c->f[8];
#pragma unroll
        for (int i = 7; i >= 0; --i) f = fma(f, z, c->f[i]);
        const double r = fma(s * z, f, s);  // asin(s)
        // pi/2 - r, 2 r, pi - 2 r
        a = big ? fma(x > 0.0 ? 2.0 : -2.0, r, x > 0.0 ? 0.0 : 0x1.921fb54442d18p+1) : 0x1.921fb54442d18p+0 - r;
    }
    const float lo = (float)(a - 0x1p-37), hi = (float)(a + 0x1p-37);
    *theta = lo;
    return (lo == hi) & in;
}
