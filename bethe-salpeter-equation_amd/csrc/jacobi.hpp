// The complex Jacobi rotation of the small Hermitian eigensolvers (per-k
// Hamiltonians, Rayleigh-Ritz), without divisions or square roots: a round of
// parallel rotations waits for its longest dependent chain.
#pragma once
#include "bse_common.hpp"

// 1/sqrt(x), x > 0: the hardware estimate and two Newton steps (1-2 ulp).
__device__ inline double jacobi_rsq(double x) {
    double r = __builtin_amdgcn_rsq(x);
    r = fma(0.5 * r, fma(-x * r, r, 1.0), r);
    return fma(0.5 * r, fma(-x * r, r, 1.0), r);
}

// Rotation of columns p, q:  p' = c p - conj(s) q,  q' = s p + c q, that
// zeroes A(p, q) = a; dl = what a(p, p) loses and a(q, q) gains.
struct JacobiRot { double c, dl; double2 s; };
__device__ inline JacobiRot jacobi_rot(double app, double aqq, double2 a) {
    // h = (a_qq - a_pp)/2, r = sqrt(h^2 + |a|^2), c^2 = (r + |h|)/(2 r),
    // s = sign(h) a / (2 r c); the pair is scaled by its size, so c and s have
    // all their digits however small a pair is (the sweeps' own convergence
    // tests form squares of the entries as they are: matrices of a size between
    // about 1e-140 and 1e150)
    JacobiRot t;
    const double h0 = 0.5 * (aqq - app);
    const double big = fmax(fabs(h0), fmax(fabs(a.x), fabs(a.y)));
    const bool act = a.x != 0.0 || a.y != 0.0;          // (a NaN goes on into c and s)
    int ex;
    (void)frexp(act ? big : 1.0, &ex);
    const double h = ldexp(h0, -ex);
    const double2 z = cmk(ldexp(a.x, -ex), ldexp(a.y, -ex));
    const double g2 = cabs2(z);
    const double ir = jacobi_rsq(act ? fma(h, h, g2) : 1.0);
    const double c2 = fma(0.5 * fabs(h), ir, 0.5);
    const double ic = jacobi_rsq(c2);
    const double f = copysign(0.5 * ir * ic, h);
    t.c = act ? c2 * ic : 1.0;
    t.s = act ? cscale(z, f) : cmk(0, 0);
    // |a| tan = sign(h) |a|^2 / (|h| + r)
    t.dl = act ? ldexp(g2 * f * ic, ex) : 0.0;
    return t;
}
