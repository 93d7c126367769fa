// sphg_roots.h -- FP64 square root and quotient of the pair sums.
#pragma once

#include <hip/hip_runtime.h>

namespace sphg {

// sqrt(x) and a / b without the scaling and the special cases that the general
// forms add, 7 and 3 FP64 instructions a pair (PCISPH, 351k particles with
// cohesion: 414 -> 407 us a step).  The hardware's estimates of 1/sqrt(x) and
// 1/b are refined by Newton steps with fma, for the root in the form that
// carries s ~ sqrt(x) and h ~ 1/(2 sqrt(x)) side by side (Goldschmidt), and the
// result is corrected by its exact residual x - s s, a - q b (P. Markstein,
// Computation of elementary functions on the IBM RISC System/6000 processor,
// IBM J. Res. Dev. 34, 1990), which rounds it correctly.  Equal to sqrt and /
// in every bit where the callers use them:
//   sqrt_n  squared distances of FP32 positions and displacements: 0 or at
//           least 2^-298, and up to h^2 (larger ones are not used).  0 is taken
//           as 1e-290, whose root is as good as zero beside 1.
//   div_n   masses and densities, quotients from 2^-60 to 2^60
__device__ inline double sqrt_n(double x) {
    x = fmax(x, 1e-290);
    const double y = __builtin_amdgcn_rsq(x);
    double h = y * 0.5, s = x * y;
    const double r = fma(-h, s, 0.5);
    s = fma(s, r, s);
    h = fma(h, r, h);
    s = fma(fma(-s, s, x), h, s);
    return fma(fma(-s, s, x), h, s);
}
__device__ inline double div_n(double a, double b) {
    double r = __builtin_amdgcn_rcp(b);
    r = fma(fma(-b, r, 1.0), r, r);
    r = fma(fma(-b, r, 1.0), r, r);
    const double q = a * r;
    return fma(fma(-b, q, a), r, q);
}

}  // namespace sphg
