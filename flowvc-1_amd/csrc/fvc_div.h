/* fvc_div.h - FP64 quotients by a divisor that many dividends share, rounded
 * to nearest as a division rounds them.
 *
 * With y = 1 / b rounded to nearest, a y is within two ulp of a / b; the
 * correction q + (a - b q) y with the residual from a fused multiply-add
 * brings it within one, and from there the same correction gives a / b
 * rounded to nearest (P. Markstein, Computation of elementary functions on
 * the IBM RISC System/6000 processor, 1990).  Five instructions where a
 * division takes twelve and more.  It holds for finite quotients and
 * residuals clear of the ends of the range: |b| in [1e-100, 1e100] (callers
 * keep y = 0 for others and divide); |a| under about 2^-900 may miss the last
 * bit, an infinite a gives NaN (callers test for it).  Compiled for the
 * device and, by the tests, for the host. */
#ifndef FVC_DIV_H
#define FVC_DIV_H

#include <math.h>

#ifdef __HIPCC__
#define FVC_DIV_HD __host__ __device__
#else
#define FVC_DIV_HD
#endif

static inline FVC_DIV_HD double fvc_near_inverse(double b) {
    return fabs(b) > 1e-100 && fabs(b) < 1e100 ? 1.0 / b : 0.0;
}

static inline FVC_DIV_HD double fvc_div_near(double a, double b, double y) {
    double q = a * y;
    q = fma(fma(-b, q, a), y, q);
    return fma(fma(-b, q, a), y, q);
}

#endif
