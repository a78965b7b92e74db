/*
 * gm_weight.h -- when a pair's mobility weight is exactly 1.0: the disorientation as the
 * device computes it, and the host's threshold for it.
 *
 * Compiled without contraction of products and sums, as everything that takes part in
 * a weight.  tests/test_weight_code.py runs both functions against the 24 candidates and the
 * weights themselves.
 */
#ifndef SCORE_GM_WEIGHT_H
#define SCORE_GM_WEIGHT_H

#include <math.h>

#include "gm_radd.h"
#include "score_gm.h"

static const double kPi = 3.1415926535897932384626433832795;
static const double kLagbHagb = ((15.0) / (180.0) * (kPi));

/* largest |component| over the six Grimmer candidates of q_def^-1 * q_rx
 * (SCORE_Math.cpp:230-239, :558-608); only + - * fabs and compares, so the
 * value is bit-identical to the host's.  The 24 candidates are the sums and
 * differences of two components times 1/sqrt(2), of all four (left to right) times
 * 1/2, and the components.  Rounding is monotone and symmetric, so no sign pattern
 * exceeds the one that adds the magnitudes, and among the pairs the two largest
 * magnitudes win: three candidates remain (24 kept 48 registers alive, which held
 * the commit pass at 12 waves a CU). */
GM_HD double grimmer_omega(const double *p, const double *q, double fac) {
    double m0 = q[0], m1 = -1.0 * q[1], m2 = -1.0 * q[2], m3 = -1.0 * q[3];
    const double a = fabs(m0 * p[0] - m1 * p[1] - m2 * p[2] - m3 * p[3]);
    const double b = fabs(p[0] * m1 + m0 * p[1] + (m2 * p[3] - m3 * p[2]));
    const double c = fabs(p[0] * m2 + m0 * p[2] + (-(m1 * p[3]) + m3 * p[1]));
    const double d = fabs(p[0] * m3 + m0 * p[3] + (m1 * p[2] - m2 * p[1]));
    const double ab = a > b ? a : b, ba = a > b ? b : a, cd = c > d ? c : d, dc = c > d ? d : c;
    const double l1 = ab > cd ? ab : cd;
    const double lo = ab > cd ? cd : ab, in = ab > cd ? ba : dc;
    const double l2 = lo > in ? lo : in;
    const double two = (l1 + l2) * fac, four = (((a + b) + c) + d) * 0.5;
    double omega = l1 > two ? l1 : two;
    if (four > omega) omega = four;
    return omega;
}

static inline double rh_weight_of_theta(const score_gm_params &p, double theta) {
    return 1.0 - (p.rh_cut * exp(-1.0 * p.rh_trans * pow((theta / kLagbHagb), p.rh_exponent)));
}

/* Largest omega for which the Rollett-Holm weight is exactly 1.0 with margin:
 * the device returns P = 1.0 for omega <= this value and asks the host otherwise.
 * Returns -1 when no safe threshold exists (shortcut disabled). */
static inline double rh_omega_threshold(const score_gm_params &p) {
    if (p.mobility_model != SCORE_GM_MOB_ROLLETTHOLM) return -1.0;
    if (!(p.rh_cut > 0.0 && p.rh_trans > 0.0 && p.rh_exponent > 0.0)) return -1.0;
    if (rh_weight_of_theta(p, kPi) != 1.0) return -1.0;
    double lo = 0.0, hi = kPi; /* invariant: weight(hi) == 1.0 */
    if (rh_weight_of_theta(p, lo) == 1.0) return 1.0; /* every pair has P == 1.0 */
    for (int it = 0; it < 200; it++) {
        double mid = 0.5 * (lo + hi);
        if (rh_weight_of_theta(p, mid) == 1.0) hi = mid;
        else lo = mid;
    }
    /* margin of 0.2 degree: the weight's deficit falls by a large factor over it */
    const double theta_hi = hi + 0.2 / 180.0 * kPi;
    if (theta_hi >= 2.0 * acos(0.85)) return -1.0; /* beyond the largest cubic disorientation */
    /* The weight is 1.0 - x with x = cut * exp(-trans * (theta / 15 deg)^n), which falls
     * with theta, and rounds to 1.0 once x <= 2^-54.  The computed x is off by at most
     * a factor 1 + arg * (n + 4) * 2^-52 (arg = trans * (theta / 15 deg)^n), which the
     * margin of 2 below covers at theta_hi and, since x falls faster than arg grows,
     * at every larger angle, while n and arg are moderate.  Other settings are checked
     * at 200,001 angles (7 of the 8 ms a handle took to create). */
    const double arg = p.rh_trans * pow((theta_hi / kLagbHagb), p.rh_exponent);
    const bool sure = p.rh_exponent <= 1000.0 && arg >= 2.0 && arg <= 700.0 && p.rh_cut * exp(-1.0 * arg) <= 0x1p-55;
    for (int i = 0; !sure && i <= 200000; i++) {
        double th = theta_hi + (kPi - theta_hi) * (double)i / 200000.0;
        if (rh_weight_of_theta(p, th) != 1.0) return -1.0;
    }
    double om = cos(0.5 * theta_hi);
    /* a few ulps below, so that 2*acos(om') >= theta_hi whatever the last-bit behaviour of acos */
    for (int i = 0; i < 4; i++) om = nextafter(om, 0.0);
    if (!(2.0 * acos(om) >= theta_hi)) return -1.0;
    return om;
}

#endif
