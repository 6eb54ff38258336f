/*
 * rc_ckbin.h -- how close to an edge of a bin the correlated-k step's quick
 * power is not trusted.
 */
#ifndef RC_CKBIN_H
#define RC_CKBIN_H

namespace rc {

/* The quick k^pwr, 1e-30 <= k <= 1e30, relative to its value.  ie = 1/pwr
 * an integer: p0 = exp2(pwr log2 k) in FP32, then p0 - p0 pwr (p0^ie - k)/k,
 * which for p0 = k^pwr (1 + eps) leaves (ie + 1)/2 eps^2.  eps: the logarithm
 * (up to 100) to an ulp and the product's rounding, 1.2e-5 pwr, then
 * the exponential to an ulp and k's rounding, 2e-7.  With those roundings
 * at their worst the error found is 3.1e-11 (ie 1), 2.8e-11 (3), 6.7e-12
 * (10) and 2.2e-12 (64): the bound is 1.3 to 5 times that, and ten times
 * the bound is the margin.  ie = 0 (any other pwr): log2 k to 1.5e-14 in
 * FP64, which the power multiplies by pwr; the margin is 60 times that. */
inline double ck_edge_margin(int ie, double pwr) {
    if (ie <= 0) return 1e-12 * (pwr > 1.0 ? pwr : 1.0);
    const double eps = 1.2e-5 / ie + 2e-7;
    return 5.0 * (ie + 1) * eps * eps;
}

}  // namespace rc

#endif
