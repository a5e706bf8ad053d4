// pow(x, y) evaluated as exp(y log x) in double-double arithmetic
// (Dekker / Knuth error-free sums and FMA products) with a 16-entry
// 2^(i/16) reduction for both the logarithm and the exponential. The result
// carries a relative error of a few 2^-70 before the final rounding, so it is
// the correctly rounded power except in rare near-halfway cases; glibc's pow
// has the same property, so the two agree on nearly every argument. Special
// operands (zero, negative or non-finite x, infinite or zero y, NaN) follow
// C99 Annex F.9.4.4 case by case, with no call to the platform pow: on the
// device its inlined body would add ~36 VGPRs to every kernel that reaches
// this function. Results below the normal range are rounded twice (once to
// 53 bits, once by ldexp), so they can differ from the correctly rounded
// subnormal by one unit (2^-1074).
//
// The same source compiles for the host (g++) and the device (hipcc).
#pragma once

#include <cmath>

#if defined(__HIPCC__)
#define MLR_HD __host__ __device__
#else
#define MLR_HD
#endif
#define MLR_CONST static constexpr

#include "ddpow_tables.hpp"

namespace mlr::ddpow {

struct alignas(16) DD {
    double hi, lo;
};

MLR_HD inline DD two_sum(double a, double b) {
    const double s = a + b;
    const double bb = s - a;
    return {s, (a - (s - bb)) + (b - bb)};
}
MLR_HD inline DD fast_two_sum(double a, double b) {
    const double s = a + b;
    return {s, b - (s - a)};
}
MLR_HD inline DD two_prod(double a, double b) {
    const double p = a * b;
    return {p, fma(a, b, -p)};
}

// n / d for several n, d and the quotients far from the exponent range's ends.
// On the device the refined reciprocal is formed once: its steps and the
// quotient's are those of one IEEE division there (reciprocal estimate, two
// Newton steps, product, remainder, correction), so the bits are the same.
struct Divider {
    double d;
#if defined(__HIP_DEVICE_COMPILE__)
    double y;
    MLR_HD explicit Divider(double den) : d(den) {
        y = __builtin_amdgcn_rcp(d);
        y = fma(y, fma(-d, y, 1.0), y);
        y = fma(y, fma(-d, y, 1.0), y);
    }
    MLR_HD double quot(double n) const {
        const double q = n * y;
        return fma(fma(-d, q, n), y, q);
    }
#else
    MLR_HD explicit Divider(double den) : d(den) {}
    MLR_HD double quot(double n) const { return n / d; }
#endif
};

// 2^(j/16), j = -8..8 (halving is exact)
#define MLR_C(i) {0.5 * kExp2Hi[i], 0.5 * kExp2Lo[i]}
#define MLR_E(i) {kExp2Hi[i], kExp2Lo[i]}
MLR_CONST DD kC[17] = {MLR_C(8), MLR_C(9), MLR_C(10), MLR_C(11), MLR_C(12), MLR_C(13), MLR_C(14), MLR_C(15), MLR_E(0),
                       MLR_E(1), MLR_E(2), MLR_E(3),  MLR_E(4),  MLR_E(5),  MLR_E(6),  MLR_E(7),  MLR_E(8)};
MLR_CONST DD kE[16] = {MLR_E(0), MLR_E(1), MLR_E(2),  MLR_E(3),  MLR_E(4),  MLR_E(5),  MLR_E(6),  MLR_E(7),
                       MLR_E(8), MLR_E(9), MLR_E(10), MLR_E(11), MLR_E(12), MLR_E(13), MLR_E(14), MLR_E(15)};
#undef MLR_C
#undef MLR_E

// nearest j with c = 2^(j/16) to m in [1/sqrt 2, sqrt 2), j in [-8, 8]: the
// thresholds m has reached. On the device 16 log2 m in FP32 decides (its error
// is below 1e-5), and the thresholds only where it lies that near to one.
MLR_HD inline int nearest_sixteenth(double m) {
#if defined(__HIP_DEVICE_COMPILE__)
    const float t = 16.0f * __builtin_amdgcn_logf((float)m), r = rintf(t);
    if (fabsf(t - r) <= 0.4995f) {
        const int j = (int)r;
        return j < -8 ? -8 : (j > 8 ? 8 : j);
    }
#endif
    int j = -8;
    for (int i = 0; i < 16; ++i) j += (m >= kThr[i]) ? 1 : 0;
    return j;
}

// ln(x) for normal x > 0 as a double-double.
MLR_HD inline DD log_dd(double x) {
    int k;
    double m = frexp(x, &k);  // [0.5, 1)
    if (m < 0.70710678118654752440) {
        m *= 2.0;
        k -= 1;
    }
    const int j = nearest_sixteenth(m);
    const double chi = kC[j + 8].hi, clo = kC[j + 8].lo;
    // s = (m - c) / (m + c) as a double-double; ln(m / c) = 2 atanh(s)
    const double n0 = m - chi;  // exact (Sterbenz)
    const DD num = two_sum(n0, -clo);
    DD den = two_sum(m, chi);
    den = fast_two_sum(den.hi, den.lo + clo);
    const Divider by_den(den.hi);
    const double shi = by_den.quot(num.hi);
    const double r = (fma(-shi, den.hi, num.hi) + num.lo) - shi * den.lo;
    const double slo = by_den.quot(r);
    const double z = shi * shi;
    // 2 s^3 (1/3 + z/5 + z^2/7 + z^3/9 + z^4/11), |s| < 0.011
    const double tail = shi * z * (2.0 / 3 + z * (2.0 / 5 + z * (2.0 / 7 + z * (2.0 / 9 + z * (2.0 / 11)))));
    const DD lm = fast_two_sum(2.0 * shi, 2.0 * slo + tail);
    // (16 k + j) ln2/16
    const double kk = (double)(16 * k + j);
    const DD kl = two_prod(kk, kLn2_16Hi);
    const double kl_lo = kk * kLn2_16Lo;
    DD s = two_sum(kl.hi, lm.hi);
    return fast_two_sum(s.hi, s.lo + (kl.lo + kl_lo + lm.lo));
}

// exp(p) for a double-double p with |p.hi| < 708.
MLR_HD inline double exp_dd(DD p) {
    const double n = rint(p.hi * (16.0 / 0.69314718055994530942));
    const DD q = two_prod(n, kLn2_16Hi);
    const double rh0 = p.hi - q.hi;  // exact for n != 0 (Sterbenz); p.hi when n = 0
    const double rl0 = (p.lo - q.lo) - n * kLn2_16Lo;
    const DD r = fast_two_sum(rh0, rl0);
    // exp(r) - 1 = r + r^2/2 + r^3 (1/6 + r/24 + ...), |r| < 0.0218
    const DD sq = two_prod(r.hi, r.hi);
    const double h = r.hi;
    const double cub = h * sq.hi *
                       (1.0 / 6 + h * (1.0 / 24 + h * (1.0 / 120 + h * (1.0 / 720 + h * (1.0 / 5040 + h * (1.0 / 40320))))));
    DD e = two_sum(h, 0.5 * sq.hi);
    e = fast_two_sum(e.hi, e.lo + (r.lo + r.lo * h + 0.5 * sq.lo + cub));
    const int ni = (int)n;
    const int i = ni & 15;
    const int sc = (ni - i) / 16;
    const double th = kE[i].hi, tl = kE[i].lo;
    // 2^(i/16) (1 + e)
    const DD a = two_prod(th, e.hi);
    const DD s = two_sum(th, a.hi);
    const double res = s.hi + (s.lo + (a.lo + tl + th * e.lo + tl * e.hi));
    return ldexp(res, sc);
}

// finite y is an integer / an odd integer (0.5 y is exact; every double
// of magnitude >= 2^53 is even)
MLR_HD inline bool is_int(double y) { return floor(y) == y; }
MLR_HD inline bool is_odd(double y) { return is_int(y) && !is_int(0.5 * y); }

// the special operands, given the power r of a finite nonzero |x| to a finite y
MLR_HD inline double pow_special(double x, double y, double r) {
    if (y == 0.0) return 1.0;               // even for a NaN operand
    if (x != x || y != y) return x + y;     // NaN
    const double ax = fabs(x);
    if (fabs(y) == INFINITY) {
        if (ax == 1.0) return 1.0;          // x = -1
        return (ax < 1.0) == (y > 0.0) ? 0.0 : INFINITY;
    }
    const bool odd = is_odd(y);
    if (x == 0.0 || ax == INFINITY) {
        // 0^y and inf^y: infinite when exactly one of (x = 0, y < 0) holds;
        // the sign of x survives for odd integer y
        const double z = (x == 0.0) == (y < 0.0) ? INFINITY : 0.0;
        return (std::signbit(x) && odd) ? -z : z;
    }
    if (x < 0.0 && !is_int(y)) return __builtin_nan("");
    return (x < 0.0 && odd) ? -r : r;
}

MLR_HD inline double pow_dd(double x, double y) {
    if (x == 1.0) return 1.0;  // even for a NaN y; whole waves of a uniform flow leave here
    // |x| finite, positive (subnormals included: frexp normalises them);
    // exactly 1 for y = 0
    const bool plain = x > 0.0 && x < INFINITY && fabs(y) < INFINITY;
    const double ax = fabs(x);
    const DD L = log_dd(ax);
    DD p = two_prod(y, L.hi);
    p = fast_two_sum(p.hi, p.lo + y * L.lo);
    double r;
    if (p.hi > 709.8) r = INFINITY;         // above ln(DBL_MAX) = 709.78...
    else if (p.hi < -745.2) r = 0.0;        // below ln(2^-1075) = -745.13...
    else r = exp_dd(p);
    return plain ? r : pow_special(x, y, r);
}

}  // namespace mlr::ddpow
