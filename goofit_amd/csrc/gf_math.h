// gf_math.h -- FP64 log for the likelihood metrics, the NLL of many events as one
// logarithm, whole powers, and the scaled complementary error function.
//
// Every event of every likelihood sweep takes one logarithm per parameter point
// (-log of the normalised PDF value), and the multi-point sweeps -- up to 16
// points per event, MIGRAD's derivative rounds and the toy batches -- are bound by
// FP64 issue.  The device library's log spends about 76 FP64 instructions (much of
// it extra-precision arithmetic); this one spends 40 and one division, with an
// error below one unit in the last place over the whole double range (measured:
// 0.9 at most) and the IEEE results at 0, +inf, negative numbers and NaN.  On
// gfx950 it runs 1.5 times the device library's throughput.  It uses only
// correctly rounded operations (fma, frexp, +, *, /, comparisons and selects), so a
// host build of this header (GF_MATH_HD empty under a plain C++ compiler) gives the
// same bits as the device; the accuracy is pinned on the host against long double.
#pragma once

#include <cmath>

#ifdef __HIPCC__
#define GF_MATH_HD __host__ __device__
#else
#define GF_MATH_HD
#endif

namespace gfmath {

// ln 2 = ln2_hi + ln2_lo: ln2_hi is ln 2 rounded to 32 fractional bits (28 significant
// bits), so e * ln2_hi is exact for every binary exponent e of a double; ln2_lo is the
// rest, rounded to double.
constexpr double ln2_hi = 0x1.62e42ffp-1;
constexpr double ln2_lo = -0x1.718432a1b0e26p-35;

// log(x).  x = m 2^e with m in [sqrt(1/2), sqrt(2)) (frexp, then one doubling); with
// f = m - 1 (exact) and s = f / (2 + f), log m = 2 atanh(s) = f - s (f - Q), where
// Q = 2 s^2 (1/3 + s^2/5 + s^4/7 + ...) -- the atanh series, |s| < 0.1716, summed to
// s^20 (the first omitted term is below 2^-57 of log m) -- since 2 s = f - s f.  The
// form keeps f exact and lets the roundings of s enter only through the correction
// s (f - Q), at most a fifth of the result.  For |e| >= 2, log x = e ln2_hi + (e ln2_lo
// + log m), one rounding of a sum that log m enters at a quarter at most.  For |e| = 1
// (x in [sqrt(2)/4, sqrt(2)/2) or [sqrt(2), 2 sqrt(2))), where e ln 2 and log m cancel
// down to half, log x = (e ln2_hi + f) - (s (f - Q) - e ln2_lo): the first sum is exact
// there (e ln2_hi has 28 significant bits and f none below the sum's last place), so
// only the small correction carries rounding error.  log(+inf) = +inf, log(0) = -inf,
// log(x < 0) = NaN, NaN propagates; subnormal inputs are normalised by frexp.
GF_MATH_HD inline double log_d(double x) {
    int e;
    double m      = frexp(x, &e);  // x = m 2^e, 0.5 <= |m| < 1 for finite nonzero x
    const bool lo = m < 0x1.6a09e667f3bcdp-1;  // sqrt(1/2)
    m             = lo ? m + m : m;
    const double ed = (double)(lo ? e - 1 : e);
    const double f  = m - 1.0;
    const double s  = f / (2.0 + f);
    const double z  = s * s;
    // 2/(2n+1) for n = 10 .. 1, each rounded to double
    double q = 0x1.8618618618618p-4;
    q        = fma(q, z, 0x1.af286bca1af28p-4);
    q        = fma(q, z, 0x1.e1e1e1e1e1e1ep-4);
    q        = fma(q, z, 0x1.1111111111111p-3);
    q        = fma(q, z, 0x1.3b13b13b13b14p-3);
    q        = fma(q, z, 0x1.745d1745d1746p-3);
    q        = fma(q, z, 0x1.c71c71c71c71cp-3);
    q        = fma(q, z, 0x1.2492492492492p-2);
    q        = fma(q, z, 0x1.999999999999ap-2);
    q        = fma(q, z, 0x1.5555555555555p-1);
    const double Q    = z * q;
    const double logm = fma(-s, f - Q, f);
    const double far  = fma(ed, ln2_hi, fma(ed, ln2_lo, logm));
    const double near = fma(ed, ln2_hi, f) - fma(s, f - Q, -(ed * ln2_lo));
    double y          = (ed == 1.0 || ed == -1.0) ? near : far;
    y                 = x == 0.0 ? -HUGE_VAL : y;
    y                 = (x < 0.0 || x != x) ? NAN : y;
    y                 = x == HUGE_VAL ? HUGE_VAL : y;
    return y;
}

// The sum of -log(v) over many values as one logarithm: sum -log(v_k) over the v_k > 0
// (the others add 0, as the NLL metric gives them) equals -log(prod v_k).  The product
// is kept as a mantissa m and a binary exponent e (an integer, held in a double: exact
// below 2^53): each factor's own mantissa (frexp, exact) multiplies m (one rounding),
// the result is renormalised into [0.5, 1) (frexp, exact) and the exponents are added,
// so the product neither overflows nor underflows, and each factor adds one rounding of
// relative size 2^-53 to it -- an absolute error in the sum of logarithms below that of
// taking each logarithm apart.  A factor v <= 0 or NaN becomes 1.0 = 0.5 * 2^1, whose
// halving is exact and undone by the renormalisation; v = +inf makes the product +inf
// (the sum -inf), as the per-value form gives.  Start from (m, e) = (1, 0).
GF_MATH_HD inline void nll_add(double &m, double &e, double v) {
    int ev, em;
    const double a = frexp(v > 0.0 ? v : 1.0, &ev);
    m              = frexp(m * a, &em);
    e += (double)(ev + em);
}
// The same product with the exponent in an integer register (no conversion per factor):
// m is the double form's m bit for bit and e its exponent's value, for any sequence of
// factors whose exponent sum stays within int range (+-2^31: over 2^20 factors at the
// extreme exponents).
GF_MATH_HD inline void nll_add(double &m, int &e, double v) {
    int ev, em;
    const double a = frexp(v > 0.0 ? v : 1.0, &ev);
    m              = frexp(m * a, &em);
    e += ev + em;
}
// sum of -log(v_k) = -(log m + e ln 2)
GF_MATH_HD inline double nll_total(double m, double e) { return -fma(e, ln2_hi, fma(e, ln2_lo, log_d(m))); }

// Powers x^n, x^(n+1), ... of the polynomials, each within half a unit in the last place and
// some 2^-100 (the power kept as an unevaluated sum h + l): six operations a power, a sum and a
// select for its value, where the library's pow, which knows nothing of whole exponents, takes
// some 200 each time.
// Where l is no number (overflow, infinite x) h alone is the power, as pow gives it.
struct Powers {
    double h = 1.0, l = 0.0;
    GF_MATH_HD void times(double bh, double bl) {
        const double p = h * bh;
        l              = fma(h, bh, -p) + (h * bl + l * bh);
        h              = p;
    }
    GF_MATH_HD void next(double x) { times(x, 0.0); }
    // from x^0 to x^n by squarings: any exponent in at most 32 steps
    GF_MATH_HD void start(double x, unsigned n) {
        Powers b;
        b.h = x;
        start(b, n);
    }
    GF_MATH_HD void start(Powers b, unsigned n) {
        while(n) {
            if(n & 1) {
                times(b.h, b.l);
                round();
            }
            if((n >>= 1)) {
                b.times(b.h, b.l);
                b.round();
            }
        }
    }
    // h again the nearest double to the sum (l grows by a rounding of h a step)
    GF_MATH_HD void round() {
        const double s = h + l;
        if(s == s && s != 0) {
            l -= s - h;
            h = s;
        }
    }
    GF_MATH_HD double value() const {
        const double s = h + l;
        return s == s ? s : h;
    }
};
// x^n by n multiplications, for the small n >= 0 of a polynomial's terms
GF_MATH_HD inline double power(double x, int n) {
    Powers p;
    for(; n > 0; --n)
        p.next(x);
    return p.value();
}
// x^n of any whole n, uniform over the wave; a negative one from the reciprocal, kept as h + l
// too (the reciprocal of x^-n is 0 once that overflows, where x^n may be subnormal yet).
GF_MATH_HD inline double powi(double x, int n) {
    Powers p, b;
    b.h = x;
    if(n < 0) {
        b.h = 1.0 / x;
        b.l = fma(-x, b.h, 1.0) * b.h;
    }
    p.start(b, n < 0 ? 0u - (unsigned)n : (unsigned)n);
    return p.value();
}

// exp(x), N arguments side by side so that each constant is read once: x = k ln 2 + r with
// |r| <= ln(2)/2 (two-part ln 2: k ln2_hi is exact), exp r = 1 + r + r^2 p(r), p the
// Chebyshev series of (exp r - 1 - r) / r^2 cut at degree 9 (1.3e-17 of exp r), then one
// ldexp.  Below one unit in the last place; overflow, underflow to 0 through the
// subnormals, infinities and NaN as the library's.  c = the table: 1 / ln 2, ln2_hi,
// ln2_lo, the coefficients of p, the highest first.
#define GF_EXP_TABLE \
    0x1.71547652b82fep+0, 0x1.62e42ffp-1, -0x1.718432a1b0e26p-35, 0x1.af4ddf7e0398cp-26, \
    0x1.28917e26a6626p-22, 0x1.71de02365785cp-19, 0x1.a019b91328958p-16, 0x1.a01a01abe6830p-13, \
    0x1.6c16c1788a55fp-10, 0x1.11111111100dep-7, 0x1.5555555553d67p-5, 0x1.5555555555557p-3, \
    0x1.0000000000001p-1
constexpr int exp_terms = 13;
template <int N, class Table>
GF_MATH_HD inline void exp_n(const double (&x)[N], double (&y)[N], Table c) {
    double k[N], r[N];
    for(int i = 0; i < N; ++i) {
        const double v = x[i] < -1000.0 ? -1000.0 : x[i] > 1000.0 ? 1000.0 : x[i];
        k[i]           = rint(v * c[0]);
        r[i]           = fma(-k[i], c[2], fma(-k[i], c[1], v));
        y[i]           = c[3];
    }
    for(int t = 4; t < exp_terms; ++t) {
        const double ct = c[t];
        for(int i = 0; i < N; ++i)
            y[i] = fma(y[i], r[i], ct);
    }
    for(int i = 0; i < N; ++i)
        y[i] = ldexp(fma(r[i], fma(r[i], y[i], 1.0), 1.0), (int)k[i]);
}

// erfcx(u) = exp(u^2) erfc(u), the tail of a Gaussian without its exponential, for u >= 0:
// (1 + u) erfcx(u) runs from 1 at u = 0 to 1/sqrt(pi) at infinity and is smooth in t =
// (u - K) / (u + K), which maps [0, inf) to [-1, 1) (Shepherd and Laframboise, Math. Comp.
// 36 (1981) 249, with K = 3.75 and 1 + 2u); its Chebyshev series in t, cut below 3e-17 of
// it, is the polynomial of degree 23 below, computed in 60 digits from erfc and written in
// powers of t, the highest first.  One reciprocal serves both quotients: r = 1 /
// erfcx_den(u) from the caller, c = the table (a copy where the caller can read it fastest).
// Within 2.5 units in the last place (0.6 rms) over [0, 1e150]; above, where erfcx u is
// 1/(sqrt(pi) u) to rounding and the denominator would overflow, the value at 1e150.  NaN
// propagates.  30 FP64 operations and the reciprocal, no branch; the device library's erfc
// evaluates its ranges' polynomials under a divergent branch and an exponential of its own.
#define GF_ERFCX_TABLE \
    0x1.b67d3cbe87cfdp-33, -0x1.3ac6917ca74d1p-30, -0x1.4b3c756e41a2cp-29, 0x1.df8b7453833dcp-27, \
    0x1.135c3e7c71fe8p-26, -0x1.d4cee07a03890p-24, -0x1.160006d6a62aap-24, 0x1.a2af86b4cd31ep-21, \
    -0x1.518d8f65de133p-23, -0x1.66b4424d30f98p-18, 0x1.0fce79c4fa4c0p-17, 0x1.cf4eb0935ef46p-16, \
    -0x1.fc0bd8648af46p-14, 0x1.2839e4434b916p-14, 0x1.c58868fcff65ap-11, -0x1.044be4278f554p-8, \
    0x1.4a003abc297dbp-7, -0x1.1b08f7c015a79p-6, 0x1.333761f87299dp-6, -0x1.964c5507e5c25p-9, \
    -0x1.4cfc268c884b0p-5, 0x1.d6351b9255894p-4, -0x1.a79726791d142p-3, 0x1.6212fee9586e8p-1
constexpr int erfcx_terms = 24;
GF_MATH_HD inline double erfcx_arg(double u) { return u > 1e150 ? 1e150 : u; }
GF_MATH_HD inline double erfcx_den(double u) { return (u + 3.75) * (1.0 + u); }
// N arguments side by side: each coefficient is read once
template <int N, class Table>
GF_MATH_HD inline void erfcx(const double (&u)[N], const double (&r)[N], double (&y)[N], Table c) {
    double t[N];
    for(int i = 0; i < N; ++i) {
        t[i] = (u[i] - 3.75) * ((1.0 + u[i]) * r[i]);
        y[i] = c[0];
    }
    for(int k = 1; k < erfcx_terms; ++k) {
        const double ck = c[k];
        for(int i = 0; i < N; ++i)
            y[i] = fma(y[i], t[i], ck);
    }
    for(int i = 0; i < N; ++i)
        y[i] *= (u[i] + 3.75) * r[i];
}

}  // namespace gfmath
