// Accuracy of gfmath::exp_n, erfcx and powi (goofit_amd/csrc/gf_math.h, built for the host
// with the same operations as on the device) against long double.
// Usage: special_check N SEED -> per function and range: n, the largest error in units of
// 2^-53 of the value and where; then the special values.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "gf_math.h"

static const double exp_table[]   = {GF_EXP_TABLE};
static const double erfcx_table[] = {GF_ERFCX_TABLE};

static double exp_1(double x) {
    const double a[1] = {x};
    double y[1];
    gfmath::exp_n(a, y, exp_table);
    return y[0];
}
static double erfcx_1(double u) {
    const double a[1] = {gfmath::erfcx_arg(u)}, r[1] = {1.0 / gfmath::erfcx_den(a[0])};
    double y[1];
    gfmath::erfcx(a, r, y, erfcx_table);
    return y[0];
}
// exp(u^2) erfc(u): below 8 the functions themselves (u^2 rounds by 64 x 2^-64), above it the
// asymptotic series 1 - z + 3 z^2 - 15 z^3 ..., z = 1 / (2 u^2) < 1/128, summed to 2^-64.
static long double erfcx_ref(long double u) {
    if(u < 8)
        return expl(u * u) * erfcl(u);
    const long double z = 1 / (2 * u * u);
    long double t = 1, s = 1;
    for(int k = 1; k < 40 && fabsl(t) > 1e-21L; ++k) {
        t *= -(2 * k - 1) * z;
        s += t;
    }
    return s / (u * 1.7724538509055160272981674833411452L);
}

struct Worst {
    double err = 0, at = 0;
    long long n = 0;
    void add(double x, double got, long double ref) {
        const double e = (double)(fabsl((long double)got - ref) / fabsl(ref)) * 0x1p53;
        ++n;
        if(!(e <= err)) {
            err = e;
            at  = x;
        }
    }
    // in units of the least subnormal, 2^-1074
    void add_tiny(double x, double got, long double ref) {
        const double e = (double)(fabsl((long double)got - ref) * 0x1p1000L * 0x1p74L);
        ++n;
        if(!(e <= err)) {
            err = e;
            at  = x;
        }
    }
    void print(const char *name) const { std::printf("%s n=%lld err=%.4f at=%.17g\n", name, n, err, at); }
};

int main(int argc, char **argv) {
    const long long N = argc > 1 ? std::atoll(argv[1]) : 1000000;
    std::mt19937_64 rng(argc > 2 ? std::strtoull(argv[2], nullptr, 10) : 1);
    std::uniform_real_distribution<double> u(0.0, 1.0);
    Worst e_all, e_small, x_low, x_mid, x_high, pw, pn, pl, pt, nt;
    for(long long i = 0; i < N; ++i) {
        double x = -707.0 + 1416.0 * u(rng);
        e_all.add(x, exp_1(x), expl((long double)x));
        x = (2 * u(rng) - 1) * std::pow(10.0, -8 * u(rng));
        e_small.add(x, exp_1(x), expl((long double)x));
        x = u(rng);
        x_low.add(x, erfcx_1(x), erfcx_ref(x));
        x = 1 + 9 * u(rng);
        x_mid.add(x, erfcx_1(x), erfcx_ref(x));
        x = std::pow(10.0, 1 + 149 * u(rng));
        x_high.add(x, erfcx_1(x), erfcx_ref(x));
        x           = (u(rng) < 0.5 ? -1 : 1) * std::pow(10.0, 4 * u(rng) - 2);
        const int n = (int)(i % 21);
        long double p = 1;
        for(int k = 0; k < n; ++k)
            p *= x;
        pw.add(x, gfmath::powi(x, n), p);
        pw.add(x, gfmath::power(x, n), p);
        pn.add(x, gfmath::powi(x, -n), 1 / p);
        // exponents to 2^31 of x with |log x^n| < 700 (not by n multiplications)
        const int big = (int)std::pow(2.0, 31 * u(rng) - 1e-9);
        x             = 1 + (2 * u(rng) - 1) * std::fmin(0.4, 500.0 / big);
        pl.add(x, gfmath::powi(x, big), powl(x, big));
        // powers in the subnormal range, of small and of huge x
        const int m = 1 + (int)(i % 6);
        x           = std::pow(10.0, (-323.0 + 15.0 * u(rng)) / m);
        if(m > 1) {
            p = 1;
            for(int k = 0; k < m; ++k)
                p *= x;
            pt.add_tiny(x, gfmath::powi(x, m), p);
        }
        x = 1 / x;
        if(m > 1) {
            p = 1;
            for(int k = 0; k < m; ++k)
                p *= x;
            nt.add_tiny(x, gfmath::powi(x, -m), 1 / p);
        }
    }
    e_all.print("exp_range");
    e_small.print("exp_small");
    x_low.print("erfcx_low");
    x_mid.print("erfcx_mid");
    x_high.print("erfcx_high");
    pw.print("powi");
    pn.print("powi_negative");
    pl.print("powi_large");
    pt.print("powi_tiny");
    nt.print("powi_negative_tiny");
    for(double x : {0.0, -0.0, 1.0, 710.0, -746.0, -745.0, 1e300, -1e300, (double)HUGE_VAL, -(double)HUGE_VAL, (double)NAN})
        std::printf("special exp x=%.17g y=%.17g library=%.17g\n", x, exp_1(x), std::exp(x));
    for(double x : {0.0, 1e200, (double)HUGE_VAL, (double)NAN})
        std::printf("special erfcx x=%.17g y=%.17g\n", x, erfcx_1(x));
    const double xs[] = {0.0, -0.0, 1e200, -1e200, (double)HUGE_VAL, -(double)HUGE_VAL, (double)NAN};
    for(double x : xs)
        for(int n : {0, 1, 2, 3, -1, -2})
            std::printf("special powi x=%.17g n=%d y=%.17g library=%.17g\n", x, n, gfmath::powi(x, n), std::pow(x, n));
    return 0;
}
