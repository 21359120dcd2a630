// gf_device.h -- per-event FP64 arithmetic of the likelihood path, for gfx950.
//
// The leaf PDFs, metrics, kinematics and truth resolution state, in the same operation order,
// what the reference's device function computes (file:line given per function), so that
// results round the same way on both sides; the library is built with -ffp-contract=off so no
// multiply-add is fused behind our back.  The lineshapes (factorised over classes of
// resonances), the three-Gaussian decay-time terms (by erfcx) and the polynomials' powers compute
// the same functions in other forms, each with its own rounding, given where it stands, as do
// the products in logarithms (k_reduce_prod).  The log, the whole powers, and exp and erfcx of
// the latter two are this library's own (gf_math.h); exp and erfc of the leaf PDFs, sqrt and the
// trigonometric functions are the device library's.
#pragma once

#include <hip/hip_runtime.h>

#include "gf_internal.h"
#include "gf_math.h"

namespace gfd {

// Wave-uniform read-only data (the program, parameter / normalisation /
// constant arrays, descriptor tables) is read through the constant address
// space: a uniform index then compiles to scalar loads through the scalar
// cache instead of per-lane vector loads followed by lane reads.  The data must
// not change while a kernel runs (it never does: it is uploaded between launches).
// The qualifier exists only in the device pass (the host pass has no address
// spaces and only parses these functions).
#if defined(__HIP_DEVICE_COMPILE__)
#define GF_CONST __attribute__((address_space(4)))
#else
#define GF_CONST
#endif
template <class T>
__device__ __forceinline__ const GF_CONST T *as_const(const T *p) {
    return (const GF_CONST T *)p;
}

// (re, im) += (cr + i ci) * (w.x + i w.y) as four fused multiply-adds (the code is
// built with contraction off, so the coherent sums ask for the fusion explicitly:
// half the instructions of separate products and sums, one rounding per step).
__device__ __forceinline__ void cmac(double &re, double &im, double cr, double ci, double2 w) {
    re = fma(cr, w.x, fma(-ci, w.y, re));
    im = fma(cr, w.y, fma(ci, w.x, im));
}

// The coherent sum sum_{i < nres} c_i W_i (device_DalitzPlot's totalAmp,
// src/PDFs/physics/Amp3Body.cu:88-108) with one fused multiply-add per real term, in
// groups of four resonances 4m .. 4m + 3: Re adds cr wr of the four, then -ci wi of
// the four; Im adds ci wr of the four, then cr wi of the four.  This is the order in
// which the FP64 matrix-core kernel adds its K terms (one 16x16x4 step takes one
// component of four resonances), so the vector and matrix-core sweeps give the same
// bits.  cpl(i) returns (cr, ci) of resonance i and is called for i < nres only; w
// holds NR >= nres waves, zero past nres.  A group that reaches past nres adds its
// terms past nres too (zero coupling, zero wave), as the matrix cores do: x + 0 is x,
// so only the sign of a zero sum could differ, which |A|^2 does not see.  Groups that
// lie wholly past nres are skipped, as the matrix-core kernel never forms them.
template <int NR, class Cpl>
__device__ __forceinline__ void coh_group(double &re, double &im, const double2 (&c)[4], const double2 *w) {
#pragma unroll
    for(int u = 0; u < 4; ++u) {
        re = fma(c[u].x, w[u].x, re);
        im = fma(c[u].y, w[u].x, im);
    }
#pragma unroll
    for(int u = 0; u < 4; ++u) {
        re = fma(-c[u].y, w[u].y, re);
        im = fma(c[u].x, w[u].y, im);
    }
}
template <int NR, class Cpl>
__device__ __forceinline__ void coh_sum(double &re, double &im, const Cpl &cpl, const double2 *w, int nres) {
    static_assert(NR % 4 == 0, "groups of four resonances");
#pragma unroll
    for(int m = 0; m < NR; m += 4) {
        double2 c[4];  // each coupling read once
        if(m + 4 <= nres) {
#pragma unroll
            for(int u = 0; u < 4; ++u)
                c[u] = cpl(m + u);
            coh_group<NR, Cpl>(re, im, c, w + m);
        } else if(m < nres) {
#pragma unroll
            for(int u = 0; u < 4; ++u)
                c[u] = m + u < nres ? cpl(m + u) : make_double2(0.0, 0.0);
            coh_group<NR, Cpl>(re, im, c, w + m);
        }
    }
}

// ------------------------------------------------------------------ grids

// Centre of local bin b of n equal bins on [lo, hi]: ((hi - lo) / n) * (b + 0.5) + lo,
// one rounding per operation in this order (MetricTaker.cu:81-84,
// SpecialResonanceIntegrator.cu:64-76).  Every grid kernel takes its cell centres
// from here, so the cells of an integral are the cells gf_grid_cells reports.
__host__ __device__ __forceinline__ double bin_centre(double lo, double hi, int n, int64_t b) {
    double x = hi - lo;
    x /= n;
    x *= ((double)b + 0.5);
    x += lo;
    return x;
}

// ---------------------------------------------------------------- leaf PDFs

// device_Gaussian, src/PDFs/basic/GaussianPdf.cu:7-17
__device__ __forceinline__ double gaussian(double x, double mean, double sigma) {
    return exp(-0.5 * (x - mean) * (x - mean) / (sigma * sigma));
}

// device_ExpGaus, src/PDFs/basic/ExpGausPdf.cu:6-24 (sqrt 2 truncated to 1.4142135623 as there)
__device__ __forceinline__ double expgaus(double x, double mean, double sigma, double alpha) {
    double ret    = 0.5 * alpha;
    double exparg = ret * (2 * mean + alpha * sigma * sigma - 2 * x);
    double erfarg = (mean + alpha * sigma * sigma - x) / (sigma * 1.4142135623);
    ret *= exp(exparg);
    ret *= erfc(erfarg);
    return ret;
}

// ------------------------------------------------------------ compensated sums

// Neumaier's variant of Kahan summation: s carries the rounded sum, c the
// accumulated rounding errors.
__device__ __forceinline__ void kb_add(double &s, double &c, double v) {
    double t = s + v;
    double d = (fabs(s) >= fabs(v)) ? ((s - t) + v) : ((v - t) + s);
    c += d;
    s = t;
}
__device__ __forceinline__ void kb_merge(double &s, double &c, double s2, double c2) {
    kb_add(s, c, s2);
    c += c2;
}
// The sum a compensated pair stands for.  Once s is infinite or NaN the
// correction is meaningless (inf - inf = NaN), and the plain sum's value -- the
// one the reference's uncompensated reduction gives -- is s itself.
__device__ __forceinline__ double kb_total(double s, double c) { return isfinite(s) ? s + c : s; }

// ------------------------------------------------------------------- metrics

// src/PDFs/MetricPointer.cu:8-58.  evt0/evt1 are the (bin entry, bin volume or
// error) of a binned event, unused for unbinned metrics.
__device__ __forceinline__ double metric(int m, double rawPdf, double evt0, double evt1, double norm,
                                         double totalEvents) {
    switch(m) {
    case 0: return rawPdf;
    case 1: rawPdf *= norm; return rawPdf > 0.0 ? -gfmath::log_d(rawPdf) : 0.0;
    case 2: return rawPdf * norm;
    case 3: {
        rawPdf *= norm;
        rawPdf *= evt1;
        if(rawPdf > 0) {
            double expEvents = totalEvents * rawPdf;
            return (expEvents - evt0 * gfmath::log_d(expEvents));
        }
        return 0;
    }
    case 4:
        rawPdf -= evt0;
        rawPdf /= evt1;
        rawPdf *= rawPdf;
        return rawPdf;
    case 5: {
        rawPdf *= norm;
        rawPdf *= evt1;
        double d = rawPdf * totalEvents - evt0;
        return d * d / (evt0 > 1 ? evt0 : 1);
    }
    default: return __builtin_nan("");
    }
}

// The NLL metric over a lane's events as one logarithm (gfmath::nll_add / nll_total): the
// kernels that reduce the NLL metric accumulate it this way, in their own event order per
// lane, in the registers of the (sum, residual) pair starting from (1, 0), so kernels that
// assign events to lanes alike give the same bits (the per-event values of
// evaluate_with_metric still use metric()).  k_reduce_prod alone does not: it adds the events'
// exponents apart and multiplies four events' other factors before each nll_add, and agrees with
// the others to the rounding of the exponents' sum.
__device__ __forceinline__ void nll_add(double &m, double &e, double rawPdf, double norm) {
    gfmath::nll_add(m, e, rawPdf * norm);
}
__device__ __forceinline__ double nll_total(double m, double e) { return gfmath::nll_total(m, e); }
constexpr int metric_nll = 1;

// --------------------------------------------------------- Dalitz kinematics

// inDalitz, src/PDFs/physics/DalitzPlotHelpers.cu:14-59
__device__ __forceinline__ bool in_dalitz(double m12, double m13, double bigM, double dm1, double dm2, double dm3) {
    double dm1pdm2  = dm1 + dm2;
    double bigMmdm3 = bigM - dm3;
    double bigMmdm1 = bigM - dm1;
    double m23      = bigM * bigM + dm1 * dm1 + dm2 * dm2 + dm3 * dm3 - m12 - m13;
    if(m23 < 0. || m23 > bigMmdm1 * bigMmdm1)
        return false;
    bool m12less     = (m12 < dm1pdm2 * dm1pdm2) ? false : true;
    bool m12grea     = (m12 > bigMmdm3 * bigMmdm3) ? false : true;
    double sqrtM12   = sqrt(m12);
    double dm11      = dm1 * dm1;
    double dm22      = dm2 * dm2;
    double dm33      = dm3 * dm3;
    double e1star    = 0.5 * (m12 - dm22 + dm11) / sqrtM12;
    double e3star    = 0.5 * (bigM * bigM - m12 - dm33) / sqrtM12;
    double rte1mdm11 = sqrt(e1star * e1star - dm11);
    double rte3mdm33 = sqrt(e3star * e3star - dm33);
    double minimum   = (e1star + e3star) * (e1star + e3star) - (rte1mdm11 + rte3mdm33) * (rte1mdm11 + rte3mdm33);
    bool m13less     = (m13 < minimum) ? false : true;
    double maximum   = (e1star + e3star) * (e1star + e3star) - (rte1mdm11 - rte3mdm33) * (rte1mdm11 - rte3mdm33);
    bool m13grea     = (m13 > maximum) ? false : true;
    return m12less && m12grea && m13less && m13grea;
}

// twoBodyCMmom, src/PDFs/physics/resonances/Resonance.cu:48-60
__host__ __device__ __forceinline__ double two_body_cm_mom(double rMassSq, double d1m, double d2m) {
    double kin1 = 1 - (d1m + d2m) * (d1m + d2m) / rMassSq;
    kin1        = kin1 >= 0 ? sqrt(kin1) : 1;
    double kin2 = 1 - (d1m - d2m) * (d1m - d2m) / rMassSq;
    kin2        = kin2 >= 0 ? sqrt(kin2) : 1;
    return 0.5 * sqrt(rMassSq) * kin1 * kin2;
}

// twoBodyCMMothermom, Resonance.cu:62-75
__host__ __device__ __forceinline__ double two_body_cm_mother_mom(double rMassSq, double dm, double d3m) {
    double kin1 = 1 - (dm + d3m) * (dm + d3m) / rMassSq;
    kin1        = kin1 >= 0 ? sqrt(kin1) : 1;
    double kin2 = 1 - (dm - d3m) * (dm - d3m) / rMassSq;
    kin2        = kin2 >= 0 ? sqrt(kin2) : 1;
    return 0.5 * rMassSq * kin1 * kin2 / dm;
}

// x^(2 spin + 1) for spin 0, 1, 2 by multiplication (the reference calls pow with
// the double exponent 2 spin + 1; products differ from pow by a few ulp, far
// inside the likelihood tolerance, and avoid FP64 pow's log/exp sequence).
__host__ __device__ __forceinline__ double odd_power(double x, int spin) {
    const double x2 = x * x;
    double r        = x;
    for(int k = 0; k < spin; ++k)
        r *= x2;
    return r;
}

// dampingFactorSquare, Resonance.cu:77-86 (spin-2 form as written there)
__device__ __forceinline__ double damping_factor_square(double cmmom, int spin, double mRadius) {
    double square  = mRadius * mRadius * cmmom * cmmom;
    double dfsq    = 2 * square;
    double dfsqres = 13 * square / ((square - 3) * (square - 3)) + 9 * square * square;
    return (spin == 2) ? dfsqres : dfsq;
}

// dampingFactorSquareNorm, Resonance.cu:88-97
__host__ __device__ __forceinline__ double damping_factor_square_norm(double cmmom, int spin, double mRadius) {
    double square  = mRadius * mRadius * cmmom * cmmom;
    double dfsq    = 1 + square;
    double dfsqres = dfsq + 8 + 2 * square + square * square;
    return (spin == 2) ? dfsqres : dfsq;
}

// hFun, dh_dsFun, fsFun, dFun: Resonance.cu:5-46 (pi truncated to 3.14159265359 as there; the
// logarithm is gf_math.h's, so that a plan filled in on the host has the device's bits)
__host__ __device__ __forceinline__ double h_fun(double s, double daug2Mass, double daug3Mass) {
    const double _pi = 3.14159265359;
    double sm        = daug2Mass + daug3Mass;
    double sqrt_s    = sqrt(s);
    double k_s       = two_body_cm_mom(s, daug2Mass, daug3Mass);
    return ((2 / _pi) * (k_s / sqrt_s) * gfmath::log_d((sqrt_s + 2 * k_s) / (sm)));
}
__host__ __device__ __forceinline__ double dh_ds_fun(double s, double daug2Mass, double daug3Mass) {
    const double _pi = 3.14159265359;
    double k_s       = two_body_cm_mom(s, daug2Mass, daug3Mass);
    return h_fun(s, daug2Mass, daug3Mass) * (1.0 / (8.0 * (k_s * k_s)) - 1.0 / (2.0 * s)) + 1.0 / (2.0 * _pi * s);
}
__host__ __device__ __forceinline__ double d_fun(double s, double daug2Mass, double daug3Mass) {
    const double _pi = 3.14159265359;
    double sm        = daug2Mass + daug3Mass;
    double sm24      = sm * sm / 4.0;
    double m         = sqrt(s);
    double k_m2      = two_body_cm_mom(s, daug2Mass, daug3Mass);
    return 3.0 / _pi * sm24 / (k_m2 * k_m2) * gfmath::log_d((m + 2 * k_m2) / sm) + m / (2 * _pi * k_m2)
           - sm24 * m / (_pi * (k_m2 * k_m2 * k_m2));
}

// ------------------------------------------------------------- lineshapes
//
// plainBW (src/PDFs/physics/resonances/RBW.cu:9-86) and gouSak (GS.cu:9-75), each
// (A + iB) / (A^2 + B^2) sqrt(F F_mother) S(spin), factorised.  With q, p the momenta of
// the daughters and of the bachelor at the point and q0, p0 at the nominal mass,
//   plain:  A = m^2 - s,         B = m^2 G (q / q0)^(2 spin + 1) F / sqrt(s)
//   GS:     A = m^2 - s + f(s),  B = m G (q / q0)^(2 spin + 1) F,  times 1 + d G / m
// and F = D(q0) / D(q) (or D'(q) without normalisation), F_mother likewise.  So B =
// kb bf and the amplitude's factor is ks sf, where bf = q^(2 spin + 1) / (D(q) sqrt(s)) and
// sf = S / sqrt(D(q) D(p)) depend on the point only and kb, ks on the mass and width only:
// line_class forms the former once for all resonances of a class, line_plan_term the latter
// once per launch, and a resonance costs one division per point.  (Evaluating each
// shape apart took 422 FP64 operations and a dozen square roots and divisions.)
// The momenta keep the thresholds' rules: a factor 1 - (ma + mb)^2 / s below zero is 1.

// The numbers of a plan's term t, with its class's and the plan's own if it is the first,
// from the current masses, widths (P) and decay constants: the nominal-mass parts of
// plainBW and gouSak.
template <class Plan>
__host__ __device__ __forceinline__ void line_plan_term(Plan &plan, int t, const double *__restrict__ P,
                                                        const GfDecay &d) {
    if(t == 0) {
        const double a = d.daug2Mass + d.daug3Mass, b = d.daug2Mass - d.daug3Mass;
        plan.m2    = d.motherMass * d.motherMass;
        plan.rm    = d.mother_meson_radius;
        plan.gsum2 = a * a;
        plan.gdif2 = b * b;
        plan.ginv  = 1.0 / a;
    }
    if(t >= plan.nterm)
        return;
    GfLineTerm &r   = plan.term[t];
    GfLineClass &c  = plan.cls[r.cls];
    const int pair  = c.pair, spin = c.spin;
    if(pair < 0)
        return;
    const double M = d.motherMass;
    // daughters and bachelor of the pair (RBW.cu:13-16), and the spin factor's A, B, C
    const double da = 2 == pair ? d.daug2Mass : d.daug1Mass;
    const double db = 0 == pair ? d.daug2Mass : d.daug3Mass;
    const double mA = 0 == pair ? d.daug1Mass : (1 == pair ? d.daug3Mass : d.daug2Mass);
    const double mB = 0 == pair ? d.daug2Mass : (1 == pair ? d.daug1Mass : d.daug3Mass);
    const double mC = 0 == pair ? d.daug3Mass : (1 == pair ? d.daug2Mass : d.daug1Mass);
    if(t == c.first) {
        const double t1 = M * M - mC * mC, t2 = mA * mA - mB * mB;
        c.sum2  = (da + db) * (da + db);
        c.dif2  = (da - db) * (da - db);
        c.mc    = mC;
        c.msum2 = (M + mC) * (M + mC);
        c.mdif2 = (M - mC) * (M - mC);
        c.r2    = d.meson_radius * d.meson_radius;
        c.rm2   = d.mother_meson_radius * d.mother_meson_radius * 0.25 / (M * M);
        c.s0    = t1 * t2;
        c.s1    = 2 * M * M + 2 * mC * mC;
        c.s2    = t1 * t1;
        c.s3    = 2 * mA * mA + 2 * mB * mB;
        c.s4    = t2 * t2;
    }
    const double m  = P[r.p], w = P[r.p + 1], m2 = m * m;
    const double q0 = two_body_cm_mom(m2, da, db);
    double kb       = (r.kind == GR_GS ? sqrt(m2) : m2) * w / odd_power(q0, spin);
    double ks       = 1.0;
    if(spin != 0 && c.norm) {
        const double p0 = two_body_cm_mother_mom(m2, M, mC);
        const double f  = damping_factor_square_norm(q0, spin, d.meson_radius);
        kb *= f;
        ks = sqrt(f) * sqrt(damping_factor_square_norm(p0, spin, d.mother_meson_radius));
    }
    if(r.kind == GR_GS) {
        // dFun and fsFun at the nominal mass (GS.cu:53-57)
        const double k0 = two_body_cm_mom(m2, d.daug2Mass, d.daug3Mass);
        ks *= 1.0 + d_fun(m2, d.daug2Mass, d.daug3Mass) * w / sqrt(m2);
        r.f0 = w * m2 / (k0 * k0 * k0);
        r.h0 = h_fun(m2, d.daug2Mass, d.daug3Mass);
        r.d0 = k0 * k0 * dh_ds_fun(m2, d.daug2Mass, d.daug3Mass);
    }
    r.m2 = m2;
    r.kb = kb;
    r.ks = ks;
}

// 1 / sqrt(x) and 1 / x of a normal x > 0, to about one unit in the last place: the
// hardware's estimate and two Newton steps.  (The barrier denominators are at least 1 and
// the propagators' are squares of masses: nothing here comes near the ends of the range
// for which the library's forms scale their operands.)
__device__ __forceinline__ double rsqrt_n(double x) {
    double y = __builtin_amdgcn_rsq(x);
    y        = fma(y, fma(-0.5 * x * y, y, 0.5), y);
    return fma(y, fma(-0.5 * x * y, y, 0.5), y);
}
__device__ __forceinline__ double rcp_n(double x) {
    double y = __builtin_amdgcn_rcp(x);
    y        = fma(y, fma(-x, y, 1.0), y);
    return fma(y, fma(-x, y, 1.0), y);
}

// 1 - t / s with the thresholds' rule (below zero: 1).  r = 1 / s; next to the threshold
// the quotient decides as the reference's division does.
__device__ __forceinline__ double threshold_factor(double t, double s, double r) {
    const double d = s - t;
    double k       = d * r;
    if(fabs(d) < 1e-14 * s)
        k = 1 - t / s;
    return k >= 0 ? k : 1;
}

// The pair's part at one point: s the pair's mass squared, r = 1 / s and the momentum
// (two_body_cm_mom), u = q / sqrt(s) and q2 = q^2.
__device__ __forceinline__ void line_pair(const GfLineClass &c, double m12, double m13, double m23, double &s,
                                          double &r, double &u, double &q2) {
    s        = 0 == c.pair ? m12 : (1 == c.pair ? m13 : m23);
    r        = 1.0 / s;
    double k = threshold_factor(c.sum2, s, r);
    if(c.dif2 != 0)  // uniform: equal daughter masses give exactly 1
        k *= threshold_factor(c.dif2, s, r);
    u  = 0.5 * sqrt(k);
    q2 = 0.25 * s * k;
}

// The class's part: bf and sf as above, from the barrier and spin factors
// (dampingFactorSquareNorm, dampingFactorSquare and spinFactor, Resonance.cu:77-155).
template <class Plan>
__device__ __forceinline__ void line_class(const GF_CONST Plan *__restrict__ plan, const GfLineClass &c,
                                           double m12, double m13, double m23, double s, double r, double u, double q2,
                                           double &bf, double &sf) {
    bf = u;
    sf = 1.0;
    if(0 == c.spin)
        return;
    for(int k = 0; k < c.spin; ++k)
        bf *= q2;
    const double z = c.r2 * q2;
    double g;  // multiplies the amplitude
    if(c.norm) {
        // the bachelor's momentum in the form of two_body_cm_mother_mom, 0.5 s / M times two
        // square roots that are 1 below s = (M - mc)^2, the end of the plot
        double k = 1.0;
        if(s >= c.mdif2 * (1 - 1e-15)) {
            const double k1 = 1 - c.msum2 / s, k2 = 1 - c.mdif2 / s;
            k = (k1 >= 0 ? k1 : 1) * (k2 >= 0 ? k2 : 1);
        }
        const double zm = c.rm2 * s * s * k;
        const double dq = 2 == c.spin ? fma(z, z + 3, 9) : 1 + z;
        const double dm = 2 == c.spin ? fma(zm, zm + 3, 9) : 1 + zm;
        g               = rsqrt_n(dq * dm);
        bf *= g * g * dm;
    } else {
        const double pm = two_body_cm_mom(plan->m2, sqrt(s), c.mc);
        const double f  = 2 == c.spin ? 13 * z / ((z - 3) * (z - 3)) + 9 * z * z : 2 * z;
        g               = sqrt(f * damping_factor_square(pm, c.spin, plan->rm));
        bf *= f;
    }
    const double sAC = 0 == c.pair ? m13 : (1 == c.pair ? m23 : m12);
    const double sBC = 0 == c.pair ? m23 : (1 == c.pair ? m12 : m13);
    double f         = -fma(r, c.s0, sBC - sAC);
    if(2 == c.spin)
        f = fma(f, f, -(fma(r, c.s2, s - c.s1) * fma(r, c.s4, s - c.s3)) * (1.0 / 3.0));
    sf = g * f;
}

// A plan in a kernel's arguments or on the device.
__device__ __forceinline__ const GF_CONST GfLinePlanArg *plan_at(const GfLinePlanArg &p) { return as_const(&p); }
__device__ __forceinline__ const GF_CONST GfLinePlan *plan_at(const GfLinePlan *p) { return as_const(p); }

// Every wave of the plan whose resonance is in mask (ALL: every one), at one point: emit(row, swap, add,
// value).  m23 is the same for the swapped point (m13, m12).  All control flow is
// uniform over the wave, and a class or term is read from the plan as a whole (one wait
// for its scalar loads).
template <bool ALL, class Plan, class Emit>
__device__ __forceinline__ void line_waves(const GF_CONST Plan *__restrict__ plan, double m12, double m13, double m23,
                                           uint32_t mask, const Emit &emit) {
    double s = 0, r = 0, u = 0, q2 = 0, bf, sf;
    int chan = -1;
    for(int ci = 0; ci < plan->nclass; ++ci) {
        const GfLineClass c = plan->cls[ci];
        if(!ALL && !(c.res & mask))
            continue;
        const int k1 = c.first + c.count;
        if(c.pair < 0) {  // nonres, NonRes.cu:8-11
            for(int k = c.first; k < k1; ++k)
                if(ALL || ((mask >> plan->term[k].res) & 1u))
                    emit(plan->term[k].res, c.swap, 0, make_double2(1.0, 0.0));
            continue;
        }
        const double x = c.swap ? m13 : m12, y = c.swap ? m12 : m13;
        if(chan != 4 * c.swap + c.pair) {
            chan = 4 * c.swap + c.pair;
            line_pair(c, x, y, m23, s, r, u, q2);
        }
        line_class(plan, c, x, y, m23, s, r, u, q2, bf, sf);
        if(c.gs) {
            // hFun takes the masses of daughters 2 and 3 in every channel, as there
            const double _pi = 3.14159265359;
            const double k   = threshold_factor(plan->gsum2, s, r) * threshold_factor(plan->gdif2, s, r);
            const double rs = sqrt(s), v = 0.5 * sqrt(k);
            const double h  = (2 / _pi) * v * gfmath::log_d(rs * fma(2, v, 1) * plan->ginv);
            for(int j = c.first; j < k1; ++j) {
                const GfLineTerm t = plan->term[j];
                const double A0 = t.m2 - s, B = t.kb * bf * rs;
                const double A = fma(t.f0, fma(0.25 * s * k, h - t.h0, A0 * t.d0), A0);
                const double C = t.ks * sf * rcp_n(fma(A, A, B * B));
                if(ALL || ((mask >> t.res) & 1u))
                    emit(t.res, c.swap, t.add, make_double2(A * C, B * C));
            }
            continue;
        }
        GfLineTerm t = plan->term[c.first];
        for(int j = c.first; j < k1; ++j) {
            const GfLineTerm next = plan->term[j + 1];  // its loads are in flight behind this term
            if(ALL || ((mask >> t.res) & 1u)) {
                const double A = t.m2 - s, B = t.kb * bf;
                const double C = t.ks * sf * rcp_n(fma(A, A, B * B));
                emit(t.res, c.swap, t.add, make_double2(A * C, B * C));
            }
            t = next;
        }
    }
}

// ------------------------------------------------------- time resolutions

// device_truth_resolution, src/PDFs/physics/TruthResolution.cu:6-27: the decay-time
// terms without smearing.
__device__ __forceinline__ double truth_resolution(double coshterm, double costerm, double sinhterm, double sinterm,
                                                   double tau, double dtime, double xmixing, double ymixing) {
    double ret = 0;
    dtime /= tau;
    ret += coshterm * cosh(ymixing * dtime);
    ret += costerm * cos(xmixing * dtime);
    ret -= 2 * sinhterm * sinh(ymixing * dtime);
    ret -= 2 * sinterm * sin(xmixing * dtime);
    ret *= exp(-dtime);
    return ret;
}

// exp and erfcx with their constants in constant memory: scalar loads next to their use.
// (As literals they are moved to the front of the event loops, some 76 scalar registers
// that are then spilled to vector lanes and read back one half at a time.)
static __constant__ double exp_table[gfmath::exp_terms]     = {GF_EXP_TABLE};
static __constant__ double erfcx_table[gfmath::erfcx_terms] = {GF_ERFCX_TABLE};
template <int N>
__device__ __forceinline__ void exp_n(const double (&x)[N], double (&y)[N]) {
    const GF_CONST double *c = as_const(exp_table);
    asm volatile("" : "+s"(c));  // not loop-invariant
    gfmath::exp_n(x, y, c);
}
template <int N>
__device__ __forceinline__ void erfcx(const double (&u)[N], double (&y)[N]) {
    const GF_CONST double *c = as_const(erfcx_table);
    asm volatile("" : "+s"(c));
    double a[N], r[N];
#pragma unroll
    for(int i = 0; i < N; ++i) {
        a[i] = gfmath::erfcx_arg(u[i]);
        r[i] = rcp_n(gfmath::erfcx_den(a[i]));
    }
    gfmath::erfcx(a, r, y, c);
}

// The decay-time terms P1..P4 (cosh, cos, sinh, sin parts) of the three-Gaussian model,
// device_threegauss_resolution, ThreeGaussResolution.cu:63-115: core, tail and outlier
// Gaussians (fractions f_c, f_t, 1 - f_c - f_t) with per-event width sigma.  R = the 13
// parameters: fractions, biases and scales, selection bias, common offsets.
//
// Per Gaussian (gaussian(), ThreeGaussResolution.cu:11-61): the terms convolved with a
// Gaussian of width s centred on the bias; cos and sin are expanded to second and third
// order in x t / tau.  With w = t / s, X = exp(-w^2/2) and, for a decay rate g, u =
// (s g - w) / sqrt(2), the integral of exp(-g t') over t' > 0 under the Gaussian is S(g) / 2,
// S(g) = exp(u^2 - w^2/2) erfc(u) = X erfcx(u); for u < 0, erfc(u) = 2 - erfc(-u) and
// u^2 - w^2/2 = s g (s g / 2 - w), formed so because u^2 and w^2/2 cancel for t >> s.  With
// g0 = 1/tau + selection bias, g+- = g0 -+ y/tau, u of g0 and R = sqrt(2) s x / tau, the
// moments' recursion in u leaves
//   P1, P3 = (S(g+) +- S(g-)) / 4,
//   P2 = S/2 - R^2/2 (S (1/2 + u^2)/2 - u h),  P4 = R (h - u S/2) - R^3/6 (h (1 + u^2) - u S (3/2 + u^2)/2),
// h = X / (2 sqrt(pi)).  Bound by FP64 issue: three erfcx and four exponentials per Gaussian
// (350 operations), X shared, where three of the library's erfc and five exponentials took
// some 1000 and the cancelling exponent cost w^2 / 2 roundings (P1 of exponential times at
// widths of 0.03 to 0.08, against 40 digits: 2.3e-14 rms and 7e-15 mean then, 1.4e-16 and
// 3e-17 now).
struct TimeTerms {
    double P1, P2, P3, P4;
};
// The resolution's parameters, of Gaussian k: fraction, bias and scale (in units of sigma).
struct GaussParams {
    const GF_CONST double *R;
    __device__ __forceinline__ double selbias() const { return R[8]; }
    __device__ __forceinline__ void get(int k, double &f, double &b, double &s) const {
        const int o = k < 1 ? 0 : 2;  // the tail and the outlier share their offsets
        f           = k < 2 ? R[k] : 1 - R[0] - R[1];
        b           = R[2 + 2 * k] + R[9 + o];
        s           = R[3 + 2 * k] * R[10 + o];
    }
};
template <class Params>
__device__ __forceinline__ TimeTerms threegauss_terms(const Params &R, double tau, double dtime, double xmixing,
                                                      double ymixing, double sigma) {
    const double G = 1 / tau, g0 = G + R.selbias(), gy = ymixing * G;
    TimeTerms P{0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
    for(int k = 0; k < 3; ++k) {
        double f, b, s;
        R.get(k, f, b, s);
        s *= sigma;
        const double w    = (dtime - b * sigma) * rcp_n(s);
        const double q[3] = {s * g0, s * (g0 - gy), s * (g0 + gy)};
        double u[3], S[3], E[4];
        {
            const double x[4] = {-0.5 * w * w, q[0] * fma(0.5, q[0], -w), q[1] * fma(0.5, q[1], -w),
                                 q[2] * fma(0.5, q[2], -w)};
            exp_n(x, E);
        }
        {
            double a[3];
#pragma unroll
            for(int i = 0; i < 3; ++i) {
                u[i] = M_SQRT1_2 * (q[i] - w);
                a[i] = fabs(u[i]);
            }
            erfcx(a, S);
        }
#pragma unroll
        for(int i = 0; i < 3; ++i) {
            S[i] *= E[0];
            S[i] = u[i] >= 0 ? S[i] : fma(2.0, E[1 + i], -S[i]);
        }
        const double h   = (0.25 * M_2_SQRTPI) * E[0], S0 = 0.5 * S[0];
        const double r   = M_SQRT2 * s * xmixing * G, r2 = r * r, u2 = u[0] * u[0];
        const double It2 = fma(S0, 0.5 + u2, -u[0] * h);
        const double It3 = fma(h, 1 + u2, -u[0] * S0 * (1.5 + u2));
        P.P1 = fma(f, 0.25 * (S[1] + S[2]), P.P1);
        P.P2 = fma(f, fma(-0.5 * r2, It2, S0), P.P2);
        P.P3 = fma(f, 0.25 * (S[1] - S[2]), P.P3);
        P.P4 = fma(f * r, fma((-1.0 / 6.0) * r2, It3, fma(-u[0], S0, h)), P.P4);
    }
    return P;
}
// ThreeGaussResolution.cu:117-122: the rate from the terms
__device__ __forceinline__ double threegauss_rate(const TimeTerms &P, double coshterm, double costerm,
                                                  double sinhterm, double sinterm) {
    double ret = 0;
    ret += coshterm * P.P1;
    ret += costerm * P.P2;
    ret -= 2 * sinhterm * P.P3;
    ret -= 2 * sinterm * P.P4;
    return ret;
}

// The resolution function of a time-dependent node, dispatched on its wave-uniform kind.
__device__ __forceinline__ double time_resolution(int kind, const GF_CONST double *__restrict__ R, double t1, double t2,
                                                  double abr, double abi, double tau, double dtime, double x,
                                                  double y, double sigma) {
    if(kind == GT_THREEGAUSS)
        return threegauss_rate(threegauss_terms(GaussParams{R}, tau, dtime, x, y, sigma), t1, t2, abr, abi);
    return truth_resolution(t1, t2, abr, abi, tau, dtime, x, y);
}

// Counter-based random numbers: splitmix64 finaliser of (key, counter).  Any
// (key, counter) pair gives the same value on every run and device.
__host__ __device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
// uniform in [0, 1) with 53 random bits
__host__ __device__ __forceinline__ double unif01(uint64_t key, uint64_t ctr) {
    return (double)(mix64(key ^ mix64(ctr)) >> 11) * (1.0 / 9007199254740992.0);
}

}  // namespace gfd
