// gf_kernels.hip -- gfx950 kernels of the likelihood path.
//
//  * k_reduce_metric / k_eval_metric: the fused per-event evaluation of a
//    compiled PDF tree over SoA event columns, the metric (NLL, Prob, ...),
//    and a compensated FP64 sum: Neumaier per thread, wave shuffles, LDS
//    across waves, one partial per block and a last-block pass that adds the
//    partials in a fixed order (deterministic for a given grid).  Replaces the
//    thrust::transform_reduce / transform over MetricTaker
//    (src/PDFs/GooPdf.cu:45-78, 112-173; src/PDFs/MetricTaker.cu:17-44).
//  * k_reduce_bins: the midpoint-grid integral of one function
//    (src/PDFs/GooPdf.cu:83-108, src/PDFs/MetricTaker.cu:48-96).
#include <hip/hip_runtime.h>

#include "gf_interp.h"

namespace {

// One workgroup: add the nparts partials in a fixed order (thread t takes
// t, t+256, ...; then the wave butterfly and the waves in order), write
// {sum, residual correction, error word} to *result (host-mapped memory),
// clear the device error word, then stamp seq.
__global__ __launch_bounds__(GF_BLOCK) void k_finish(const Partial *partials, int nparts, GfResult *result,
                                                     int32_t *err, uint32_t seq) {
    double ts = 0.0, tc = 0.0;
    for(int i = threadIdx.x; i < nparts; i += GF_BLOCK)
        gfd::kb_merge(ts, tc, partials[i].s, partials[i].c);
    block_reduce(ts, tc);
    if(threadIdx.x == 0) {
        const int32_t e = *err;
        result->sum     = gfd::kb_total(ts, tc);
        result->comp    = tc;
        result->err     = e;
        if(e)
            *err = 0;
        __threadfence_system();
        __hip_atomic_store(&result->seq, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

__global__ __launch_bounds__(256) void k_fuse_init(unsigned long long *slots) {
    for(int i = blockIdx.x * blockDim.x + threadIdx.x; i < 2 * GF_MAX_PARTIALS; i += gridDim.x * blockDim.x)
        slots[i] = GF_SLOT_EMPTY;
}

// ------------------------------------------------------------- event kernels

template <int EPT, bool INL, int FEAT>
__global__ __launch_bounds__(GF_BLOCK) void k_reduce_metric(GfProgArgs A, GfInline I, int metric, Partial *partials) {
    const double *__restrict__ P  = INL ? I.p : A.params;
    const double *__restrict__ Nm = INL ? I.n : A.norms;
    const int64_t n    = A.nevents;
    const int64_t tile = (int64_t)GF_BLOCK * EPT;
    const double norm  = Nm[1];
    const bool binned  = metric >= GF_METRIC_BINAVG_CODE;
    const bool nll     = metric == gfd::metric_nll;
    double s = nll ? 1.0 : 0.0, c = 0.0;  // the NLL as a product: (mantissa, exponent)
    for(int64_t base = (int64_t)blockIdx.x * tile; base < n; base += (int64_t)gridDim.x * tile) {
        ColSrc<EPT> src;
        src.cols = A.cols;
        int64_t row[EPT];
        bool valid[EPT];
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            int64_t e  = base + (int64_t)j * GF_BLOCK + threadIdx.x;
            valid[j]   = e < n;
            row[j]     = valid[j] ? e : n - 1;
            src.idx[j] = row[j];
        }
        double T[EPT];
        run<EPT, FEAT>(A, P, Nm, 0, src, row, valid, T);
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            if(nll) {
                if(valid[j])
                    gfd::nll_add(s, c, T[j], norm);
                continue;
            }
            double e0 = 0.0, e1 = 0.0;
            if(binned) {
                e0 = A.cols[A.nobs - 2][row[j]];
                e1 = A.cols[A.nobs - 1][row[j]];
            }
            double v = gfd::metric(metric, T[j], e0, e1, norm, A.total_events);
            if(valid[j])
                gfd::kb_add(s, c, v);
        }
    }
    if(nll)
        s = gfd::nll_total(s, c), c = 0.0;
    store_partial(s, c, partials);
}

// ------------------------------------------- a time-dependent node at the root

// The reduction of a lone Amp3Body_TD -- [TDDP, MULTI_POLY, TDDP_END, END] -- with run()'s
// arithmetic (device_Tddp, src/PDFs/physics/Amp3Body_TD.cu:41-257), one event per lane.
// Bound by reading the waves (2 x 16 bytes per resonance and event) as long as the
// decay-time terms, some thousand FP64 operations which need no wave, run while they
// arrive: the first 2 x TD_CHUNK resonances are loaded before the terms, the following
// ones each as soon as a chunk is used up.  That takes 168 registers, three waves on a
// SIMD; in 128, for four, a dozen values per event spill and the sweep is slower (216 us).
// 1e6 events, 16 resonances, three Gaussians: 194 us in the interpreter with the library's
// exp and erfc, 160 with these terms there, 129 here (4.2 TB/s), on grids of three
// workgroups a CU (134 on four).
constexpr int TD_CHUNK = 4;
struct TdChunk {
    double2 a[TD_CHUNK], b[TD_CHUNK];
    // past the last resonance: the last one's again, not used
    __device__ __forceinline__ void load(const GfDalitzSlot &dz, int i0, int nres, int64_t e) {
        if(i0 >= nres)
            return;
#pragma unroll
        for(int u = 0; u < TD_CHUNK; ++u) {
            const int64_t o = (int64_t)(i0 + u < nres ? i0 + u : nres - 1) * dz.ncache + e;
            a[u]            = dz.wave[o];
            b[u]            = dz.wave_b[o];
        }
    }
    __device__ __forceinline__ void add(const GF_CONST double *__restrict__ C, int i0, int nres, double2 &sa,
                                        double2 &sb) const {
#pragma unroll
        for(int u = 0; u < TD_CHUNK; ++u)
            if(i0 + u < nres) {
                const double cr = C[2 * (i0 + u)], ci = C[2 * (i0 + u) + 1];
                gfd::cmac(sa.x, sa.y, cr, ci, a[u]);
                gfd::cmac(sb.x, sb.y, cr, ci, b[u]);
            }
    }
};

// What every event needs and no event changes, in LDS: held in registers across the loop
// (the compiler moves all of it in front) it would cost 40 vector registers of 128.
struct TdShared {
    double f[3], b[3], s[3], sb;
    GfDecay decay;
    __device__ __forceinline__ double selbias() const { return sb; }
    __device__ __forceinline__ void get(int k, double &fk, double &bk, double &sk) const {
        fk = f[k];
        bk = b[k];
        sk = s[k];
    }
};

template <bool INL, bool GAUSS>
__global__ __launch_bounds__(GF_BLOCK, 3) void k_td_reduce(GfProgArgs A, GfInline I, int metric, Partial *partials) {
    const GF_CONST double *__restrict__ P  = gfd::as_const(INL ? I.p : A.params);
    const GF_CONST double *__restrict__ Nm = gfd::as_const(INL ? I.n : A.norms);
    const GfIns td        = gfd::as_const(A.ins)[0];
    const GfIns eff       = gfd::as_const(A.ins)[1];
    const GfDalitzSlot dz = gfd::as_const(A.dz)[td.x];
    const auto cols       = gfd::as_const(A.cols);
    const GF_CONST double *__restrict__ C = P + td.p + 5;
    const GF_CONST double *__restrict__ R = P + dz.res_p;
    const int nres     = td.a;
    const int64_t n    = A.nevents;
    const double norm  = Nm[1];
    const bool nll     = metric == gfd::metric_nll;
    const double xfix = 0.0039, yfix = 0.0065, taufix = 0.4101;
    __shared__ TdShared sh;
    if(threadIdx.x == 0) {
        if(GAUSS)
            for(int k = 0; k < 3; ++k)
                gfd::GaussParams{R}.get(k, sh.f[k], sh.b[k], sh.s[k]);
        sh.sb    = GAUSS ? R[8] : 0.0;
        sh.decay = A.decay;
    }
    __syncthreads();
    double s = nll ? 1.0 : 0.0, c = 0.0;  // the NLL as a product: (mantissa, exponent)
    for(int64_t base = (int64_t)blockIdx.x * GF_BLOCK; base < n; base += (int64_t)gridDim.x * GF_BLOCK) {
        const int64_t row = base + threadIdx.x < n ? base + threadIdx.x : n - 1;
        const bool valid  = base + threadIdx.x < n;
        const double m12 = cols[dz.col_m12][row], m13 = cols[dz.col_m13][row];
        const double t = cols[dz.col_time][row], sg = cols[dz.col_sigma][row];
        const int tag      = dz.col_tag >= 0 ? (int)cols[dz.col_tag][row] : 0;
        const double mis   = dz.col_mis >= 0 ? cols[dz.col_mis][row] : 0.0;
        asm volatile("" ::: "memory");  // sh is read in each pass
        const GfDecay &D   = sh.decay;
        const bool inside  = gfd::in_dalitz(m12, m13, D.motherMass, D.daug1Mass, D.daug2Mass, D.daug3Mass);
        int64_t e          = A.identity_num ? row : (int64_t)floor(0.5 + cols[dz.col_num][row]);
        if(e < 0 || e >= dz.ncache) {
            if(inside && valid)
                atomicOr(A.err, 1);
            e = 0;
        }
        TdChunk w0, w1;
        w0.load(dz, 0, nres, e);
        w1.load(dz, TD_CHUNK, nres, e);
        const double tau = P[td.p], x0 = P[td.p + 1], y0 = P[td.p + 2], dx = P[td.p + 3], dy = P[td.p + 4];
        const double x = tag == 1 ? x0 + dx : (tag == -1 ? x0 - dx : x0);
        const double y = tag == 1 ? y0 + dy : (tag == -1 ? y0 - dy : y0);
        gfd::TimeTerms Pt{}, Pf{};
        if constexpr(GAUSS) {
            Pt = gfd::threegauss_terms(sh, tau, t, x, y, sg);
            if(mis > 0)
                Pf = gfd::threegauss_terms(sh, taufix, t, xfix, yfix, sg);
        }
        double2 sa = make_double2(0.0, 0.0), sb = make_double2(0.0, 0.0);
        for(int i0 = 0; i0 < nres; i0 += 2 * TD_CHUNK) {
            w0.add(C, i0, nres, sa, sb);
            w0.load(dz, i0 + 2 * TD_CHUNK, nres, e);
            w1.add(C, i0 + TD_CHUNK, nres, sa, sb);
            w1.load(dz, i0 + 3 * TD_CHUNK, nres, e);
        }
        const double nA = sa.x * sa.x + sa.y * sa.y;
        const double nB = sb.x * sb.x + sb.y * sb.y;
        const double t1 = nA + nB, t2 = nA - nB;
        const double abr = sa.x * sb.x + sa.y * sb.y;  // A conj(B)
        const double abi = sa.y * sb.x - sa.x * sb.y;
        double ret;
        if constexpr(GAUSS)
            ret = gfd::threegauss_rate(Pt, t1, t2, abr, abi);
        else
            ret = gfd::truth_resolution(t1, t2, abr, abi, tau, t, x, y);
        if(mis > 0) {  // A <-> B with fixed lifetime and mixing (Amp3Body_TD.cu:226-248)
            ret *= (1 - 2 * mis);
            if constexpr(GAUSS) {
                ret += mis * gfd::threegauss_rate(Pf, t1, -t2, abr, -abi);
                ret += mis * gfd::threegauss_rate(Pf, t1, t2, abr, abi);
            } else {
                ret += mis * gfd::truth_resolution(t1, -t2, abr, -abi, taufix, t, xfix, yfix);
                ret += mis * gfd::truth_resolution(t1, t2, abr, abi, taufix, t, xfix, yfix);
            }
        }
        const double v = inside ? ret * multipoly_at(eff, A, P, row) : 0.0;
        if(!valid)
            continue;
        if(nll)
            gfd::nll_add(s, c, v, norm);
        else
            gfd::kb_add(s, c, gfd::metric(metric, v, 0.0, 0.0, norm, A.total_events));
    }
    if(nll)
        s = gfd::nll_total(s, c), c = 0.0;
    store_partial(s, c, partials);
}

// ------------------------------------------------------------ flat trees

// The event columns of a flat program (at most GF_FLAT_COLS), loaded for the whole
// tile before any of them is used: a lane has every load of the tile in flight at
// once instead of waiting for one column per leaf.
template <int EPT>
struct FlatSrc {
    double v[EPT][GF_FLAT_COLS];
    __device__ __forceinline__ double get(int a, int j) const {
        switch(a) {
        case 0: return v[j][0];
        case 1: return v[j][1];
        case 2: return v[j][2];
        default: return v[j][3];
        }
    }
};

// A leaf of a flat program into T: the arithmetic of run()'s leaf cases.
template <int EPT>
__device__ __forceinline__ void flat_leaf(const GfIns &in, const GF_CONST double *__restrict__ P,
                                          const FlatSrc<EPT> &src, double (&T)[EPT]) {
    switch(in.op) {
    case GI_GAUSS: {
        const double m = P[in.p], sg = P[in.p + 1];
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            T[j] = gfd::gaussian(src.get(in.a, j), m, sg);
    } break;
    case GI_EXP: {
        const double al = P[in.p];
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            T[j] = exp(al * src.get(in.a, j));
    } break;
    case GI_EXP_OFF: {
        const double x0 = P[in.p], al = P[in.p + 1];
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            double x = src.get(in.a, j);
            x -= x0;
            T[j] = exp(al * x);
        }
    } break;
    default: {  // GI_EXPGAUS
        const double m = P[in.p], sg = P[in.p + 1], al = P[in.p + 2];
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            T[j] = gfd::expgaus(src.get(in.a, j), m, sg, al);
    } break;
    }
}

// A flat program over the events in src: run()'s arithmetic with one accumulator, the caller's
// (as a local of this function it costs k_reduce_flat<4> 14 registers and its fourth wave, or
// held to four waves a fourteenth of its time: 30.5 us against 28.5 for a sum of two over 4e6
// events).
template <int EPT>
__device__ __forceinline__ void flat_run(const GF_CONST GfIns *__restrict__ prog, const GF_CONST double *__restrict__ P,
                                         const GF_CONST double *__restrict__ Nm, const FlatSrc<EPT> &src,
                                         double (&T)[EPT], double (&acc)[EPT]) {
#pragma unroll
    for(int j = 0; j < EPT; ++j)
        T[j] = acc[j] = 0.0;
    for(int pc = 0;; ++pc) {
        const GfIns in = prog[pc];
        if(in.op == GI_END)
            break;
        if(in.op < GI_LVL) {
            flat_leaf<EPT>(in, P, src, T);
            continue;
        }
        switch((in.op - GI_LVL) >> 2) {
        case GK_PUSH0:
#pragma unroll
            for(int j = 0; j < EPT; ++j)
                acc[j] = 0.0;
            break;
        case GK_PUSH1:
#pragma unroll
            for(int j = 0; j < EPT; ++j)
                acc[j] = 1.0;
            break;
        case GK_ADD_ACC: {
            const double w = P[in.p], nm = Nm[in.n];
#pragma unroll
            for(int j = 0; j < EPT; ++j)
                acc[j] += w * T[j] * nm;
        } break;
        case GK_ADD_LAST: {
            double tw = 0;
            for(int i = 0; i < in.k; ++i)
                tw += P[in.p + i];
            const double nm = Nm[in.n];
#pragma unroll
            for(int j = 0; j < EPT; ++j)
                acc[j] += (1 - tw) * T[j] * nm;
        } break;
        case GK_ADDEXT_END: {
            double tw = 0;
            for(int i = 0; i < in.k; ++i)
                tw += P[in.p + i];
#pragma unroll
            for(int j = 0; j < EPT; ++j)
                T[j] = acc[j] / tw;
        } break;
        case GK_PROD_ACC: {
            const double nm = Nm[in.n];
#pragma unroll
            for(int j = 0; j < EPT; ++j) {
                double cur = T[j] * nm;
                acc[j] *= cur;
            }
        } break;
        default:  // GK_POP
#pragma unroll
            for(int j = 0; j < EPT; ++j)
                T[j] = acc[j];
            break;
        }
    }
}

// The reduction of a flat program -- one leaf, or one AddPdf / ProdPdf level over
// Gaussian, Exp, Exp-with-offset and ExpGaus leaves, reading columns 0 .. ncols-1
// (ncols <= GF_FLAT_COLS) -- with run()'s arithmetic in the same order (the same
// bits as k_reduce_metric) but one accumulator instead of a stack of levels, no
// Dalitz or polynomial cases, and the tile's columns loaded up front.
template <int EPT, bool INL>
__global__ __launch_bounds__(GF_BLOCK) void k_reduce_flat(GfProgArgs A, GfInline I, int metric, int ncols,
                                                         Partial *partials) {
    const GF_CONST double *__restrict__ P    = gfd::as_const(INL ? I.p : A.params);
    const GF_CONST double *__restrict__ Nm   = gfd::as_const(INL ? I.n : A.norms);
    const GF_CONST GfIns *__restrict__ prog  = gfd::as_const(A.ins);
    const auto cols                          = gfd::as_const(A.cols);
    const int64_t n    = A.nevents;
    const int64_t tile = (int64_t)GF_BLOCK * EPT;
    const double norm  = Nm[1];
    const bool nll     = metric == gfd::metric_nll;
    double s = nll ? 1.0 : 0.0, c = 0.0;  // the NLL as a product: (mantissa, exponent)
    FlatSrc<EPT> src;
#pragma unroll
    for(int j = 0; j < EPT; ++j)
#pragma unroll
        for(int k = 0; k < GF_FLAT_COLS; ++k)
            src.v[j][k] = 0.0;
    for(int64_t base = (int64_t)blockIdx.x * tile; base < n; base += (int64_t)gridDim.x * tile) {
        int64_t row[EPT];
        bool valid[EPT];
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            const int64_t e = base + (int64_t)j * GF_BLOCK + threadIdx.x;
            valid[j]        = e < n;
            row[j]          = valid[j] ? e : n - 1;
        }
#pragma unroll
        for(int k = 0; k < GF_FLAT_COLS; ++k)
            if(k < ncols) {
                const double *__restrict__ col = cols[k];
#pragma unroll
                for(int j = 0; j < EPT; ++j)
                    src.v[j][k] = col[row[j]];
            }
        double T[EPT], acc[EPT];
        flat_run<EPT>(prog, P, Nm, src, T, acc);
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            if(nll) {
                if(valid[j])
                    gfd::nll_add(s, c, T[j], norm);
                continue;
            }
            const double v = gfd::metric(metric, T[j], 0.0, 0.0, norm, A.total_events);
            if(valid[j])
                gfd::kb_add(s, c, v);
        }
    }
    if(nll)
        s = gfd::nll_total(s, c), c = 0.0;
    if(A.fuse_slots)
        finish_in_kernel(s, c, A);
    else
        store_partial(s, c, partials);
}

// The NLL of one leaf or of a product of leaves on a large set.  Such a sweep is bound by FP64
// issue in k_reduce_flat's form (257 operations an event for a Gaussian, an exponential and
// an ExpGaus, which are 24 bytes: 112 us for 1e7 events); here the leaves' exponents are
// added and not exponentiated, an ExpGaus leaves its erfcx, and a tile's exponents and factors
// meet in one compensated sum and one product: 70 us (3.4 TB/s).  125 registers, four waves on
// a SIMD; loading the next tile ahead takes a wave's place (155 registers: 81 us), two
// events a lane with the next two ahead also 81.  Taken from 2^20 events on, where k_reduce_flat
// goes to four events per lane: 16 us against 19 there, with the first tile's columns requested
// before the plan is formed.
//
// An event takes this way if no partial product of the reference's form can leave the normal
// range: its leaves' negative exponents add up to more than -616, the positive ones to less than
// 600, an ExpGaus' u < 24 (erfc above 1e-253, its exponential below e^577), the norms (positive)
// within 2^+-60, so each within 2^+-120 (the caller's part: prod_norms).  It adds nothing if one
// of its leaves is certain to round to 0 (an exponent below -750, an ExpGaus' u > 28): the
// product is then 0, or NaN if another leaf is infinite.  The loop tests less: the exponents'
// sum above -520, each Exp's below 80 / their number and each ExpGaus' below 1.  Any other event
// is noted and evaluated after the loop as k_reduce_flat does, on full waves.  A wave that meets
// more than GF_PROD_MISSES of them in a tile, or has noted GF_PROD_NOTES, evaluates this tile and
// its remaining ones so.  What is left of k_reduce_flat's speed on samples that meet these bounds, at
// 1e7 events: 72 us where any share of the events is certain to be 0, 70 with decay times to 330
// widths of the resolution, 137 (k_reduce_flat 115) where a fifth of all events lies between; at 2^20
// events 16, 16 and 27 (19).  (Giving up a whole tile for one event, and bounding u from below:
// 239, 175 and 241; 37, 35 and 37.)
struct ProdPlan {
    int ngauss, nexp, nexpgaus;  // leaves by kind, Gaussians first, then exponentials
    double K, rise;                     // the event-independent factor, the bound of an Exp's exponent
    int col[GF_PROD_LEAVES];
    double p[GF_PROD_LEAVES][5];        // mean, width^2, 1 / width^2; offset, alpha; see prod_plan
};
#define GF_PROD_MISSES 96
#define GF_PROD_NOTES 1024

// By the lanes of one wave, an instruction each (a product's program has at most 2 x
// GF_PROD_LEAVES + 3 of them): one lane alone took 3 us of its dependent loads and divisions.
__device__ __forceinline__ void prod_plan(ProdPlan &S, const GF_CONST GfIns *__restrict__ prog, int nins,
                                          const GF_CONST double *__restrict__ P,
                                          const GF_CONST double *__restrict__ Nm) {
    static_assert(2 * GF_PROD_LEAVES + 3 <= 64, "an instruction per lane");
    const int lane = threadIdx.x;
    GfIns in{};
    in.op = GI_END;
    if(lane < nins)
        in = prog[lane];
    const bool leaf = in.op != GI_END && in.op < GI_LVL;
    const int kind  = in.op == GI_GAUSS ? 0 : in.op == GI_EXPGAUS ? 2 : 1;
    int first = 0, count[3];
    double K = lane == 0 ? Nm[1] : 1.0;
    for(int k = 0; k < 3; ++k) {
        const unsigned long long m = __ballot(leaf && kind == k);
        count[k]                   = __popcll(m);
        if(leaf && kind == k) {
            const int at = first + __popcll(m & ((1ull << lane) - 1ull));
            double *q    = S.p[at];
            S.col[at]    = in.a;
            if(k == 0) {
                const double v = P[in.p + 1] * P[in.p + 1];
                q[0] = P[in.p];
                q[1] = v;
                q[2] = 1 / v;
            } else if(k == 1) {
                q[0] = in.op == GI_EXP_OFF ? P[in.p] : 0.0;
                q[1] = in.op == GI_EXP_OFF ? P[in.p + 1] : P[in.p];
            } else {  // expgaus(): exp(q3 (q4 - 2 x)) erfc((q0 - x) / q1)
                const double m = P[in.p], sg = P[in.p + 1], al = P[in.p + 2], w = sg * 1.4142135623;
                q[0] = m + al * sg * sg;
                q[1] = w;
                q[2] = 1 / w;
                q[3] = 0.5 * al;
                q[4] = 2 * m + al * sg * sg;
                K *= q[3];
            }
        }
        first += count[k];
    }
    if(in.op >= GI_LVL && (in.op - GI_LVL) >> 2 == GK_PROD_ACC)
        K = Nm[in.n];
    for(int off = 32; off > 0; off >>= 1)
        K *= __shfl_xor(K, off, 64);
    if(lane == 0) {
        S.ngauss   = count[0];
        S.nexp     = count[1];
        S.nexpgaus = count[2];
        S.K        = K;
        S.rise     = 80.0 / count[1];
    }
}

template <int EPT, bool INL>
__global__ __launch_bounds__(GF_BLOCK, 4) void k_reduce_prod(GfProgArgs A, GfInline I, int ncols, Partial *partials) {
    const GF_CONST double *__restrict__ P   = gfd::as_const(INL ? I.p : A.params);
    const GF_CONST double *__restrict__ Nm  = gfd::as_const(INL ? I.n : A.norms);
    const GF_CONST GfIns *__restrict__ prog = gfd::as_const(A.ins);
    const auto cols                         = gfd::as_const(A.cols);
    __shared__ ProdPlan S;
    __shared__ unsigned note[GF_BLOCK / 64][GF_PROD_NOTES];  // 64 (pass EPT + event of the lane) + lane
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t n    = A.nevents;
    const int64_t tile = (int64_t)GF_BLOCK * EPT;
    const double norm  = Nm[1];
    double s = 1.0, c = 0.0, es = 0.0, ec = 0.0;  // the factors' product, the exponents' sum
    FlatSrc<EPT> src;
#pragma unroll
    for(int j = 0; j < EPT; ++j)
#pragma unroll
        for(int k = 0; k < GF_FLAT_COLS; ++k)
            src.v[j][k] = 0.0;
    const auto load = [&](int64_t base, bool full) {
#pragma unroll
        for(int k = 0; k < GF_FLAT_COLS; ++k)
            if(k < ncols) {
                const double *__restrict__ col = cols[k] + base;
#pragma unroll
                for(int j = 0; j < EPT; ++j) {
                    const int o = j * GF_BLOCK + threadIdx.x;
                    src.v[j][k] = col[full || base + o < n ? o : n - 1 - base];
                }
            }
    };
    const int64_t base0 = (int64_t)blockIdx.x * tile, stride = (int64_t)gridDim.x * tile;
    const int npass     = base0 < n ? (int)((n - base0 + stride - 1) / stride) : 0;
    if(npass)
        load(base0, base0 + tile <= n);
    if(wave == 0)
        prod_plan(S, prog, A.flat_prod, P, Nm);
    __syncthreads();
    const int ng = __builtin_amdgcn_readfirstlane(S.ngauss), ne = ng + __builtin_amdgcn_readfirstlane(S.nexp);
    const int nl = ne + __builtin_amdgcn_readfirstlane(S.nexpgaus);
    int pass = 0, notes = 0;
    while(pass < npass) {
        const int64_t base = base0 + pass * stride;
        const bool full    = base + tile <= n;
        asm volatile("" ::: "memory");  // the plan is read where it is used
        double E[EPT], G[EPT];  // exponents, factors
        const double rise = S.rise;
        bool ok           = full;
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            E[j] = 0.0;
            G[j] = S.K;
        }
        for(int l = 0; l < ng; ++l) {
            const int a    = __builtin_amdgcn_readfirstlane(S.col[l]);
            const double m = S.p[l][0], v = S.p[l][1], r = S.p[l][2];
#pragma unroll
            for(int j = 0; j < EPT; ++j) {
                const double d = src.get(a, j) - m, t = -0.5 * d * d, q = t * r;
                E[j] += fma(fma(-q, v, t), r, q);  // t / v, rounded once
            }
        }
        for(int l = ng; l < ne; ++l) {
            const int a     = __builtin_amdgcn_readfirstlane(S.col[l]);
            const double x0 = S.p[l][0], al = S.p[l][1];
#pragma unroll
            for(int j = 0; j < EPT; ++j) {
                const double e = al * (src.get(a, j) - x0);
                ok             = ok && e < rise;
                E[j] += e;
            }
        }
        // exp(e) erfc(u): for u >= 0 exp(e - u^2) erfcx(u), else exp(e) (2 - exp(-u^2) erfcx(-u)),
        // for any u below 0: far below, the second term is 0
        for(int l = ne; l < nl; ++l) {
            const int a = __builtin_amdgcn_readfirstlane(S.col[l]);
            double u[EPT], y[EPT], t[EPT], g[EPT];
            {
                const double c0 = S.p[l][0], v = S.p[l][1], r = S.p[l][2], h = S.p[l][3], c2 = S.p[l][4];
#pragma unroll
                for(int j = 0; j < EPT; ++j) {
                    const double x = src.get(a, j), d = c0 - x, q = d * r;
                    double e       = h * (c2 - 2 * x);
                    u[j]           = fma(fma(-q, v, d), r, q);
                    e              = u[j] >= 0 ? fma(-u[j], u[j], e) : e;
                    ok             = ok && u[j] < 24.0 && e < 1.0;
                    E[j] += e;
                    t[j] = -u[j] * u[j];
                    y[j] = fabs(u[j]);
                }
            }
            gfd::exp_n(t, g);
#pragma unroll
            for(int j = 0; j < EPT; ++j)
                g[j] = u[j] >= 0 ? 0.0 : g[j];
            gfd::erfcx(y, t);
#pragma unroll
            for(int j = 0; j < EPT; ++j)
                G[j] *= u[j] >= 0 ? t[j] : fma(-g[j], t[j], 2.0);
        }
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            ok = ok && E[j] > -520.0;
        if(!__all(ok)) {  // which events, by the bounds themselves
            unsigned long long miss[EPT];
            int misses = 0;
#pragma unroll
            for(int j = 0; j < EPT; ++j) {
                bool in = E[j] == E[j], zero = !(base + j * GF_BLOCK + threadIdx.x < n);
                double fall = 0.0, rise = 0.0;  // the negative and the positive exponents' sums
                for(int l = 0; l < nl; ++l) {
                    const double x = src.get(__builtin_amdgcn_readfirstlane(S.col[l]), j);
                    double e;
                    if(l < ng) {
                        e    = -0.5 * (x - S.p[l][0]) * (x - S.p[l][0]) * S.p[l][2];
                        zero = zero || e < -750.0;
                    } else if(l < ne) {
                        e    = S.p[l][1] * (x - S.p[l][0]);
                        zero = zero || e < -750.0;
                    } else {
                        const double u = (S.p[l][0] - x) * S.p[l][2];
                        e              = S.p[l][3] * (S.p[l][4] - 2 * x);
                        zero           = zero || e < -750.0 || u > 28.0;
                        in             = in && u < 24.0;
                        e              = u >= 0 ? e - u * u : e;
                    }
                    fall += e < 0 ? e : 0.0;
                    rise += e < 0 ? 0.0 : e;
                }
                in      = in && fall > -616.0 && rise < 600.0;
                miss[j] = __ballot(!in && !zero);
                misses += __popcll(miss[j]);
                E[j] = in && !zero ? E[j] : 0.0;
                G[j] = in && !zero ? G[j] : 1.0;
            }
            if(misses > GF_PROD_MISSES || notes + misses > GF_PROD_NOTES)
                break;
#pragma unroll
            for(int j = 0; j < EPT; ++j) {
                if((miss[j] >> lane) & 1)
                    note[wave][notes + __popcll(miss[j] & ((1ull << lane) - 1ull))] = 64 * (pass * EPT + j) + lane;
                notes += __popcll(miss[j]);
            }
        }
        double e = 0.0, g = 1.0;
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            e += E[j];
            g *= G[j];
        }
        const double t = es + e, b = t - es;
        ec += (es - (t - b)) + (e - b);
        es = t;
        gfmath::nll_add(s, c, g);
        if(++pass < npass)
            load(base + stride, base + stride + tile <= n);
    }
    // The other form, after the loop: inside it the compiler holds the library functions' constants
    // in vector registers throughout (187 registers, two waves on a SIMD).  First the tiles from
    // the one on at which the wave stopped, which is still in registers, then the notes.
    for(bool kept = true; pass < npass; ++pass, kept = false) {
        const int64_t base = base0 + pass * stride;
        if(!kept)
            load(base, base + tile <= n);
        double T[EPT], acc[EPT];
        flat_run<EPT>(prog, P, Nm, src, T, acc);
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            if(base + j * GF_BLOCK + threadIdx.x < n)
                gfd::nll_add(s, c, T[j], norm);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for(int i = 0; i < notes; i += 64) {
        const unsigned id = note[wave][i + lane < notes ? i + lane : 0];
        const int64_t row = base0 + (int64_t)(id / (64 * EPT)) * stride + id / 64 % EPT * GF_BLOCK + 64 * wave + id % 64;
        FlatSrc<1> one;
        double T[1], acc[1];
#pragma unroll
        for(int k = 0; k < GF_FLAT_COLS; ++k)
            one.v[0][k] = k < ncols ? cols[k][row] : 0.0;
        flat_run<1>(prog, P, Nm, one, T, acc);
        if(i + lane < notes)
            gfd::nll_add(s, c, T[0], norm);
    }
    s = gfd::nll_total(s, c);
    c = 0.0;
    gfd::kb_add(s, c, -es);
    c -= ec;
    if(A.fuse_slots)
        finish_in_kernel(s, c, A);
    else
        store_partial(s, c, partials);
}

template <int EPT, bool INL, int FEAT>
__global__ __launch_bounds__(GF_BLOCK) void k_eval_metric(GfProgArgs A, GfInline I, int metric, double *out) {
    const double *__restrict__ P  = INL ? I.p : A.params;
    const double *__restrict__ Nm = INL ? I.n : A.norms;
    const int64_t n    = A.nevents;
    const int64_t tile = (int64_t)GF_BLOCK * EPT;
    const double norm  = Nm[1];
    const bool binned  = metric >= GF_METRIC_BINAVG_CODE;
    for(int64_t base = (int64_t)blockIdx.x * tile; base < n; base += (int64_t)gridDim.x * tile) {
        ColSrc<EPT> src;
        src.cols = A.cols;
        int64_t row[EPT];
        bool valid[EPT];
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            int64_t e  = base + (int64_t)j * GF_BLOCK + threadIdx.x;
            valid[j]   = e < n;
            row[j]     = valid[j] ? e : n - 1;
            src.idx[j] = row[j];
        }
        double T[EPT];
        run<EPT, FEAT>(A, P, Nm, 0, src, row, valid, T);
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            double e0 = 0.0, e1 = 0.0;
            if(binned) {
                e0 = A.cols[A.nobs - 2][row[j]];
                e1 = A.cols[A.nobs - 1][row[j]];
            }
            double v = gfd::metric(metric, T[j], e0, e1, norm, A.total_events);
            if(valid[j])
                out[row[j]] = v;
        }
    }
}

}  // namespace

// Grid description of k_reduce_bins (by value; indexed only by unrolled constants).
struct GfGrid {
    double lo[GF_MAX_OBS], hi[GF_MAX_OBS];
    int nb[GF_MAX_OBS];
    int slot[GF_MAX_OBS];
    int k;
};

namespace {

// The centres of global bin `bin` of grid G in every dimension (MetricTaker.cu:76-86:
// the first observable varies fastest, local bin = bin % n, then bin /= n).
__device__ __forceinline__ void grid_point(const GfGrid &G, int64_t bin, double (&x)[GF_MAX_OBS]) {
#pragma unroll
    for(int d = 0; d < GF_MAX_OBS; ++d) {
        x[d] = 0.0;
        if(d < G.k) {
            const int64_t localBin = bin % G.nb[d];
            x[d]                   = gfd::bin_centre(G.lo[d], G.hi[d], G.nb[d], localBin);
            bin /= G.nb[d];
        }
    }
}

// The synthetic event of grid bin `bin` in slot j of src: every observable slot 0,
// then each grid dimension's centre at its observable slot.
template <int EPT>
__device__ __forceinline__ void grid_event(const GfGrid &G, int64_t bin, RegSrc<EPT> &src, int j) {
    double x[GF_MAX_OBS];
    grid_point(G, bin, x);
#pragma unroll
    for(int o = 0; o < GF_MAX_OBS; ++o)
        src.v[j][o] = 0.0;
#pragma unroll
    for(int d = 0; d < GF_MAX_OBS; ++d)
        if(d < G.k)
            src.set(G.slot[d], j, x[d]);
}

template <int EPT>
__global__ __launch_bounds__(GF_BLOCK) void k_reduce_bins(GfProgArgs A, int pc0, GfGrid G, int64_t total,
                                                          Partial *partials) {
    const int64_t tile = (int64_t)GF_BLOCK * EPT;
    double s = 0.0, c = 0.0;
    for(int64_t base = (int64_t)blockIdx.x * tile; base < total; base += (int64_t)gridDim.x * tile) {
        RegSrc<EPT> src;
        int64_t row[EPT];
        bool valid[EPT];
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            int64_t b = base + (int64_t)j * GF_BLOCK + threadIdx.x;
            valid[j]  = b < total;
            row[j]    = valid[j] ? b : 0;
            grid_event(G, row[j], src, j);
        }
        double T[EPT];
        run<EPT>(A, A.params, A.norms, pc0, src, row, valid, T);
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            if(valid[j])
                gfd::kb_add(s, c, T[j]);
    }
    store_partial(s, c, partials);
}

// Per-bin raw values of the subprogram at pc0 over grid G: the transform that
// k_reduce_bins sums (same cells, same evaluation), written to out[bin].
template <int EPT>
__global__ __launch_bounds__(GF_BLOCK) void k_eval_bins(GfProgArgs A, int pc0, GfGrid G, int64_t total, double *out) {
    const int64_t tile = (int64_t)GF_BLOCK * EPT;
    for(int64_t base = (int64_t)blockIdx.x * tile; base < total; base += (int64_t)gridDim.x * tile) {
        RegSrc<EPT> src;
        int64_t row[EPT];
        bool valid[EPT];
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            int64_t b = base + (int64_t)j * GF_BLOCK + threadIdx.x;
            valid[j]  = b < total;
            row[j]    = valid[j] ? b : 0;
            grid_event(G, row[j], src, j);
        }
        double T[EPT];
        run<EPT>(A, A.params, A.norms, pc0, src, row, valid, T);
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            if(valid[j])
                out[row[j]] = T[j];
    }
}

// The cell centres of grid G: out[d * total + bin] = coordinate d of bin.
__global__ __launch_bounds__(256) void k_grid_cells(GfGrid G, int64_t total, double *out) {
    for(int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; b < total; b += (int64_t)gridDim.x * blockDim.x) {
        double x[GF_MAX_OBS];
        grid_point(G, b, x);
#pragma unroll
        for(int d = 0; d < GF_MAX_OBS; ++d)
            if(d < G.k)
                out[(int64_t)d * total + b] = x[d];
    }
}

// One v_mfma_f64_16x16x4f64 on given per-lane operands: out[4*lane + r] is
// D-register r of the lane.  Used to establish the operand/result lane layout.
__global__ __launch_bounds__(64) void k_mfma_probe(const double *__restrict__ a, const double *__restrict__ b,
                                                   double *out) {
    const int l    = threadIdx.x;
    gf_double4 acc = {0, 0, 0, 0};
    acc            = __builtin_amdgcn_mfma_f64_16x16x4f64(a[l], b[l], acc, 0, 0, 0);
    out[4 * l + 0] = acc[0];
    out[4 * l + 1] = acc[1];
    out[4 * l + 2] = acc[2];
    out[4 * l + 3] = acc[3];
}

// flag stays 1 only if floor(0.5 + col[i]) == i for every row (Amp3Body.cu:82-84).
__global__ __launch_bounds__(256) void k_identity_check(const double *__restrict__ col, int64_t n, int32_t *flag) {
    bool ok = true;
    for(int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        ok = ok && ((int64_t)floor(0.5 + col[i]) == i);
    if(!ok)
        atomicAnd(flag, 0);
}

}  // namespace

// ------------------------------------------------------------------ launchers

namespace gfk {

// Add the nblocks partials of the launch before it on stream s into *result.
// A non-null a.mark event is recorded between the two launches (timing).
int launch_finish(const GfProgArgs &a, Partial *partials, int nblocks, GfResult *result, hipStream_t s) {
    int rc = check(hipGetLastError());
    if(rc)
        return rc;
    if(a.mark && (rc = check(hipEventRecord((hipEvent_t)a.mark, s))))
        return rc;
    if(a.sweep_only || a.fuse_slots)  // a fused sweep has finished itself
        return 0;
    hipLaunchKernelGGL(k_finish, dim3(1), dim3(GF_BLOCK), 0, s, partials, nblocks, result, a.err, a.seq);
    return check(hipGetLastError());
}


int launch_reduce_metric(const GfProgArgs &a, const GfInline *inl, int metric, Partial *partials, GfResult *result,
                         int nblocks, void *stream) {
    hipStream_t s = (hipStream_t)stream;
    if(a.fuse_slots)  // the interpreter has no in-kernel finish
        return -1;
    // a lone time-dependent node: its own kernel; other trees that hold one: the kernels compiled
    // with the TD ops; programs without Dalitz nodes: the kernels compiled without them
    const dim3 g(nblocks), b(GF_BLOCK);
    const GfInline none{};
    if(a.lone_td && metric < GF_METRIC_BINAVG_CODE) {
        switch((a.lone_td - 1) * 2 + (inl ? 1 : 0)) {
        case 0: hipLaunchKernelGGL((k_td_reduce<false, false>), g, b, 0, s, a, none, metric, partials); break;
        case 1: hipLaunchKernelGGL((k_td_reduce<true, false>), g, b, 0, s, a, *inl, metric, partials); break;
        case 2: hipLaunchKernelGGL((k_td_reduce<false, true>), g, b, 0, s, a, none, metric, partials); break;
        default: hipLaunchKernelGGL((k_td_reduce<true, true>), g, b, 0, s, a, *inl, metric, partials); break;
        }
        return launch_finish(a, partials, nblocks, result, s);
    }
    switch(feature_level(a) * 2 + (inl ? 1 : 0)) {
    case 0: hipLaunchKernelGGL((k_reduce_metric<2, false, 0>), g, b, 0, s, a, none, metric, partials); break;
    case 1: hipLaunchKernelGGL((k_reduce_metric<2, true, 0>), g, b, 0, s, a, *inl, metric, partials); break;
    case 2: hipLaunchKernelGGL((k_reduce_metric<2, false, 1>), g, b, 0, s, a, none, metric, partials); break;
    case 3: hipLaunchKernelGGL((k_reduce_metric<2, true, 1>), g, b, 0, s, a, *inl, metric, partials); break;
    case 4: hipLaunchKernelGGL((k_reduce_metric<2, false, 2>), g, b, 0, s, a, none, metric, partials); break;
    default: hipLaunchKernelGGL((k_reduce_metric<2, true, 2>), g, b, 0, s, a, *inl, metric, partials); break;
    }
    return launch_finish(a, partials, nblocks, result, s);
}
int launch_reduce_flat(const GfProgArgs &a, const GfInline *inl, int metric, int ncols, int ept, Partial *partials,
                       GfResult *result, int nblocks, void *stream) {
    hipStream_t s = (hipStream_t)stream;
    if(ncols < 1 || ncols > GF_FLAT_COLS || metric >= GF_METRIC_BINAVG_CODE)
        return -1;
    const dim3 g(nblocks), b(GF_BLOCK);
    const GfInline none{};
    if(ept == 4 && a.flat_prod && metric == gfd::metric_nll) {
        if(inl)
            hipLaunchKernelGGL((k_reduce_prod<4, true>), g, b, 0, s, a, *inl, ncols, partials);
        else
            hipLaunchKernelGGL((k_reduce_prod<4, false>), g, b, 0, s, a, none, ncols, partials);
        return launch_finish(a, partials, nblocks, result, s);
    }
    switch((ept == 4 ? 2 : 0) + (inl ? 1 : 0)) {
    case 0: hipLaunchKernelGGL((k_reduce_flat<2, false>), g, b, 0, s, a, none, metric, ncols, partials); break;
    case 1: hipLaunchKernelGGL((k_reduce_flat<2, true>), g, b, 0, s, a, *inl, metric, ncols, partials); break;
    case 2: hipLaunchKernelGGL((k_reduce_flat<4, false>), g, b, 0, s, a, none, metric, ncols, partials); break;
    default: hipLaunchKernelGGL((k_reduce_flat<4, true>), g, b, 0, s, a, *inl, metric, ncols, partials); break;
    }
    return launch_finish(a, partials, nblocks, result, s);
}

int launch_eval_metric(const GfProgArgs &a, const GfInline *inl, int metric, double *out, int nblocks, void *stream) {
    hipStream_t s = (hipStream_t)stream;
    const dim3 g(nblocks), b(GF_BLOCK);
    const GfInline none{};
    switch(feature_level(a) * 2 + (inl ? 1 : 0)) {
    case 0: hipLaunchKernelGGL((k_eval_metric<2, false, 0>), g, b, 0, s, a, none, metric, out); break;
    case 1: hipLaunchKernelGGL((k_eval_metric<2, true, 0>), g, b, 0, s, a, *inl, metric, out); break;
    case 2: hipLaunchKernelGGL((k_eval_metric<2, false, 1>), g, b, 0, s, a, none, metric, out); break;
    case 3: hipLaunchKernelGGL((k_eval_metric<2, true, 1>), g, b, 0, s, a, *inl, metric, out); break;
    case 4: hipLaunchKernelGGL((k_eval_metric<2, false, 2>), g, b, 0, s, a, none, metric, out); break;
    default: hipLaunchKernelGGL((k_eval_metric<2, true, 2>), g, b, 0, s, a, *inl, metric, out); break;
    }
    return check(hipGetLastError());
}

static GfGrid make_grid(const double *ranges, const int *slots, int k) {
    GfGrid G;
    for(int d = 0; d < GF_MAX_OBS; ++d) {
        G.lo[d]   = d < k ? ranges[3 * d + 0] : 0.0;
        G.hi[d]   = d < k ? ranges[3 * d + 1] : 1.0;
        G.nb[d]   = d < k ? (int)floor(ranges[3 * d + 2] + 0.5) : 1;
        G.slot[d] = (d < k && slots) ? slots[d] : 0;
    }
    G.k = k;
    return G;
}

int launch_reduce_bins(const GfProgArgs &a, int pc0, const double *ranges, const int *slots, int k, int64_t total,
                       Partial *partials, GfResult *result, int nblocks, void *stream) {
    const GfGrid G = make_grid(ranges, slots, k);
    hipStream_t s  = (hipStream_t)stream;
    if(a.fuse_slots)  // no in-kernel finish here
        return -1;
    hipLaunchKernelGGL(k_reduce_bins<2>, dim3(nblocks), dim3(GF_BLOCK), 0, s, a, pc0, G, total, partials);
    return launch_finish(a, partials, nblocks, result, s);
}

int launch_eval_bins(const GfProgArgs &a, int pc0, const double *ranges, const int *slots, int k, int64_t total,
                     double *out, int nblocks, void *stream) {
    const GfGrid G = make_grid(ranges, slots, k);
    hipLaunchKernelGGL(k_eval_bins<2>, dim3(nblocks), dim3(GF_BLOCK), 0, (hipStream_t)stream, a, pc0, G, total, out);
    return check(hipGetLastError());
}


int launch_grid_cells(const double *ranges, int k, int64_t total, double *out, void *stream) {
    const GfGrid G = make_grid(ranges, nullptr, k);
    hipLaunchKernelGGL(k_grid_cells, dim3(cell_blocks(total)), dim3(256), 0, (hipStream_t)stream, G, total, out);
    return check(hipGetLastError());
}

int launch_fuse_init(unsigned long long *slots, void *stream) {
    hipLaunchKernelGGL(k_fuse_init, dim3(2 * GF_MAX_PARTIALS / 256), dim3(256), 0, (hipStream_t)stream, slots);
    return check(hipGetLastError());
}

int launch_identity_check(const double *col, int64_t n, int32_t *flag, void *stream) {
    int64_t nb = (n + 255) / 256;
    if(nb > 2048)
        nb = 2048;
    if(nb < 1)
        nb = 1;
    hipLaunchKernelGGL(k_identity_check, dim3((unsigned)nb), dim3(256), 0, (hipStream_t)stream, col, n, flag);
    return check(hipGetLastError());
}

int mfma_probe(const double *dev_a, const double *dev_b, double *dev_out, void *stream) {
    hipLaunchKernelGGL(k_mfma_probe, dim3(1), dim3(64), 0, (hipStream_t)stream, dev_a, dev_b, dev_out);
    return check(hipGetLastError());
}


}  // namespace gfk
