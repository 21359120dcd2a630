// gf_interp.h -- the per-event interpreter of a compiled PDF tree and the compensated
// reductions that the kernels of gf_kernels.hip, gf_coherent.hip and gf_lines.hip share.
#pragma once

#include <hip/hip_runtime.h>

#include "gf_device.h"
#include "gf_internal.h"

namespace {

using gfk::Partial;

// ------------------------------------------------------------ event sources

// Events read from the SoA columns in HBM.
template <int EPT>
struct ColSrc {
    const double *const *cols;
    int64_t idx[EPT];
    __device__ __forceinline__ double get(int a, int j) const { return gfd::as_const(cols)[a][idx[j]]; }
};

// Synthetic events held in registers (grid points); slot chosen by a
// wave-uniform switch so no register array is indexed dynamically.
template <int EPT>
struct RegSrc {
    double v[EPT][GF_MAX_OBS];
    __device__ __forceinline__ double get(int a, int j) const {
        switch(a) {
        case 0: return v[j][0];
        case 1: return v[j][1];
        case 2: return v[j][2];
        case 3: return v[j][3];
        case 4: return v[j][4];
        case 5: return v[j][5];
        case 6: return v[j][6];
        default: return v[j][7];
        }
    }
    __device__ __forceinline__ void set(int a, int j, double x) {
        switch(a) {
        case 0: v[j][0] = x; break;
        case 1: v[j][1] = x; break;
        case 2: v[j][2] = x; break;
        case 3: v[j][3] = x; break;
        case 4: v[j][4] = x; break;
        case 5: v[j][5] = x; break;
        case 6: v[j][6] = x; break;
        default: v[j][7] = x; break;
        }
    }
};

// Per-level accumulators of the combining nodes.  The few operations of a sum or product are a
// case per level, on that level's registers.  A Dalitz node is compiled once, its level's
// accumulator taken and put back by selects on the wave-uniform level (four copies of the
// time-dependent node had 960 scalar registers spilled to vector lanes); with selects for
// sums and products too, trees three levels deep took a seventh longer (1000 events 23.0 us,
// 20.4 as cases; an integral over 2e5 cells 30.4 and 25.8), with a switch on the level and one
// on the kind 21.7 and 27.4.  The time-dependent kernels keep the selects: the
// cases spill there (3e5 events 57.6 us, 59.4 as cases).
template <int EPT>
struct Acc {
    double v[4][EPT];
    __device__ __forceinline__ void take(int l, double (&a)[EPT]) const {
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            a[j] = l == 0 ? v[0][j] : l == 1 ? v[1][j] : l == 2 ? v[2][j] : v[3][j];
    }
    __device__ __forceinline__ void put(int l, const double (&a)[EPT]) {
#pragma unroll
        for(int k = 0; k < 4; ++k)
#pragma unroll
            for(int j = 0; j < EPT; ++j)
                v[k][j] = l == k ? a[j] : v[k][j];
    }
};

// ------------------------------------------------------------ interpreter

// One step of a sum or product on the accumulator a of its level.
template <int EPT>
__device__ __forceinline__ void sum_step(int kind, const GfIns &in, const GF_CONST double *__restrict__ P,
                                         const GF_CONST double *__restrict__ Nm, double (&a)[EPT], double (&T)[EPT]) {
    switch(kind) {
    case GK_PUSH0:
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            a[j] = 0.0;
        break;
    case GK_PUSH1:
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            a[j] = 1.0;
        break;
    case GK_ADD_ACC: {
        // device_AddPdfs / device_AddPdfsExt: ret += weight * curr * norm
        const double w = P[in.p], nm = Nm[in.n];
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            a[j] += w * T[j] * nm;
    } break;
    case GK_ADD_LAST: {
        // AddPdf.cu:43-48: ret += (1 - totalWeight) * last * normFactor
        double tw = 0;
        for(int i = 0; i < in.k; ++i)
            tw += P[in.p + i];
        const double nm = Nm[in.n];
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            a[j] += (1 - tw) * T[j] * nm;
    } break;
    case GK_ADDEXT_END: {
        // AddPdf.cu:76: ret /= totalWeight
        double tw = 0;
        for(int i = 0; i < in.k; ++i)
            tw += P[in.p + i];
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            T[j] = a[j] / tw;
    } break;
    case GK_PROD_ACC: {
        // ProdPdf.cu:19-23: curr *= norm; ret *= curr
        const double nm = Nm[in.n];
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            double cur = T[j] * nm;
            a[j] *= cur;
        }
    } break;
    case GK_POP:
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            T[j] = a[j];
        break;
    default: break;
    }
}

// One step of a Dalitz node (or of a sum or product, where no case of its own takes it) on the
// accumulator a of its level.  FEAT: the node kinds compiled
// in -- 0 none of the Dalitz nodes, 1 the time-integrated Dalitz node, 2 also the
// time-dependent one -- so that each kernel carries only the register budget of
// the programs it runs (a Dalitz node met by a kernel without it sets bit 1 of
// the error word instead of being skipped silently).
template <int EPT, int FEAT, class Src>
__device__ __forceinline__ void node_step(int kind, const GfIns &in, const GfProgArgs &A,
                                          const GF_CONST double *__restrict__ P,
                                          const GF_CONST double *__restrict__ Nm, const Src &src,
                                          const int64_t (&row)[EPT], const bool (&valid)[EPT], double (&a)[EPT],
                                          double (&T)[EPT]) {
    switch(kind) {
    case GK_DALITZ: {
        if constexpr(FEAT < 1) {
            atomicOr(A.err, 2);
            break;
        }
        // device_DalitzPlot, src/PDFs/physics/Amp3Body.cu:60-122
        const GfDalitzSlot dz = gfd::as_const(A.dz)[in.x];
        const GfDecay &D      = A.decay;
        int64_t en[EPT];
        bool inside[EPT];
        double re[EPT], im[EPT];
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            const double m12 = src.get(dz.col_m12, j), m13 = src.get(dz.col_m13, j);
            inside[j] = gfd::in_dalitz(m12, m13, D.motherMass, D.daug1Mass, D.daug2Mass, D.daug3Mass);
            int64_t e = A.identity_num ? row[j] : (int64_t)floor(0.5 + src.get(dz.col_num, j));
            if(e < 0 || e >= dz.ncache) {
                if(inside[j] && valid[j])
                    atomicOr(A.err, 1);
                e = 0;
            }
            en[j] = e;
            re[j] = 0.0;
            im[j] = 0.0;
        }
        // Loads of GF_DZ_CHUNK resonances are issued back to back before any of them is
        // consumed, so each wave keeps 8 * EPT 16-byte loads in flight; the terms are
        // added in gfd::coh_sum's order (groups of four resonances), as every other
        // coherent-sum kernel adds them.
        constexpr int GF_DZ_CHUNK = 8;
        for(int i0 = 0; i0 < in.a; i0 += GF_DZ_CHUNK) {
            double2 w[GF_DZ_CHUNK][EPT];
#pragma unroll
            for(int u = 0; u < GF_DZ_CHUNK; ++u) {
                const bool use              = i0 + u < in.a;
                const double2 *__restrict__ b = dz.wave + (int64_t)(use ? i0 + u : 0) * dz.ncache;
#pragma unroll
                for(int j = 0; j < EPT; ++j)
                    w[u][j] = use ? b[en[j]] : make_double2(0.0, 0.0);
            }
#pragma unroll
            for(int j = 0; j < EPT; ++j) {
                double2 wj[GF_DZ_CHUNK];
#pragma unroll
                for(int u = 0; u < GF_DZ_CHUNK; ++u)
                    wj[u] = w[u][j];
                gfd::coh_sum<GF_DZ_CHUNK>(
                    re[j], im[j],
                    [&](int u) { return make_double2(P[in.p + 2 * (i0 + u)], P[in.p + 2 * (i0 + u) + 1]); }, wj,
                    in.a - i0);
            }
        }
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            a[j] = inside[j] ? re[j] * re[j] + im[j] * im[j] : -1.0;
    } break;
    case GK_DALITZ_END:
        // Amp3Body.cu:118-121: ret *= eff (0 for events outside the Dalitz region)
#pragma unroll
        for(int j = 0; j < EPT; ++j)
            T[j] = (a[j] == -1.0) ? 0.0 : a[j] * T[j];
        break;
    case GK_TDDP:
        if constexpr(FEAT >= 2) {
            // device_Tddp, src/PDFs/physics/Amp3Body_TD.cu:41-257.  in.p: tau (then x, y,
            // dx, dy and the couplings); in.a: resonance count; in.x: node slot.
            const GfDalitzSlot dz = gfd::as_const(A.dz)[in.x];
            const GfDecay &D      = A.decay;
            int64_t en[EPT];
            double sar[EPT], sai[EPT], sbr[EPT], sbi[EPT];
#pragma unroll
            for(int j = 0; j < EPT; ++j) {
                const double m12 = src.get(dz.col_m12, j), m13 = src.get(dz.col_m13, j);
                const bool inside = gfd::in_dalitz(m12, m13, D.motherMass, D.daug1Mass, D.daug2Mass, D.daug3Mass);
                int64_t e = A.identity_num ? row[j] : (int64_t)floor(0.5 + src.get(dz.col_num, j));
                if(e < 0 || e >= dz.ncache) {
                    if(inside && valid[j])
                        atomicOr(A.err, 1);
                    e = 0;
                }
                en[j]  = e;
                sar[j] = sai[j] = sbr[j] = sbi[j] = 0.0;
            }
            // A += a_i * c_i, B += b_i * c_i (Amp3Body_TD.cu:91-110).  The A and B waves of
            // GF_TD_CHUNK resonances are loaded before any is consumed (2 x 4 x EPT 16-byte
            // loads in flight per lane); the sums still run over i = 0, 1, ... in order.
            constexpr int GF_TD_CHUNK = 4;
            for(int i0 = 0; i0 < in.a; i0 += GF_TD_CHUNK) {
                double2 wa[GF_TD_CHUNK][EPT], wb[GF_TD_CHUNK][EPT];
#pragma unroll
                for(int u = 0; u < GF_TD_CHUNK; ++u) {
                    const bool use = i0 + u < in.a;
                    const int64_t off = (int64_t)(use ? i0 + u : 0) * dz.ncache;
#pragma unroll
                    for(int j = 0; j < EPT; ++j) {
                        wa[u][j] = use ? dz.wave[off + en[j]] : make_double2(0.0, 0.0);
                        wb[u][j] = use ? dz.wave_b[off + en[j]] : make_double2(0.0, 0.0);
                    }
                }
#pragma unroll
                for(int u = 0; u < GF_TD_CHUNK; ++u) {
                    if(i0 + u < in.a) {
                        const double cr = P[in.p + 5 + 2 * (i0 + u)], ci = P[in.p + 6 + 2 * (i0 + u)];
#pragma unroll
                        for(int j = 0; j < EPT; ++j) {
                            gfd::cmac(sar[j], sai[j], cr, ci, wa[u][j]);
                            gfd::cmac(sbr[j], sbi[j], cr, ci, wb[u][j]);
                        }
                    }
                }
            }
            const double tau = P[in.p], x0 = P[in.p + 1], y0 = P[in.p + 2], dx = P[in.p + 3], dy = P[in.p + 4];
            const GF_CONST double *__restrict__ R = P + dz.res_p;
            // mistag terms: A <-> B with fixed lifetime and mixing (Amp3Body_TD.cu:226-248)
            const double xfix = 0.0039, yfix = 0.0065, taufix = 0.4101;
#pragma unroll
            for(int j = 0; j < EPT; ++j) {
                const int tag = dz.col_tag >= 0 ? (int)src.get(dz.col_tag, j) : 0;
                const double x = tag == 1 ? x0 + dx : (tag == -1 ? x0 - dx : x0);
                const double y = tag == 1 ? y0 + dy : (tag == -1 ? y0 - dy : y0);
                const double t = src.get(dz.col_time, j), sg = src.get(dz.col_sigma, j);
                const double nA = sar[j] * sar[j] + sai[j] * sai[j];
                const double nB = sbr[j] * sbr[j] + sbi[j] * sbi[j];
                const double t1 = nA + nB, t2 = nA - nB;
                const double abr = sar[j] * sbr[j] + sai[j] * sbi[j];  // A conj(B)
                const double abi = sai[j] * sbr[j] - sar[j] * sbi[j];
                double ret = gfd::time_resolution(dz.res_kind, R, t1, t2, abr, abi, tau, t, x, y, sg);
                const double mis = dz.col_mis >= 0 ? src.get(dz.col_mis, j) : 0.0;
                if(mis > 0) {
                    ret *= (1 - 2 * mis);
                    if(dz.res_kind == GT_THREEGAUSS) {
                        // both mistag calls take the same (taufix, t, xfix, yfix, sigma): their
                        // Gaussian terms are evaluated once and combined twice (same values)
                        const gfd::TimeTerms Pf = gfd::threegauss_terms(gfd::GaussParams{R}, taufix, t, xfix, yfix, sg);
                        ret += mis * gfd::threegauss_rate(Pf, t1, -t2, abr, -abi);
                        ret += mis * gfd::threegauss_rate(Pf, t1, t2, abr, abi);
                    } else {
                        ret += mis * gfd::truth_resolution(t1, -t2, abr, -abi, taufix, t, xfix, yfix);
                        ret += mis * gfd::truth_resolution(t1, t2, abr, abi, taufix, t, xfix, yfix);
                    }
                }
                a[j] = ret;
            }
        } else {
            atomicOr(A.err, 2);
        }
        break;
    case GK_TDDP_END:
        if constexpr(FEAT >= 2) {
            // Amp3Body_TD.cu:61-76, 253-255: ret *= eff inside, 0 outside
            const GfDalitzSlot dz = gfd::as_const(A.dz)[in.x];
            const GfDecay &D      = A.decay;
#pragma unroll
            for(int j = 0; j < EPT; ++j) {
                const bool inside = gfd::in_dalitz(src.get(dz.col_m12, j), src.get(dz.col_m13, j), D.motherMass,
                                                   D.daug1Mass, D.daug2Mass, D.daug3Mass);
                T[j] = inside ? a[j] * T[j] : 0.0;
            }
        } else {
            atomicOr(A.err, 2);
        }
        break;
    default:
        if constexpr(FEAT == 2)
            sum_step<EPT>(kind, in, P, Nm, a, T);
        break;
    }
}


// Run the compiled program from instruction pc0 for EPT events per lane; the
// value of the tree ends up in T.  row[] are the event rows (used as wave-cache
// index when the event-number column is the identity), valid[] masks tail lanes.
template <int EPT, int FEAT = 1, class Src>
__device__ __forceinline__ void run(const GfProgArgs &A, const double *__restrict__ P_, const double *__restrict__ Nm_,
                                    int pc0, const Src &src, const int64_t (&row)[EPT], const bool (&valid)[EPT],
                                    double (&T)[EPT]) {
    const GF_CONST double *__restrict__ P  = gfd::as_const(P_);
    const GF_CONST double *__restrict__ Nm = gfd::as_const(Nm_);
    const GF_CONST double *__restrict__ Cn = gfd::as_const(A.consts);
    const GF_CONST GfIns *__restrict__ prog = gfd::as_const(A.ins);
    Acc<EPT> acc;
#pragma unroll
    for(int j = 0; j < EPT; ++j)
        T[j] = acc.v[0][j] = acc.v[1][j] = acc.v[2][j] = acc.v[3][j] = 0.0;
    for(int pc = pc0;; ++pc) {
        const GfIns in = prog[pc];
        // the time-dependent kernels take every level's step by the default case
        switch(FEAT == 2 && in.op >= GI_LVL ? GF_LVL_OP(GK_DALITZ, 0) : in.op) {
        case GI_END: return;
        case GI_GAUSS: {
            const double m = P[in.p], s = P[in.p + 1];
#pragma unroll
            for(int j = 0; j < EPT; ++j)
                T[j] = gfd::gaussian(src.get(in.a, j), m, s);
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
        case GI_EXP_POLY: {
#pragma unroll
            for(int j = 0; j < EPT; ++j) {
                double x = src.get(in.a, j), e = 0;
                gfmath::Powers xi;
                for(int i = 0; i < in.k; ++i, xi.next(x))
                    e += xi.value() * P[in.p + i];
                T[j] = exp(e);
            }
        } break;
        case GI_EXP_POLY_OFF: {
#pragma unroll
            for(int j = 0; j < EPT; ++j) {
                double x = src.get(in.a, j), e = 0;
                x -= P[in.p];
                gfmath::Powers xi;
                for(int i = 1; i < in.k; ++i) {
                    xi.next(x);
                    e += xi.value() * P[in.p + i];
                }
                T[j] = exp(e);
            }
        } break;
        case GI_EXPGAUS: {
            const double m = P[in.p], s = P[in.p + 1], al = P[in.p + 2];
#pragma unroll
            for(int j = 0; j < EPT; ++j)
                T[j] = gfd::expgaus(src.get(in.a, j), m, s, al);
        } break;
        case GI_POLY:
        case GI_OFF_POLY: {
            // the powers from lowest on (a negative one apart); the two coefficients in
            // front of an offset polynomial's are no terms of it
            const int lowest = (int)Cn[in.c], i0 = in.op == GI_OFF_POLY ? 2 : 0;
#pragma unroll
            for(int j = 0; j < EPT; ++j) {
                const double x = src.get(in.a, j);
                double r       = 0;
                gfmath::Powers xi;
                if(lowest > 0)
                    xi.start(x, (unsigned)lowest);
                for(int i = i0; i < in.k; ++i) {
                    const int n = lowest + i - i0;
                    r += P[in.p + i] * (n < 0 ? gfmath::powi(x, n) : xi.value());
                    if(n >= 0)
                        xi.next(x);
                }
                T[j] = r;
            }
        } break;
        case GI_MULTI_POLY: {
            // device_MultiPolynomial, src/PDFs/basic/PolynomialPdf.cu:47-118
            const int nobs      = in.a;
            const int maxDegree = (int)Cn[in.c] + 1;
            int numBoxes        = 1;
            for(int i = 0; i < nobs; ++i)
                numBoxes *= maxDegree;
#pragma unroll
            for(int j = 0; j < EPT; ++j) {
                int coeff = nobs;
                double r  = P[in.p + coeff];
                coeff++;
                for(int i = 1; i < numBoxes; ++i) {
                    double term = 1;
                    int ci = i, sum = 0;
                    for(int o = 0; o < nobs; ++o) {
                        double x = src.get(gfd::as_const(A.obsid)[in.x + o], j);
                        x -= P[in.p + o];
                        int pw = ci % maxDegree;
                        ci /= maxDegree;
                        term *= gfmath::power(x, pw);
                        sum += pw;
                    }
                    if(sum >= maxDegree)
                        continue;
                    term *= P[in.p + coeff];
                    coeff++;
                    r += term;
                }
                T[j] = r;
            }
        } break;
#define GF_SUM_CASE(k)                                                     \
    case GF_LVL_OP(k, 0): sum_step<EPT>(k, in, P, Nm, acc.v[0], T); break; \
    case GF_LVL_OP(k, 1): sum_step<EPT>(k, in, P, Nm, acc.v[1], T); break; \
    case GF_LVL_OP(k, 2): sum_step<EPT>(k, in, P, Nm, acc.v[2], T); break; \
    case GF_LVL_OP(k, 3): sum_step<EPT>(k, in, P, Nm, acc.v[3], T); break;
            GF_SUM_CASE(GK_PUSH0)
            GF_SUM_CASE(GK_PUSH1)
            GF_SUM_CASE(GK_ADD_ACC)
            GF_SUM_CASE(GK_ADD_LAST)
            GF_SUM_CASE(GK_ADDEXT_END)
            GF_SUM_CASE(GK_PROD_ACC)
            GF_SUM_CASE(GK_POP)
#undef GF_SUM_CASE
        default:
            if(in.op >= (FEAT == 2 ? GI_LVL : GF_LVL_OP(GK_DALITZ, 0))) {
                double a[EPT];
                acc.take((in.op - GI_LVL) & 3, a);
                node_step<EPT, FEAT>((in.op - GI_LVL) >> 2, in, A, P, Nm, src, row, valid, a, T);
                acc.put((in.op - GI_LVL) & 3, a);
                break;
            }
            return;
        }
    }
}

// Multivariate polynomial of one event (device_MultiPolynomial,
// src/PDFs/basic/PolynomialPdf.cu:47-118), columns read at row e.
__device__ __forceinline__ double multipoly_at(const GfIns &in, const GfProgArgs &A,
                                               const GF_CONST double *__restrict__ P, int64_t e) {
    const int nobs      = in.a;
    const int maxDegree = (int)gfd::as_const(A.consts)[in.c] + 1;
    int numBoxes        = 1;
    for(int i = 0; i < nobs; ++i)
        numBoxes *= maxDegree;
    int coeff = nobs;
    double r  = P[in.p + coeff];
    coeff++;
    for(int i = 1; i < numBoxes; ++i) {
        double term = 1;
        int ci = i, sum = 0;
        for(int o = 0; o < nobs; ++o) {
            double x = gfd::as_const(A.cols)[gfd::as_const(A.obsid)[in.x + o]][e];
            x -= P[in.p + o];
            int pw = ci % maxDegree;
            ci /= maxDegree;
            term *= gfmath::power(x, pw);
            sum += pw;
        }
        if(sum >= maxDegree)
            continue;
        term *= P[in.p + coeff];
        coeff++;
        r += term;
    }
    return r;
}

// the four result registers of a lane of v_mfma_f64_16x16x4f64
typedef double gf_double4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------- reductions

// Reduce (s, c) over the block; the result is valid in thread 0.
__device__ __forceinline__ void block_reduce(double &s, double &c) {
    __shared__ double ls[GF_BLOCK / 64], lc[GF_BLOCK / 64];
#pragma unroll
    for(int off = 32; off > 0; off >>= 1) {
        double s2 = __shfl_xor(s, off, 64);
        double c2 = __shfl_xor(c, off, 64);
        gfd::kb_merge(s, c, s2, c2);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if(lane == 0) {
        ls[wave] = s;
        lc[wave] = c;
    }
    __syncthreads();
    if(threadIdx.x == 0) {
        s = ls[0];
        c = lc[0];
        for(int w = 1; w < (int)(blockDim.x >> 6); ++w)
            gfd::kb_merge(s, c, ls[w], lc[w]);
    }
    __syncthreads();
}

// Reduce (s, c) over the 16 lanes of a lane's group (lanes 16 g .. 16 g + 15 of its
// wave): the result is valid in every lane of the group.
__device__ __forceinline__ void group_reduce(double &s, double &c) {
#pragma unroll
    for(int off = 8; off > 0; off >>= 1) {
        double s2 = __shfl_xor(s, off, 64);
        double c2 = __shfl_xor(c, off, 64);
        gfd::kb_merge(s, c, s2, c2);
    }
}

// Reduce the block's (sum, residual) pair and store it as partial blockIdx.x.
// No fence and no atomic: on a multi-XCD device an agent-scope release per
// workgroup writes back the XCD's L2 each time, which costs more than the
// whole sweep over the events once there are thousands of workgroups.  The
// partials are added by k_finish, whose launch orders it after every store.
__device__ __forceinline__ void store_partial(double s, double c, Partial *partials) {
    block_reduce(s, c);
    if(threadIdx.x == 0) {
        partials[blockIdx.x].s = s;
        partials[blockIdx.x].c = c;
    }
}

// The in-kernel finish: k_finish's work done inside the sweep by its last
// workgroup (the highest index), with no second launch.  Every other workgroup
// stores its (sum, residual) pair into its slot with agent-scope atomic stores
// (coherent across the XCDs' L2 caches) and exits.  Workgroups are dispatched in
// index order on each XCD, so the last one starts after every workgroup it waits
// for has been placed and holds no resource they need.  It reads the slots with
// agent-scope atomic loads -- a thread's slots t, t+256, ... four at a time, all
// eight loads in flight together -- until none is GF_SLOT_EMPTY, adds them exactly
// as k_finish does (same order, same bits; its own pair taken from LDS), empties
// them for the next launch and writes the result block.  No workgroup runs a
// release fence: on this device an agent-scope release writes back the XCD's L2,
// once per workgroup.  The wait is bounded; a slot still empty after it sets
// GF_DEVERR_FINISH in the result's error word.
// finish_reduced: the same for a workgroup whose pair is reduced already (valid in
// thread 0); every thread of the workgroup calls it.
__device__ __forceinline__ void finish_reduced(double s, double c, const GfProgArgs &A) {
    constexpr uint32_t spin_limit = 1u << 18;
    constexpr int group           = 4;
    __shared__ double own_s, own_c;
    unsigned long long *slots = A.fuse_slots;
    const int nparts          = (int)gridDim.x;
    const int mine            = nparts - 1;
    if((int)blockIdx.x != mine) {
        if(threadIdx.x == 0) {
            __hip_atomic_store(slots + 2 * blockIdx.x, (unsigned long long)__double_as_longlong(s),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(slots + 2 * blockIdx.x + 1, (unsigned long long)__double_as_longlong(c),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return;
    }
    if(threadIdx.x == 0) {
        own_s = s;
        own_c = c;
    }
    __syncthreads();
    double ts = 0.0, tc = 0.0;
    int late  = 0;
    for(int i0 = threadIdx.x; i0 < nparts; i0 += group * GF_BLOCK) {
        unsigned long long vs[group], vc[group];
#pragma unroll
        for(int g = 0; g < group; ++g)
            vs[g] = vc[g] = GF_SLOT_EMPTY;
        for(uint32_t spin = 0;; ++spin) {
#pragma unroll
            for(int g = 0; g < group; ++g) {
                const int i = i0 + g * GF_BLOCK;
                if(i < mine && (vs[g] == GF_SLOT_EMPTY || vc[g] == GF_SLOT_EMPTY)) {
                    vs[g] = __hip_atomic_load(slots + 2 * i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    vc[g] = __hip_atomic_load(slots + 2 * i + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            bool done = true;
#pragma unroll
            for(int g = 0; g < group; ++g)
                if(i0 + g * GF_BLOCK < mine && (vs[g] == GF_SLOT_EMPTY || vc[g] == GF_SLOT_EMPTY))
                    done = false;
            if(done)
                break;
            if(spin == spin_limit) {
                late = 1;
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
#pragma unroll
        for(int g = 0; g < group; ++g) {
            const int i = i0 + g * GF_BLOCK;
            if(i < mine) {
                gfd::kb_merge(ts, tc, __longlong_as_double((long long)vs[g]), __longlong_as_double((long long)vc[g]));
                __hip_atomic_store(slots + 2 * i, GF_SLOT_EMPTY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(slots + 2 * i + 1, GF_SLOT_EMPTY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else if(i == mine) {
                gfd::kb_merge(ts, tc, own_s, own_c);
            }
        }
    }
    late = __syncthreads_or(late);
    block_reduce(ts, tc);
    if(threadIdx.x == 0) {
        GfResult *result = A.fuse_result;
        const int32_t e  = *A.err;  // written by earlier launches only
        result->sum      = gfd::kb_total(ts, tc);
        result->comp     = tc;
        result->err      = e | (late ? GF_DEVERR_FINISH : 0);
        if(e)
            *A.err = 0;
        __threadfence_system();
        __hip_atomic_store(&result->seq, A.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

__device__ __forceinline__ void finish_in_kernel(double s, double c, const GfProgArgs &A) {
    block_reduce(s, c);
    finish_reduced(s, c, A);
}

// Node kinds a program needs compiled in (FEAT of the interpreter kernels).
inline int feature_level(const GfProgArgs &a) { return a.td ? 2 : (a.has_dz ? 1 : 0); }

inline unsigned cell_blocks(int64_t total) {
    int64_t nb = (total + 255) / 256;
    return (unsigned)(nb > 8192 ? 8192 : (nb < 1 ? 1 : nb));
}

inline int check(hipError_t e) { return e == hipSuccess ? 0 : (int)e; }

}  // namespace
