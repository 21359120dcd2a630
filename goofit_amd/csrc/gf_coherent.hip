// gf_coherent.hip -- coherent-sum sweeps of a lone Amp3Body (single and multi-point, on
// the vector ALUs and on the FP64 matrix cores) and the toy batches, for gfx950
// (src/PDFs/GooPdf.cu:45-78, src/PDFs/physics/Amp3Body.cu:60-122).
#include <hip/hip_runtime.h>

#include "gf_interp.h"

namespace {

// ------------------------------------------------------ coherent-sum fast path

// |sum_i c_i W_i[e]|^2 * eff for a Dalitz node at the root of the tree.  All
// wave loads of an event are issued before any arithmetic (16 x 16 bytes per lane
// in flight); the rest is device_DalitzPlot's arithmetic, the coherent sum in
// gfd::coh_sum's grouped order (the matrix-core kernel's).
// ZERO_OUT (constant efficiency, cache filled from these events): the waves of an event
// outside the Dalitz region are all 0, so |A|^2 eff is the reference's 0 there without
// reading m12 and m13 (256 instead of 272 bytes per event).
template <bool WRITE, bool INL, bool CONST_EFF, bool ZERO_OUT = false>
__global__ __launch_bounds__(256) void k_dalitz_fast(GfProgArgs A, GfInline I, int metric, Partial *partials,
                                                     double *out) {
    const double *__restrict__ P  = INL ? I.p : A.params;
    const double *__restrict__ Nm = INL ? I.n : A.norms;
    const GfIns dzi       = A.ins[0];
    const GfIns effi      = A.ins[1];
    const GfDalitzSlot dz = A.dz[dzi.x];
    const GfDecay &D      = A.decay;
    const int nres        = dzi.a;
    const int64_t n       = A.nevents;
    const double norm     = Nm[1];
    const double *__restrict__ c12 = A.cols[dz.col_m12];
    const double *__restrict__ c13 = A.cols[dz.col_m13];
    const bool nll        = !WRITE && metric == gfd::metric_nll;
    // the events of the NLL grouped as k_coh_mx groups a set's (the multi-point sums of
    // these parameters run there): lanes 0-15 of a wave hold the products, below
    const bool grp        = nll && CONST_EFF && ZERO_OUT && A.coh_group;
    double s = nll ? 1.0 : 0.0, c = 0.0;  // the NLL as a product: (mantissa, exponent)
    for(int64_t base = (int64_t)blockIdx.x * blockDim.x; base < n; base += (int64_t)gridDim.x * blockDim.x) {
        const int64_t e0 = base + threadIdx.x;
        const bool valid = e0 < n;
        const int64_t e  = valid ? e0 : n - 1;
        double2 w[GF_MAX_RES];
#pragma unroll
        for(int i = 0; i < GF_MAX_RES; ++i)
            w[i] = (i < nres) ? dz.wave[(int64_t)i * dz.ncache + e] : make_double2(0.0, 0.0);
        const double m12 = ZERO_OUT ? 0.0 : c12[e];
        const double m13 = ZERO_OUT ? 0.0 : c13[e];
        double re = 0.0, im = 0.0;
        gfd::coh_sum<GF_MAX_RES>(
            re, im, [&](int i) { return make_double2(P[dzi.p + 2 * i], P[dzi.p + 2 * i + 1]); }, w, nres);
        const bool inside =
            ZERO_OUT || gfd::in_dalitz(m12, m13, D.motherMass, D.daug1Mass, D.daug2Mass, D.daug3Mass);
        // a degree-0 polynomial is its constant coefficient (numBoxes == 1)
        const double eff = CONST_EFF ? P[effi.p + effi.a] : multipoly_at(effi, A, gfd::as_const(P), e);
        const double T   = inside ? (re * re + im * im) * eff : 0.0;
        if(WRITE) {
            if(valid)
                out[e] = gfd::metric(metric, T, 0.0, 0.0, norm, A.total_events);
        } else if(grp) {
            // k_coh_mx's grouping: lane (0, j) takes events 16 t + j of the wave, in tile order
            const int64_t w0 = base + (threadIdx.x & ~63);
#pragma unroll
            for(int t = 0; t < 4; ++t) {
                const double v = t == 0 ? T : __shfl(T, 16 * t + (threadIdx.x & 15), 64);
                if((threadIdx.x & 63) < 16 && w0 + 16 * t + (threadIdx.x & 15) < n)
                    gfd::nll_add(s, c, v, norm);
            }
        } else if(nll) {
            if(valid)
                gfd::nll_add(s, c, T, norm);
        } else if(valid) {
            gfd::kb_add(s, c, gfd::metric(metric, T, 0.0, 0.0, norm, A.total_events));
        }
    }
    if(!WRITE && grp) {
        // as k_coh_mx reduces a set: the 16 lanes of the group, then the four waves in order
        __shared__ double gls[4], glc[4];
        double sv = (threadIdx.x & 63) < 16 ? gfd::nll_total(s, c) : 0.0, cv = 0.0;
        group_reduce(sv, cv);
        if((threadIdx.x & 63) == 0) {
            gls[threadIdx.x >> 6] = sv;
            glc[threadIdx.x >> 6] = cv;
        }
        __syncthreads();
        if(threadIdx.x == 0) {
            sv = gls[0];
            cv = glc[0];
            for(int wv = 1; wv < 4; ++wv)
                gfd::kb_merge(sv, cv, gls[wv], glc[wv]);
        }
        if(A.fuse_slots) {
            finish_reduced(sv, cv, A);
        } else if(threadIdx.x == 0) {
            partials[blockIdx.x].s = sv;
            partials[blockIdx.x].c = cv;
        }
    } else if(!WRITE) {
        if(nll)
            s = gfd::nll_total(s, c), c = 0.0;
        if(A.fuse_slots)
            finish_in_kernel(s, c, A);
        else
            store_partial(s, c, partials);
    }
}

// The coherent-sum metric sum of up to GF_MULTI_PTS parameter sets over the same
// events in one sweep: an event's waves are loaded once and every set's term is
// taken with the arithmetic, the event-to-lane assignment and the reduction
// order of k_dalitz_fast on the same grid, so each set's partials equal that
// kernel's for the same parameters bit for bit.  params / norms: npts
// consecutive copies of the flattened arrays (np and nn doubles each).
// partials: [npts][gridDim.x].
// The parameter sets of one multi-set sweep as the event loop reads them: the
// couplings of set p at c[p][i] (zero for resonances i >= nres, so that a resonance
// loop unrolled to NR >= nres adds exact zeros past nres), each set's constant
// efficiency and normalisation.  Staged once per workgroup in LDS (4.3 KB): the
// loop then reads them with broadcast LDS loads instead of one scalar load and
// wait per coupling.
struct MultiSets {
    // one row per set, padded by one entry: 16 lanes reading resonance i of sets 0..15
    // (the matrix-core kernels' A operands) then hit 16 different bank groups
    double2 c[GF_MULTI_PTS][GF_MAX_RES + 1];
    double eff[GF_MULTI_PTS], norm[GF_MULTI_PTS];
};
static_assert(GF_MULTI_PTS * GF_MAX_RES == 256, "one staging thread per (set, resonance)");

// Fill S from cnt sets: set p's parameter array at P0 + p * pstride, its
// normalisation array at N0 + p * nstride; couplings from index pc, the constant
// efficiency (CONST_EFF) at index pe.  All 256 threads of the workgroup take part.
template <bool CONST_EFF>
__device__ __forceinline__ void stage_sets(MultiSets &S, const double *__restrict__ P0, int64_t pstride,
                                           const double *__restrict__ N0, int64_t nstride, int cnt, int pc, int pe,
                                           int nres) {
    const int t = threadIdx.x, p = t >> 4, i = t & 15;
    double2 v   = make_double2(0.0, 0.0);
    if(p < cnt && i < nres) {
        const GF_CONST double *__restrict__ P = gfd::as_const(P0 + p * pstride);
        v                                     = make_double2(P[pc + 2 * i], P[pc + 2 * i + 1]);
    }
    S.c[p][i] = v;
    if(t < GF_MULTI_PTS) {
        S.eff[t]  = (CONST_EFF && t < cnt) ? gfd::as_const(P0 + t * pstride)[pe] : 0.0;
        S.norm[t] = t < cnt ? gfd::as_const(N0 + t * nstride)[1] : 0.0;
    }
    __syncthreads();
}

// The coherent-sum metric of up to GF_MULTI_PTS parameter sets over the same
// events in one sweep: an event's waves are loaded once and every set's term is
// taken with the arithmetic, the event-to-lane assignment and the reduction
// order of k_dalitz_fast on the same grid, so each set's partials equal that
// kernel's for the same parameters bit for bit (the resonance loop runs to
// NR >= nres with zero couplings and waves past nres, whose fused terms add
// exact zeros).  params / norms: npts consecutive copies of the flattened arrays
// (np and nn doubles each).  partials: [npts][gridDim.x].
template <bool CONST_EFF, bool ZERO_OUT, int NR, bool NLL>
__global__ __launch_bounds__(256) void k_dalitz_multi(GfProgArgs A, const double *__restrict__ params, int np,
                                                      const double *__restrict__ norms, int nn, int npts, int metric,
                                                      Partial *partials) {
    __shared__ MultiSets S;
    const GfIns dzi       = A.ins[0];
    const GfIns effi      = A.ins[1];
    const GfDalitzSlot dz = gfd::as_const(A.dz)[dzi.x];
    const GfDecay &D      = A.decay;
    const int nres        = dzi.a;
    const int64_t n       = A.nevents;
    const double *__restrict__ c12 = A.cols[dz.col_m12];
    const double *__restrict__ c13 = A.cols[dz.col_m13];
    stage_sets<CONST_EFF>(S, params, np, norms, nn, npts, dzi.p, effi.p + effi.a, nres);
    constexpr bool nll = NLL;  // the launcher sets it for metric == NLL
    double s[GF_MULTI_PTS], c[GF_MULTI_PTS];  // per set: (sum, residual), or the NLL's (mantissa, exponent)
#pragma unroll
    for(int p = 0; p < GF_MULTI_PTS; ++p) {
        s[p] = nll ? 1.0 : 0.0;
        c[p] = 0.0;
    }
    for(int64_t base = (int64_t)blockIdx.x * blockDim.x; base < n; base += (int64_t)gridDim.x * blockDim.x) {
        // keep the LDS reads of the sets inside the loop: hoisted, the 16 x NR
        // loop-invariant couplings would not fit in registers
        asm volatile("" ::: "memory");
        const int64_t e0 = base + threadIdx.x;
        const bool valid = e0 < n;
        const int64_t e  = valid ? e0 : n - 1;
        double2 w[NR];
#pragma unroll
        for(int i = 0; i < NR; ++i)
            w[i] = (i < nres) ? dz.wave[(int64_t)i * dz.ncache + e] : make_double2(0.0, 0.0);
        const double m12  = ZERO_OUT ? 0.0 : c12[e];
        const double m13  = ZERO_OUT ? 0.0 : c13[e];
        const bool inside =
            ZERO_OUT || gfd::in_dalitz(m12, m13, D.motherMass, D.daug1Mass, D.daug2Mass, D.daug3Mass);
#pragma unroll
        for(int p = 0; p < GF_MULTI_PTS; ++p) {
            if(p < npts) {
                double re = 0.0, im = 0.0;
                gfd::coh_sum<NR>(re, im, [&](int i) { return S.c[p][i]; }, w, nres);
                const double eff =
                    CONST_EFF ? S.eff[p] : multipoly_at(effi, A, gfd::as_const(params + (int64_t)p * np), e);
                const double T = inside ? (re * re + im * im) * eff : 0.0;
                if(nll) {
                    if(valid)
                        gfd::nll_add(s[p], c[p], T, S.norm[p]);
                } else if(valid) {
                    gfd::kb_add(s[p], c[p], gfd::metric(metric, T, 0.0, 0.0, S.norm[p], A.total_events));
                }
            }
        }
    }
#pragma unroll
    for(int p = 0; p < GF_MULTI_PTS; ++p) {
        if(p < npts) {
            double ss = s[p], cc = c[p];
            if(nll)
                ss = gfd::nll_total(ss, cc), cc = 0.0;
            block_reduce(ss, cc);
            if(threadIdx.x == 0) {
                partials[(int64_t)p * gridDim.x + blockIdx.x].s = ss;
                partials[(int64_t)p * gridDim.x + blockIdx.x].c = cc;
            }
        }
    }
}

// ------------------------------------------------------- coherent sums on MFMA
//
// The NLL of up to 16 coupling sets over the same events, constant efficiency, waves 0
// outside the Dalitz region (the k_dalitz_multi<true, true, NR, true> case), with the
// coherent sums of a wave's 64 events formed on the FP64 matrix cores.  Per tile of 16
// events, Re_p and Im_p are rows of real matrix products M W over K = 2 NR terms, on
// v_mfma_f64_16x16x4f64 (NR / 2 steps of K = 4).  The instruction adds its K terms to
// the accumulator one after the other, each as a fused multiply-add.  K-step 2 m takes
// the real parts of the waves of resonances 4 m .. 4 m + 3 (Re: cr wr; Im: ci wr),
// K-step 2 m + 1 their imaginary parts (Re: -ci wi; Im: cr wi): the order of
// gfd::coh_sum, so every element equals the vector sweeps' sum bit for bit.
// Operand layouts (gfx950; the host uses this kernel only after its probe of the
// instruction found the result layout assumed here): lane l supplies A[l % 16][l / 16]
// and B[l / 16][l % 16] of a K-step and holds D[4 r + l / 16][l % 16] in result register
// r.  The couplings are loop-invariant A operands (16 doubles a lane, read from LDS once).
// Lane (g = l / 16, j = l % 16) loads the wave of resonance 4 m + g of event 16 t + j
// (one 16-byte load per group of four resonances: a 256-byte run of 16 events per
// resonance) and gives its real part to K-step 2 m and its imaginary part to 2 m + 1,
// for both products.  Lane (g, j) ends tile t holding |A|^2 eff of sets 4 r + g of event
// 16 t + j, and multiplies it into those sets' NLL products: per set, lane (g, j) takes
// events 16 t + j of each of the wave's tiles in order.  The sets are then reduced over
// the 16 lanes of their group (xor 8, 4, 2, 1) and the four waves in order, partials
// [p][b].  k_dalitz_fast groups the events of a set the same way whenever this kernel
// serves the multi-point sums (GfProgArgs::coh_group), so a multi-point sum equals the
// single sweep of the same parameters.  The register budget is that of three waves per
// SIMD, the occupancy the grid of three workgroups per CU asks for.
//
// coh_mx_rows runs the tiles of this workgroup's events (rows first + k stride +
// 0..255 below end, wave w taking rows 64 w .. 64 w + 63 of each) for the NSG x 16 sets
// staged in S[0 .. NSG - 1] (npts of them in all) and leaves set p's (sum, residual) of
// the workgroup in ls[p], lc[p] (every thread returns after the workgroup barrier).
// With two set groups the wave loads of a tile serve both (the HBM bytes of a sweep are
// shared by 32 sets); the first group's couplings stay in registers, the second's are
// read from LDS per tile, so the kernel keeps three waves per SIMD.  Every set is
// reduced over the same lanes and events in the same order whichever group it is in.
// All 256 threads call it.
template <int NR, int NSG>
__device__ __forceinline__ void coh_mx_rows(const MultiSets *S, const GfDalitzSlot &dz, int nres, int64_t first,
                                            int64_t stride, int64_t end, int npts, double *ls, double *lc) {
    static_assert(NR % 4 == 0 && NR <= GF_MAX_RES, "NR: 4, 8, 12 or 16");
    static_assert(NSG == 1 || NSG == 2, "one or two groups of 16 sets");
    constexpr int NG = NR / 4;  // groups of four resonances: K-steps 2 m (real parts), 2 m + 1 (imaginary)
    __shared__ double wls[4][GF_MX_SETS], wlc[4][GF_MX_SETS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, j = lane & 15;
    // A[j][k]: set j's factor of K term k = 4 kk + g (resonance 4 (kk / 2) + g): K-step 2 m
    // takes (cr | ci) against wr, 2 m + 1 (-ci | cr) against wi
    auto a_ops = [&](const double2 c, double &ar0, double &ai0, double &ar1, double &ai1) {
        ar0 = c.x;   // Re: cr wr
        ai0 = c.y;   // Im: ci wr
        ar1 = -c.y;  // Re: -ci wi
        ai1 = c.x;   // Im: cr wi
    };
    double are[2 * NG], aim[2 * NG];
#pragma unroll
    for(int m = 0; m < NG; ++m)
        a_ops(S[0].c[j][4 * m + g], are[2 * m], aim[2 * m], are[2 * m + 1], aim[2 * m + 1]);
    double m_[4 * NSG];  // per set: the NLL product's mantissa and (integer) exponent
    int ex[4 * NSG];
#pragma unroll
    for(int r = 0; r < 4 * NSG; ++r) {
        m_[r] = 1.0;
        ex[r] = 0;
    }
    // The wave's tiles in order: tile q = 4 p + t covers rows first + p stride + 64 wave +
    // 16 t + (0..15) (pass p of the strided loop, quarter t of the wave's 64 rows).
    // Tile q + 2's waves (q + 1's with two set groups) are requested before tile q's
    // products start, so loads stay in flight behind the matrix cores; a tile past the end
    // reads row end - 1 (one line per resonance) and is never used.
    const double2 *__restrict__ wv = dz.wave;
    const int64_t ntile            = first < end ? 4 * ((end - 1 - first) / stride + 1) : 0;
    auto tile_event = [&](int64_t q) { return first + (q >> 2) * stride + 64 * wave + 16 * (q & 3) + j; };
    // Only the last group can reach past nres (NR - 4 < nres <= NR): there the load reads
    // resonance nres - 1 and the value is replaced by zero, without a branch around it.
    auto load_tile = [&](int64_t q, double2(&w)[NG]) {
        const int64_t ev  = tile_event(q);
        const int64_t row = ev < end ? ev : end - 1;  // loads stay in bounds; the row is masked below
#pragma unroll
        for(int m = 0; m < NG; ++m) {
            const int i  = 4 * m + g;
            const int ir = (m == NG - 1 && i >= nres) ? nres - 1 : i;
            w[m]         = wv[(int64_t)ir * dz.ncache + row];
        }
    };
    auto run_tile = [&](int64_t q, const double2(&w)[NG]) {
        const bool live     = tile_event(q) < end;
        const bool all_live = tile_event(q) - j + 15 < end;  // uniform over the wave
#pragma unroll
        for(int sg = 0; sg < NSG; ++sg) {
            gf_double4 re = {0, 0, 0, 0}, im = {0, 0, 0, 0};
#pragma unroll
            for(int m = 0; m < NG; ++m) {
                const bool pad   = m == NG - 1 && 4 * m + g >= nres;
                const double2 wk = pad ? make_double2(0.0, 0.0) : w[m];
                double ar0, ai0, ar1, ai1;
                if(sg == 0) {
                    ar0 = are[2 * m], ai0 = aim[2 * m], ar1 = are[2 * m + 1], ai1 = aim[2 * m + 1];
                } else {
                    a_ops(S[sg].c[j][4 * m + g], ar0, ai0, ar1, ai1);
                }
                re = __builtin_amdgcn_mfma_f64_16x16x4f64(ar0, wk.x, re, 0, 0, 0);
                im = __builtin_amdgcn_mfma_f64_16x16x4f64(ai0, wk.x, im, 0, 0, 0);
                re = __builtin_amdgcn_mfma_f64_16x16x4f64(ar1, wk.y, re, 0, 0, 0);
                im = __builtin_amdgcn_mfma_f64_16x16x4f64(ai1, wk.y, im, 0, 0, 0);
            }
            // The sets' efficiencies and normalisations are read from LDS per tile (held in
            // registers they would cost the occupancy of three waves per SIMD).  A set past
            // npts has efficiency and normalisation 0 (stage_sets), so its factor is 0, which
            // the product takes as exactly 1 (mantissa 1/2, exponent +1, renormalised back:
            // the pair is unchanged); a lane past the last row is given the factor 1 outright,
            // in the one tile per wave that reaches past it.
            asm volatile("" ::: "memory");
            double ef[4], nm[4];
#pragma unroll
            for(int r = 0; r < 4; ++r) {
                ef[r] = S[sg].eff[4 * r + g];
                nm[r] = S[sg].norm[4 * r + g];
            }
            if(all_live) {
#pragma unroll
                for(int r = 0; r < 4; ++r)
                    gfmath::nll_add(m_[4 * sg + r], ex[4 * sg + r], ((re[r] * re[r] + im[r] * im[r]) * ef[r]) * nm[r]);
            } else {
#pragma unroll
                for(int r = 0; r < 4; ++r) {
                    const double v = ((re[r] * re[r] + im[r] * im[r]) * ef[r]) * nm[r];
                    gfmath::nll_add(m_[4 * sg + r], ex[4 * sg + r], live ? v : 1.0);
                }
            }
        }
    };
    if(ntile > 0 && NSG == 1) {
        double2 wa[NG], wb[NG], wc[NG];
        load_tile(0, wa);
        load_tile(1, wb);
        for(int64_t q = 0;; q += 3) {
            load_tile(q + 2, wc);
            run_tile(q, wa);
            if(q + 1 >= ntile)
                break;
            load_tile(q + 3, wa);
            run_tile(q + 1, wb);
            if(q + 2 >= ntile)
                break;
            load_tile(q + 4, wb);
            run_tile(q + 2, wc);
            if(q + 3 >= ntile)
                break;
        }
    } else if(ntile > 0) {
        // two groups: a tile's products take twice as long, so one tile of loads ahead
        // covers the same time (and the registers of a third buffer are not there)
        double2 wa[NG], wb[NG];
        load_tile(0, wa);
        for(int64_t q = 0;; q += 2) {
            load_tile(q + 1, wb);
            run_tile(q, wa);
            if(q + 1 >= ntile)
                break;
            load_tile(q + 2, wa);
            run_tile(q + 1, wb);
            if(q + 2 >= ntile)
                break;
        }
    }
    // set p: the 16 lanes of its group (xor 8, 4, 2, 1), then the four waves in order
#pragma unroll
    for(int r = 0; r < 4 * NSG; ++r) {
        double sv = gfd::nll_total(m_[r], (double)ex[r]), cv = 0.0;
        group_reduce(sv, cv);
        if(j == 0) {
            const int p    = GF_MULTI_PTS * (r >> 2) + 4 * (r & 3) + g;
            wls[wave][p]   = sv;
            wlc[wave][p]   = cv;
        }
    }
    __syncthreads();
    if((int)threadIdx.x < npts) {
        const int p = threadIdx.x;
        double sv   = wls[0][p], cv = wlc[0][p];
        for(int w = 1; w < 4; ++w)
            gfd::kb_merge(sv, cv, wls[w][p], wlc[w][p]);
        ls[p] = sv;
        lc[p] = cv;
    }
    __syncthreads();
}

// Up to NSG x 16 sets per sweep (partials [p][b]); NSG = 2 shares each wave load
// between two groups of 16 sets.
template <int NR, int NSG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_coh_mx(
    GfProgArgs A, const double *__restrict__ params, int np, const double *__restrict__ norms, int nn, int npts,
    Partial *partials) {
    __shared__ MultiSets S[NSG];
    __shared__ double ls[GF_MX_SETS], lc[GF_MX_SETS];
    const GfIns dzi       = A.ins[0];
    const GfIns effi      = A.ins[1];
    const GfDalitzSlot dz = gfd::as_const(A.dz)[dzi.x];
    const int nres        = dzi.a;
#pragma unroll
    for(int sg = 0; sg < NSG; ++sg)
        stage_sets<true>(S[sg], params + (int64_t)GF_MULTI_PTS * sg * np, np, norms + (int64_t)GF_MULTI_PTS * sg * nn,
                         nn, min(max(npts - GF_MULTI_PTS * sg, 0), GF_MULTI_PTS), dzi.p, effi.p + effi.a, nres);
    coh_mx_rows<NR, NSG>(S, dz, nres, (int64_t)blockIdx.x * blockDim.x, (int64_t)gridDim.x * blockDim.x, A.nevents,
                         npts, ls, lc);
    if((int)threadIdx.x < npts) {
        const int p                                    = threadIdx.x;
        partials[(int64_t)p * gridDim.x + blockIdx.x].s = ls[p];
        partials[(int64_t)p * gridDim.x + blockIdx.x].c = lc[p];
    }
}

// k_finish for several sums: workgroup p adds the nparts partials of set p in the
// order k_finish uses and writes {sum, residual} to out[2p] (host-mapped memory that
// the host polls): the residual, a system-scope fence, then the sum over the empty
// marker the host left there.
__global__ __launch_bounds__(GF_BLOCK) void k_finish_multi(const Partial *partials, int nparts, double *out) {
    const Partial *q = partials + (int64_t)blockIdx.x * nparts;
    double ts = 0.0, tc = 0.0;
    for(int i = threadIdx.x; i < nparts; i += GF_BLOCK)
        gfd::kb_merge(ts, tc, q[i].s, q[i].c);
    block_reduce(ts, tc);
    if(threadIdx.x == 0) {
        out[2 * blockIdx.x + 1] = tc;
        __threadfence_system();
        __hip_atomic_store((unsigned long long *)(out + 2 * blockIdx.x),
                           (unsigned long long)__double_as_longlong(gfd::kb_total(ts, tc)), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ------------------------------------------------------------- toy batches

// One entry of a batch's work table: rows [start, end) of toy `toy`.
// (GfBatchWork is declared in gf_internal.h)

// The metric sum over rows [w.start, w.end) of one toy with parameter array P and
// normalisation array Nm, accumulated per thread in the tile order of
// k_batch_metric (EPT rows per thread per tile).
template <int EPT, int FEAT>
__device__ __forceinline__ void batch_rows(const GfProgArgs &A, const GfBatchWork &w, const double *__restrict__ P,
                                           const double *__restrict__ Nm, int metric, double &s, double &c) {
    const double norm  = Nm[1];
    const bool binned  = metric >= GF_METRIC_BINAVG_CODE;
    const bool nll     = metric == gfd::metric_nll;
    const int64_t tile = (int64_t)GF_BLOCK * EPT;
    if(nll)  // the NLL as a product: (mantissa, exponent)
        s = 1.0, c = 0.0;
    for(int64_t base = w.start; base < w.end; base += tile) {
        ColSrc<EPT> src;
        src.cols = A.cols;
        int64_t row[EPT];
        bool valid[EPT];
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            const int64_t r = base + (int64_t)j * GF_BLOCK + threadIdx.x;
            valid[j]        = r < w.end;
            row[j]          = valid[j] ? r : w.start;
            src.idx[j]      = row[j];
        }
        double T[EPT];
        run<EPT, FEAT>(A, P, Nm, 0, src, row, valid, T);
#pragma unroll
        for(int j = 0; j < EPT; ++j) {
            if(!valid[j])
                continue;
            if(nll) {
                gfd::nll_add(s, c, T[j], norm);
                continue;
            }
            double e0 = 0.0, e1 = 0.0;
            if(binned) {
                e0 = A.cols[A.nobs - 2][row[j]];
                e1 = A.cols[A.nobs - 1][row[j]];
            }
            gfd::kb_add(s, c, gfd::metric(metric, T[j], e0, e1, norm, w.total));
        }
    }
    if(nll)
        s = gfd::nll_total(s, c), c = 0.0;
}

// Metric sums of many toys in one launch: workgroup b evaluates the rows of
// work[b] with its toy's parameter and normalisation arrays (P = params +
// toy * np, Nm = norms + toy * nn) and stores one partial; workgroups of
// inactive toys store zero.  FEAT as for k_reduce_metric.
template <int EPT, int FEAT>
__global__ __launch_bounds__(GF_BLOCK) void k_batch_metric(GfProgArgs A, const GfBatchWork *__restrict__ work,
                                                           const double *__restrict__ params, int np,
                                                           const double *__restrict__ norms, int nn,
                                                           const uint8_t *__restrict__ active, int metric,
                                                           Partial *partials) {
    const GfBatchWork w = work[blockIdx.x];
    double s = 0.0, c = 0.0;
    if(active[w.toy])
        batch_rows<EPT, FEAT>(A, w, params + (int64_t)w.toy * np, norms + (int64_t)w.toy * nn, metric, s, c);
    store_partial(s, c, partials);
}

// Several points per toy, any program: workgroup (b, g) evaluates the rows of
// work[b] once per point p in [16 g, min(16 g + 16, npts)) of its toy and stores
// partial (b, p).  Each point's sum takes the path of k_batch_metric.
template <int EPT, int FEAT>
__global__ __launch_bounds__(GF_BLOCK) void k_batch_points(GfProgArgs A, const GfBatchWork *__restrict__ work,
                                                           const double *__restrict__ stage, int np, int nn,
                                                           const int *__restrict__ tbl, int metric,
                                                           Partial *partials) {
    const GfBatchWork w = work[blockIdx.x];
    const int slot0     = tbl[2 * w.toy];
    const int npts      = tbl[2 * w.toy + 1];
    const int p0        = (int)blockIdx.y * GF_MULTI_PTS;
    const int p1        = min(npts, p0 + GF_MULTI_PTS);
    for(int p = p0; p < p1; ++p) {
        const double *__restrict__ P = stage + (int64_t)(slot0 + p) * (np + nn);
        double s = 0.0, c = 0.0;
        batch_rows<EPT, FEAT>(A, w, P, P + np, metric, s, c);
        block_reduce(s, c);
        if(threadIdx.x == 0) {
            partials[(int64_t)blockIdx.x * GF_BATCH_PTS + p].s = s;
            partials[(int64_t)blockIdx.x * GF_BATCH_PTS + p].c = c;
        }
    }
}

// Several points per toy, coherent-sum program (as k_dalitz_multi): workgroup
// (b, g) reads the waves of each row of work[b] once and adds the row's metric
// for every point p in [16 g, min(16 g + 16, npts)) of its toy.  A group of
// mx_min points or more is left to k_batch_coh_mx (launched over the same grid).
template <bool CONST_EFF, bool ZERO_OUT, int NR, bool NLL>
__global__ __launch_bounds__(GF_BLOCK) void k_batch_dalitz_points(GfProgArgs A, const GfBatchWork *__restrict__ work,
                                                                  const double *__restrict__ stage, int np, int nn,
                                                                  const int *__restrict__ tbl, int metric,
                                                                  int mx_min, Partial *partials) {
    __shared__ MultiSets S;
    const GfBatchWork w = work[blockIdx.x];
    const int slot0     = tbl[2 * w.toy];
    const int npts      = tbl[2 * w.toy + 1];
    const int p0        = (int)blockIdx.y * GF_MULTI_PTS;
    const int cnt       = min(npts - p0, GF_MULTI_PTS);
    if(cnt <= 0 || cnt >= mx_min)
        return;  // uniform over the workgroup
    const GfIns dzi       = A.ins[0];
    const GfIns effi      = A.ins[1];
    const GfDalitzSlot dz = gfd::as_const(A.dz)[dzi.x];
    const GfDecay &D      = A.decay;
    const int nres        = dzi.a;
    const int64_t W       = np + nn;
    const double *__restrict__ S0  = stage + (int64_t)(slot0 + p0) * W;
    const double *__restrict__ c12 = A.cols[dz.col_m12];
    const double *__restrict__ c13 = A.cols[dz.col_m13];
    stage_sets<CONST_EFF>(S, S0, W, S0 + np, W, cnt, dzi.p, effi.p + effi.a, nres);
    constexpr bool nll = NLL;  // the launcher sets it for metric == NLL
    double s[GF_MULTI_PTS], c[GF_MULTI_PTS];  // per point: (sum, residual), or the NLL's (mantissa, exponent)
#pragma unroll
    for(int p = 0; p < GF_MULTI_PTS; ++p) {
        s[p] = nll ? 1.0 : 0.0;
        c[p] = 0.0;
    }
    for(int64_t base = w.start; base < w.end; base += GF_BLOCK) {
        asm volatile("" ::: "memory");  // the set reads stay in the loop (as k_dalitz_multi)
        const int64_t e0 = base + threadIdx.x;
        const bool valid = e0 < w.end;
        const int64_t e  = valid ? e0 : w.start;
        double2 wv[NR];
#pragma unroll
        for(int i = 0; i < NR; ++i)
            wv[i] = (i < nres) ? dz.wave[(int64_t)i * dz.ncache + e] : make_double2(0.0, 0.0);
        const double m12  = ZERO_OUT ? 0.0 : c12[e];
        const double m13  = ZERO_OUT ? 0.0 : c13[e];
        const bool inside =
            ZERO_OUT || gfd::in_dalitz(m12, m13, D.motherMass, D.daug1Mass, D.daug2Mass, D.daug3Mass);
#pragma unroll
        for(int p = 0; p < GF_MULTI_PTS; ++p) {
            if(p < cnt) {
                // a toy's points are compared with one another, never with the single
                // sweep, so the sum keeps the per-resonance order (fewer live registers)
                double re = 0.0, im = 0.0;
#pragma unroll
                for(int i = 0; i < NR; ++i) {
                    const double2 cp = S.c[p][i];
                    gfd::cmac(re, im, cp.x, cp.y, wv[i]);
                }
                const double eff = CONST_EFF ? S.eff[p] : multipoly_at(effi, A, gfd::as_const(S0 + p * W), e);
                const double T   = inside ? (re * re + im * im) * eff : 0.0;
                if(nll) {
                    if(valid)
                        gfd::nll_add(s[p], c[p], T, S.norm[p]);
                } else if(valid) {
                    gfd::kb_add(s[p], c[p], gfd::metric(metric, T, 0.0, 0.0, S.norm[p], w.total));
                }
            }
        }
    }
#pragma unroll
    for(int p = 0; p < GF_MULTI_PTS; ++p) {
        if(p < cnt) {
            double ss = s[p], cc = c[p];
            if(nll)
                ss = gfd::nll_total(ss, cc), cc = 0.0;
            block_reduce(ss, cc);
            if(threadIdx.x == 0) {
                partials[(int64_t)blockIdx.x * GF_BATCH_PTS + p0 + p].s = ss;
                partials[(int64_t)blockIdx.x * GF_BATCH_PTS + p0 + p].c = cc;
            }
        }
    }
}

// The groups of k_batch_dalitz_points with mx_min points or more, for the NLL of a
// lone Amp3Body with constant efficiency and waves 0 outside the Dalitz region: the
// coherent sums on the FP64 matrix cores (coh_mx_rows over the rows of the
// workgroup's chunk, as k_coh_mx runs them over the whole sample).  A smaller group
// (a line-search point, say) exits here and is taken by the vector kernel.  A
// point's value depends on the size of the group it came in, deterministically; the
// points of a toy meet only in its minimiser, which sees differences of an ulp.
template <int NR>
__global__ __launch_bounds__(GF_BLOCK) void k_batch_coh_mx(GfProgArgs A, const GfBatchWork *__restrict__ work,
                                                           const double *__restrict__ stage, int np, int nn,
                                                           const int *__restrict__ tbl, int mx_min,
                                                           Partial *partials) {
    const GfBatchWork w = work[blockIdx.x];
    const int npts      = tbl[2 * w.toy + 1];
    const int p0        = (int)blockIdx.y * GF_MULTI_PTS;
    const int cnt       = min(npts - p0, GF_MULTI_PTS);
    if(cnt < mx_min)
        return;  // uniform over the workgroup
    __shared__ MultiSets S[1];
    __shared__ double ls[GF_MULTI_PTS], lc[GF_MULTI_PTS];
    const GfIns dzi                = A.ins[0];
    const GfIns effi               = A.ins[1];
    const GfDalitzSlot dz          = gfd::as_const(A.dz)[dzi.x];
    const int nres                 = dzi.a;
    const int64_t W                = np + nn;
    const double *__restrict__ S0  = stage + (int64_t)(tbl[2 * w.toy] + p0) * W;
    stage_sets<true>(S[0], S0, W, S0 + np, W, cnt, dzi.p, effi.p + effi.a, nres);
    coh_mx_rows<NR, 1>(S, dz, nres, w.start, GF_BLOCK, w.end, cnt, ls, lc);
    if((int)threadIdx.x < cnt) {
        const int p                                             = threadIdx.x;
        partials[(int64_t)blockIdx.x * GF_BATCH_PTS + p0 + p].s = ls[p];
        partials[(int64_t)blockIdx.x * GF_BATCH_PTS + p0 + p].c = lc[p];
    }
}

// The normalisation arrays of staged batch points, one lane per point: the template,
// then norms[op.out] = 1 / I for each op with I from the point's parameters in the
// host's operation order (GooPdf::normalize: ret = 1 * integral, norm = 1 / ret;
// GaussianPdf.cu:28-35, ExpPdf.cu:121-132, Amp3Body.cu:334-358).
__global__ __launch_bounds__(256) void k_batch_norms(double *__restrict__ stage, int nslots, int np, int nn,
                                                     const double *__restrict__ tmpl,
                                                     const GfNormOp *__restrict__ ops, int nops,
                                                     const double *__restrict__ table) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if(k >= nslots)
        return;
    const double *__restrict__ P = stage + (int64_t)k * (np + nn);
    double *__restrict__ Nm      = stage + (int64_t)k * (np + nn) + np;
    for(int i = 0; i < nn; ++i)
        Nm[i] = tmpl[i];
    for(int o = 0; o < nops; ++o) {
        const GfNormOp op = ops[o];
        double integral;
        if(op.kind == GN_SCALE) {
            integral = P[op.p];
            integral *= op.c0;
        } else if(op.kind == GN_EXP) {
            const double a = P[op.p];
            if(0 == a) {
                integral = op.c1 - op.c0;
            } else {
                integral = exp(a * op.c1) - exp(a * op.c0);
                integral /= a;
            }
        } else {
            // sum_ij c_i conj(c_j) T_ij, each complex product written out
            const double *__restrict__ cp = P + op.p;
            const double *__restrict__ T  = table + op.g;
            double sum_re = 0;
            for(int i = 0; i < op.n; ++i) {
                const double ar = cp[2 * i], ai = cp[2 * i + 1];
                for(int j = 0; j < op.n; ++j) {
                    const double br = cp[2 * j], bi = -cp[2 * j + 1];
                    const double pr = ar * br - ai * bi, pi = ar * bi + ai * br;
                    const double ir = T[2 * (i * op.n + j)], ii = T[2 * (i * op.n + j) + 1];
                    sum_re += pr * ir - pi * ii;
                }
            }
            integral = sum_re;
            integral *= op.c0;
        }
        double ret = 1;
        ret *= integral;
        Nm[op.out] = 1.0 / ret;
    }
}

// One workgroup per toy: for each of its points, the partials of the toy's work
// entries [first[t], first[t + 1]) in the order of k_finish_toys into
// result[2 (t GF_BATCH_PTS + p) ..] (host-mapped).
__global__ __launch_bounds__(GF_BLOCK) void k_finish_toy_points(const Partial *__restrict__ partials,
                                                                const int *__restrict__ first,
                                                                const int *__restrict__ tbl,
                                                                double *__restrict__ result) {
    const int t    = blockIdx.x;
    const int npts = tbl[2 * t + 1];
    const int f0 = first[t], f1 = first[t + 1];
    if(f1 - f0 <= 64) {  // uniform over the workgroup
        // Every partial of the toy lies in wave 0 of block_reduce's layout (thread i holds
        // entry i), and waves 1-3 hold exact (+0, +0) pairs.  So one wave per point gives
        // block_reduce's bits -- the same butterfly, then three zero pairs merged in
        // order -- and the four waves take the points in turn, without a barrier.
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        for(int p = wave; p < npts; p += GF_BLOCK / 64) {
            double s = 0.0, c = 0.0;
            if(f0 + lane < f1)
                gfd::kb_merge(s, c, partials[(int64_t)(f0 + lane) * GF_BATCH_PTS + p].s,
                              partials[(int64_t)(f0 + lane) * GF_BATCH_PTS + p].c);
#pragma unroll
            for(int off = 32; off > 0; off >>= 1) {
                double s2 = __shfl_xor(s, off, 64);
                double c2 = __shfl_xor(c, off, 64);
                gfd::kb_merge(s, c, s2, c2);
            }
            if(lane == 0) {
                for(int w = 1; w < GF_BLOCK / 64; ++w)
                    gfd::kb_merge(s, c, 0.0, 0.0);
                result[2 * ((int64_t)t * GF_BATCH_PTS + p)]     = gfd::kb_total(s, c);
                result[2 * ((int64_t)t * GF_BATCH_PTS + p) + 1] = c;
            }
        }
        return;
    }
    for(int p = 0; p < npts; ++p) {
        double s = 0.0, c = 0.0;
        for(int i = first[t] + threadIdx.x; i < first[t + 1]; i += GF_BLOCK)
            gfd::kb_merge(s, c, partials[(int64_t)i * GF_BATCH_PTS + p].s, partials[(int64_t)i * GF_BATCH_PTS + p].c);
        block_reduce(s, c);
        if(threadIdx.x == 0) {
            result[2 * ((int64_t)t * GF_BATCH_PTS + p)]     = gfd::kb_total(s, c);
            result[2 * ((int64_t)t * GF_BATCH_PTS + p) + 1] = c;
        }
    }
}

// One workgroup per toy: the toy's partials [first[t], first[t + 1]) in order
// into result[2t] = sum, result[2t + 1] = residual (host-mapped).
__global__ __launch_bounds__(GF_BLOCK) void k_finish_toys(const Partial *__restrict__ partials,
                                                          const int *__restrict__ first,
                                                          const uint8_t *__restrict__ active,
                                                          double *__restrict__ result) {
    const int t = blockIdx.x;
    if(!active[t])
        return;
    double s = 0.0, c = 0.0;
    for(int i = first[t] + threadIdx.x; i < first[t + 1]; i += GF_BLOCK)
        gfd::kb_merge(s, c, partials[i].s, partials[i].c);
    block_reduce(s, c);
    if(threadIdx.x == 0) {
        result[2 * t]     = gfd::kb_total(s, c);
        result[2 * t + 1] = c;
    }
}

// Completion stamp after the toys' results: counter + 1 into the mapped word.
__global__ void k_stamp(uint32_t *__restrict__ counter, uint32_t *__restrict__ mapped) {
    const uint32_t v = *counter + 1u;
    *counter         = v;
    __threadfence_system();
    __hip_atomic_store(mapped, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

namespace gfk {

template <bool WRITE, bool INL, bool CE, bool ZO = false>
static void launch_fast_t(const GfProgArgs &a, const GfInline *inl, int metric, Partial *partials, double *out,
                          int nblocks, hipStream_t s) {
    hipLaunchKernelGGL((k_dalitz_fast<WRITE, INL, CE, ZO>), dim3(nblocks), dim3(256), 0, s, a,
                       inl ? *inl : GfInline{}, metric, partials, out);
}

// The multi-set kernels for nres resonances: the resonance loop unrolled to the
// next multiple of 4 (NR), the variant by efficiency and zero-outside use.
#define GF_MULTI_CASES(KERNEL, NLLB, ...)                                                                           \
    switch(v_ * 4 + nr_ / 4 - 1) {                                                                                   \
    case 0: hipLaunchKernelGGL((KERNEL<false, false, 4, NLLB>), __VA_ARGS__); break;                                \
    case 1: hipLaunchKernelGGL((KERNEL<false, false, 8, NLLB>), __VA_ARGS__); break;                                \
    case 2: hipLaunchKernelGGL((KERNEL<false, false, 12, NLLB>), __VA_ARGS__); break;                               \
    case 3: hipLaunchKernelGGL((KERNEL<false, false, 16, NLLB>), __VA_ARGS__); break;                               \
    case 4: hipLaunchKernelGGL((KERNEL<true, false, 4, NLLB>), __VA_ARGS__); break;                                 \
    case 5: hipLaunchKernelGGL((KERNEL<true, false, 8, NLLB>), __VA_ARGS__); break;                                 \
    case 6: hipLaunchKernelGGL((KERNEL<true, false, 12, NLLB>), __VA_ARGS__); break;                                \
    case 7: hipLaunchKernelGGL((KERNEL<true, false, 16, NLLB>), __VA_ARGS__); break;                                \
    case 8: hipLaunchKernelGGL((KERNEL<true, true, 4, NLLB>), __VA_ARGS__); break;                                  \
    case 9: hipLaunchKernelGGL((KERNEL<true, true, 8, NLLB>), __VA_ARGS__); break;                                  \
    case 10: hipLaunchKernelGGL((KERNEL<true, true, 12, NLLB>), __VA_ARGS__); break;                                \
    default: hipLaunchKernelGGL((KERNEL<true, true, 16, NLLB>), __VA_ARGS__); break;                                \
    }
// The variant for nres resonances (loop unrolled to the next multiple of 4), the
// efficiency / zero-outside use, and whether the metric is the NLL (its own
// accumulation, compiled apart so that each variant holds only its own path).
#define GF_MULTI_SWITCH(KERNEL, NRES, CE, ZO, NLL, ...)                                                             \
    do {                                                                                                             \
        const int nr_ = (NRES) <= 4 ? 4 : (NRES) <= 8 ? 8 : (NRES) <= 12 ? 12 : 16;                                  \
        const int v_  = (CE) ? ((ZO) ? 2 : 1) : 0;                                                                   \
        if(NLL) {                                                                                                    \
            GF_MULTI_CASES(KERNEL, true, __VA_ARGS__)                                                                \
        } else {                                                                                                     \
            GF_MULTI_CASES(KERNEL, false, __VA_ARGS__)                                                               \
        }                                                                                                            \
    } while(0)

// k_batch_coh_mx for nres resonances (NR = nres rounded up to 4).
#define GF_COH_MX(KERNEL, NRES, ...)                                                                                 \
    do {                                                                                                             \
        switch((NRES) <= 4 ? 4 : (NRES) <= 8 ? 8 : (NRES) <= 12 ? 12 : 16) {                                         \
        case 4: hipLaunchKernelGGL((KERNEL<4>), __VA_ARGS__); break;                                                \
        case 8: hipLaunchKernelGGL((KERNEL<8>), __VA_ARGS__); break;                                                \
        case 12: hipLaunchKernelGGL((KERNEL<12>), __VA_ARGS__); break;                                              \
        default: hipLaunchKernelGGL((KERNEL<16>), __VA_ARGS__); break;                                              \
        }                                                                                                            \
    } while(0)

// k_coh_mx<NR, NSG> for nres resonances (NR = nres rounded up to 4).
template <int NSG>
static void launch_coh_mx(int nres, int nblocks, hipStream_t s, const GfProgArgs &a, const double *params, int np,
                          const double *norms, int nn, int npts, Partial *partials) {
    const dim3 grid(nblocks), block(256);
    switch(nres <= 4 ? 4 : nres <= 8 ? 8 : nres <= 12 ? 12 : 16) {
    case 4: hipLaunchKernelGGL((k_coh_mx<4, NSG>), grid, block, 0, s, a, params, np, norms, nn, npts, partials); break;
    case 8: hipLaunchKernelGGL((k_coh_mx<8, NSG>), grid, block, 0, s, a, params, np, norms, nn, npts, partials); break;
    case 12:
        hipLaunchKernelGGL((k_coh_mx<12, NSG>), grid, block, 0, s, a, params, np, norms, nn, npts, partials);
        break;
    default:
        hipLaunchKernelGGL((k_coh_mx<16, NSG>), grid, block, 0, s, a, params, np, norms, nn, npts, partials);
        break;
    }
}

int launch_dalitz_multi(const GfProgArgs &a, int nres, const double *params, int np, const double *norms, int nn,
                        int npts, bool const_eff, bool zero_outside, int metric, Partial *partials, double *out,
                        int nblocks, void *stream) {
    hipStream_t s = (hipStream_t)stream;
    const bool mx = a.coh_mx_nres > 0 && const_eff && zero_outside && metric == gfd::metric_nll;
    if(npts < 1 || npts > (mx ? GF_MX_SETS : GF_MULTI_PTS) || nres < 1 || nres > GF_MAX_RES)
        return -1;
    if(mx) {
        if(npts > GF_MULTI_PTS)
            launch_coh_mx<2>(nres, nblocks, s, a, params, np, norms, nn, npts, partials);
        else
            launch_coh_mx<1>(nres, nblocks, s, a, params, np, norms, nn, npts, partials);
        int rc = check(hipGetLastError());
        if(rc)
            return rc;
        hipLaunchKernelGGL(k_finish_multi, dim3(npts), dim3(GF_BLOCK), 0, s, partials, nblocks, out);
        return check(hipGetLastError());
    }
    GF_MULTI_SWITCH(k_dalitz_multi, nres, const_eff, zero_outside && const_eff, metric == gfd::metric_nll, dim3(nblocks), dim3(256), 0, s, a,
                    params, np, norms, nn, npts, metric, partials);
    int rc = check(hipGetLastError());
    if(rc)
        return rc;
    hipLaunchKernelGGL(k_finish_multi, dim3(npts), dim3(GF_BLOCK), 0, s, partials, nblocks, out);
    return check(hipGetLastError());
}

int launch_dalitz_fast(const GfProgArgs &a, const GfInline *inl, bool const_eff, bool zero_outside, int metric,
                       Partial *partials, GfResult *result, double *out, int nblocks, void *stream) {
    hipStream_t s = (hipStream_t)stream;
    const int v   = (out ? 4 : 0) | (inl ? 2 : 0) | (const_eff ? 1 : 0);
    if(zero_outside && const_eff) {
        switch(v) {
        case 1: launch_fast_t<false, false, true, true>(a, inl, metric, partials, out, nblocks, s); break;
        case 3: launch_fast_t<false, true, true, true>(a, inl, metric, partials, out, nblocks, s); break;
        case 5: launch_fast_t<true, false, true, true>(a, inl, metric, partials, out, nblocks, s); break;
        default: launch_fast_t<true, true, true, true>(a, inl, metric, partials, out, nblocks, s); break;
        }
        if(out)
            return check(hipGetLastError());
        return launch_finish(a, partials, nblocks, result, s);
    }
    switch(v) {
    case 0: launch_fast_t<false, false, false>(a, inl, metric, partials, out, nblocks, s); break;
    case 1: launch_fast_t<false, false, true>(a, inl, metric, partials, out, nblocks, s); break;
    case 2: launch_fast_t<false, true, false>(a, inl, metric, partials, out, nblocks, s); break;
    case 3: launch_fast_t<false, true, true>(a, inl, metric, partials, out, nblocks, s); break;
    case 4: launch_fast_t<true, false, false>(a, inl, metric, partials, out, nblocks, s); break;
    case 5: launch_fast_t<true, false, true>(a, inl, metric, partials, out, nblocks, s); break;
    case 6: launch_fast_t<true, true, false>(a, inl, metric, partials, out, nblocks, s); break;
    default: launch_fast_t<true, true, true>(a, inl, metric, partials, out, nblocks, s); break;
    }
    if(out)
        return check(hipGetLastError());
    return launch_finish(a, partials, nblocks, result, s);
}

int launch_batch(const GfProgArgs &a, const GfBatchWork *work, int nblocks, const double *params, int np,
                 const double *norms, int nn, const uint8_t *active, int metric, Partial *partials, const int *first,
                 int ntoys, double *result, uint32_t *counter, uint32_t *stamp, void *stream) {
    hipStream_t s = (hipStream_t)stream;
    switch(feature_level(a)) {
    case 0:
        hipLaunchKernelGGL((k_batch_metric<2, 0>), dim3(nblocks), dim3(GF_BLOCK), 0, s, a, work, params, np, norms, nn,
                           active, metric, partials);
        break;
    case 1:
        hipLaunchKernelGGL((k_batch_metric<2, 1>), dim3(nblocks), dim3(GF_BLOCK), 0, s, a, work, params, np, norms, nn,
                           active, metric, partials);
        break;
    default:
        hipLaunchKernelGGL((k_batch_metric<2, 2>), dim3(nblocks), dim3(GF_BLOCK), 0, s, a, work, params, np, norms, nn,
                           active, metric, partials);
        break;
    }
    int rc = check(hipGetLastError());
    if(rc)
        return rc;
    hipLaunchKernelGGL(k_finish_toys, dim3(ntoys), dim3(GF_BLOCK), 0, s, partials, first, active, result);
    if((rc = check(hipGetLastError())))
        return rc;
    hipLaunchKernelGGL(k_stamp, dim3(1), dim3(1), 0, s, counter, stamp);
    return check(hipGetLastError());
}

int launch_batch_norms(double *stage, int nslots, int np, int nn, const double *tmpl, const GfNormOp *ops, int nops,
                       const double *table, void *stream) {
    if(nslots <= 0)
        return 0;
    hipLaunchKernelGGL(k_batch_norms, dim3((nslots + 255) / 256), dim3(256), 0, (hipStream_t)stream, stage, nslots, np,
                       nn, tmpl, ops, nops, table);
    return check(hipGetLastError());
}

int launch_batch_points(const GfProgArgs &a, int nres, const GfBatchWork *work, int nblocks, int groups,
                        const double *stage, int np, int nn, const int *tbl, bool fast, bool const_eff,
                        bool zero_outside, int metric, int mx_min, Partial *partials, const int *first, int ntoys,
                        double *result, uint32_t *counter, uint32_t *stamp, void *stream) {
    hipStream_t s = (hipStream_t)stream;
    if(groups < 1 || groups * GF_MULTI_PTS > GF_BATCH_PTS || (fast && (nres < 1 || nres > GF_MAX_RES)))
        return -1;
    const dim3 grid(nblocks, groups);
    if(!fast && feature_level(a) == 2)
        hipLaunchKernelGGL((k_batch_points<2, 2>), grid, dim3(GF_BLOCK), 0, s, a, work, stage, np, nn, tbl, metric,
                           partials);
    else if(!fast && feature_level(a) == 1)
        hipLaunchKernelGGL((k_batch_points<2, 1>), grid, dim3(GF_BLOCK), 0, s, a, work, stage, np, nn, tbl, metric,
                           partials);
    else if(!fast)
        hipLaunchKernelGGL((k_batch_points<2, 0>), grid, dim3(GF_BLOCK), 0, s, a, work, stage, np, nn, tbl, metric,
                           partials);
    else {
        // groups of mx_min points or more on the matrix cores, the others on the vector ALUs
        const bool mx = mx_min > 0 && const_eff && zero_outside && metric == gfd::metric_nll;
        if(mx) {
            GF_COH_MX(k_batch_coh_mx, nres, grid, dim3(GF_BLOCK), 0, s, a, work, stage, np, nn, tbl, mx_min,
                      partials);
            int rc = check(hipGetLastError());
            if(rc)
                return rc;
        }
        GF_MULTI_SWITCH(k_batch_dalitz_points, nres, const_eff, zero_outside && const_eff, metric == gfd::metric_nll, grid, dim3(GF_BLOCK), 0, s,
                        a, work, stage, np, nn, tbl, metric, mx ? mx_min : GF_MULTI_PTS + 1, partials);
    }
    int rc = check(hipGetLastError());
    if(rc)
        return rc;
    hipLaunchKernelGGL(k_finish_toy_points, dim3(ntoys), dim3(GF_BLOCK), 0, s, partials, first, tbl, result);
    if((rc = check(hipGetLastError())))
        return rc;
    hipLaunchKernelGGL(k_stamp, dim3(1), dim3(1), 0, s, counter, stamp);
    return check(hipGetLastError());
}
}  // namespace gfk
