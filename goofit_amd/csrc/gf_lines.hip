// gf_lines.hip -- gfx950 kernels that evaluate the resonance lineshapes.
//
//  * k_dalitz_cache: the resonance lineshape cache W_i[e]
//    (src/PDFs/physics/Amp3Body.cu:292-310, detail/SpecialResonanceCalculator.cu:12-46).
//  * k_gram: the per-amplitude normalisation integrals as one FP64-MFMA Gram
//    A^H diag(eff*w) A over grid cells, phase-space points or the data cache
//    (src/PDFs/physics/Amp3Body.cu:312-330 and 376-428,
//    detail/SpecialResonanceIntegrator.cu:7-121).
//  * k_dalitz_candidates / k_compact: accept-reject generation from an Amp3Body.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gf_interp.h"

namespace {

// ------------------------------------------------------------- Dalitz cache

// The numbers of a plan kept on the device, one lane per term.
__global__ __launch_bounds__(GF_MAX_TERMS) void k_line_plan(GfLinePlan *plan, const double *__restrict__ P, GfDecay d) {
    gfd::line_plan_term(*plan, threadIdx.x, P, d);
}

// The wave cache (ALL: every resonance of the plan).  16 shapes over 1e6 events: 59 us on
// average, 1045 vector instructions per wave of 64 events (29 us of issue) beside 256 MB of
// stores (40 us at the fill rate); 290 us with each shape evaluated by itself.
template <bool ALL, class Plan>
__global__ __launch_bounds__(256) void k_dalitz_cache(GfProgArgs A, int slot, int64_t offset, int64_t n, uint32_t mask,
                                                      const Plan plan) {
    const GfDalitzSlot dz = gfd::as_const(A.dz)[slot];
    const GfDecay D       = A.decay;
    double2 *wave         = const_cast<double2 *>(dz.wave);
    double2 *wave_b       = const_cast<double2 *>(dz.wave_b);  // time-dependent nodes only
    const double *c12     = A.cols[dz.col_m12];
    const double *c13     = A.cols[dz.col_m13];
    for(int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
        const double m12  = c12[offset + e];
        const double m13  = c13[offset + e];
        const bool inside = gfd::in_dalitz(m12, m13, D.motherMass, D.daug1Mass, D.daug2Mass, D.daug3Mass);
        // SpecialResonanceCalculator.cu:36-37; the B wave is at the reversed point with the
        // same m23 (SpecialWaveCalculator.cu:55-58)
        const double m23 = D.motherMass * D.motherMass + D.daug1Mass * D.daug1Mass + D.daug2Mass * D.daug2Mass
                           + D.daug3Mass * D.daug3Mass - m12 - m13;
        gfd::line_waves<ALL>(gfd::plan_at(plan), m12, m13, m23, mask, [&](int i, int swap, int add, double2 v) {
            double2 *w = (swap ? wave_b : wave) + (int64_t)i * dz.ncache + e;
            if(add) {
                v.x += w->x;
                v.y += w->y;
            }
            *w = make_double2(inside ? v.x : 0.0, inside ? v.y : 0.0);
        });
    }
}

// ------------------------------------------------------------- event generation

// Accept-reject generation from an Amp3Body: candidate i of the counter-based stream is
// uniform in the box; its value is |sum_r c_r B_r(m12, m13)|^2 * eff (0 outside the Dalitz
// plot, as device_DalitzPlot, Amp3Body.cu:60-122, with lineshapes computed directly);
// accepted when u_i * fmax < value.

__device__ __forceinline__ void gen_point(const GfGenBox &B, uint64_t key, uint64_t i, double &m12, double &m13) {
    m12 = B.l12 + gfd::unif01(key, 2 * i) * (B.u12 - B.l12);
    m13 = B.l13 + gfd::unif01(key, 2 * i + 1) * (B.u13 - B.l13);
}

// One workgroup takes GF_GEN_BLOCK candidates: all its lanes draw and test them against
// the plot, the points inside (about half of a box around it) are gathered in LDS, and
// only those are evaluated, on full waves -- the lineshapes are nine tenths of the work.
// Out: the accepted candidates as bits, their number and the largest value (to check the
// envelope).  Nothing is done once st->have has reached limit.  A pass of 2^22 candidates
// with 16 shapes: 130 us; 208 us with every candidate evaluated in its own lane.
template <bool GEN_EFF, class Plan>
__global__ __launch_bounds__(256) void k_dalitz_candidates(GfProgArgs A, const Plan plan,
                                                           int p_coup, int eff_pc, double eff_const, int id12,
                                                           int id13, GfGenBox B, uint64_t key, int64_t base,
                                                           const GfGenState *__restrict__ st, int64_t limit,
                                                           uint32_t *__restrict__ bits, int *__restrict__ bcount,
                                                           double *__restrict__ bmax) {
    __shared__ double x12[GF_GEN_BLOCK], x13[GF_GEN_BLOCK];
    __shared__ uint16_t at[GF_GEN_BLOCK];
    __shared__ uint32_t word[GF_GEN_BLOCK / 32];
    __shared__ int inside_n, scount[4];
    __shared__ double smax[4];
    if(st->have >= limit)
        return;  // uniform over the launch
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const GfDecay D    = A.decay;
    const double fmax  = st->fmax;
    const int64_t base0 = base + (int64_t)blockIdx.x * GF_GEN_BLOCK;
    if(t == 0)
        inside_n = 0;
    if(t < GF_GEN_BLOCK / 32)
        word[t] = 0;
    __syncthreads();
    for(int j = t; j < GF_GEN_BLOCK; j += 256) {
        double m12, m13;
        gen_point(B, key, (uint64_t)(base0 + j), m12, m13);
        const bool in = gfd::in_dalitz(m12, m13, D.motherMass, D.daug1Mass, D.daug2Mass, D.daug3Mass);
        const unsigned long long ball = __ballot(in);
        int first = 0;
        if(lane == 0)
            first = atomicAdd(&inside_n, __popcll(ball));
        first = __shfl(first, 0, 64);
        if(in) {  // in any order: what follows does not depend on it
            const int k = first + __popcll(ball & ((1ull << lane) - 1ull));
            x12[k] = m12;
            x13[k] = m13;
            at[k]  = (uint16_t)j;
        }
    }
    __syncthreads();
    const int n = inside_n;
    const GF_CONST double *__restrict__ P = gfd::as_const(A.params) + p_coup;
    double vm   = 0.0;
    int count   = 0;
    for(int k = t; k < n; k += 256) {
        const double m12 = x12[k], m13 = x13[k];
        const double m23 = D.motherMass * D.motherMass + D.daug1Mass * D.daug1Mass + D.daug2Mass * D.daug2Mass
                           + D.daug3Mass * D.daug3Mass - m12 - m13;
        double re = 0.0, im = 0.0;
        gfd::line_waves<true>(gfd::plan_at(plan), m12, m13, m23, ~0u, [&](int r, int, int, double2 b) {
            const double ar = P[2 * r], ai = P[2 * r + 1];
            re = fma(ar, b.x, fma(-ai, b.y, re));
            im = fma(ar, b.y, fma(ai, b.x, im));
        });
        double eff = eff_pc == -2 ? eff_const : 1.0;
        if constexpr(GEN_EFF) {
            RegSrc<1> ev;
#pragma unroll
            for(int o = 0; o < GF_MAX_OBS; ++o)
                ev.v[0][o] = 0.0;
            ev.set(id12, 0, m12);
            ev.set(id13, 0, m13);
            const int64_t r0[1] = {0};
            const bool v0[1]    = {true};
            double T[1];
            run<1>(A, A.params, A.norms, eff_pc, ev, r0, v0, T);
            eff = T[0];
        }
        const double value = (re * re + im * im) * eff;
        vm                 = ::fmax(vm, value);
        const int j        = at[k];
        if(gfd::unif01(key ^ 0xD1B54A32D192ED03ull, (uint64_t)(base0 + j)) * fmax < value) {
            atomicOr(&word[j >> 5], 1u << (j & 31));
            ++count;
        }
    }
    for(int off = 32; off > 0; off >>= 1) {
        vm = ::fmax(vm, __shfl_xor(vm, off, 64));
        count += __shfl_xor(count, off, 64);
    }
    if(lane == 0) {
        scount[wave] = count;
        smax[wave]   = vm;
    }
    __syncthreads();
    if(t < GF_GEN_BLOCK / 32)
        bits[(int64_t)blockIdx.x * (GF_GEN_BLOCK / 32) + t] = word[t];
    if(t == 0) {
        for(int w = 1; w < 4; ++w) {
            count += scount[w];
            vm = ::fmax(vm, smax[w]);
        }
        bcount[blockIdx.x] = count;
        bmax[blockIdx.x]   = vm;
    }
}

// One workgroup after a pass: its largest value and accepted count into *out (host-mapped),
// and the state of the next one.  GF_GEN_ENVELOPE: the pass sets the envelope, 1.25 x its
// largest value; otherwise boff[b] = the row of block b's first accepted candidate.
// nblk 0: no pass, the envelope is `value`.
__global__ __launch_bounds__(1024) void k_gen_scan(int envelope, double value, const int *__restrict__ bcount,
                                                   const double *__restrict__ bmax, int nblk, int64_t limit,
                                                   int64_t *__restrict__ boff, GfGenState *st, GfGenPass *out) {
    __shared__ int64_t wsum[16];
    __shared__ double wmax[16];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if(nblk == 0) {
        if(t == 0) {
            st->fmax = value;
            st->have = 0;
        }
        return;
    }
    const int64_t have = st->have;
    const int per = (nblk + 1023) / 1024, b0 = t * per, b1 = min(nblk, b0 + per);
    if(have >= limit) {  // the pass did nothing and has no rows to write
        for(int b = b0; b < b1 && !envelope; ++b)
            boff[b] = limit;
        if(t == 0)
            out->count = 0, out->mx = 0.0;
        return;
    }
    int64_t sum = 0;
    double m    = 0.0;
    for(int b = b0; b < b1; ++b) {
        sum += bcount[b];
        m = ::fmax(m, bmax[b]);
    }
    int64_t incl = sum;  // inclusive scan over the wave
    for(int off = 1; off < 64; off <<= 1) {
        const int64_t v = __shfl_up(incl, off, 64);
        if(lane >= off)
            incl += v;
    }
    for(int off = 32; off > 0; off >>= 1)
        m = ::fmax(m, __shfl_xor(m, off, 64));
    if(lane == 63)
        wsum[wave] = incl;
    if(lane == 0)
        wmax[wave] = m;
    __syncthreads();
    int64_t before = have, total = 0;
    for(int w = 0; w < 16; ++w) {
        if(w < wave)
            before += wsum[w];
        total += wsum[w];
        m = ::fmax(m, wmax[w]);
    }
    int64_t row = before + incl - sum;
    for(int b = b0; b < b1; ++b) {
        boff[b] = row;
        row += bcount[b];
    }
    if(t == 0) {
        out->count = total;
        out->mx    = m;
        if(envelope)
            st->fmax = 1.25 * m;
        else
            st->have = have + total;
    }
}

// Write a pass's accepted candidates in the stream's order: block b's to boff[b] + their
// rank in the block; rows >= limit are dropped.  The points are drawn again from their
// counters (a few in a hundred candidates) instead of kept for every candidate.
__global__ __launch_bounds__(256) void k_compact(const uint32_t *__restrict__ bits, GfGenBox B, uint64_t key,
                                                 int64_t base, const int64_t *__restrict__ boff, int64_t limit,
                                                 double *__restrict__ o12, double *__restrict__ o13) {
    static_assert(GF_GEN_BLOCK == 256 * 8, "a byte of the mask per lane");
    __shared__ int wcount[4];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    uint32_t m   = (bits[(int64_t)blockIdx.x * (GF_GEN_BLOCK / 32) + (t >> 2)] >> (8 * (t & 3))) & 0xFFu;
    const int c  = __popc(m);
    int incl     = c;
    for(int off = 1; off < 64; off <<= 1) {
        const int v = __shfl_up(incl, off, 64);
        if(lane >= off)
            incl += v;
    }
    if(lane == 63)
        wcount[wave] = incl;
    __syncthreads();
    int64_t dst = boff[blockIdx.x] + incl - c;
    for(int w = 0; w < wave; ++w)
        dst += wcount[w];
    const int64_t i0 = base + (int64_t)blockIdx.x * GF_GEN_BLOCK + 8 * t;
    for(; m && dst < limit; m &= m - 1, ++dst) {
        double m12, m13;
        gen_point(B, key, (uint64_t)(i0 + __ffs(m) - 1), m12, m13);
        o12[dst] = m12;
        o13[dst] = m13;
    }
}

// ------------------------------------------------------------- FP64-MFMA Gram


#define GG_LD 65  // padded LDS row (doubles): 16 lanes reading one column hit distinct banks

struct GramSrc {
    int mode;  // 0 grid, 1 points, 2 data cache
    double l12, u12, l13, u13;
    int n12, n13;
    const double *m12, *m13, *w;
    int64_t npoints;
    int slot;          // mode 2
    int id_m12, id_m13;
    int eff_pc;        // >= 0: efficiency subprogram; -1: efficiency 1; -2: constant eff_const
    double eff_const;
    int td;            // grid of a time-dependent node: m13 bin count n13 (SpecialDalitzIntegrator.cu:75-82)
};

// Centre (m12, m13) of integration cell p of a Dalitz grid (SpecialResonanceIntegrator.cu:61-76:
// m12 fastest; the m13 bin count is read from the m12 entry there, numBinsM13 = numBinsM12,
// reproduced here; a time-dependent node's integrator reads its own m13 count,
// SpecialDalitzIntegrator.cu:75-82).  The cell index is an int there, as here.
__device__ __forceinline__ void dalitz_cell(const GramSrc &S, int64_t p, double &m12, double &m13) {
    int globalBinNumber  = (int)p;
    const int numBinsM12 = S.n12;
    const int binM12     = globalBinNumber % numBinsM12;
    m12                  = gfd::bin_centre(S.l12, S.u12, numBinsM12, binM12);
    globalBinNumber /= numBinsM12;
    const int numBinsM13 = S.td ? S.n13 : S.n12;
    m13                  = gfd::bin_centre(S.l13, S.u13, numBinsM13, globalBinNumber);
}

// The centres of the first npoints cells of the grid in S (mode 0).
__global__ __launch_bounds__(256) void k_dalitz_cells(GramSrc S, double *m12, double *m13) {
    for(int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < S.npoints; p += (int64_t)gridDim.x * blockDim.x)
        dalitz_cell(S, p, m12[p], m13[p]);
}

// Each wave takes 64 points at a time, on its own: a lane computes the 16 complex
// amplitudes of its point (wave-uniform control flow) and stages them in the wave's LDS
// rows component-major, then the wave multiplies its 64 points as 16 MFMA k-steps for
// each of three 16x16 output tiles: RR = R^T E R, II = I^T E I, RI = R^T E I, with
// E = diag(eff * weight).  No barrier until the four waves' tiles are added at the end.
// A point outside the Dalitz plot adds nothing, so a wave with none inside moves on (two
// fifths of the waves over a box around the plot).  16 shapes on 1414 x 1414 cells: 116 us
// (40 us of vector and 24 us of matrix-core issue; the 16.5 KB of LDS per wave leave two
// waves per SIMD, so latency shows), 450-520 us with each shape evaluated by itself over
// every cell.  Partials: 3 tiles x 64 lanes x 4 values per block.
template <bool GEN_EFF, class Plan>
__global__ __launch_bounds__(GG_BLOCK) __attribute__((amdgpu_waves_per_eu(2))) void k_gram(
    GfProgArgs A, GramSrc S, const Plan plan, int nres, double *partials) {
    __shared__ double Xr[GG_BLOCK / 64][16][GG_LD];
    __shared__ double Xi[GG_BLOCK / 64][16][GG_LD];
    __shared__ double Ew[GG_BLOCK / 64][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const GfDecay D = A.decay;
    gf_double4 RR = {0, 0, 0, 0}, II = {0, 0, 0, 0}, RI = {0, 0, 0, 0};
    const int64_t npts = S.npoints;
    for(int i = 0; i < 16; ++i)  // rows past nres stay 0
        Xr[wave][i][lane] = Xi[wave][i][lane] = 0.0;
    for(int64_t base = (int64_t)blockIdx.x * GG_BLOCK + 64 * wave; base < npts;
        base += (int64_t)gridDim.x * GG_BLOCK) {
        const int64_t p  = base + lane;
        const bool valid = p < npts;
        double ew = 0.0;
        if(S.mode == 2) {
            const GfDalitzSlot dz = A.dz[S.slot];
            const int64_t q       = valid ? p : 0;
            for(int i = 0; i < nres; ++i) {
                const double2 b   = dz.wave[(int64_t)i * dz.ncache + q];
                Xr[wave][i][lane] = b.x;
                Xi[wave][i][lane] = b.y;
            }
            ew = valid ? 1.0 : 0.0;
        } else {
            double m12 = 0.0, m13 = 0.0, wt = 1.0;
            if(S.mode == 0) {
                dalitz_cell(S, valid ? p : 0, m12, m13);
            } else {
                m12 = valid ? S.m12[p] : 0.0;
                m13 = valid ? S.m13[p] : 0.0;
                wt  = (valid && S.w) ? S.w[p] : 1.0;
            }
            const bool inside = valid && gfd::in_dalitz(m12, m13, D.motherMass, D.daug1Mass, D.daug2Mass, D.daug3Mass);
            if(!__any(inside))
                continue;
            const double m23  = D.motherMass * D.motherMass + D.daug1Mass * D.daug1Mass + D.daug2Mass * D.daug2Mass
                               + D.daug3Mass * D.daug3Mass - m12 - m13;
            gfd::line_waves<true>(gfd::plan_at(plan), m12, m13, m23, ~0u, [&](int i, int, int add, double2 b) {
                if(add) {
                    b.x += Xr[wave][i][lane];
                    b.y += Xi[wave][i][lane];
                }
                Xr[wave][i][lane] = inside ? b.x : 0.0;
                Xi[wave][i][lane] = inside ? b.y : 0.0;
            });
            double eff = S.eff_pc == -2 ? S.eff_const : 1.0;
            if constexpr(GEN_EFF) {
                // The fake event of SpecialResonanceIntegrator.cu:97-101: slot 0 = 2,
                // then m12 and m13 at their observable slots; other slots 0.
                RegSrc<1> ev;
#pragma unroll
                for(int o = 0; o < GF_MAX_OBS; ++o)
                    ev.v[0][o] = 0.0;
                ev.v[0][0] = 2.0;
                ev.set(S.id_m12, 0, m12);
                ev.set(S.id_m13, 0, m13);
                const int64_t r0[1] = {0};
                const bool v0[1]    = {true};
                double T[1];
                run<1>(A, A.params, A.norms, S.eff_pc, ev, r0, v0, T);
                eff = T[0];
            }
            ew = inside ? eff * wt : 0.0;
        }
        Ew[wave][lane] = ew;
        // the wave's own LDS rows: its LDS operations complete in order, the fences keep the
        // compiler from moving them across
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // A operand lane l: A[i = l%16][k = l/16]; B operand lane l: B[k = l/16][j = l%16].
        const int comp = lane & 15, sub = lane >> 4;
#pragma unroll
        for(int kk = 0; kk < 16; ++kk) {
            const int pt    = 4 * kk + sub;
            const double ar = Xr[wave][comp][pt];
            const double ai = Xi[wave][comp][pt];
            const double e  = Ew[wave][pt];
            const double br = e * ar, bi = e * ai;
            RR = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, br, RR, 0, 0, 0);
            II = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, bi, II, 0, 0, 0);
            RI = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, bi, RI, 0, 0, 0);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    // add the waves' tiles in order through LDS, then write this block's partial
    __syncthreads();
    double *stage = &Xr[0][0][0];  // 4 * 16 * 65 doubles >= 3 * 768
    if(wave > 0) {
        double *mine = stage + (wave - 1) * 768;
#pragma unroll
        for(int r = 0; r < 4; ++r) {
            mine[(0 * 4 + r) * 64 + lane] = RR[r];
            mine[(1 * 4 + r) * 64 + lane] = II[r];
            mine[(2 * 4 + r) * 64 + lane] = RI[r];
        }
    }
    __syncthreads();
    if(wave == 0) {
        double *out = partials + (int64_t)blockIdx.x * 768;
#pragma unroll
        for(int r = 0; r < 4; ++r) {
            double t[3] = {RR[r], II[r], RI[r]};
#pragma unroll
            for(int q = 0; q < 3; ++q) {
                for(int w = 0; w < GG_BLOCK / 64 - 1; ++w)
                    t[q] += stage[w * 768 + (q * 4 + r) * 64 + lane];
                out[(q * 4 + r) * 64 + lane] = t[q];
            }
        }
    }
}

// Sum the per-block Gram partials: a workgroup takes 8 output elements (64 bytes of each
// block's row), 32 lanes each with a fixed stride of blocks, then the lanes' sums in order
// (deterministic for a given grid).
__global__ __launch_bounds__(256) void k_gram_final(const double *__restrict__ partials, int nblocks, double *out) {
    __shared__ double ls[32][8], lc[32][8];
    const int e = threadIdx.x & 7, row = threadIdx.x >> 3;
    double s = 0.0, c = 0.0;
#pragma unroll 4
    for(int b = row; b < nblocks; b += 32)
        gfd::kb_add(s, c, partials[(int64_t)b * 768 + 8 * blockIdx.x + e]);
    ls[row][e] = s;
    lc[row][e] = c;
    __syncthreads();
    if(row == 0) {
        for(int k = 1; k < 32; ++k)
            gfd::kb_merge(s, c, ls[k][e], lc[k][e]);
        out[8 * blockIdx.x + e] = gfd::kb_total(s, c);
    }
}

}  // namespace

namespace gfk {

int launch_line_plan(const GfProgArgs &a, const GfLinePlanRef &plan, void *stream) {
    if(plan.arg)
        return 0;
    hipLaunchKernelGGL(k_line_plan, dim3(1), dim3(GF_MAX_TERMS), 0, (hipStream_t)stream, plan.dev, a.params, a.decay);
    return check(hipGetLastError());
}

// f(plan) with the plan in the form in which the kernels take it.
template <class F>
static void with_plan(const GfLinePlanRef &plan, const F &f) {
    if(plan.arg)
        f(*plan.arg);
    else
        f((const GfLinePlan *)plan.dev);
}

int launch_dalitz_candidates(const GfProgArgs &a, const GfLinePlanRef &plan, int p_coup, int eff_pc, double eff_const,
                             int id12, int id13, const GfGenBox &box, uint64_t key, int64_t base, int nblocks,
                             const GfGenState *st, int64_t limit, uint32_t *bits, int *bcount, double *bmax,
                             void *stream) {
    with_plan(plan, [&](const auto &p) {
        using Plan = std::decay_t<decltype(p)>;
        if(eff_pc >= 0)
            hipLaunchKernelGGL((k_dalitz_candidates<true, Plan>), dim3(nblocks), dim3(256), 0, (hipStream_t)stream, a, p,
                               p_coup, eff_pc, eff_const, id12, id13, box, key, base, st, limit, bits, bcount, bmax);
        else
            hipLaunchKernelGGL((k_dalitz_candidates<false, Plan>), dim3(nblocks), dim3(256), 0, (hipStream_t)stream, a, p,
                               p_coup, eff_pc, eff_const, id12, id13, box, key, base, st, limit, bits, bcount, bmax);
    });
    return check(hipGetLastError());
}

int launch_gen_scan(bool envelope, double value, const int *bcount, const double *bmax, int nblocks, int64_t limit,
                    int64_t *boff, GfGenState *st, GfGenPass *out, void *stream) {
    hipLaunchKernelGGL(k_gen_scan, dim3(1), dim3(1024), 0, (hipStream_t)stream, envelope ? 1 : 0, value, bcount, bmax,
                       nblocks, limit, boff, st, out);
    return check(hipGetLastError());
}

int launch_compact(const uint32_t *bits, const GfGenBox &box, uint64_t key, int64_t base, int nblocks,
                   const int64_t *boff, int64_t limit, double *o12, double *o13, void *stream) {
    hipLaunchKernelGGL(k_compact, dim3(nblocks), dim3(256), 0, (hipStream_t)stream, bits, box, key, base, boff, limit,
                       o12, o13);
    return check(hipGetLastError());
}

int launch_dalitz_cache(const GfProgArgs &a, int slot, int64_t offset, int64_t n, uint32_t mask, bool all,
                        const GfLinePlanRef &plan, int nblocks, void *stream) {
    hipStream_t s = (hipStream_t)stream;
    const dim3 g(nblocks), b(256);
    const GfLinePlan *dev = plan.dev;
    const int rc          = launch_line_plan(a, plan, stream);
    if(rc)
        return rc;
    if(plan.arg)
        hipLaunchKernelGGL((k_dalitz_cache<true, GfLinePlanArg>), g, b, 0, s, a, slot, offset, n, mask, *plan.arg);
    else if(all)
        hipLaunchKernelGGL((k_dalitz_cache<true, const GfLinePlan *>), g, b, 0, s, a, slot, offset, n, mask, dev);
    else
        hipLaunchKernelGGL((k_dalitz_cache<false, const GfLinePlan *>), g, b, 0, s, a, slot, offset, n, mask, dev);
    return check(hipGetLastError());
}

int launch_gram(const GfProgArgs &a, int mode, const double *grid6, const double *m12, const double *m13,
                const double *w, int64_t npoints, int slot, int id_m12, int id_m13, int eff_pc, double eff_const,
                int td_grid, const GfLinePlanRef &plan, int nres, double *partials, double *tiles_dev, int nblocks,
                void *stream) {
    GramSrc S;
    S.mode = mode;
    S.td   = td_grid;
    S.l12 = S.u12 = S.l13 = S.u13 = 0.0;
    S.n12 = S.n13 = 1;
    if(grid6) {
        S.l12 = grid6[0];
        S.u12 = grid6[1];
        S.n12 = (int)floor(grid6[2] + 0.5);
        S.l13 = grid6[3];
        S.u13 = grid6[4];
        S.n13 = (int)floor(grid6[5] + 0.5);
    }
    S.m12     = m12;
    S.m13     = m13;
    S.w       = w;
    S.npoints = npoints;
    S.slot    = slot;
    S.id_m12  = id_m12;
    S.id_m13  = id_m13;
    S.eff_pc    = eff_pc;
    S.eff_const = eff_const;
    hipStream_t s = (hipStream_t)stream;
    int rc = mode == 2 ? 0 : launch_line_plan(a, plan, s);
    if(rc)
        return rc;
    with_plan(plan, [&](const auto &p) {
        using Plan = std::decay_t<decltype(p)>;
        if(eff_pc >= 0)
            hipLaunchKernelGGL((k_gram<true, Plan>), dim3(nblocks), dim3(GG_BLOCK), 0, s, a, S, p, nres, partials);
        else
            hipLaunchKernelGGL((k_gram<false, Plan>), dim3(nblocks), dim3(GG_BLOCK), 0, s, a, S, p, nres, partials);
    });
    if((rc = check(hipGetLastError())))
        return rc;
    hipLaunchKernelGGL(k_gram_final, dim3(768 / 8), dim3(256), 0, s, partials, nblocks, tiles_dev);
    return check(hipGetLastError());
}

int launch_dalitz_cells(const double *grid6, int td_grid, int64_t ncells, double *m12, double *m13, void *stream) {
    GramSrc S{};
    S.mode    = 0;
    S.td      = td_grid;
    S.l12     = grid6[0];
    S.u12     = grid6[1];
    S.n12     = (int)floor(grid6[2] + 0.5);
    S.l13     = grid6[3];
    S.u13     = grid6[4];
    S.n13     = (int)floor(grid6[5] + 0.5);
    S.npoints = ncells;
    hipLaunchKernelGGL(k_dalitz_cells, dim3(cell_blocks(ncells)), dim3(256), 0, (hipStream_t)stream, S, m12, m13);
    return check(hipGetLastError());
}
}  // namespace gfk
