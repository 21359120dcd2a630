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

#include "gf_interp.h"

namespace {

// ------------------------------------------------------------- Dalitz cache

__global__ __launch_bounds__(256) void k_dalitz_cache(GfProgArgs A, int slot, int64_t offset, int64_t n,
                                                      uint32_t mask, const GfResDesc *__restrict__ res, int nres) {
    const GfDalitzSlot dz = A.dz[slot];
    const GfDecay D       = A.decay;
    double2 *wave         = const_cast<double2 *>(dz.wave);
    double2 *wave_b       = const_cast<double2 *>(dz.wave_b);  // time-dependent nodes only
    const double *c12     = A.cols[dz.col_m12];
    const double *c13     = A.cols[dz.col_m13];
    for(int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
        const double m12  = c12[offset + e];
        const double m13  = c13[offset + e];
        const bool inside = gfd::in_dalitz(m12, m13, D.motherMass, D.daug1Mass, D.daug2Mass, D.daug3Mass);
        // SpecialResonanceCalculator.cu:36-37
        const double m23 = D.motherMass * D.motherMass + D.daug1Mass * D.daug1Mass + D.daug2Mass * D.daug2Mass
                           + D.daug3Mass * D.daug3Mass - m12 - m13;
        for(int i = 0; i < nres; ++i) {
            if(!((mask >> i) & 1u))
                continue;
            double2 w = make_double2(0.0, 0.0);
            if(inside)
                w = gfd::lineshape(res[i], A.params, A.consts, D, m12, m13, m23);
            wave[(int64_t)i * dz.ncache + e] = w;
            if(wave_b) {
                // SpecialWaveCalculator.cu:55-58: the B wave at the reversed point, same m23
                double2 v = make_double2(0.0, 0.0);
                if(inside)
                    v = gfd::lineshape(res[i], A.params, A.consts, D, m13, m12, m23);
                wave_b[(int64_t)i * dz.ncache + e] = v;
            }
        }
    }
}

// ------------------------------------------------------------- event generation

// Candidates for accept-reject generation from an Amp3Body: point i of the
// counter-based stream is uniform in the box; its value is
// |sum_r c_r B_r(m12, m13)|^2 * eff (0 outside the Dalitz plot, as
// device_DalitzPlot, Amp3Body.cu:60-122, with lineshapes computed directly);
// accepted when u_i * fmax < value.  Per block: accepted count and the largest
// value (to check the envelope).
template <bool GEN_EFF>
__global__ __launch_bounds__(256) void k_dalitz_candidates(GfProgArgs A, const GfResDesc *__restrict__ res, int nres,
                                                           int p_coup, int eff_pc, double eff_const, int id12,
                                                           int id13, double l12,
                                                           double u12, double l13, double u13, uint64_t key,
                                                           int64_t base, int64_t nc, double fmax,
                                                           double *__restrict__ c12, double *__restrict__ c13,
                                                           uint8_t *__restrict__ flag, int *__restrict__ bcount,
                                                           double *__restrict__ bmax) {
    __shared__ int scount[4];
    __shared__ double smax[4];
    const int64_t i   = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid  = i < nc;
    const GfDecay D   = A.decay;
    const uint64_t ct = (uint64_t)(base + (valid ? i : 0));
    const double m12  = l12 + gfd::unif01(key, 2 * ct) * (u12 - l12);
    const double m13  = l13 + gfd::unif01(key, 2 * ct + 1) * (u13 - l13);
    double value      = 0.0;
    if(valid && gfd::in_dalitz(m12, m13, D.motherMass, D.daug1Mass, D.daug2Mass, D.daug3Mass)) {
        const double m23 = D.motherMass * D.motherMass + D.daug1Mass * D.daug1Mass + D.daug2Mass * D.daug2Mass
                           + D.daug3Mass * D.daug3Mass - m12 - m13;
        double re = 0.0, im = 0.0;
#pragma unroll 1
        for(int r = 0; r < nres; ++r) {
            const double2 b = gfd::lineshape(res[r], A.params, A.consts, D, m12, m13, m23);
            const double ar = A.params[p_coup + 2 * r], ai = A.params[p_coup + 2 * r + 1];
            re += ar * b.x - ai * b.y;
            im += ar * b.y + ai * b.x;
        }
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
        value = (re * re + im * im) * eff;
    }
    const bool acc = valid && gfd::unif01(key ^ 0xD1B54A32D192ED03ull, ct) * fmax < value;
    if(valid) {
        c12[i]  = m12;
        c13[i]  = m13;
        flag[i] = acc ? 1 : 0;
    }
    // block totals: count of accepted, largest value
    const unsigned long long ball = __ballot(acc);
    double vm = value;
    for(int off = 32; off > 0; off >>= 1)
        vm = ::fmax(vm, __shfl_xor(vm, off, 64));
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if(lane == 0) {
        scount[wave] = __popcll(ball);
        smax[wave]   = vm;
    }
    __syncthreads();
    if(threadIdx.x == 0) {
        int c    = 0;
        double m = 0.0;
        for(int w = 0; w < 4; ++w) {
            c += scount[w];
            m = ::fmax(m, smax[w]);
        }
        bcount[blockIdx.x] = c;
        bmax[blockIdx.x]   = m;
    }
}

// Write the accepted candidates in order: block b's go to boff[b] + their rank
// in the block (waves in order, lanes in order); rows >= limit are dropped.
__global__ __launch_bounds__(256) void k_compact(const double *__restrict__ c12, const double *__restrict__ c13,
                                                 const uint8_t *__restrict__ flag, int64_t nc,
                                                 const int64_t *__restrict__ boff, int64_t limit,
                                                 double *__restrict__ o12, double *__restrict__ o13) {
    __shared__ int wcount[4];
    const int64_t i  = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool acc   = i < nc && flag[i];
    const unsigned long long ball = __ballot(acc);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if(lane == 0)
        wcount[wave] = __popcll(ball);
    __syncthreads();
    int before = 0;
    for(int w = 0; w < wave; ++w)
        before += wcount[w];
    const unsigned long long lower = lane ? (ball & ((1ull << lane) - 1ull)) : 0ull;
    const int64_t dst = boff[blockIdx.x] + before + __popcll(lower);
    if(acc && dst < limit) {
        o12[dst] = c12[i];
        o13[dst] = c13[i];
    }
}

// ------------------------------------------------------------- FP64-MFMA Gram


#define GG_BLOCK 128  // two waves
#define GG_LD 65      // padded LDS row (doubles): 16 lanes reading one column hit distinct banks

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

// One block: 128 points per pass; each lane computes the 16 complex amplitudes of
// its point (wave-uniform control flow), stages them in LDS component-major,
// and each wave multiplies its 64 points as 16 MFMA k-steps for each of three
// 16x16 output tiles: RR = R^T E R, II = I^T E I, RI = R^T E I, with
// E = diag(eff * weight).  Partials: 3 tiles x 64 lanes x 4 values per block.
template <bool GEN_EFF>
__global__ __launch_bounds__(GG_BLOCK) void k_gram(GfProgArgs A, GramSrc S, const GfResDesc *__restrict__ res,
                                                   int nres, double *partials) {
    __shared__ double Xr[2][16][GG_LD];
    __shared__ double Xi[2][16][GG_LD];
    __shared__ double Ew[2][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const GfDecay D = A.decay;
    gf_double4 RR = {0, 0, 0, 0}, II = {0, 0, 0, 0}, RI = {0, 0, 0, 0};
    const int64_t npts = S.npoints;
    for(int64_t base = (int64_t)blockIdx.x * GG_BLOCK; base < npts; base += (int64_t)gridDim.x * GG_BLOCK) {
        const int64_t p  = base + tid;
        const bool valid = p < npts;
        double m12 = 0.0, m13 = 0.0, wt = 1.0;
        if(S.mode == 0) {
            dalitz_cell(S, valid ? p : 0, m12, m13);
        } else if(S.mode == 1) {
            m12 = valid ? S.m12[p] : 0.0;
            m13 = valid ? S.m13[p] : 0.0;
            wt  = (valid && S.w) ? S.w[p] : 1.0;
        }
        double ew = 0.0;
        if(S.mode == 2) {
            const GfDalitzSlot dz = A.dz[S.slot];
            const int64_t q       = valid ? p : 0;
            for(int i = 0; i < GF_MAX_RES; ++i) {
                double2 b = (i < nres) ? dz.wave[(int64_t)i * dz.ncache + q] : make_double2(0.0, 0.0);
                Xr[wave][i][lane] = b.x;
                Xi[wave][i][lane] = b.y;
            }
            ew = valid ? 1.0 : 0.0;
        } else {
            const bool inside = valid && gfd::in_dalitz(m12, m13, D.motherMass, D.daug1Mass, D.daug2Mass, D.daug3Mass);
            const double m23  = D.motherMass * D.motherMass + D.daug1Mass * D.daug1Mass + D.daug2Mass * D.daug2Mass
                               + D.daug3Mass * D.daug3Mass - m12 - m13;
            // one lineshape body in the loop (not 16 inlined copies): registers for occupancy
#pragma unroll 1
            for(int i = 0; i < GF_MAX_RES; ++i) {
                double2 b = make_double2(0.0, 0.0);
                if(i < nres && inside) {
                    const bool sw = res[i].swap != 0;  // B wave of a time-dependent node
                    b = gfd::lineshape(res[i], A.params, A.consts, D, sw ? m13 : m12, sw ? m12 : m13, m23);
                }
                Xr[wave][i][lane] = b.x;
                Xi[wave][i][lane] = b.y;
            }
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
            ew = valid ? eff * wt : 0.0;
        }
        Ew[wave][lane] = ew;
        __syncthreads();
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
        __syncthreads();
    }
    // add wave 1 into wave 0 through LDS, then write this block's partial
    double *stage = &Xr[0][0][0];  // 2*16*65 doubles >= 64*12
    if(wave == 1) {
#pragma unroll
        for(int r = 0; r < 4; ++r) {
            stage[(0 * 4 + r) * 64 + lane] = RR[r];
            stage[(1 * 4 + r) * 64 + lane] = II[r];
            stage[(2 * 4 + r) * 64 + lane] = RI[r];
        }
    }
    __syncthreads();
    if(wave == 0) {
        double *out = partials + (int64_t)blockIdx.x * 768;
#pragma unroll
        for(int r = 0; r < 4; ++r) {
            out[(0 * 4 + r) * 64 + lane] = RR[r] + stage[(0 * 4 + r) * 64 + lane];
            out[(1 * 4 + r) * 64 + lane] = II[r] + stage[(1 * 4 + r) * 64 + lane];
            out[(2 * 4 + r) * 64 + lane] = RI[r] + stage[(2 * 4 + r) * 64 + lane];
        }
    }
}

// Sum the per-block Gram partials: one block per output element, each thread a
// fixed stride of blocks, then a fixed-order tree (deterministic for a given grid).
__global__ __launch_bounds__(256) void k_gram_final(const double *__restrict__ partials, int nblocks, double *out) {
    const int e = blockIdx.x;  // 0..767
    double s = 0.0, c = 0.0;
    for(int b = threadIdx.x; b < nblocks; b += blockDim.x)
        gfd::kb_add(s, c, partials[(int64_t)b * 768 + e]);
    block_reduce(s, c);
    if(threadIdx.x == 0)
        out[e] = gfd::kb_total(s, c);
}

}  // namespace

namespace gfk {

int launch_dalitz_candidates(const GfProgArgs &a, const GfResDesc *res, int nres, int p_coup, int eff_pc,
                             double eff_const, int id12, int id13, const double box[4], uint64_t key, int64_t base,
                             int64_t nc, double fmax, double *c12, double *c13, uint8_t *flag, int *bcount,
                             double *bmax, void *stream) {
    const int nb = (int)((nc + 255) / 256);
    if(eff_pc >= 0)
        hipLaunchKernelGGL(k_dalitz_candidates<true>, dim3(nb), dim3(256), 0, (hipStream_t)stream, a, res, nres,
                           p_coup, eff_pc, eff_const, id12, id13, box[0], box[1], box[2], box[3], key, base, nc, fmax,
                           c12, c13, flag, bcount, bmax);
    else
        hipLaunchKernelGGL(k_dalitz_candidates<false>, dim3(nb), dim3(256), 0, (hipStream_t)stream, a, res, nres,
                           p_coup, eff_pc, eff_const, id12, id13, box[0], box[1], box[2], box[3], key, base, nc, fmax,
                           c12, c13, flag, bcount, bmax);
    return check(hipGetLastError());
}

int launch_compact(const double *c12, const double *c13, const uint8_t *flag, int64_t nc, const int64_t *boff,
                   int64_t limit, double *o12, double *o13, void *stream) {
    const int nb = (int)((nc + 255) / 256);
    hipLaunchKernelGGL(k_compact, dim3(nb), dim3(256), 0, (hipStream_t)stream, c12, c13, flag, nc, boff, limit, o12,
                       o13);
    return check(hipGetLastError());
}

int launch_dalitz_cache(const GfProgArgs &a, int slot, int64_t offset, int64_t n, uint32_t mask, const GfResDesc *res,
                        int nres, int nblocks, void *stream) {
    hipLaunchKernelGGL(k_dalitz_cache, dim3(nblocks), dim3(256), 0, (hipStream_t)stream, a, slot, offset, n, mask, res,
                       nres);
    return check(hipGetLastError());
}

int launch_gram(const GfProgArgs &a, int mode, const double *grid6, const double *m12, const double *m13,
                const double *w, int64_t npoints, int slot, int id_m12, int id_m13, int eff_pc, double eff_const,
                int td_grid, const GfResDesc *res, int nres, double *partials, double *tiles_dev, int nblocks,
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
    if(eff_pc >= 0)
        hipLaunchKernelGGL(k_gram<true>, dim3(nblocks), dim3(GG_BLOCK), 0, s, a, S, res, nres, partials);
    else
        hipLaunchKernelGGL(k_gram<false>, dim3(nblocks), dim3(GG_BLOCK), 0, s, a, S, res, nres, partials);
    int rc = check(hipGetLastError());
    if(rc)
        return rc;
    hipLaunchKernelGGL(k_gram_final, dim3(768), dim3(256), 0, s, partials, nblocks, tiles_dev);
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
