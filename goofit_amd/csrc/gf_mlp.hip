// Learned importance-sampling proposal for the Dalitz normalisation integrals.
//
// A 2 -> 128 -> 128 -> 1 SiLU network f(u, v) over the unit square (the Dalitz
// box [l12, u12] x [l13, u13] mapped to [0, 1]^2) is trained by maximum
// likelihood on events the model generated: loss = -mean_data f + log mean_unif
// exp(f), the second term a Monte-Carlo estimate of the normaliser over the box.
// The 128 x 128 layer and both of its backward products run on BF16 MFMA
// (v_mfma_f32_16x16x32_bf16, FP32 accumulation); the rest is FP32 VALU.
//
// Sampling: exp(f) tabulated on a G x G grid of cell centres, mixed with the
// uniform density (weight alpha, so every cell has probability >= alpha/G^2),
// sampled by inverse CDF (cell) and uniformly inside the cell.  The proposal's
// density is exactly that piecewise-constant table, so the weights
// w = 1 / (N q(x)) make sum_p w_p F(x_p) an unbiased estimate of the integral of
// F over the box whatever the network learned.
//
// No reference counterpart: GooFit normalises Amp3Body on a fixed midpoint grid
// (src/PDFs/physics/detail/SpecialResonanceIntegrator.cu:52-121).

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "gf_device.h"
#include "gf_mlp.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// Row of the 16 x 16 MFMA result held by register r of lane l (the column is
// l % 16).  gfx950 result layout of v_mfma_f32_16x16x32_bf16, checked by
// gf_mlp_layout_check against a host product.
__device__ __forceinline__ int d_row(int l, int r) { return GF_BF16_D_ROW(l, r); }

// fp32 -> bf16 bits, round to nearest even (finite inputs)
__device__ __forceinline__ uint16_t f2bf(float x) {
    uint32_t b = __float_as_uint(x);
    b += 0x7FFFu + ((b >> 16) & 1u);
    return (uint16_t)(b >> 16);
}

__device__ __forceinline__ float sigm(float z) { return 1.0f / (1.0f + expf(-z)); }
using gfd::mix64;
__device__ __forceinline__ double unif(uint64_t key, uint64_t ctr) { return gfd::unif01(key, ctr); }

__device__ __forceinline__ bf16x8 load8(const uint16_t *p) {
    const uint4 q = *reinterpret_cast<const uint4 *>(p);  // 16-byte aligned
    bf16x8 v;
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for(int t = 0; t < 4; ++t) {
        v[2 * t]     = __builtin_bit_cast(__bf16, (uint16_t)(w[t] & 0xFFFFu));
        v[2 * t + 1] = __builtin_bit_cast(__bf16, (uint16_t)(w[t] >> 16));
    }
    return v;
}

// ----------------------------------------------------------------- batches

// Sample s of a training batch: rows [0, nd) are data events drawn with replacement, rows
// from nd on uniform points of the unit square.  Inputs to the network are x = 2u - 1,
// y = 2v - 1.
__device__ __forceinline__ float2 train_sample(const GfTrainBatch &T, uint64_t key, int s) {
    double u, v;
    if(s < T.nd) {
        const int64_t e = (int64_t)(mix64(key ^ mix64(2 * (uint64_t)s)) % (uint64_t)T.ndata);
        u = (T.m12[e] - T.box.l12) / (T.box.u12 - T.box.l12);
        v = (T.m13[e] - T.box.l13) / (T.box.u13 - T.box.l13);
    } else {
        u = unif(key + 1, 2 * (uint64_t)s);
        v = unif(key + 1, 2 * (uint64_t)s + 1);
    }
    return make_float2((float)(2.0 * u - 1.0), (float)(2.0 * v - 1.0));
}

// Cell centres of a G x G grid over the unit square, cell c = cx + G * cy.
__global__ __launch_bounds__(256) void k_batch_grid(int G, int64_t ncell, float2 *__restrict__ xy) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if(c >= ncell)
        return;
    const double u = ((double)(c % G) + 0.5) / G, v = ((double)(c / G) + 0.5) / G;
    xy[c] = make_float2((float)(2.0 * u - 1.0), (float)(2.0 * v - 1.0));
}

// A training step is four launches: k_forward, k_loss, k_backward and k_update.  At the batch of
// 8192 each kernel is a chain of latencies over a few hundred workgroups, so a step costs
// what its launches and passes through memory cost: ten kernels (a step's state, the batch,
// two layers, the loss, three backward products, the sum and Adam) took 80 us a step, these
// four 34 us (8 + 5 + 16 + 4 on the device).
// What crosses between them is z2 (the layer-2 pre-activations); the first layer is formed
// again where it is needed (two products and a sigmoid an element: storing the sigmoids cost
// more than it saved).

// W1 and b1 as one LDS row per neuron.
__device__ __forceinline__ void stage_layer1(float4 *w1, const float *__restrict__ P) {
    for(int k = threadIdx.x; k < GF_MLP_H; k += blockDim.x)
        w1[k] = make_float4(P[GF_MLP_W1 + 2 * k], P[GF_MLP_W1 + 2 * k + 1], P[GF_MLP_B1 + k], 0.f);
}
__device__ __forceinline__ float layer1(const float4 w, float2 x) { return w.x * x.x + w.y * x.y + w.z; }

// ----------------------------------------------------------------- forward

// Layer 1 (2 -> 128, SiLU, FP32), layer 2 (128 -> 128, SiLU, BF16 MFMA) and the output
// layer (128 -> 1).  A workgroup of 8 waves takes 32 samples; four waves share 16 rows, each
// forming a quarter of their h1 and a quarter of their layer-2 neurons (two tiles of 4 MFMAs
// over K = 128): the sigmoids, some 40 instructions each, are the work, and 16 a lane on two
// waves per SIMD take less than 64 a lane on one.  The output's products go through LDS and
// are added per sample over neurons 16 t + i, t = 0 .. 7, then over the 16 i.  TRAIN: draws
// the samples first, and workgroup 0 sets the step's learning rate (cosine-decayed,
// lr0 (0.05 + 0.95 (1 + cos(pi k / steps)) / 2)) and Adam corrections for k_update.  z2 null:
// not stored.  n is a multiple of 64.
template <bool TRAIN>
__global__ __launch_bounds__(512) void k_forward(GfTrainBatch T, GfTrainState *st,
                                                 float2 *__restrict__ xy, const uint16_t *__restrict__ w2b,
                                                 const float *__restrict__ P, float *__restrict__ z2,
                                                 float *__restrict__ out) {
    __shared__ float4 w1[GF_MLP_H];
    __shared__ float2 sx[32];
    __shared__ __align__(16) uint16_t h1[32][GF_MLP_H + 8];
    __shared__ float po[32][GF_MLP_H + 1];
    const int t = threadIdx.x, l = t & 63, w = t >> 6, li = l & 15, lg = l >> 4;
    const int s0 = blockIdx.x * 32, row0 = 16 * (w >> 2), quarter = w & 3;
    // layer 2's operands and biases: in flight behind the first layer
    bf16x8 b[2][4];
    float bj[2], wj[2];
#pragma unroll
    for(int u = 0; u < 2; ++u) {
        const int j = 32 * quarter + 16 * u + li;  // this lane's column (neuron)
#pragma unroll
        for(int c = 0; c < 4; ++c)
            b[u][c] = load8(w2b + (int64_t)j * GF_MLP_H + 32 * c + 8 * lg);  // B[k][j] = W2[j][k]
        bj[u] = P[GF_MLP_B2 + j];
        wj[u] = P[GF_MLP_W3 + j];
    }
    stage_layer1(w1, P);
    if(t < 32) {
        float2 x;
        if(TRAIN) {
            x          = train_sample(T, st->seed * 0x9E3779B97F4A7C15ull + 2ull * (uint64_t)st->k + 1ull, s0 + t);
            xy[s0 + t] = x;
        } else {
            x = xy[s0 + t];
        }
        sx[t] = x;
    } else if(TRAIN && blockIdx.x == 0 && t == 64) {
        const int k    = st->k, at = st->adam_t + 1;
        const double c = 0.5 * (1.0 + cos(3.141592653589793 * (double)k / (double)st->steps));
        st->lr         = (float)(st->lr0 * (0.05 + 0.95 * c));
        st->c1         = 1.f - powf(st->b1, (float)at);
        st->c2         = 1.f - powf(st->b2, (float)at);
        st->next_k     = k + 1;  // committed by k_update, when nothing reads k any more
        st->next_t     = at;
    }
    __syncthreads();
    {
        const float2 x = sx[row0 + li];
        const int k0   = 32 * quarter + 8 * lg;
        uint32_t ph[4];
#pragma unroll
        for(int q = 0; q < 8; ++q) {
            const float z     = layer1(w1[k0 + q], x);
            const uint32_t hb = f2bf(z * sigm(z));
            ph[q >> 1]        = (q & 1) ? ph[q >> 1] | (hb << 16) : hb;
        }
        *reinterpret_cast<uint4 *>(&h1[row0 + li][32 * quarter + 8 * lg]) = make_uint4(ph[0], ph[1], ph[2], ph[3]);
    }
    __syncthreads();
    bf16x8 a[4];
#pragma unroll
    for(int c = 0; c < 4; ++c)
        a[c] = load8(&h1[row0 + li][32 * c + 8 * lg]);
#pragma unroll
    for(int u = 0; u < 2; ++u) {
        const int j = 32 * quarter + 16 * u + li;
        floatx4 d   = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for(int c = 0; c < 4; ++c)
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[c], b[u][c], d, 0, 0, 0);
#pragma unroll
        for(int r = 0; r < 4; ++r) {
            const int row = row0 + d_row(l, r);
            const float z = d[r] + bj[u], sg = sigm(z);
            if(z2)
                z2[(int64_t)(s0 + row) * GF_MLP_H + j] = z;
            po[row][j] = wj[u] * (z * sg);
        }
    }
    __syncthreads();
    const int row = t >> 4, i = t & 15;  // 32 rows of 16 lanes
    float acc     = 0.f;
#pragma unroll
    for(int u = 0; u < GF_MLP_H / 16; ++u)
        acc += po[row][16 * u + i];
#pragma unroll
    for(int off = 1; off < 16; off <<= 1)
        acc += __shfl_xor(acc, off, 64);
    if(i == 0)
        out[s0 + row] = acc + P[GF_MLP_B3];
}

// ----------------------------------------------------------------- loss

// One workgroup: per-sample output gradients of the loss
//   L = -(1/nd) sum_data f + log((1/nu) sum_unif exp f)
// (data: -1/nd; uniform: softmax weight), and L itself.  Lane t takes the samples t + 1024 i;
// the first eight f are loaded together (they were written through another XCD's L2, so each
// load waits for memory) and their exponentials kept.
__global__ __launch_bounds__(1024) void k_loss(const float *__restrict__ out, int nd, int nu, float *__restrict__ coef,
                                               float *__restrict__ loss) {
    constexpr int KEEP = 8;
    __shared__ float rm[16];
    __shared__ double rs[16], rd[16];
    const int t = threadIdx.x, w = t >> 6, l = t & 63, n = nd + nu;
    float v[KEEP];
#pragma unroll
    for(int i = 0; i < KEEP; ++i)
        v[i] = t + 1024 * i < n ? out[t + 1024 * i] : 0.f;
    float m = -INFINITY;
#pragma unroll
    for(int i = 0; i < KEEP; ++i)
        if(t + 1024 * i >= nd && t + 1024 * i < n)
            m = fmaxf(m, v[i]);
    for(int s = t + 1024 * KEEP; s < n; s += 1024)
        if(s >= nd)
            m = fmaxf(m, out[s]);
    for(int off = 32; off > 0; off >>= 1)
        m = fmaxf(m, __shfl_xor(m, off, 64));
    if(l == 0)
        rm[w] = m;
    __syncthreads();
    for(int q = 0; q < 16; ++q)
        m = fmaxf(m, rm[q]);
    double se = 0.0, sd = 0.0, e[KEEP];
#pragma unroll
    for(int i = 0; i < KEEP; ++i) {
        const int s = t + 1024 * i;
        e[i]        = 0.0;
        if(s < nd) {
            sd += v[i];
        } else if(s < n) {
            e[i] = exp((double)(v[i] - m));
            se += e[i];
        }
    }
    for(int s = t + 1024 * KEEP; s < n; s += 1024) {
        if(s < nd)
            sd += out[s];
        else
            se += exp((double)(out[s] - m));
    }
    for(int off = 32; off > 0; off >>= 1) {
        se += __shfl_xor(se, off, 64);
        sd += __shfl_xor(sd, off, 64);
    }
    if(l == 0) {
        rs[w] = se;
        rd[w] = sd;
    }
    __syncthreads();
    double z = 0.0;
    for(int q = 0; q < 16; ++q)
        z += rs[q];
#pragma unroll
    for(int i = 0; i < KEEP; ++i) {
        const int s = t + 1024 * i;
        if(s < n)
            coef[s] = s < nd ? -1.0f / nd : (float)(e[i] / z);
    }
    for(int s = t + 1024 * KEEP; s < n; s += 1024)
        coef[s] = s < nd ? -1.0f / nd : (float)(exp((double)(out[s] - m)) / z);
    if(t == 0) {
        sd = 0.0;
        for(int q = 0; q < 16; ++q)
            sd += rd[q];
        *loss = (float)(-sd / nd + (double)m + log(z / nu));
    }
}

// ----------------------------------------------------------------- backward

// The gradient of sum_s coef_s f(x_s).  Workgroup (b, h) takes the samples of the 32-sample
// chunks [b cpb, (b + 1) cpb), 128 at a time, and the neurons k of half h of layer 1:
//   delta2 = coef w3 silu'(z2) (bf16), and h = 0 writes the sums of dL/dw3, dL/db2, dL/db3
//     over every 16 samples;
//   dh1[s][k] = sum_j delta2[s][j] W2[j][k] (BF16 MFMA, W2^T rows), dz1 = dh1 silu'(z1),
//     and the sums of dL/dW1, dL/db1 over every 16 samples;
//   dW2[j][k] = sum_s delta2[s][j] h1[s][k] (BF16 MFMA, K = samples in chunk order), from
//     sample-contiguous copies of delta2 and h1 in LDS (16-byte operand reads), one 128 x 64
//     part per workgroup.
#define GF_BK 128
__global__ __launch_bounds__(1024) void k_backward(const float2 *__restrict__ xy, const float *__restrict__ z2,
                                                   const float *__restrict__ coef,
                                                   const uint16_t *__restrict__ w2t, const float *__restrict__ P, int n,
                                                   int cpb, float *__restrict__ part_in, float *__restrict__ part_w2,
                                                   float *__restrict__ part_out) {
    constexpr int HALF = GF_MLP_H / 2;
    __shared__ float4 w1[GF_MLP_H];
    __shared__ __align__(16) uint16_t dT[GF_MLP_H][GF_BK + 8];  // delta2, a neuron's samples in a row
    __shared__ __align__(16) uint16_t hT[HALF][GF_BK + 8];      // h1 of this half, likewise
    __shared__ __align__(16) uint16_t dR[GF_BK][GF_MLP_H + 8];  // delta2, a sample's neurons in a row
    __shared__ float2 sx[GF_BK];
    __shared__ float sc[GF_BK];
    const int t = threadIdx.x, l = t & 63, w = t >> 6, li = l & 15, lg = l >> 4;
    const int k0 = HALF * blockIdx.y;
    const int j = t % GF_MLP_H, g = t / GF_MLP_H;  // delta2: neuron j on samples 16 g ..
    const int rt = w & 7, half = w >> 3;           // the products: row tile, two of the four column tiles
    const float wj = P[GF_MLP_W3 + j];
    stage_layer1(w1, P);
    floatx4 acc[2];
#pragma unroll
    for(int q = 0; q < 2; ++q)
        acc[q] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int s_begin = blockIdx.x * cpb * 32, s_end = min(n, s_begin + cpb * 32);
    for(int s0 = s_begin; s0 < s_end; s0 += GF_BK) {
        const int cnt = min(GF_BK, s_end - s0);  // a multiple of 32
        const bool mine = 16 * g < cnt;
        float z[16];
#pragma unroll
        for(int q = 0; q < 16; ++q) {
            z[q]   = mine ? z2[(int64_t)(s0 + 16 * g + q) * GF_MLP_H + j] : 0.f;
        }
        __syncthreads();
        if(t < cnt) {
            sx[t] = xy[s0 + t];
            sc[t] = coef[s0 + t];
        }
        __syncthreads();
        if(mine) {
            float gw3 = 0.f, gb2 = 0.f, gb3 = 0.f;
#pragma unroll
            for(int q8 = 0; q8 < 2; ++q8) {
                uint32_t pd[4];
#pragma unroll
                for(int q = 0; q < 8; ++q) {
                    const int s    = 16 * g + 8 * q8 + q;
                    const float zz = z[8 * q8 + q];
                    const float sg = sigm(zz), cs = sc[s];
                    const float d  = cs * wj * (sg * (1.0f + zz * (1.0f - sg)));
                    const uint32_t db = f2bf(d);
                    dR[s][j]          = (uint16_t)db;
                    pd[q >> 1]        = (q & 1) ? pd[q >> 1] | (db << 16) : db;
                    gw3 += cs * (zz * sg);
                    gb2 += d;
                    gb3 += cs;
                }
                *reinterpret_cast<uint4 *>(&dT[j][16 * g + 8 * q8]) = make_uint4(pd[0], pd[1], pd[2], pd[3]);
            }
            if(blockIdx.y == 0) {
                float *po        = part_out + (int64_t)(s0 / 16 + g) * GF_MLP_PART_OUT;
                po[j]            = gw3;
                po[GF_MLP_H + j] = gb2;
                if(j == 0)
                    po[2 * GF_MLP_H] = gb3;
            }
        }
        if(8 * w < cnt) {  // h1: neuron k0 + l on samples 8 w ..
            const float4 wk = w1[k0 + l];
            uint32_t ph[4];
#pragma unroll
            for(int q = 0; q < 8; ++q) {
                const float zz    = layer1(wk, sx[8 * w + q]);
                const uint32_t hb = f2bf(zz * sigm(zz));
                ph[q >> 1]        = (q & 1) ? ph[q >> 1] | (hb << 16) : hb;
            }
            *reinterpret_cast<uint4 *>(&hT[l][8 * w]) = make_uint4(ph[0], ph[1], ph[2], ph[3]);
        }
        __syncthreads();
        if(16 * rt < cnt) {
            bf16x8 a[4];
#pragma unroll
            for(int c = 0; c < 4; ++c)
                a[c] = load8(&dR[16 * rt + li][32 * c + 8 * lg]);
            float *pi = part_in + (int64_t)(s0 / 16 + rt) * GF_MLP_PART_IN;
#pragma unroll
            for(int u = 0; u < 2; ++u) {
                const int k = k0 + 32 * half + 16 * u + li;
                floatx4 d   = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for(int c = 0; c < 4; ++c) {
                    const bf16x8 b = load8(w2t + (int64_t)k * GF_MLP_H + 32 * c + 8 * lg);  // B[j][k] = W2t[k][j]
                    d              = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[c], b, d, 0, 0, 0);
                }
                const float4 wk = w1[k];
                float g0 = 0.f, g1 = 0.f, gb = 0.f;
#pragma unroll
                for(int r = 0; r < 4; ++r) {
                    const int row  = 16 * rt + d_row(l, r);
                    const float2 x = sx[row];
                    const float zz = layer1(wk, x), sg = sigm(zz);
                    const float dz = d[r] * (sg * (1.0f + zz * (1.0f - sg)));
                    g0 += dz * x.x;
                    g1 += dz * x.y;
                    gb += dz;
                }
                // lanes l, l+16, l+32, l+48 share column k
#pragma unroll
                for(int off = 16; off < 64; off <<= 1) {
                    g0 += __shfl_xor(g0, off, 64);
                    g1 += __shfl_xor(g1, off, 64);
                    gb += __shfl_xor(gb, off, 64);
                }
                if(lg == 0) {
                    pi[2 * k]            = g0;
                    pi[2 * k + 1]        = g1;
                    pi[2 * GF_MLP_H + k] = gb;
                }
            }
        }
        for(int c = 0; c < cnt / 32; ++c) {
            const bf16x8 av = load8(&dT[16 * rt + li][32 * c + 8 * lg]);
#pragma unroll
            for(int u = 0; u < 2; ++u)
                acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    av, load8(&hT[32 * half + 16 * u + li][32 * c + 8 * lg]), acc[u], 0, 0, 0);
        }
    }
    float *p2 = part_w2 + (int64_t)blockIdx.x * GF_MLP_H * GF_MLP_H + k0 + 32 * half;
#pragma unroll
    for(int u = 0; u < 2; ++u)
#pragma unroll
        for(int r = 0; r < 4; ++r)
            p2[(16 * rt + d_row(l, r)) * GF_MLP_H + 16 * u + li] = acc[u][r];
}

// The gradient as the sum of its parts, and (ADAM) the Adam step on the FP32 master
// parameters with the bf16 copies of W2 and W2^T.  A workgroup takes 64 parameters; its 8
// waves sum the parts b = w, w + 8, w + 16, ..., and the eight sums are added in a fixed order
// (waves w and w + 4, then those four).  W1, b1, b2, w3, b3 have a part per 16 samples, taken
// four at a time (nb = n / 64 of those); W2 has nb_w2.
template <bool ADAM>
__global__ __launch_bounds__(512) void k_update(const float *__restrict__ p_in, const float *__restrict__ p_out, int nb,
                                                const float *__restrict__ p_w2, int nb_w2, float *__restrict__ grad,
                                                float *__restrict__ P, float *__restrict__ m, float *__restrict__ v,
                                                GfTrainState *st, uint16_t *__restrict__ w2b,
                                                uint16_t *__restrict__ w2t) {
    __shared__ float red[8][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i    = blockIdx.x * 64 + lane;
    float s0 = 0.f;
    if(i >= GF_MLP_W2 && i < GF_MLP_B2) {
        const float *base = p_w2 + (i - GF_MLP_W2);
        constexpr int64_t stride = (int64_t)GF_MLP_H * GF_MLP_H;
#pragma unroll 8
        for(int b = w; b < nb_w2; b += 8)
            s0 += base[(int64_t)b * stride];
    } else if(i < GF_MLP_NPARAM) {
        // W1 (interleaved k, input) then b1; the output parts are [w3 | b2 | b3]
        const bool in    = i < GF_MLP_W2;
        const int64_t st4 = in ? GF_MLP_PART_IN : GF_MLP_PART_OUT;
        const float *base = in ? p_in + i
                               : p_out + (i < GF_MLP_W3 ? GF_MLP_H + (i - GF_MLP_B2)
                                                        : i < GF_MLP_B3 ? i - GF_MLP_W3 : 2 * GF_MLP_H);
#pragma unroll 4
        for(int b = w; b < nb; b += 8) {
            const float *q = base + 4 * (int64_t)b * st4;
            s0 += ((q[0] + q[st4]) + q[2 * st4]) + q[3 * st4];
        }
    }
    red[w][lane] = s0;
    __syncthreads();
    if(w != 0 || i >= GF_MLP_NPARAM)
        return;
    const float gi = (((red[0][lane] + red[4][lane]) + (red[1][lane] + red[5][lane])) + (red[2][lane] + red[6][lane]))
                     + (red[3][lane] + red[7][lane]);
    if(!ADAM) {
        grad[i] = gi;
        return;
    }
    const float lr = st->lr, b1 = st->b1, b2 = st->b2, eps = st->eps, c1 = st->c1, c2 = st->c2;
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i]           = mi;
    v[i]           = vi;
    const float p  = P[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    P[i]           = p;
    if(i >= GF_MLP_W2 && i < GF_MLP_B2) {
        const int jk = i - GF_MLP_W2, j = jk / GF_MLP_H, k = jk % GF_MLP_H;
        const uint16_t h = f2bf(p);
        w2b[jk]                = h;
        w2t[k * GF_MLP_H + j]  = h;
    }
    if(i == 0) {
        st->k      = st->next_k;
        st->adam_t = st->next_t;
    }
}

// bf16 copies of W2 and W2^T from the master parameters.
__global__ __launch_bounds__(256) void k_w2_bf16(const float *__restrict__ P, uint16_t *__restrict__ w2b,
                                                 uint16_t *__restrict__ w2t) {
    const int jk = blockIdx.x * blockDim.x + threadIdx.x;
    if(jk >= GF_MLP_H * GF_MLP_H)
        return;
    const int j = jk / GF_MLP_H, k = jk % GF_MLP_H;
    const uint16_t h = f2bf(P[GF_MLP_W2 + jk]);
    w2b[jk]               = h;
    w2t[k * GF_MLP_H + j] = h;
}

// ----------------------------------------------------------------- sampling

// n points of the tabulated proposal: cell by binary search of the FP64 CDF
// (cdf[c] = P(cell <= c), cdf[G*G - 1] = 1), position uniform in the cell;
// w = box area / (n * p_cell * G^2) = 1 / (n q(x)).
__global__ __launch_bounds__(256) void k_sample(const double *__restrict__ cdf, const double *__restrict__ pcell,
                                                int G, GfBox box, int64_t n, uint64_t key, double *__restrict__ m12,
                                                double *__restrict__ m13, double *__restrict__ wt) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n)
        return;
    const int64_t ncell = (int64_t)G * G;
    const double r = unif(key, 3 * (uint64_t)i);
    int64_t lo = 0, hi = ncell - 1;  // first c with cdf[c] > r
    while(lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if(cdf[mid] > r)
            hi = mid;
        else
            lo = mid + 1;
    }
    const int64_t c = lo;
    const double u = ((double)(c % G) + unif(key, 3 * (uint64_t)i + 1)) / G;
    const double v = ((double)(c / G) + unif(key, 3 * (uint64_t)i + 2)) / G;
    const double area = (box.u12 - box.l12) * (box.u13 - box.l13);
    m12[i] = box.l12 + u * (box.u12 - box.l12);
    m13[i] = box.l13 + v * (box.u13 - box.l13);
    wt[i]  = area / ((double)n * pcell[c] * (double)ncell);
}

// Uniform points of the box with w = area / n.
__global__ __launch_bounds__(256) void k_sample_uniform(GfBox box, int64_t n, uint64_t key, double *__restrict__ m12,
                                                        double *__restrict__ m13, double *__restrict__ wt) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n)
        return;
    const double area = (box.u12 - box.l12) * (box.u13 - box.l13);
    m12[i] = box.l12 + unif(key, 2 * (uint64_t)i) * (box.u12 - box.l12);
    m13[i] = box.l13 + unif(key, 2 * (uint64_t)i + 1) * (box.u13 - box.l13);
    wt[i]  = area / (double)n;
}

// Probe of the MFMA operand/result layout: lane l feeds a8[l][0..7], b8[l][0..7]
// and writes its 4 result registers.
__global__ void k_bf16_probe(const uint16_t *a8, const uint16_t *b8, float *d) {
    const int l = threadIdx.x;
    bf16x8 av, bv;
#pragma unroll
    for(int t = 0; t < 8; ++t) {
        av[t] = __builtin_bit_cast(__bf16, a8[8 * l + t]);
        bv[t] = __builtin_bit_cast(__bf16, b8[8 * l + t]);
    }
    floatx4 r = {0.f, 0.f, 0.f, 0.f};
    r         = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, r, 0, 0, 0);
#pragma unroll
    for(int t = 0; t < 4; ++t)
        d[4 * l + t] = r[t];
}

inline int nblk(int64_t n, int b) { return (int)((n + b - 1) / b); }

}  // namespace

namespace gfm {

int check(hipError_t e) { return e == hipSuccess ? 0 : (int)e; }

// The backward kernel over n samples: at most GF_MLP_W2_BLOCKS workgroups per half, each a
// whole number of 32-sample chunks.
static void back_grid(int n, int &nb, int &cpb) {
    const int chunks = n / 32;
    nb  = chunks < GF_MLP_W2_BLOCKS ? chunks : GF_MLP_W2_BLOCKS;
    cpb = (chunks + nb - 1) / nb;
}

int launch_train_step(const GfMlpDev &D, const double *m12, const double *m13, int64_t ndata, GfBox box, int batch,
                      hipStream_t s) {
    const int half = batch / 2;
    int nb, cpb;
    back_grid(batch, nb, cpb);
    const GfTrainBatch T{m12, m13, ndata, box, half};
    hipLaunchKernelGGL(k_forward<true>, dim3(batch / 32), dim3(512), 0, s, T, D.state, D.xy,
                       (const uint16_t *)D.w2b, (const float *)D.P, D.z2, D.out);
    int rc = check(hipGetLastError());
    if(rc)
        return rc;
    hipLaunchKernelGGL(k_loss, dim3(1), dim3(1024), 0, s, D.out, half, half, D.coef, D.loss);
    if((rc = check(hipGetLastError())))
        return rc;
    hipLaunchKernelGGL(k_backward, dim3(nb, 2), dim3(1024), 0, s, D.xy, D.z2, D.coef, D.w2t, D.P, batch, cpb,
                       D.part_in, D.part_w2, D.part_out);
    if((rc = check(hipGetLastError())))
        return rc;
    hipLaunchKernelGGL(k_update<true>, dim3(nblk(GF_MLP_NPARAM, 64)), dim3(512), 0, s, D.part_in, D.part_out,
                       batch / 64, D.part_w2, nb, (float *)nullptr, D.P, D.m, D.v, D.state, D.w2b, D.w2t);
    return check(hipGetLastError());
}

int launch_batch_grid(int G, float2 *xy, hipStream_t s) {
    const int64_t nc = (int64_t)G * G;
    hipLaunchKernelGGL(k_batch_grid, dim3(nblk(nc, 256)), dim3(256), 0, s, G, nc, xy);
    return check(hipGetLastError());
}

int launch_forward(const GfMlpDev &D, float2 *xy, int n, float *out, bool keep, hipStream_t s) {
    hipLaunchKernelGGL(k_forward<false>, dim3(n / 32), dim3(512), 0, s, GfTrainBatch{}, (GfTrainState *)nullptr,
                       xy, (const uint16_t *)D.w2b, (const float *)D.P, keep ? D.z2 : (float *)nullptr, out);
    return check(hipGetLastError());
}

int launch_backward(const GfMlpDev &D, const float2 *xy, const float *coef, int n, float *grad, hipStream_t s) {
    int nb, cpb;
    back_grid(n, nb, cpb);
    hipLaunchKernelGGL(k_backward, dim3(nb, 2), dim3(1024), 0, s, xy, D.z2, coef, D.w2t, D.P, n, cpb, D.part_in,
                       D.part_w2, D.part_out);
    int rc = check(hipGetLastError());
    if(rc)
        return rc;
    hipLaunchKernelGGL(k_update<false>, dim3(nblk(GF_MLP_NPARAM, 64)), dim3(512), 0, s, D.part_in, D.part_out, n / 64,
                       D.part_w2, nb, grad, (float *)nullptr, (float *)nullptr, (float *)nullptr,
                       (GfTrainState *)nullptr, (uint16_t *)nullptr, (uint16_t *)nullptr);
    return check(hipGetLastError());
}

int launch_w2_bf16(const GfMlpDev &D, hipStream_t s) {
    hipLaunchKernelGGL(k_w2_bf16, dim3(nblk(GF_MLP_H * GF_MLP_H, 256)), dim3(256), 0, s, D.P, D.w2b, D.w2t);
    return check(hipGetLastError());
}

int launch_sample(const double *cdf, const double *pcell, int G, GfBox box, int64_t n, uint64_t key, double *m12,
                  double *m13, double *w, hipStream_t s) {
    hipLaunchKernelGGL(k_sample, dim3(nblk(n, 256)), dim3(256), 0, s, cdf, pcell, G, box, n, key, m12, m13, w);
    return check(hipGetLastError());
}

int launch_sample_uniform(GfBox box, int64_t n, uint64_t key, double *m12, double *m13, double *w, hipStream_t s) {
    hipLaunchKernelGGL(k_sample_uniform, dim3(nblk(n, 256)), dim3(256), 0, s, box, n, key, m12, m13, w);
    return check(hipGetLastError());
}

int launch_bf16_probe(const uint16_t *a8, const uint16_t *b8, float *d, hipStream_t s) {
    hipLaunchKernelGGL(k_bf16_probe, dim3(1), dim3(64), 0, s, a8, b8, d);
    return check(hipGetLastError());
}

}  // namespace gfm
