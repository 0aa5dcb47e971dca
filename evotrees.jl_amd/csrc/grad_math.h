// A row's gradients and the running maxima they raise, for the kernels that pass over the rows.
#pragma once
#include "evt_internal.h"

// Maximum of the 64 lanes' values, none of them negative or NaN (their bit patterns order as they do), by VALU moves as in split_math.h's prefix
// scan: seven outputs' fourteen maxima as cross-lane shuffles were 84 trips through the LDS crossbar, one after the other (60k rows of 7 classes: the
// gradient pass 13.2 -> 10.1 us).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t max_step(uint32_t v) {
    const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xf, false);
    return o > v ? o : v;
}
__device__ __forceinline__ float wave_max_f32(float x) {
    uint32_t v = __float_as_uint(x);
    v = max_step<0x111, 0xf>(v); // row_shr:1
    v = max_step<0x112, 0xf>(v); // row_shr:2
    v = max_step<0x114, 0xf>(v); // row_shr:4
    v = max_step<0x118, 0xf>(v); // row_shr:8
    v = max_step<0x142, 0xa>(v); // row_bcast:15 into rows 1 and 3
    v = max_step<0x143, 0xc>(v); // row_bcast:31 into rows 2 and 3
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)v, 63));
}

__device__ __forceinline__ float dev_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float dev_softplus(float x) { return fmaxf(x, 0.0f) + log1pf(expf(-fabsf(x))); }

// mle2p_grad_hess, src/loss.jl:194-217: GaussianMLE (LOSS 2) and LogisticMLE (LOSS 7); raw is the unconstrained scale.
template <int LOSS>
__device__ __forceinline__ void mle2p_grad_hess(float loc, float raw, float y, float &g_loc, float &g_scale, float &h_loc, float &h_scale) {
    const float scale = dev_softplus(raw);
    const float dscale = dev_sigmoid(raw);
    const float ds = dscale / scale;
    if (LOSS == 2) {
        const float resid = loc - y;
        const float s2 = scale * scale;
        g_loc = resid / s2;
        g_scale = (1.0f - (resid * resid) / s2) * dscale / scale;
        h_loc = 1.0f / s2;
        h_scale = 2.0f * (ds * ds);
    } else {
        const float z = (y - loc) / scale;
        const float th = tanhf(z / 2.0f);
        g_loc = -th / scale;
        g_scale = (1.0f - z * th) * dscale / scale;
        h_loc = 1.0f / (3.0f * (scale * scale));
        h_scale = (3.14159274f * 3.14159274f + 3.0f) / 9.0f * (ds * ds); // oftype(scale, pi)^2
    }
}

// Raises the running maximum of gradient row k.  Same-address atomics from thousands of blocks queue up one behind the
// other (about 20 ns each - 40 us for the 2048 blocks of a gradient pass), so the maximum is kept in
// EVT_ABSMAX_STRIPES copies on different cache lines, a block raises the copy its index selects, and the one reader
// (the quantisation pass, k_quantize) takes the largest.  The value only grows while a pass runs: a block whose own maximum is already
// covered by what a device-scope load shows skips the atomic.
__device__ __forceinline__ void absmax_raise(uint32_t *absmax, int k, float m) {
    if (!(m > 0.0f)) return;
    uint32_t *p = absmax + (blockIdx.x % EVT_ABSMAX_STRIPES) * EVT_MC_MAX_NK + k;
    const uint32_t u = __float_as_uint(m);
    if (__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < u) atomicMax(p, u);
}

// Raises the maxima by those of a block, a thread's in mx; s_m: a row of the block's wavefronts (16 at most)
template <int ROWS>
__device__ __forceinline__ void absmax_raise_block(const float *mx, float (*s_m)[ROWS], uint32_t *absmax) {
#pragma unroll
    for (int k = 0; k < ROWS; k++) {
        const float m = wave_max_f32(mx[k]);
        if ((threadIdx.x & 63) == 0) s_m[threadIdx.x >> 6][k] = m;
    }
    __syncthreads();
    if (threadIdx.x < ROWS) {
        const int k = threadIdx.x;
        float m = s_m[0][k];
        for (int w = 1; w < (int)blockDim.x >> 6; w++) m = fmaxf(m, s_m[w][k]);
        absmax_raise(absmax, k, m);
    }
}

// LOSS: 0 mse (src/loss.jl:52), 1 logloss (:54-57), 2 gaussian_mle (:194-203), 3 poisson (:59-62),
// 4 gamma (:64-67), 5 tweedie with rho = 1.5 (:69-76), 8 mae (:78), 9 cred_var / cred_std (:80-83).
// pr: the row's outputs (two of an MLE loss); out: g, then h of each, times the row's weight.
template <int LOSS>
__device__ __forceinline__ void grad_row(const float *pr, float y, float w, float *out) {
    if (LOSS == 0) {
        const float gg = 2.0f * (pr[0] - y);
        out[0] = gg * w;
        out[1] = 2.0f * w;
    } else if (LOSS == 1) {
        const float s = dev_sigmoid(pr[0]);
        out[0] = (s - y) * w;
        out[1] = (s * (1.0f - s)) * w;
    } else if (LOSS == 3) {
        const float e = expf(pr[0]);
        out[0] = (e - y) * w;
        out[1] = e * w;
    } else if (LOSS == 4) {
        const float e = expf(pr[0]);
        out[0] = (2.0f * (1.0f - y / e)) * w;
        out[1] = (2.0f * y / e) * w;
    } else if (LOSS == 5) {
        const float e = expf(pr[0]);
        const float a = powf(e, 0.5f), b = powf(e, -0.5f);
        out[0] = (2.0f * (a - y * b)) * w;
        out[1] = (2.0f * (0.5f * a - (-0.5f) * y * b)) * w;
    } else if (LOSS == 8) { // mae (src/loss.jl:78): the residual, no second-order row
        out[0] = (y - pr[0]) * w;
        out[1] = 0.0f * w;
    } else if (LOSS == 9) { // credibility losses (src/loss.jl:80-83): residual and its square
        const float d = y - pr[0];
        out[0] = d * w;
        out[1] = (d * d) * w;
    } else {
        float g1, g2, h1, h2;
        mle2p_grad_hess<LOSS>(pr[0], pr[1], y, g1, g2, h1, h2);
        out[0] = g1 * w;
        out[1] = g2 * w;
        out[2] = h1 * w;
        out[3] = h2 * w;
    }
}

// grad_row's LOSS for the gradients of a handle, -1 where they are not those of one target
inline int grad_row_loss(const evt_ctx *c) {
    if (EVT_IS_QUANTILE(c->loss) || c->loss == EVT_LOSS_MLOGLOSS || c->K != (EVT_IS_MLE2P(c->loss) ? 2 : 1)) return -1;
    return EVT_IS_CRED(c->loss) ? 9 : c->loss;
}
// A tree's last kernel computes the next round's gradients: those that would be queued behind the tree (tree_close), of one target
inline bool grads_with_tree(const evt_ctx *c, const evt_params *p) {
    return c->grads_ahead && p->update_pred && p->bagging_size == 1 && grad_row_loss(c) >= 0;
}
// LAUNCH(LOSS) for the handle's loss
#define EVT_GRAD_ROW_CASES(c, LAUNCH) \
    switch (grad_row_loss(c)) {       \
    case 0: LAUNCH(0); break;         \
    case 1: LAUNCH(1); break;         \
    case 2: LAUNCH(2); break;         \
    case 3: LAUNCH(3); break;         \
    case 4: LAUNCH(4); break;         \
    case 5: LAUNCH(5); break;         \
    case 7: LAUNCH(7); break;         \
    case 8: LAUNCH(8); break;         \
    default: LAUNCH(9); break;        \
    }

// Exponent of gradient row t for its fixed-point words: ilogb(max |row t|) + 1, 0 for an all-zero row, from the striped maxima of one pass.
__device__ __forceinline__ int quant_exponent(const uint32_t *__restrict__ absmax, int t) {
    uint32_t mu = 0u;
#pragma unroll
    for (int st = 0; st < EVT_ABSMAX_STRIPES; st++) {
        const uint32_t v = absmax[st * EVT_MC_MAX_NK + t]; // non-negative floats order as their bit patterns
        mu = v > mu ? v : mu;
    }
    const float m = __uint_as_float(mu);
    int e = 0;
    if (m > 0.0f) {
        e = ilogbf(m) + 1;
        if (e > 128) e = 128;
        if (e < -140) e = -140;
    }
    return e;
}
// gradient row of global channel ag: one-target mse / mae have {g, w}, otherwise the rows as they are
__device__ __forceinline__ int quant_row(int loss, int K, int ag) { return EVT_TWO_CHAN(loss, K) && ag == 1 ? 2 : ag; }

// lanes that share a row's channels, as a power of two (60k rows of 14 channels, set-up and quantisation in one launch: one lane a row 11.7 us,
// four 9.3)
__host__ __device__ inline int quant_lanes_sh(int na) { return na > EVT_MAX_NA ? 2 : 0; }

struct QuantArgs {
    const float *grad;
    unsigned long long *gq;
    int64_t N;
    int NK, NA, NAg, loss, two, unit_w, pack, pack_wide;
    int stride; // words from row to row of gq, 0: planes of N words
    const uint32_t *absmax;
    uint32_t *absmax_next;
    const int32_t *qbits;
    int32_t *qexp;
    double *qscale; // decode scales per global channel, then EVT_MC_MAX_NK on the multipliers per gradient row
};
void quant_args(evt_ctx *c, QuantArgs &Q);             // behind quant_set
unsigned quant_blocks(const evt_ctx *c, int threads);
void quant_taken(evt_ctx *c);                          // behind the launch

// Quantisation tables of a gradient pass and the fixed-point words the histogram kernel adds, in one pass.
// qexp[k] = ilogb(max |row k|) + 1 (0 for an all-zero row); qmul[k] = 2^(qbits - qexp) encodes, qscale decodes.  Every block
// derives the multipliers from the striped maxima itself (a few dozen cached loads: no kernel of its own in front of this one);
// block 0 also writes the tables for the readers that follow (split search, read-back).  The maxima live in two sets: a
// gradient pass raises one, this kernel reads it and clears the other - which nobody uses at that moment - for the next pass,
// so no pass starts from maxima an earlier one left behind.  The weight row (last) is written once and keeps its maximum.
// Word a of a row is q = rint(v * 2^(qbits - qexp)) of gradient row chan_k[a]; with unit weights word 0 also carries
// the row count in its low 16 bits ((q << 16) + 1) so that one 64-bit LDS add serves both.  A row's words go to planes, or side by side (gq_rows).
// absmax == nullptr: the words are made again, in the other layout, with the tables there are.
// Channel a reads gradient row a, except for mse whose channels are {g, w} = rows {0, 2}.
// `block` of `blocks`: of a kernel of its own, or of one that sets a tree up meanwhile (kernels_part.hip).
__device__ __forceinline__ void quant_rows(const QuantArgs &Q, int block, int blocks) {
    __shared__ double s_qmul[EVT_MC_MAX_NK];
    __shared__ int s_qexp[EVT_MC_MAX_NK], s_qbits[EVT_MC_MAX_NK];
    const int t = threadIdx.x, nthr = blockDim.x, NK = Q.NK;
    if (t < NK) {
        if (Q.absmax) {
            const int e = quant_exponent(Q.absmax, t);
            const int qb = Q.qbits[t];
            s_qexp[t] = e;
            s_qbits[t] = qb;
            s_qmul[t] = scalbn(1.0, qb - e);
        } else {
            s_qmul[t] = Q.qscale[EVT_MC_MAX_NK + t];
        }
    }
    __syncthreads();
    if (block == 0 && Q.absmax) {
        if (t < NK) {
            Q.qexp[t] = s_qexp[t];
            Q.qscale[EVT_MC_MAX_NK + t] = s_qmul[t];
            if (t < NK - 1)
                for (int st = 0; st < EVT_ABSMAX_STRIPES; st++) Q.absmax_next[st * EVT_MC_MAX_NK + t] = 0u;
        }
        if (t < Q.NAg) {
            const int kk = quant_row(Q.loss, (NK - 1) / 2, t); // the last channel is w (or the row count)
            if (t == Q.NAg - 1 && Q.unit_w) Q.qscale[t] = 1.0;
            else Q.qscale[t] = scalbn(1.0, s_qexp[kk] - s_qbits[kk]);
        }
    }
    // a block takes many rows (grid-stride), so that the prologue above is paid a couple of thousand times, not once per 256 rows
    const int sh = quant_lanes_sh(Q.NA), part = t & ((1 << sh) - 1);
    for (int64_t w = (int64_t)block * nthr + t; w < Q.N << sh; w += (int64_t)blocks * nthr) {
        const int64_t i = w >> sh;
        const float *g = Q.grad + (size_t)NK * i;
        if (Q.stride) { // 16 bytes, two channels, at a time
#pragma unroll 3
            for (int a = 2 * part; a < Q.NA; a += 2 << sh) {
                long long q0 = __double2ll_rn((double)g[a] * s_qmul[a]);
                const int a1 = a + 1 < Q.NA ? a + 1 : a, k1 = (Q.two && a1 == 1) ? 2 : a1;
                const long long q1 = __double2ll_rn((double)g[k1] * s_qmul[k1]);
                if (a == 0 && Q.unit_w) q0 = (long long)(((unsigned long long)q0 << EVT_PACK_CNT_BITS) + 1ull);
                *reinterpret_cast<ulonglong2 *>(Q.gq + (size_t)i * Q.stride + a) = make_ulonglong2((unsigned long long)q0, (unsigned long long)q1);
            }
            continue;
        }
#pragma unroll 5
        for (int a = part; a < Q.NA; a += 1 << sh) { // several channels' words in flight
            const int k = (Q.two && a == 1) ? 2 : a;
            long long q = __double2ll_rn((double)g[k] * s_qmul[k]);
            if (a == 0 && Q.pack) { // 30 bits: staged as a 32-bit word, widened to (q << 16) + 1 (the row count) by the histogram kernel
                reinterpret_cast<int32_t *>(Q.gq)[i] = (int32_t)q;
                continue;
            }
            if (a == 0 && Q.pack_wide) q = (long long)(((unsigned long long)q << EVT_PACK_CNT_BITS) + 1ull); // the same word, for kernels that read every channel alike
            Q.gq[(size_t)a * Q.N + i] = (unsigned long long)q;
        }
    }
}
