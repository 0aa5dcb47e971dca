// Gradient kernels: fused per-loss gradient + hessian rows, |max| reduction, fixed-point staging.
//
// Streaming work, HBM bound: per row the kernel reads pred (4K B), y (4 B) and the weight
// (4 B, last row of the gradient matrix) and writes 8K B.
//
// A tree grown on every row leaves its leaf values pending: growing recorded the leaf of each row and
// the addition to the prediction (predict!, src/predict.jl:1-46) happens here, in row order, as the
// first thing the next gradient pass does (4 B of node id read and 4K B written more per row) - or in
// k_apply_leaf when something else needs the predictions first.
#include "grad_math.h"
#include <algorithm>

// Maxima of any number of outputs (mx[k] and mx[EVT_MAX_K + k]: gradient row k and K + k), by a whole block of 256 threads: a thread raises a
// row, all rows side by side, where one thread raising them in turn took two barriers and a trip to memory for each (60k rows of 7 classes:
// the pass 22.4 -> 13.7 us).
__device__ __forceinline__ void raise_maxima(const float *mx, int K, uint32_t *absmax) {
    __shared__ float s_m[4][2 * EVT_MAX_K];
#pragma unroll
    for (int k = 0; k < 2 * EVT_MAX_K; k++) {
        if ((k < EVT_MAX_K ? k : k - EVT_MAX_K) < K) { // uniform
            const float m = wave_max_f32(mx[k]);
            if ((threadIdx.x & 63) == 0) s_m[threadIdx.x >> 6][k] = m;
        }
    }
    __syncthreads();
    const int t = threadIdx.x, k = t < EVT_MAX_K ? t : t - EVT_MAX_K;
    if (t < 2 * EVT_MAX_K && k < K)
        absmax_raise(absmax, t < EVT_MAX_K ? k : K + k, fmaxf(fmaxf(s_m[0][t], s_m[1][t]), fmaxf(s_m[2][t], s_m[3][t])));
}

// grad rows: [g_1..g_K, h_1..h_K, w]; every written value is multiplied by w (src/loss.jl:104-108, :223-233).
// Blocks of 256 threads, or of 1024 where the grid fills the chip: the blocks of a whole generation raise their maxima at the same time, and a
// quarter of them queue for a quarter as long (1M rows, blocks of 256 | 1024: 8.4 | 6.5 us).
template <int LOSS>
__global__ __launch_bounds__(1024) void k_grads(float *__restrict__ pred, const float *__restrict__ y, float *__restrict__ grad, int64_t N,
                                              uint32_t *absmax, const uint32_t *__restrict__ pend_nidx,
                                              const float *__restrict__ pend_leaf, int unit_w) {
    constexpr int K = (LOSS == 2 || LOSS == 7) ? 2 : 1;
    constexpr int NK = 2 * K + 1;
    float mx[2 * K];
#pragma unroll
    for (int k = 0; k < 2 * K; k++) mx[k] = 0.0f;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (int64_t)gridDim.x * blockDim.x) {
        float out[2 * K];
        float *g = grad + (size_t)NK * i;
        const float w = unit_w ? 1.0f : g[NK - 1]; // unit weights: the weight row (all ones) is not read
        if (pend_nidx) evt_add_leaf(pred + (size_t)K * i, pend_leaf + (size_t)K * (pend_nidx[i] - 1), K, LOSS);
        grad_row<LOSS>(pred + (size_t)K * i, y[i], w, out);
#pragma unroll
        for (int k = 0; k < 2 * K; k++) {
            g[k] = out[k];
            mx[k] = fmaxf(mx[k], fabsf(out[k]));
        }
    }
    // per gradient row max |v| -> exponent bound of the fixed-point histogram.
    // One atomic per block and row: contended same-address atomics serialise in L2.
    __shared__ float s_m[16][2 * K];
    absmax_raise_block<2 * K>(mx, s_m, absmax);
}

// Several targets at once (y is T x N, one column per row of data; src/loss.jl:49-50, :100-111, :219-236): the same
// per-target expressions as k_grads with K = T outputs (2T for gaussian_mle, whose rows are
// [g_loc_1, g_scale_1, g_loc_2, ..., h_loc_1, h_scale_1, ..., w]).
template <int LOSS>
__device__ __forceinline__ void grad_hess_one(float pk, float yk, float &g, float &h) {
    if (LOSS == 0) {
        g = 2.0f * (pk - yk);
        h = 2.0f;
    } else if (LOSS == 1) {
        const float s = dev_sigmoid(pk);
        g = s - yk;
        h = s * (1.0f - s);
    } else if (LOSS == 3) {
        const float e = expf(pk);
        g = e - yk;
        h = e;
    } else if (LOSS == 4) {
        const float e = expf(pk);
        g = 2.0f * (1.0f - yk / e);
        h = 2.0f * yk / e;
    } else if (LOSS == 8) {
        g = yk - pk;
        h = 0.0f;
    } else if (LOSS == 9) {
        const float d = yk - pk;
        g = d;
        h = d * d;
    } else {
        const float e = expf(pk);
        const float a = powf(e, 0.5f), b = powf(e, -0.5f);
        g = 2.0f * (a - yk * b);
        h = 2.0f * (0.5f * a - (-0.5f) * yk * b);
    }
}

template <int LOSS>
__global__ __launch_bounds__(256) void k_grads_mt(float *__restrict__ pred, const float *__restrict__ y, float *__restrict__ grad, int64_t N,
                                                 int K, uint32_t *absmax, const uint32_t *__restrict__ pend_nidx,
                                                 const float *__restrict__ pend_leaf, int unit_w) {
    const int NK = 2 * K + 1;
    constexpr bool MLE2P = (LOSS == 2 || LOSS == 7);
    const int T = MLE2P ? K / 2 : K; // target columns
    float mx[2 * EVT_MAX_K];
#pragma unroll
    for (int k = 0; k < 2 * EVT_MAX_K; k++) mx[k] = 0.0f;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < N; i += (int64_t)gridDim.x * 256) {
        float *pr = pred + (size_t)K * i;
        float *g = grad + (size_t)NK * i;
        const float *yi = y + (size_t)T * i;
        const float w = unit_w ? 1.0f : g[NK - 1];
        if (pend_nidx) evt_add_leaf(pr, pend_leaf + (size_t)K * (pend_nidx[i] - 1), K, LOSS);
#pragma unroll
        for (int k = 0; k < EVT_MAX_K; k++) {
            if (k < K) {
                float gg, hh;
                if (MLE2P) {
                    // output k of pair t = k / 2: even = location, odd = raw scale
                    const int t = k >> 1;
                    float g1, g2, h1, h2;
                    mle2p_grad_hess<MLE2P ? LOSS : 2>(pr[2 * t], pr[2 * t + 1], yi[t], g1, g2, h1, h2);
                    gg = (((k & 1) == 0) ? g1 : g2) * w;
                    hh = (((k & 1) == 0) ? h1 : h2) * w;
                } else {
                    float g1, h1;
                    grad_hess_one<MLE2P ? 0 : LOSS>(pr[k], yi[k], g1, h1);
                    gg = g1 * w;
                    hh = h1 * w;
                }
                g[k] = gg;
                g[K + k] = hh;
                mx[k] = fmaxf(mx[k], fabsf(gg));
                mx[EVT_MAX_K + k] = fmaxf(mx[EVT_MAX_K + k], fabsf(hh));
            }
        }
    }
    raise_maxima(mx, K, absmax);
}

// Multi-class log loss (src/loss.jl:93-98, :113-128): prob_k = exp(p_k) / sum_j exp(p_j); g_k = (prob_k - [y == k]) w,
// h_k = prob_k (1 - prob_k) w; y holds the 1-based class.
// KM: a bound of K, 4, 8 or 16; a row's words are requested together (those past the last class read it again), where a request per class behind a
// branch each was a trip to memory per class.  60k rows of 7 classes 13.7 -> 13.2 us.
template <int KM>
__global__ __launch_bounds__(256) void k_grads_mlogloss(float *__restrict__ pred, const float *__restrict__ y, float *__restrict__ grad,
                                                       int64_t N, int K, uint32_t *absmax, const uint32_t *__restrict__ pend_nidx,
                                                       const float *__restrict__ pend_leaf, int unit_w) {
    const int NK = 2 * K + 1;
    float mx[2 * EVT_MAX_K];
#pragma unroll
    for (int k = 0; k < 2 * EVT_MAX_K; k++) mx[k] = 0.0f;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < N; i += (int64_t)gridDim.x * 256) {
        float *pr = pred + (size_t)K * i;
        float *g = grad + (size_t)NK * i;
        const float w = unit_w ? 1.0f : g[NK - 1]; // unit weights: the weight row (all ones) is not read
        const int cls = (int)y[i];
        float e[KM]; // the row's predictions, then their exponentials: read and written once
#pragma unroll
        for (int k = 0; k < KM; k++) e[k] = pr[k < K ? k : K - 1];
        if (pend_nidx) { // evt_add_leaf
            const float *lp = pend_leaf + (size_t)K * (pend_nidx[i] - 1);
            float l[KM], m = -INFINITY;
#pragma unroll
            for (int k = 0; k < KM; k++) l[k] = lp[k < K ? k : K - 1];
#pragma unroll
            for (int k = 0; k < KM; k++) {
                e[k] += l[k];
                m = fmaxf(m, e[k]);
            }
#pragma unroll
            for (int k = 0; k < KM; k++)
                if (k < K) {
                    e[k] = fmaxf(-15.0f, e[k] - m);
                    pr[k] = e[k];
                }
        }
        float isum = 0.0f;
#pragma unroll
        for (int k = 0; k < KM; k++) {
            if (k < K) {
                e[k] = expf(e[k]);
                isum += e[k];
            }
        }
#pragma unroll
        for (int k = 0; k < KM; k++) {
            if (k < K) {
                const float prob = e[k] / isum;
                const float gg = ((cls == k + 1) ? prob - 1.0f : prob) * w;
                const float hh = (prob * (1.0f - prob)) * w;
                g[k] = gg;
                g[K + k] = hh;
                mx[k] = fmaxf(mx[k], fabsf(gg));
                mx[EVT_MAX_K + k] = fmaxf(mx[EVT_MAX_K + k], fabsf(hh));
            }
        }
    }
    raise_maxima(mx, K, absmax);
}

// The quantile losses (src/loss.jl:85-91, :144-171): row k = (alpha or alpha - 1, a Float64) * w, row K + k = the raw
// residual (not weighted: the leaf pass takes its quantile).  multi: one target column and a level per output
// (multiquantile); otherwise one level and a target column per output (quantile).
__global__ __launch_bounds__(256) void k_grads_quantile(float *__restrict__ pred, const float *__restrict__ y, float *__restrict__ grad, int64_t N,
                                                       int K, int multi, const double *__restrict__ alphas, uint32_t *absmax,
                                                       const uint32_t *__restrict__ pend_nidx, const float *__restrict__ pend_leaf, int unit_w) {
    const int NK = 2 * K + 1;
    const int T = multi ? 1 : K;
    float mx[2 * EVT_MAX_K];
#pragma unroll
    for (int k = 0; k < 2 * EVT_MAX_K; k++) mx[k] = 0.0f;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < N; i += (int64_t)gridDim.x * 256) {
        float *pr = pred + (size_t)K * i;
        float *g = grad + (size_t)NK * i;
        const float *yi = y + (size_t)T * i;
        const float w = unit_w ? 1.0f : g[NK - 1];
        if (pend_nidx) evt_add_leaf(pr, pend_leaf + (size_t)K * (pend_nidx[i] - 1), K, EVT_LOSS_QUANTILE);
#pragma unroll
        for (int k = 0; k < EVT_MAX_K; k++) {
            if (k < K) {
                const double alpha = multi ? alphas[k] : alphas[0];
                const float diff = (multi ? yi[0] : yi[k]) - pr[k];
                const float gg = (float)((diff > 0.0f ? alpha : alpha - 1.0) * (double)w);
                g[k] = gg;
                g[K + k] = diff;
                mx[k] = fmaxf(mx[k], fabsf(gg));
                mx[EVT_MAX_K + k] = fmaxf(mx[EVT_MAX_K + k], fabsf(diff));
            }
        }
    }
    raise_maxima(mx, K, absmax);
}

// max |v| of every gradient row of an existing gradient matrix (injected gradients, weight row)
__global__ __launch_bounds__(256) void k_absmax(const float *__restrict__ grad, int64_t N, int NK, int k0, int k1, uint32_t *absmax) {
    // one gradient row at a time: any number of rows without per-thread arrays
    for (int k = k0; k < k1; k++) {
        float m = 0.0f;
        for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < N; i += (int64_t)gridDim.x * 256)
            m = fmaxf(m, fabsf(grad[(size_t)NK * i + k]));
        const float v = wave_max_f32(m);
        if ((threadIdx.x & 63) == 0) absmax_raise(absmax, k, v);
    }
}

// The quantisation as a kernel of its own (quant_rows)
__global__ __launch_bounds__(256) void k_quantize(QuantArgs Q) { quant_rows(Q, blockIdx.x, gridDim.x); }

// the set of striped maxima the next gradient pass raises (and the quantisation behind it reads)
uint32_t *absmax_set(evt_ctx *c, int which) { return c->absmax + (size_t)which * EVT_ABSMAX_STRIPES * EVT_MC_MAX_NK; }

int launch_grads(evt_ctx *c) {
    // the maxima of the rows this kernel writes start from zero (cleared at creation and by the quantisation pass before last)
    uint32_t *const am = absmax_set(c, c->absmax_cur);
    int64_t nb = (c->N + 255) / 256;
    if (nb > 2048) nb = 2048;
    dim3 grid((unsigned)nb);
    const uint32_t *pn = c->pend_pred ? c->nidx : nullptr; // the last tree's leaf values are added on the way
    c->pend_pred = false;
    if (EVT_IS_QUANTILE(c->loss)) {
        hipLaunchKernelGGL(k_grads_quantile, grid, dim3(256), 0, c->stream, c->pred, c->y, c->grad, c->N, c->K, c->loss == EVT_LOSS_MULTIQUANTILE ? 1 : 0,
                           c->alphas, am, pn, c->tree.pred, c->unit_w ? 1 : 0);
        HIPCHK(hipGetLastError());
        return EVT_OK;
    }
    const bool multi_target = c->loss != EVT_LOSS_MLOGLOSS && c->K > (EVT_IS_MLE2P(c->loss) ? 2 : 1);
    if (multi_target) {
#define MT(L_) hipLaunchKernelGGL(k_grads_mt<L_>, grid, dim3(256), 0, c->stream, c->pred, c->y, c->grad, c->N, c->K, am, pn, c->tree.pred, c->unit_w ? 1 : 0)
        switch (c->loss) {
        case EVT_LOSS_MSE: MT(0); break;
        case EVT_LOSS_LOGLOSS: MT(1); break;
        case EVT_LOSS_GAUSSIAN_MLE: MT(2); break;
        case EVT_LOSS_POISSON: MT(3); break;
        case EVT_LOSS_GAMMA: MT(4); break;
        case EVT_LOSS_LOGISTIC_MLE: MT(7); break;
        case EVT_LOSS_MAE: MT(8); break;
        case EVT_LOSS_CRED_VAR:
        case EVT_LOSS_CRED_STD: MT(9); break;
        default: MT(5); break;
        }
#undef MT
        HIPCHK(hipGetLastError());
        return EVT_OK;
    }
    const bool wide = nb == 2048;
    const dim3 grid1(wide ? 512u : (unsigned)nb), block1(wide ? 1024u : 256u);
    if (c->loss == EVT_LOSS_MSE)
        hipLaunchKernelGGL(k_grads<0>, grid1, block1, 0, c->stream, c->pred, c->y, c->grad, c->N, am, pn, c->tree.pred, c->unit_w ? 1 : 0);
    else if (c->loss == EVT_LOSS_LOGLOSS)
        hipLaunchKernelGGL(k_grads<1>, grid1, block1, 0, c->stream, c->pred, c->y, c->grad, c->N, am, pn, c->tree.pred, c->unit_w ? 1 : 0);
    else if (c->loss == EVT_LOSS_LOGISTIC_MLE)
        hipLaunchKernelGGL(k_grads<7>, grid1, block1, 0, c->stream, c->pred, c->y, c->grad, c->N, am, pn, c->tree.pred, c->unit_w ? 1 : 0);
    else if (c->loss == EVT_LOSS_GAUSSIAN_MLE)
        hipLaunchKernelGGL(k_grads<2>, grid1, block1, 0, c->stream, c->pred, c->y, c->grad, c->N, am, pn, c->tree.pred, c->unit_w ? 1 : 0);
    else if (c->loss == EVT_LOSS_POISSON)
        hipLaunchKernelGGL(k_grads<3>, grid1, block1, 0, c->stream, c->pred, c->y, c->grad, c->N, am, pn, c->tree.pred, c->unit_w ? 1 : 0);
    else if (c->loss == EVT_LOSS_GAMMA)
        hipLaunchKernelGGL(k_grads<4>, grid1, block1, 0, c->stream, c->pred, c->y, c->grad, c->N, am, pn, c->tree.pred, c->unit_w ? 1 : 0);
    else if (c->loss == EVT_LOSS_MAE)
        hipLaunchKernelGGL(k_grads<8>, grid1, block1, 0, c->stream, c->pred, c->y, c->grad, c->N, am, pn, c->tree.pred, c->unit_w ? 1 : 0);
    else if (EVT_IS_CRED(c->loss))
        hipLaunchKernelGGL(k_grads<9>, grid1, block1, 0, c->stream, c->pred, c->y, c->grad, c->N, am, pn, c->tree.pred, c->unit_w ? 1 : 0);
    else if (c->loss == EVT_LOSS_MLOGLOSS)
#define ML(KM_) hipLaunchKernelGGL(k_grads_mlogloss<KM_>, grid, dim3(256), 0, c->stream, c->pred, c->y, c->grad, c->N, c->K, am, pn, c->tree.pred, c->unit_w ? 1 : 0)
        if (c->K <= 4) ML(4);
        else if (c->K <= 8) ML(8);
        else ML(16);
#undef ML
    else
        hipLaunchKernelGGL(k_grads<5>, grid1, block1, 0, c->stream, c->pred, c->y, c->grad, c->N, am, pn, c->tree.pred, c->unit_w ? 1 : 0);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

// Adds the pending leaf values of the last tree to the predictions, row by row.
__global__ __launch_bounds__(256) void k_apply_leaf(float *__restrict__ pred, const uint32_t *__restrict__ nidx,
                                                   const float *__restrict__ leaf, int64_t N, int K, int loss) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < N; i += (int64_t)gridDim.x * 256)
        evt_add_leaf(pred + (size_t)K * i, leaf + (size_t)K * (nidx[i] - 1), K, loss);
}

int launch_apply_pending(evt_ctx *c) {
    if (!c->pend_pred) return EVT_OK;
    int64_t nb = (c->N + 255) / 256;
    if (nb > 4096) nb = 4096;
    hipLaunchKernelGGL(k_apply_leaf, dim3((unsigned)nb), dim3(256), 0, c->stream, c->pred, c->nidx, c->tree.pred, c->N, c->K, c->loss);
    HIPCHK(hipGetLastError());
    c->pend_pred = false;
    return EVT_OK;
}

// Unit weights: the row count stands for the weight in every histogram, so a gradient matrix handed in from outside
// must carry ones in its weight row.  Flags the first kind of violation it sees.
__global__ __launch_bounds__(256) void k_check_unit_weight(const float *__restrict__ grad, int64_t N, int NK, int32_t *errflag) {
    bool bad = false;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < N; i += (int64_t)gridDim.x * 256) bad |= grad[(size_t)NK * i + NK - 1] != 1.0f;
    if (__ballot(bad) != 0ull && (threadIdx.x & 63) == 0) *errflag = 1;
}
int launch_check_unit_weight(evt_ctx *c) {
    int64_t nb = (c->N + 255) / 256;
    if (nb > 4096) nb = 4096;
    hipLaunchKernelGGL(k_check_unit_weight, dim3((unsigned)nb), dim3(256), 0, c->stream, c->grad, c->N, c->NK, c->errflag);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

__global__ void k_absmax_clear(uint32_t *absmax, int k0, int k1) {
    const int n = k1 - k0;
    for (int i = threadIdx.x; i < n * EVT_ABSMAX_STRIPES; i += blockDim.x) absmax[(i / n) * EVT_MC_MAX_NK + k0 + i % n] = 0u;
}

// absmax over rows [k0, k1) of the current gradient matrix, into the set the next quantisation reads; the weight row's
// maximum (row NK - 1) is kept in both sets, since no gradient pass renews it
int launch_absmax_rows(evt_ctx *c, int k0, int k1) {
    int64_t nb = (c->N + 255) / 256;
    if (nb > 2048) nb = 2048;
    for (int pass = 0; pass < 2; pass++) {
        uint32_t *am = absmax_set(c, pass == 0 ? c->absmax_cur : c->absmax_other);
        const int a0 = pass == 0 ? k0 : std::max(k0, c->NK - 1);
        if (a0 >= k1) continue;
        hipLaunchKernelGGL(k_absmax_clear, dim3(1), dim3(256), 0, c->stream, am, a0, k1);
        HIPCHK(hipGetLastError());
        hipLaunchKernelGGL(k_absmax, dim3((unsigned)nb), dim3(256), 0, c->stream, c->grad, c->N, c->NK, a0, k1, am);
        HIPCHK(hipGetLastError());
    }
    return EVT_OK;
}

// The tables the gradients at hand are quantised with: the set the last grown tree does not use, whose histogram stays decodable
void quant_set(evt_ctx *c) {
    c->q_cur = c->q_tree ^ 1;
    c->qexp = c->qexp_buf[c->q_cur];
    c->qscale = c->qscale_buf[c->q_cur];
}

void quant_args(evt_ctx *c, QuantArgs &Q) {
    Q.grad = c->grad;
    Q.gq = c->gq;
    Q.N = c->N;
    Q.NK = c->NK; Q.NA = c->NA; Q.NAg = c->NAg; Q.loss = c->loss;
    Q.two = EVT_TWO_CHAN(c->loss, c->K) ? 1 : 0;
    Q.unit_w = c->unit_w ? 1 : 0;
    Q.pack = (c->unit_w && c->NA <= EVT_MAX_NA) ? 1 : 0;
    Q.pack_wide = (c->unit_w && c->NA > EVT_MAX_NA) ? 1 : 0;
    Q.stride = c->gq_rows ? EVT_GQ_STRIDE(c->NA) : 0;
    Q.absmax = absmax_set(c, c->absmax_cur);
    Q.absmax_next = absmax_set(c, c->absmax_other);
    Q.qbits = c->qbits;
    Q.qexp = c->qexp;
    Q.qscale = c->qscale;
}

// Blocks of `threads` that quantise.  Every block derives the multipliers first: fewer where a row is one word (1M rows, at most 1024 | 4096 blocks of
// 256: 5.4 | 6.5 us; four words a row at 500k rows 7.8 | 6.9, one word at 10M 27.6 | 25.5)
unsigned quant_blocks(const evt_ctx *c, int threads) {
    const int64_t most = (c->NA == 1 && c->N <= (int64_t)4 << 20 ? 1024 : 4096) * 256 / threads;
    return (unsigned)std::min<int64_t>(most, ((c->N << quant_lanes_sh(c->NA)) + threads - 1) / threads);
}

void quant_taken(evt_ctx *c) {
    c->quant_pending = false;
    std::swap(c->absmax_cur, c->absmax_other); // the next gradient pass raises the set that the quantisation cleared
}

int launch_quantize(evt_ctx *c) {
    quant_set(c);
    QuantArgs Q;
    quant_args(c, Q);
    hipLaunchKernelGGL(k_quantize, dim3(quant_blocks(c, 256)), dim3(256), 0, c->stream, Q);
    HIPCHK(hipGetLastError());
    quant_taken(c);
    return EVT_OK;
}

// The layout that a tree's kernels read.  Words that are still to be made are made in it; words that an earlier tree has made in the other (a
// tree of the other form on the same gradients) are made again.
int gq_layout(evt_ctx *c, bool rows) {
    rows = rows && c->NA > 1;
    if (c->gq_rows == rows) return EVT_OK;
    c->gq_rows = rows;
    if (c->quant_pending) return EVT_OK;
    QuantArgs Q;
    quant_args(c, Q);
    Q.absmax = nullptr;
    hipLaunchKernelGGL(k_quantize, dim3(quant_blocks(c, 256)), dim3(256), 0, c->stream, Q);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

// ---- evaluation metric ------------------------------------------------------------------------
// Per row value of src/metrics.jl:1-28 (:88-91 for gaussian_mle) in Float32, weighted as eval[i] = w * v / K
// (:43, :111), accumulated in Float64.  Two stages with a fixed shape (EVT_METRIC_BLOCKS partial sums, then one
// block's) keep the summation order, hence the result, independent of scheduling.
__device__ __forceinline__ float metric_value_one(int metric, float pk, float yk);
// T: target columns of y (K, or 1 when every output is measured against the one target: _target(y::AbstractVector, k, i) = y[i],
// src/loss.jl:49).  alphas: the levels of the quantile metrics as Float32 (src/callback.jl:62-66).
__device__ __forceinline__ float metric_value(int metric, int K, int T, const float *__restrict__ pred, const float *__restrict__ y, int64_t i,
                                              const float *__restrict__ alphas) {
    if (metric == EVT_METRIC_QUANTILE || metric == EVT_METRIC_MULTIQUANTILE) { // src/metrics.jl:4-6, :83-84, :117-134
        float acc = 0.0f;
        for (int k = 0; k < K; k++) {
            const float pk = pred[(size_t)K * i + k], yk = y[(size_t)T * i + (T == 1 ? 0 : k)];
            const float alpha = (metric == EVT_METRIC_MULTIQUANTILE) ? alphas[k] : alphas[0];
            acc += alpha * fmaxf(yk - pk, 0.0f) + (1.0f - alpha) * fmaxf(pk - yk, 0.0f);
        }
        return acc;
    }
    if (metric == EVT_METRIC_MLOGLOSS) { // src/metrics.jl:59-77
        float isum = 0.0f;
        for (int k = 0; k < K; k++) isum += expf(pred[(size_t)K * i + k]);
        return logf(isum) - pred[(size_t)K * i + (int)y[i] - 1];
    }
    if (metric == EVT_METRIC_GAUSSIAN_MLE || metric == EVT_METRIC_LOGISTIC_MLE) { // src/metrics.jl:84-114: summed over the targets
        const int T = K / 2;
        float acc = 0.0f;
        for (int t = 0; t < T; t++) {
            const float loc = pred[(size_t)K * i + 2 * t], scale = dev_softplus(pred[(size_t)K * i + 2 * t + 1]);
            if (metric == EVT_METRIC_GAUSSIAN_MLE) {
                const float d = y[(size_t)T * i + t] - loc;
                acc += -(logf(scale) + (d * d) / (2.0f * (scale * scale)));
            } else {
                const float az = fabsf((y[(size_t)T * i + t] - loc) / scale);
                acc += -logf(scale) - az - 2.0f * log1pf(expf(-az));
            }
        }
        return acc;
    }
    float acc = 0.0f; // src/metrics.jl:39-43: the per-target values are added in Float32, starting from zero
    for (int k = 0; k < K; k++) acc += metric_value_one(metric, pred[(size_t)K * i + k], y[(size_t)T * i + (T == 1 ? 0 : k)]);
    return acc;
}

__device__ __forceinline__ float metric_value_one(int metric, float pk, float yk) {
    switch (metric) {
    case EVT_METRIC_MSE:
    case EVT_METRIC_RMSE: return (pk - yk) * (pk - yk);
    case EVT_METRIC_MAE: return fabsf(pk - yk);
    case EVT_METRIC_LOGLOSS: {
        const float s = dev_sigmoid(pk);
        return -yk * logf(s) + (yk - 1.0f) * logf(1.0f - s);
    }
    case EVT_METRIC_POISSON: {
        const float e = expf(pk);
        return 2.0f * (yk * logf(yk / e + 7.105427357601002e-15f) + e - yk); // eps(Float32(1e-7)) = 2^-47
    }
    case EVT_METRIC_GAMMA: {
        const float e = expf(pk);
        return 2.0f * (logf(e / yk) + yk / e - 1.0f);
    }
    default: {
        const float e = expf(pk);
        return 2.0f * (powf(yk, 0.5f) / (-0.5f) / 0.5f - yk * powf(e, -0.5f) / (-0.5f) + powf(e, 0.5f) / 0.5f);
    }
    }
}

__device__ __forceinline__ double block_sum_f64(double v, double *s_red) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = v;
    __syncthreads();
    return (s_red[0] + s_red[1]) + (s_red[2] + s_red[3]);
}

// The block that leaves its sums last adds them up and stores the metric in host memory: two launches fewer per round than with a kernel for that and one
// for the store (and a tree goes up in one copy): 100k x 10 with 25k eval rows, 200 rounds 20.8 -> 19.9 ms.
__global__ __launch_bounds__(256) void k_metric(const float *__restrict__ pred, const float *__restrict__ y,
                                                       const float *__restrict__ grad, int64_t N, int NK, int K, int T, int metric, float kdiv,
                                                       const float *__restrict__ alphas, double *partial, int *count, double *out) {
    __shared__ double s_red[4];
    __shared__ int s_last;
    double num = 0.0, den = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < N; i += (int64_t)gridDim.x * 256) {
        const float w = grad[(size_t)NK * i + NK - 1];
        const float ev = w * metric_value(metric, K, T, pred, y, i, alphas) / kdiv;
        num += (double)ev;
        den += (double)w;
    }
    num = block_sum_f64(num, s_red);
    den = block_sum_f64(den, s_red);
    if (threadIdx.x == 0) { // past the caches that are not shared, and in memory before the block is counted
        __hip_atomic_store(partial + 2 * blockIdx.x, num, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(partial + 2 * blockIdx.x + 1, den, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        s_last = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1;
    }
    __syncthreads();
    if (!s_last) return;
    num = den = 0.0;
    for (int b = threadIdx.x; b < (int)gridDim.x; b += 256) {
        num += __hip_atomic_load(partial + 2 * b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        den += __hip_atomic_load(partial + 2 * b + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    num = block_sum_f64(num, s_red);
    den = block_sum_f64(den, s_red);
    if (threadIdx.x == 0) {
        const double r = num / den;
        out[0] = (metric == EVT_METRIC_RMSE) ? sqrt(r) : r;
        *count = 0; // for the next launch
    }
}

// the metric lands in `out`, the caller's pinned buffer
int launch_eval_metric(evt_ctx *c, int metric, double *out) {
    int64_t nb = (c->N + 255) / 256;
    if (nb > EVT_METRIC_BLOCKS) nb = EVT_METRIC_BLOCKS;
    const float kdiv = (metric == EVT_METRIC_MLOGLOSS) ? 1.0f : (float)((metric == EVT_METRIC_GAUSSIAN_MLE || metric == EVT_METRIC_LOGISTIC_MLE) ? c->K / 2 : c->K);
    // y has K columns for the losses whose outputs each have a target; the multi-class, two-parameter and multiquantile
    // metrics index their own layouts
    const int T = (c->loss == EVT_LOSS_MULTIQUANTILE) ? 1 : c->K;
    hipLaunchKernelGGL(k_metric, dim3((unsigned)nb), dim3(256), 0, c->stream, c->pred, c->y, c->grad, c->N, c->NK, c->K, T, metric, kdiv,
                       c->alphas_f, c->metric_partial, reinterpret_cast<int *>(c->metric_partial + 2 * EVT_METRIC_BLOCKS), out);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}
