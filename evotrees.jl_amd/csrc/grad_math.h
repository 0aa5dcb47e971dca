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
