// What the split-search kernels share: wavefront primitives and the Float64 gain algebra (src/split.jl:1-141; src/predict.jl:198-262).
#pragma once
#include "evt_internal.h"
#include <float.h>

#define NO_BIN 0x7fffffff

// ---- wavefront primitives -----------------------------------------------------------------
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ long long dpp_move_i64(long long x) {
    int lo = (int)(x & 0xffffffffll), hi = (int)(x >> 32);
    lo = __builtin_amdgcn_update_dpp(0, lo, CTRL, ROW_MASK, 0xf, false);
    hi = __builtin_amdgcn_update_dpp(0, hi, CTRL, ROW_MASK, 0xf, false);
    return ((long long)hi << 32) | (unsigned int)lo;
}

// Inclusive prefix sum over the 64 lanes of a wavefront.
// row_shr:1,2,4,8 scan each row of 16 lanes; row_bcast:15 then row_bcast:31 carry row totals forward.
__device__ __forceinline__ long long wave_incl_scan_i64(long long x) {
    x += dpp_move_i64<0x111, 0xf>(x); // row_shr:1
    x += dpp_move_i64<0x112, 0xf>(x); // row_shr:2
    x += dpp_move_i64<0x114, 0xf>(x); // row_shr:4
    x += dpp_move_i64<0x118, 0xf>(x); // row_shr:8
    x += dpp_move_i64<0x142, 0xa>(x); // row_bcast:15 into rows 1 and 3
    x += dpp_move_i64<0x143, 0xc>(x); // row_bcast:31 into rows 2 and 3
    return x;
}

__device__ __forceinline__ long long readlane_i64(long long x, int lane) {
    const int lo = __builtin_amdgcn_readlane((int)(x & 0xffffffffll), lane), hi = __builtin_amdgcn_readlane((int)(x >> 32), lane);
    return ((long long)hi << 32) | (unsigned int)lo;
}

// Sum over the wavefront, in every lane: the scan's last lane (VALU moves; twelve cross-lane shuffles are as many trips through the LDS crossbar)
__device__ __forceinline__ long long wave_sum_i64(long long x) { return readlane_i64(wave_incl_scan_i64(x), 63); }

// Maximum over the 64 lanes of a wavefront (ROW: over the first 16), no value a NaN: the scan's moves, a lane without a source meeting itself.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double max_step_f64(double g) {
    const long long v = __double_as_longlong(g);
    const int lo = (int)(v & 0xffffffffll), hi = (int)(v >> 32);
    const double o = __longlong_as_double(((long long)__builtin_amdgcn_update_dpp(hi, hi, CTRL, ROW_MASK, 0xf, false) << 32) |
                                          (unsigned int)__builtin_amdgcn_update_dpp(lo, lo, CTRL, ROW_MASK, 0xf, false));
    double m;
    asm("v_max_f64 %0, %1, %2" : "=v"(m) : "v"(g), "v"(o)); // fmax first makes a quiet NaN of either that is a signalling one
    return m;
}
template <bool ROW = false>
__device__ __forceinline__ double wave_max_f64(double g) {
    g = max_step_f64<0x111, 0xf>(g); // row_shr:1
    g = max_step_f64<0x112, 0xf>(g); // row_shr:2
    g = max_step_f64<0x114, 0xf>(g); // row_shr:4
    g = max_step_f64<0x118, 0xf>(g); // row_shr:8
    if (!ROW) {
        g = max_step_f64<0x142, 0xa>(g); // row_bcast:15 into rows 1 and 3
        g = max_step_f64<0x143, 0xc>(g); // row_bcast:31 into rows 2 and 3
    }
    return __longlong_as_double(readlane_i64(__double_as_longlong(g), ROW ? 15 : 63));
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ int min_step(int v) {
    const int o = __builtin_amdgcn_update_dpp(v, v, CTRL, ROW_MASK, 0xf, false);
    return o < v ? o : v;
}

// Arg-max over the 64 lanes of a wavefront (ROW: the first 16): highest gain, of equal gains the lowest bin (NO_BIN: no gain); every lane gets the result.
// The maximum alone goes through the moves; which lane has it is a ballot, and the lowest bin is looked for only where several have it.  Gain and bin taken
// through the moves together cost 80 instructions for 45.  us a launch of the split search: 10M x 100, depth 11, whose deep levels are bound by their instructions, 15.4 -> 14.6, 800k x 28 of
// 128 bins 9.6 -> 9.15, 500k x 50 of two outputs, oblivious, 9.5 -> 9.1, 7 classes 9.55 -> 8.9; k_small_level 11.0 -> 10.7, k_small_final 8.6 -> 8.25 (100k x 10).
template <bool ROW = false>
__device__ __forceinline__ void wave_argmax(double &g, int &b) {
    const double m = wave_max_f64<ROW>(g);
    unsigned long long who = __ballot(g == m && b != NO_BIN);
    if (ROW) who &= 0xFFFFull;
    if (who == 0ull) {
        g = m;
        b = NO_BIN;
        return;
    }
    if (who & (who - 1ull)) {
        int v = (who >> (threadIdx.x & 63)) & 1ull ? b : NO_BIN;
        v = min_step<0x111, 0xf>(v);
        v = min_step<0x112, 0xf>(v);
        v = min_step<0x114, 0xf>(v);
        v = min_step<0x118, 0xf>(v);
        v = min_step<0x142, 0xa>(v);
        v = min_step<0x143, 0xc>(v);
        const int lowest = __builtin_amdgcn_readlane(v, 63);
        who &= __ballot(b == lowest);
    }
    const int lane = __builtin_ctzll(who);
    g = __longlong_as_double(readlane_i64(__double_as_longlong(g), lane));
    b = __builtin_amdgcn_readlane(b, lane);
}

// ---- Float64 gain algebra, expression order as in the reference ------------------------------
__device__ __forceinline__ double term_gh(double g, double h, double w, double lambda, double L2) {
    double d = h + lambda * w + L2;
    if (!(d > DBL_EPSILON)) d = DBL_EPSILON;
    return g * g / d / 2.0;
}

// fixed-point channel sums -> the 2K+1 Float64 statistics [g.., h.., w]
__device__ __forceinline__ void decode_vals(const long long *q, const double *sc, int loss, int NK, double *out) {
    if (EVT_TWO_CHAN(loss, (NK - 1) / 2)) { // one-target mse / mae: channels {g, w}; h = 2w (mse), 0 (mae)
        double w = (double)q[1] * sc[1];
        out[0] = (double)q[0] * sc[0];
        out[1] = (loss == EVT_LOSS_MSE) ? 2.0 * w : 0.0;
        out[2] = w;
    } else {
        for (int k = 0; k < NK; k++) out[k] = (double)q[k] * sc[k];
    }
}

// _term_cred with _cred_Z (src/split.jl:3-4, src/loss.jl:275-290): Z |m1| / (1 + L2 / w), Z = VHM / (VHM + EVPV) for
// cred_var and the same ratio of square roots for cred_std, VHM = (m1 / w)^2, EVPV = max(eps, m2 / w - VHM)
__device__ __forceinline__ double term_cred(int loss, double m1, double m2, double w, double L2) {
    const double mean = m1 / w;
    const double VHM = mean * mean;
    double EVPV = m2 / w - VHM;
    if (!(EVPV > DBL_EPSILON)) EVPV = DBL_EPSILON;
    const double Z = (loss == EVT_LOSS_CRED_VAR) ? VHM / (VHM + EVPV) : sqrt(VHM) / (sqrt(VHM) + sqrt(EVPV));
    return Z * fabs(m1) / (1.0 + L2 / w);
}

// One output's term of node_gain (src/split.jl:58-78): zero for mae.
__device__ __forceinline__ double node_gain_k(int loss, double g, double h, double w, double lambda, double L2) {
    if (EVT_IS_SHIFT(loss)) return 0.0;
    if (EVT_IS_CRED(loss)) return term_cred(loss, g, h, w, L2);
    return term_gh(g, h, w, lambda, L2);
}

// One output's term of split_gain (src/split.jl:108-141): left + right.  (Sg, Sh, w_p) are the node's totals.  mae:
// _term_shift (src/split.jl:2), |g / w - mu_p| w / d on either side with d = max(eps, 1 + lambda + L2 / w).
__device__ __forceinline__ double split_gain_k(int loss, double Sg, double Sh, double w_p, double g_l, double h_l, double w_l, double w_r,
                                               double lambda, double L2) {
    if (EVT_IS_SHIFT(loss)) {
        double d_l = 1.0 + lambda + L2 / w_l, d_r = 1.0 + lambda + L2 / w_r;
        if (!(d_l > DBL_EPSILON)) d_l = DBL_EPSILON;
        if (!(d_r > DBL_EPSILON)) d_r = DBL_EPSILON;
        const double mu_p = Sg / w_p;
        return fabs(g_l / w_l - mu_p) * w_l / d_l + fabs((Sg - g_l) / w_r - mu_p) * w_r / d_r;
    }
    if (EVT_IS_CRED(loss)) return term_cred(loss, g_l, h_l, w_l, L2) + term_cred(loss, Sg - g_l, Sh - h_l, w_r, L2);
    return term_gh(g_l, h_l, w_l, lambda, L2) + term_gh(Sg - g_l, Sh - h_l, w_r, lambda, L2);
}

// pred_leaf_cpu! / pred_scalar (src/predict.jl:198-262) for output k
__device__ __forceinline__ double leaf_value(int loss, const double *S, int k, int K, double eta, int bagging, double lambda, double L2) {
    if (EVT_IS_QUANTILE(loss)) return 0.0; // valued from the leaf's rows once the tree is complete (launch_quantile_leaves)
    if (EVT_IS_CRED(loss)) return eta / (double)bagging * S[k] / (S[2 * K] + L2);
    if (loss == EVT_LOSS_MAE) {
        double d = S[2 * K] + lambda * S[2 * K] + L2;
        if (!(d > DBL_EPSILON)) d = DBL_EPSILON;
        return eta / (double)bagging * S[k] / d;
    }
    double d = S[K + k] + lambda * S[2 * K] + L2;
    if (!(d > DBL_EPSILON)) d = DBL_EPSILON;
    return -eta / (double)bagging * S[k] / d;
}
