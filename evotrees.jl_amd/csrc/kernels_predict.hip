// Tree traversal: predict! (src/predict.jl:1-46), predict_leaf_idx! (:138-154), _predict (:118-136).
//
// A node is packed in one 32-bit word (feat | cond_bin << 16 | split << 24 | numeric << 25) so that each
// visited node costs one 4-byte load and nothing else has to be looked up.  Rows are independent; per row the
// walk reads one bin byte per level, from the column-major x_bin (neighbouring rows share 64-byte sectors of
// a column) or, in the whole-model kernel, from a copy of the block's rows in LDS.
#include "grad_math.h"
#include <algorithm>

__device__ __forceinline__ int walk_packed(const uint32_t *__restrict__ nodes, const uint8_t *__restrict__ xcm, int64_t N, int64_t i) {
    int nid = 1;
    uint32_t nd = nodes[0];
    while (nd & EVT_NODE_SPLIT) {
        const int feat = (int)(nd & 0xFFFFu);
        const uint32_t cb = (nd >> 16) & 0xFFu;
        const uint32_t xb = xcm[(size_t)(feat - 1) * N + i];
        const bool cond = (nd & EVT_NODE_NUMERIC) ? (xb <= cb) : (xb == cb);
        nid = (nid << 1) + (cond ? 0 : 1);
        nd = nodes[nid - 1];
    }
    return nid;
}

// one tree added to pred (K x N), all rows.  blob.blocks extra blocks at the end of the grid send the finished tree to the host, when this is its last kernel.
// A row's walk is a chain of dependent loads (node word, bin byte, node word, ...), so the kernel is paced by latency, not by
// the bytes it moves: the first n_lds node words (the upper levels of the heap, all of it for depths up to 13) are copied to
// LDS, where a lookup costs a fraction of a trip to the caches, and a thread walks R rows side by side - R bin bytes are
// requested before the first is used.  Rows of a thread are 256 apart: the threads of a wavefront read neighbouring bytes.
// LOSS >= 0: the next round's gradients are computed as well, as k_grads<LOSS> would from the predictions it read again; what they need is requested
// ahead of the walk (walk + gradients, us: 1M rows, depth 6 9.8 + 5.8 and a launch -> 11.8; 1M rows, depth 8 10.9 + 5.5 -> 14.2).
struct GradOut {
    const float *y;
    float *grad;
    uint32_t *absmax;
    int unit_w;
};
template <int R, int LOSS>
__global__ __launch_bounds__(LOSS < 0 ? 256 : 1024) void k_predict_tree(const uint32_t *__restrict__ nodes, int n_lds, const float *__restrict__ leaf_pred,
                                                     const uint8_t *__restrict__ xcm, int64_t N, int K, int loss, float *pred,
                                                     BlobOut blob, GradOut O) {
    extern __shared__ uint32_t s_nodes[];
    constexpr bool GRADS = LOSS >= 0;
    constexpr int KG = LOSS == 2 || LOSS == 7 ? 2 : 1, NKG = 2 * KG + 1;
    const int nthr = GRADS ? (int)blockDim.x : 256;
    const int64_t G = (int64_t)gridDim.x - blob.blocks;
    if ((int64_t)blockIdx.x >= G) {
        blob_send(blob, (int)(blockIdx.x - G));
        return;
    }
    const int64_t i0 = (int64_t)blockIdx.x * (nthr * R) + threadIdx.x;
    float pr[R][KG], y[R], w[R];
    if constexpr (GRADS) {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int64_t i = i0 + nthr * r < N ? i0 + nthr * r : N - 1;
#pragma unroll
            for (int k = 0; k < KG; k++) pr[r][k] = pred[(size_t)KG * i + k];
            y[r] = O.y[i];
            w[r] = 1.0f;
            if (!O.unit_w) w[r] = O.grad[(size_t)NKG * i + NKG - 1];
        }
    }
    for (int k = threadIdx.x; k < n_lds; k += nthr) s_nodes[k] = nodes[k];
    __syncthreads();
    int nid[R];
    uint32_t nd[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        nid[r] = 1;
        nd[r] = (i0 + nthr * r < N) ? s_nodes[0] : 0u; // a row past the end walks nothing
    }
    for (;;) {
        uint32_t xb[R];
        bool any = false;
#pragma unroll
        for (int r = 0; r < R; r++) {
            xb[r] = 0;
            if (nd[r] & EVT_NODE_SPLIT) {
                xb[r] = xcm[(size_t)((nd[r] & 0xFFFFu) - 1) * N + (i0 + nthr * r)];
                any = true;
            }
        }
        if (!any) break;
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (nd[r] & EVT_NODE_SPLIT) {
                const uint32_t cb = (nd[r] >> 16) & 0xFFu;
                const bool cond = (nd[r] & EVT_NODE_NUMERIC) ? (xb[r] <= cb) : (xb[r] == cb);
                nid[r] = (nid[r] << 1) + (cond ? 0 : 1);
                nd[r] = (nid[r] - 1 < n_lds) ? s_nodes[nid[r] - 1] : nodes[nid[r] - 1];
            }
        }
    }
    if constexpr (GRADS) {
        __shared__ float s_m[16][2 * KG];
        float mx[2 * KG];
#pragma unroll
        for (int k = 0; k < 2 * KG; k++) mx[k] = 0.0f;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int64_t i = i0 + nthr * r;
            float out[2 * KG];
            evt_add_leaf(pr[r], leaf_pred + (size_t)KG * (nid[r] - 1), KG, LOSS);
            grad_row<LOSS>(pr[r], y[r], w[r], out);
            if (i < N) {
#pragma unroll
                for (int k = 0; k < KG; k++) pred[(size_t)KG * i + k] = pr[r][k];
#pragma unroll
                for (int k = 0; k < 2 * KG; k++) {
                    O.grad[(size_t)NKG * i + k] = out[k];
                    mx[k] = fmaxf(mx[k], fabsf(out[k]));
                }
            }
        }
        absmax_raise_block<2 * KG>(mx, s_m, O.absmax);
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int64_t i = i0 + nthr * r;
            if (i < N) evt_add_leaf(pred + (size_t)K * i, leaf_pred + (size_t)K * (nid[r] - 1), K, loss);
        }
    }
}

// rows per thread: four once the rows fill the device several times over, one for small inputs (more blocks)
// grads: with the next round's gradients.  Blocks raise the maxima one after the other, so that those of large inputs are wide and walk two rows a thread (1M rows,
// depth 6 | depth 8: blocks of 256 15.1 | 17.7 us, 512 14.1 | 16.3, 1024 13.1 | 15.3, 1024 and two rows 11.8 | 14.2).
static int launch_predict_tree_any(evt_ctx *c, const uint32_t *nodes, int nnodes, const float *leaf_pred, const BlobOut &blob, bool grads) {
    const int n_lds = nnodes < 8192 ? nnodes : 8192;
    const size_t lds = (size_t)n_lds * sizeof(uint32_t);
    const GradOut O = {c->y, c->grad, absmax_set(c, c->absmax_cur), c->unit_w ? 1 : 0};
    const bool wide = grads && c->N > 2047 * 256;
    const int R = c->N >= ((int64_t)1 << 21) ? 4 : wide ? 2 : 1, threads = wide ? 1024 : 256;
    const dim3 grid((unsigned)((c->N + threads * R - 1) / (threads * R)) + (unsigned)blob.blocks);
#define PT(R_, LOSS_)                                                                                                                               \
    hipLaunchKernelGGL((k_predict_tree<R_, LOSS_>), grid, dim3(threads), lds, c->stream, nodes, n_lds, leaf_pred, c->xcm, c->N, c->K, c->loss, c->pred, \
                       blob, O)
#define PT1(LOSS_) PT(1, LOSS_)
#define PT2(LOSS_) PT(2, LOSS_)
#define PT4(LOSS_) PT(4, LOSS_)
    if (!grads) {
        if (R == 4) PT4(-1);
        else PT1(-1);
    } else if (R == 4) {
        EVT_GRAD_ROW_CASES(c, PT4)
    } else if (R == 2) {
        EVT_GRAD_ROW_CASES(c, PT2)
    } else {
        EVT_GRAD_ROW_CASES(c, PT1)
    }
#undef PT4
#undef PT2
#undef PT1
#undef PT
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

// node each sampled row of the last tree ended in (0 outside the sample): the walk reproduces the
// partition's decisions row by row (update_nodes_idx!, ext/EvoTreesKernelAbstractionsExt/fit-utils.jl:9-31)
__global__ __launch_bounds__(256) void k_nidx_from_tree(const uint32_t *__restrict__ nodes, const uint8_t *__restrict__ xcm, int64_t N,
                                                       const uint8_t *__restrict__ mask, uint32_t cond, uint32_t *out) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= N) return;
    uint32_t r = 0;
    if (!mask || mask[i] <= cond) r = (uint32_t)walk_packed(nodes, xcm, N, i);
    out[i] = r;
}

int launch_nidx_from_tree(evt_ctx *c, bool use_mask, uint8_t cond) {
    hipLaunchKernelGGL(k_nidx_from_tree, dim3((unsigned)((c->N + 255) / 256)), dim3(256), 0, c->stream, c->tree.packed, c->xcm, c->N,
                       use_mask ? c->mask : nullptr, (uint32_t)cond, c->nidx);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

int launch_predict_tree_cache(evt_ctx *c, bool send_blob, bool grads) {
    BlobOut blob = {};
    if (send_blob) blob_out(c, blob);
    const int r = launch_predict_tree_any(c, c->tree.packed, c->nnodes, c->tree.pred, blob, grads);
    if (r != EVT_OK) return r;
    if (send_blob) c->step.blob_sent = true;
    if (grads) c->step.grads_done = true;
    return EVT_OK;
}

int launch_predict_tree_nodes(evt_ctx *c, const uint32_t *nodes_dev, int nnodes, const float *leaf_pred_dev) {
    return launch_predict_tree_any(c, nodes_dev, nnodes, leaf_pred_dev, BlobOut{}, false);
}

// apply_prediction_link!, src/predict.jl:105-116 (softmax!: :187-195)
template <int KMAX>
__device__ __forceinline__ void apply_link(float *acc, int K, int loss) {
    if (loss == EVT_LOSS_LOGLOSS) {
        for (int k = 0; k < K; k++) acc[k] = 1.0f / (1.0f + expf(-acc[k]));
    } else if (EVT_IS_MLE2P(loss)) {
        for (int k = 1; k < K; k += 2) acc[k] = fmaxf(acc[k], 0.0f) + log1pf(expf(-fabsf(acc[k])));
    } else if (loss == EVT_LOSS_MLOGLOSS) {
        float isum = 0.0f;
#pragma unroll
        for (int k = 0; k < KMAX; k++) {
            if (k < K) {
                acc[k] = expf(acc[k]);
                isum += acc[k];
            }
        }
#pragma unroll
        for (int k = 0; k < KMAX; k++) acc[k] /= isum;
    } else if (loss >= EVT_LOSS_POISSON && loss <= EVT_LOSS_TWEEDIE) {
        for (int k = 0; k < K; k++) acc[k] = expf(acc[k]);
    }
}

// acc += leaf values of one tree, with the per-tree clamps of predict! (src/predict.jl:1-84)
template <int KMAX>
__device__ __forceinline__ void add_tree(float *acc, const float *lp, int K, int loss) {
    if (KMAX <= 4) {
        evt_add_leaf(acc, lp, K, loss);
    } else { // many outputs: constant trip counts keep the running prediction in registers
        float m = -INFINITY;
#pragma unroll
        for (int k = 0; k < KMAX; k++) {
            if (k < K) {
                acc[k] += lp[k];
                m = fmaxf(m, acc[k]);
            }
        }
        if (loss == EVT_LOSS_MLOGLOSS) {
#pragma unroll
            for (int k = 0; k < KMAX; k++) acc[k] = fmaxf(-15.0f, acc[k] - m);
        } else if (loss == EVT_LOSS_LOGLOSS) { // several targets: each clamped to [-15, 15]
#pragma unroll
            for (int k = 0; k < KMAX; k++) acc[k] = fminf(fmaxf(acc[k], -15.0f), 15.0f);
        } else if (EVT_IS_MLE2P(loss)) { // (location, raw scale) pairs: the scale outputs are floored at -15
#pragma unroll
            for (int k = 1; k < KMAX; k += 2) acc[k] = fmaxf(-15.0f, acc[k]);
        }
    }
}

// whole model: trees concatenated, tree t owns nodes [off[t], off[t+1]); the running prediction
// stays in registers and is written once.  The per-tree clamps are applied after every tree, as
// predict! does.  This variant gathers bin bytes from global memory: any tree size, any feature count.
template <int KMAX>
__global__ __launch_bounds__(256) void k_predict_model(const uint32_t *__restrict__ nodes, const float *__restrict__ leaf_pred,
                                                      const int64_t *__restrict__ off, int ntrees, const uint8_t *__restrict__ xcm, int64_t N,
                                                      int K, int loss, int link, float *out, const int32_t *__restrict__ skip_flag) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= N) return;
    if (skip_flag && *skip_flag) return; // the model was packed on the device and found invalid: nothing is walked
    float acc[KMAX];
#pragma unroll
    for (int k = 0; k < KMAX; k++) acc[k] = 0.0f;
    for (int t = 0; t < ntrees; t++) {
        const int64_t o = off[t];
        const int nid = walk_packed(nodes + o, xcm, N, i);
        add_tree<KMAX>(acc, leaf_pred + (size_t)K * (o + nid - 1), K, loss);
    }
    if (link) apply_link<KMAX>(acc, K, loss);
#pragma unroll
    for (int k = 0; k < KMAX; k++)
        if (k < K) out[(size_t)K * i + k] = acc[k];
}

// Whole model with the walk entirely in LDS, over trees the host has completed: every leaf above a tree's last
// level is replaced by a chain of nodes that always go left down to that level and carry its value there, so every
// row walks exactly depth - 1 levels of every tree.  No lane leaves the loop early, nothing is tested but the bin,
// and the leaf is found by position.  (Leaf indices of the original tree are what evt_predict_leaf_idx is for.)
//
// A block copies its RB rows into LDS once - the only pass over x_bin - laid out so that row r of a wavefront owns
// LDS bank r: word k of the row (features 4k .. 4k+3) sits at word (wave * S4 + k) * 64 + lane, so the 64 lanes read
// their bin bytes without bank conflicts whatever features their nodes test.  A tree's internal nodes sit in LDS too,
// double buffered (the next tree's words are requested before the walk and stored after it): a level costs two LDS
// reads and no trip to memory.  A node word is byte offset of the feature inside the row's words | cond_bin << 16 |
// numeric << 25.  The leaf values of a tree are requested after its walk and added after the next tree's, in order.
template <bool ALLNUM>
__device__ __forceinline__ uint32_t step_node(uint32_t nid, uint32_t nd, uint32_t xb) {
    const uint32_t cb = (nd >> 16) & 0xFFu;
    if (ALLNUM) return __builtin_amdgcn_alignbit(nid, cb - xb, 31); // (nid << 1) | (bin > cond_bin)
    const bool right = (nd & EVT_NODE_NUMERIC) ? (xb > cb) : (xb != cb);
    return 2 * nid + (right ? 1u : 0u);
}

struct ModelTree {
    int32_t node_off; // first internal node in the node array
    int32_t leaf_off; // first last-level leaf in the value array
    int32_t levels;   // depth - 1: levels walked
    int32_t n_int;    // internal nodes: 2^levels - 1
};

// NT trees are walked side by side (NT independent chains of LDS reads per lane hide each other's latency); groups of
// NT trees are double buffered.  PRE = words of the next group each thread carries across the walk (>= NT * max_int / RB).
template <int KMAX, int RB, int NT, int PRE, bool ALLNUM>
__global__ __launch_bounds__(RB) void k_predict_model_lds(const uint32_t *__restrict__ cnodes, const float *__restrict__ cleaf,
                                                         const ModelTree *__restrict__ meta, int ntrees, const uint8_t *__restrict__ xcm,
                                                         int64_t N, int F, int S4, int max_int, int K, int ks, int loss, int link, float *out) {
    extern __shared__ uint32_t smem[];
    uint32_t *T = smem;                                                        // [2][NT][max_int]
    uint8_t *R = reinterpret_cast<uint8_t *>(smem + 2 * (size_t)NT * max_int); // [RB / 64][S4][64] words
    const int tid = threadIdx.x;
    const int64_t i = (int64_t)blockIdx.x * RB + tid;
    const bool live = i < N;
    const int64_t ic = live ? i : N - 1;
    uint8_t *Rw = R + ((size_t)(tid >> 6) * S4 * 64 + (tid & 63)) * 4; // byte f of this row: Rw[(f >> 2) * 256 + (f & 3)]
    // a column at a time (RB consecutive bytes per request), 16 columns requested before the first is stored: the copy
    // costs F / 16 trips to memory, not F
    for (int f0 = 0; f0 < F; f0 += 16) {
        uint8_t v[16];
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const int f = f0 + j < F ? f0 + j : F - 1;
            v[j] = xcm[(size_t)f * N + ic];
        }
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const int f = f0 + j;
            if (f < F) Rw[(f >> 2) * 256 + (f & 3)] = v[j];
        }
    }
    const int ngroups = (ntrees + NT - 1) / NT;
    const int gw = NT * max_int; // words of one group's buffer
    // The host padded every tree to max_int words and the tree list to a whole number of groups (with trees of no
    // levels), so group g's LDS image is the plain run cnodes[g * gw, (g + 1) * gw) and meta has ngroups * NT entries.
    for (int w = tid; w < gw; w += RB) T[w] = cnodes[w];
    __syncthreads();
    float acc[KMAX], lpv[NT][KMAX];
#pragma unroll
    for (int k = 0; k < KMAX; k++) {
        acc[k] = 0.0f;
#pragma unroll
        for (int j = 0; j < NT; j++) lpv[j][k] = 0.0f;
    }
    int nprev = 0; // trees whose values wait in lpv
    for (int g = 0; g < ngroups; g++) {
        const uint32_t *Tc = T + (size_t)(g & 1) * gw;
        uint32_t *Tn = T + (size_t)((g + 1) & 1) * gw;
        ModelTree m[NT];
#pragma unroll
        for (int j = 0; j < NT; j++) m[j] = meta[g * NT + j];
        // the next group's words: requested now, stored after the walk
        uint32_t pre[PRE];
        if (g + 1 < ngroups) {
            const uint32_t *src = cnodes + (size_t)(g + 1) * gw;
#pragma unroll
            for (int q = 0; q < PRE; q++) {
                const int w = q * RB + tid;
                pre[q] = src[w < gw ? w : 0];
            }
        }
        // heap index of the node reached (1-based; children of n are 2n and 2n + 1): the sign of cond_bin - bin is the
        // step to the right, shifted in with one v_alignbit when every feature is numeric
        uint32_t nid[NT];
#pragma unroll
        for (int j = 0; j < NT; j++) nid[j] = 1;
        bool same = true;
#pragma unroll
        for (int j = 1; j < NT; j++) same = same && (m[j].levels == m[0].levels);
        if (same) { // the usual case: NT chains advance level by level together
            for (int l = 0; l < m[0].levels; l++) {
                uint32_t nd[NT], xb[NT];
#pragma unroll
                for (int j = 0; j < NT; j++) nd[j] = Tc[j * max_int + nid[j] - 1];
#pragma unroll
                for (int j = 0; j < NT; j++) xb[j] = Rw[nd[j] & 0xFFFFu];
#pragma unroll
                for (int j = 0; j < NT; j++) nid[j] = step_node<ALLNUM>(nid[j], nd[j], xb[j]);
            }
        } else {
#pragma unroll
            for (int j = 0; j < NT; j++) {
                for (int l = 0; l < m[j].levels; l++) {
                    const uint32_t nd = Tc[j * max_int + nid[j] - 1];
                    const uint32_t xb = Rw[nd & 0xFFFFu];
                    nid[j] = step_node<ALLNUM>(nid[j], nd, xb);
                }
            }
        }
        uint32_t pos[NT]; // position in the last level
#pragma unroll
        for (int j = 0; j < NT; j++) pos[j] = nid[j] - (1u << m[j].levels);
        // the previous group's values go in (tree order), then this group's are requested
#pragma unroll
        for (int j = 0; j < NT; j++)
            if (j < nprev) add_tree<KMAX>(acc, lpv[j], K, loss);
        nprev = ntrees - g * NT < NT ? ntrees - g * NT : NT;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const float *lp = cleaf + (size_t)ks * (m[j].leaf_off + pos[j]);
            if (KMAX > 4 && (ks & 3) == 0) { // rows of 4 values: 16-byte loads (the value array starts on an allocation boundary)
#pragma unroll
                for (int k = 0; k < KMAX; k += 4) {
                    if (k < K) {
                        const float4 v = *reinterpret_cast<const float4 *>(lp + k);
                        lpv[j][k] = v.x; lpv[j][k + 1] = v.y; lpv[j][k + 2] = v.z; lpv[j][k + 3] = v.w;
                    }
                }
            } else {
#pragma unroll
                for (int k = 0; k < KMAX; k++)
                    if (k < K) lpv[j][k] = lp[k];
            }
        }
        if (g + 1 < ngroups) {
#pragma unroll
            for (int q = 0; q < PRE; q++) {
                const int w = q * RB + tid;
                if (w < gw) Tn[w] = pre[q];
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < NT; j++)
        if (j < nprev) add_tree<KMAX>(acc, lpv[j], K, loss);
    if (link) apply_link<KMAX>(acc, K, loss);
    if (live) {
#pragma unroll
        for (int k = 0; k < KMAX; k++)
            if (k < K) out[(size_t)K * i + k] = acc[k];
    }
}

__global__ __launch_bounds__(256) void k_leaf_idx_model(const uint32_t *__restrict__ nodes, const int64_t *__restrict__ off, int ntrees,
                                                       const uint8_t *__restrict__ xcm, int64_t N, uint32_t *out) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= N) return;
    for (int t = 0; t < ntrees; t++) out[(size_t)t * N + i] = (uint32_t)walk_packed(nodes + off[t], xcm, N, i);
}

template <int KMAX, int RB, int NT, int PRE, bool ALLNUM>
static int launch_model_lds(hipStream_t s, const uint32_t *cnodes, const float *cleaf, const void *meta, int ntrees, const uint8_t *xcm, int64_t N,
                            int F, int max_int, int K, int ks, int loss, int apply_link, float *out) {
    static EvtDevOnce once;
    const int dev = EvtDevOnce::current();
    if (once.pending(dev)) {
        HIPCHK(hipFuncSetAttribute(reinterpret_cast<const void *>(k_predict_model_lds<KMAX, RB, NT, PRE, ALLNUM>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        once.mark(dev);
    }
    const int S4 = (F + 3) >> 2;
    const size_t lds = (size_t)RB * S4 * 4 + 8 * (size_t)NT * max_int;
    hipLaunchKernelGGL((k_predict_model_lds<KMAX, RB, NT, PRE, ALLNUM>), dim3((unsigned)((N + RB - 1) / RB)), dim3(RB), lds, s, cnodes, cleaf,
                       static_cast<const ModelTree *>(meta), ntrees, xcm, N, F, S4, max_int, K, ks, loss, apply_link, out);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

// Launch shape of the LDS kernel for this model: 1 = 1024 rows per block, 4 trees side by side (one block per CU);
// 2 = 512 rows, 2 trees (two blocks per CU); 3 = 512 rows, 1 tree; 4 = 256 rows, 1 tree; 0 = does not apply.
// A row's running prediction and the leaf values of the trees walked side by side live in registers: up to 4 outputs
// take any shape, 5 - 8 outputs at most two trees side by side, 9 - 16 outputs one tree at a time.
int predict_lds_shape(int F, int max_int, int K, int hint) {
    if (K > EVT_MAX_K || F >= 1024 || max_int < 0) return 0;
    const size_t S = 4 * (size_t)((F + 3) >> 2), mi = (size_t)(max_int > 0 ? max_int : 1);
    const int first = K <= 4 ? 1 : (K <= 8 ? 2 : 3);
    const bool fits[5] = {false, 4 * mi <= 8 * 1024 && 1024 * S + 32 * mi <= 150 * 1024, 2 * mi <= 8 * 512 && 512 * S + 16 * mi <= 80 * 1024,
                          mi <= 8 * 512 && 512 * S + 8 * mi <= 80 * 1024, mi <= 16 * 256 && 256 * S + 8 * mi <= 80 * 1024};
    if (hint >= first && hint <= 4 && fits[hint]) return hint; // a sweep's choice, when the shape allows it
    for (int sh = first; sh <= 4; sh++)
        if (fits[sh]) return sh;
    return 0;
}

// Completed trees (see k_predict_model_lds): cnodes / cleaf / meta as the host prepared them; a leaf's K values lie ks apart.
int launch_predict_model_lds(hipStream_t s, const uint32_t *cnodes, const float *cleaf, const void *meta, int ntrees, const uint8_t *xcm, int64_t N,
                             int F, int max_int, int K, int ks, int loss, int apply_link, int all_numeric, int shape, float *out) {
    const int mi = max_int > 0 ? max_int : 1;
    shape = predict_lds_shape(F, max_int, K, shape);
#define EVT_PM(KM_, RB_, NT_, PRE_)                                                                                                          \
    return all_numeric ? launch_model_lds<KM_, RB_, NT_, PRE_, true>(s, cnodes, cleaf, meta, ntrees, xcm, N, F, mi, K, ks, loss, apply_link, out) \
                       : launch_model_lds<KM_, RB_, NT_, PRE_, false>(s, cnodes, cleaf, meta, ntrees, xcm, N, F, mi, K, ks, loss, apply_link, out)
    if (K <= 4) {
        if (shape == 1) { EVT_PM(4, 1024, 4, 8); }
        if (shape == 2) { EVT_PM(4, 512, 2, 8); }
        if (shape == 3) { EVT_PM(4, 512, 1, 8); }
        if (shape == 4) { EVT_PM(4, 256, 1, 16); }
    } else if (K <= 8) {
        if (shape == 2) { EVT_PM(8, 512, 2, 8); }
        if (shape == 3) { EVT_PM(8, 512, 1, 8); }
        if (shape == 4) { EVT_PM(8, 256, 1, 16); }
    } else {
        if (shape == 3) { EVT_PM(16, 512, 1, 8); }
        if (shape == 4) { EVT_PM(16, 256, 1, 16); }
    }
#undef EVT_PM
    evt_set_error("internal: model shape does not fit the LDS predict kernel");
    return EVT_ERR_ARG;
}

int launch_predict_model(hipStream_t s, const uint32_t *nodes, const float *leaf_pred, const int64_t *off, int ntrees, const uint8_t *xcm, int64_t N,
                         int K, int loss, int apply_link, float *out, const int32_t *skip_flag) {
    if (K <= 4)
        hipLaunchKernelGGL(k_predict_model<4>, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, nodes, leaf_pred, off, ntrees, xcm, N, K, loss,
                           apply_link, out, skip_flag);
    else
        hipLaunchKernelGGL(k_predict_model<EVT_MAX_K>, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, nodes, leaf_pred, off, ntrees, xcm, N, K,
                           loss, apply_link, out, skip_flag);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

int launch_leaf_idx_model(hipStream_t s, const uint32_t *nodes, const int64_t *off, int ntrees, const uint8_t *xcm, int64_t N, uint32_t *out) {
    hipLaunchKernelGGL(k_leaf_idx_model, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, nodes, off, ntrees, xcm, N, out);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

// the leaf values of n trees for one row (tree t's at v + t * step) added to its running prediction in tree order, with predict!'s
// clamps after each tree (src/predict.jl:1-84); values are read a few trees ahead of their use
template <int KMAX, typename ADD>
__device__ __forceinline__ void add_run(float *acc, const float *v, int step, int n, ADD add) {
    int t = 0;
    constexpr int U = KMAX <= 2 ? 8 : (KMAX <= 4 ? 4 : 2);
    for (; t + U <= n; t += U) {
        float lp[U][KMAX];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int k = 0; k < KMAX; k++) lp[u][k] = v[(t + u) * step + k];
#pragma unroll
        for (int u = 0; u < U; u++) add(acc, lp[u]);
    }
    for (; t < n; t++) {
        float lp[KMAX];
#pragma unroll
        for (int k = 0; k < KMAX; k++) lp[k] = v[t * step + k];
        add(acc, lp);
    }
}
// one or two outputs of a row, by one lane
template <int KMAX>
__device__ __forceinline__ void add_trees(float *acc, const float *v, int step, int n, int K, int loss) {
    if (loss == EVT_LOSS_LOGLOSS) {
        add_run<KMAX>(acc, v, step, n, [](float *a, const float *lp) {
#pragma unroll
            for (int k = 0; k < KMAX; k++) a[k] = fminf(fmaxf(a[k] + lp[k], -15.0f), 15.0f);
        });
    } else if (EVT_IS_MLE2P(loss)) {
        add_run<KMAX>(acc, v, step, n, [](float *a, const float *lp) {
#pragma unroll
            for (int k = 0; k < KMAX; k++) a[k] = (k & 1) ? fmaxf(-15.0f, a[k] + lp[k]) : a[k] + lp[k];
        });
    } else if (loss == EVT_LOSS_MLOGLOSS) {
        add_run<KMAX>(acc, v, step, n, [K](float *a, const float *lp) {
            float m = -INFINITY;
#pragma unroll
            for (int k = 0; k < KMAX; k++) {
                a[k] += lp[k];
                m = k < K ? fmaxf(m, a[k]) : m;
            }
#pragma unroll
            for (int k = 0; k < KMAX; k++) a[k] = fmaxf(-15.0f, a[k] - m);
        });
    } else {
        add_run<KMAX>(acc, v, step, n, [](float *a, const float *lp) {
#pragma unroll
            for (int k = 0; k < KMAX; k++) a[k] += lp[k];
        });
    }
}

// The largest of the values of KMAX neighbouring lanes (4, 8 or 16 of a DPP row), in all of them.  Written out, since as a move and a maximum of
// its own each step costs three dependent instructions; a DPP read waits two states for the write before it.
#define EVT_MAX_DPP(CTRL_) asm("s_nop 1\n\tv_max_f32_dpp %0, %1, %1 " CTRL_ " row_mask:0xf bank_mask:0xf" : "=v"(x) : "v"(x))
template <int KMAX>
__device__ __forceinline__ float group_max(float x) {
    EVT_MAX_DPP("quad_perm:[1,0,3,2]"); // the neighbour
    EVT_MAX_DPP("quad_perm:[2,3,0,1]"); // the other pair of the quad
    if (KMAX >= 8) EVT_MAX_DPP("row_half_mirror"); // the other quad of eight
    if (KMAX >= 16) EVT_MAX_DPP("row_mirror");     // the other eight
    return x;
}
#undef EVT_MAX_DPP
// More outputs: a lane adds one output of one row (the row's outputs side by side), P rows at a time, with the clamps of add_trees; the
// lanes of a row meet where classes are shifted by their maximum.
template <int P, typename ADD>
__device__ __forceinline__ void add_run_lane(float *acc, const float *v, int step, int per, int n, ADD add) {
    constexpr int U = 8 / P > 0 ? 8 / P : 1; // trees read ahead of their use
    int t = 0;
    for (; t + U <= n; t += U) {
        float lp[U][P];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int p = 0; p < P; p++) lp[u][p] = v[(t + u) * step + p * per];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int p = 0; p < P; p++) acc[p] = add(acc[p] + lp[u][p]);
    }
    for (; t < n; t++)
#pragma unroll
        for (int p = 0; p < P; p++) acc[p] = add(acc[p] + v[t * step + p * per]);
}
// k: the lane's output; lanes past the last one stay at minus infinity where classes are shifted, and are not written out
template <int KMAX, int P>
__device__ __forceinline__ void add_trees_lane(float *acc, const float *v, int step, int per, int n, int k, int K, int loss, bool first) {
    if (loss == EVT_LOSS_MLOGLOSS) {
        const float least = k < K ? -15.0f : -INFINITY;
        if (first && k >= K)
#pragma unroll
            for (int p = 0; p < P; p++) acc[p] = -INFINITY;
        add_run_lane<P>(acc, v, step, per, n, [least](float a) { return fmaxf(least, a - group_max<KMAX>(a)); });
    } else if (loss == EVT_LOSS_LOGLOSS) {
        add_run_lane<P>(acc, v, step, per, n, [](float a) { return fminf(fmaxf(a, -15.0f), 15.0f); });
    } else if (EVT_IS_MLE2P(loss)) {
        add_run_lane<P>(acc, v, step, per, n, [k](float a) { return (k & 1) ? fmaxf(-15.0f, a) : a; });
    } else {
        add_run_lane<P>(acc, v, step, per, n, [](float a) { return a; });
    }
}

// Few rows, many trees: a block takes R rows and spreads the trees over its 256 / R lanes per row, so that a handful of rows still
// occupies whole wavefronts (and a few thousand rows the chip), where a row per lane leaves a single chain of dependent reads.  A lane
// walks WALK_U trees side by side over the completed trees (fixed depth, nodes from the caches: a model of 200 trees of
// depth 8 is 100 KB); the leaf values of a run of trees meet in LDS, and one lane per row adds them in tree order,
// so the sum has the bits of the sequential one - or, of more than two outputs, a lane per row and output: one lane went through all outputs of
// a row while most of its block waited (16 700 rows, 100 trees, 7 classes: 50.8 -> 33.5 us, one row 27.0 -> 11.1).  The bins may lie in pinned host memory, and so may the output.
// With a single row per block the nodes are first touched all at once: one trip to memory instead of one per level.
// LEAF: the leaf's node id of every row and tree instead, tree by tree, in LB-byte words.
// A leaf's values lie KMAX apart, those past the last output zero, and move in pieces of up to 16 bytes (word by word a tree's values were more
// requests than its walk).
#define WALK_U 4
int walk_leaf_stride(int K) { return K <= 2 ? K : K <= 4 ? 4 : K <= 8 ? 8 : EVT_MAX_K; }
template <int KMAX, int R, bool LEAF, int LB>
__global__ __launch_bounds__(256) void k_walk_rows(const uint32_t *__restrict__ cnodes, int stride, const ModelTree *__restrict__ meta,
                                                  const float *__restrict__ cleaf, const uint32_t *__restrict__ cid, int ntrees, int run,
                                                  const uint8_t *__restrict__ x, int64_t ldx, int64_t n, int F, int wide, int K, int loss, int link,
                                                  float *__restrict__ out, void *__restrict__ leaf_out, int64_t leaf_ld) {
    constexpr int G = 256 / R;
    extern __shared__ float4 smem4[];
    float *s_v = reinterpret_cast<float *>(smem4);                                      // [run][R][KMAX]
    uint8_t *s_x = reinterpret_cast<uint8_t *>(s_v + (LEAF ? 0 : (size_t)run * R * KMAX)); // [F][R]
    const int tid = threadIdx.x, r = tid % R, g = tid / R;
    const int64_t i0 = (int64_t)blockIdx.x * R;
    if (R == 1) {
        const int words = ntrees * stride < 8192 ? ntrees * stride : 8192;
        uint32_t seen = 0;
        for (int w = tid * 16; w < words; w += 256 * 16) seen |= cnodes[w];
        asm volatile("" ::"v"(seen));
    }
    for (int k = tid; k < F * R; k += 256) {
        const int64_t i = i0 + k % R;
        s_x[k] = x[(size_t)(k / R) * ldx + (i < n ? i : n - 1)];
    }
    __syncthreads();
    constexpr bool WIDE = KMAX > 2; // a lane per row and output
    constexpr int L = R * KMAX < 256 ? R * KMAX : 256, P = R * KMAX / L; // lanes that add, and what each of them adds
    float acc[WIDE ? P : KMAX];
#pragma unroll
    for (int k = 0; k < (WIDE ? P : KMAX); k++) acc[k] = 0.0f;
    for (int t0 = 0; t0 < ntrees; t0 += run) {
        const int t1 = t0 + run < ntrees ? t0 + run : ntrees;
        for (int tb = t0 + g; tb < t1; tb += G * WALK_U) {
            uint32_t nid[WALK_U], at[WALK_U];
            int levels[WALK_U], most = 0;
            const uint32_t *cn[WALK_U];
#pragma unroll
            for (int u = 0; u < WALK_U; u++) {
                const int t = tb + u * G < t1 ? tb + u * G : tb; // past the end: this lane's first tree again
                const int4 m = *reinterpret_cast<const int4 *>(meta + t);
                nid[u] = 1;
                cn[u] = cnodes + (size_t)(uint32_t)m.x;
                at[u] = (uint32_t)m.y;
                levels[u] = m.z;
                most = m.z > most ? m.z : most;
            }
            for (int l = 0; l < most; l++) {
                uint32_t nd[WALK_U];
#pragma unroll
                for (int u = 0; u < WALK_U; u++) nd[u] = cn[u][l < levels[u] ? nid[u] - 1 : 0];
#pragma unroll
                for (int u = 0; u < WALK_U; u++) {
                    const uint32_t f = wide ? nd[u] & 0xFFFFu : ((nd[u] >> 6) & 0x3FCu) | (nd[u] & 3u);
                    const uint32_t next = step_node<false>(nid[u], nd[u], s_x[f * R + r]);
                    nid[u] = l < levels[u] ? next : nid[u];
                }
            }
#pragma unroll
            for (int u = 0; u < WALK_U; u++) at[u] += nid[u] - (1u << levels[u]);
            if (LEAF) {
                uint32_t id[WALK_U];
#pragma unroll
                for (int u = 0; u < WALK_U; u++) id[u] = cid[at[u]];
#pragma unroll
                for (int u = 0; u < WALK_U; u++) {
                    const int t = tb + u * G;
                    const size_t o = (size_t)t * leaf_ld + i0 + r;
                    if (t < t1 && i0 + r < n) {
                        if (LB == 1) static_cast<uint8_t *>(leaf_out)[o] = (uint8_t)id[u];
                        else if (LB == 2) static_cast<uint16_t *>(leaf_out)[o] = (uint16_t)id[u];
                        else static_cast<uint32_t *>(leaf_out)[o] = id[u];
                    }
                }
            } else {
                alignas(16) float lv[WALK_U][KMAX];
                if constexpr (WIDE) {
#pragma unroll
                    for (int u = 0; u < WALK_U; u++)
#pragma unroll
                        for (int k = 0; k < KMAX; k += 4) *reinterpret_cast<float4 *>(&lv[u][k]) = *reinterpret_cast<const float4 *>(cleaf + (size_t)at[u] * KMAX + k);
#pragma unroll
                    for (int u = 0; u < WALK_U; u++)
                        if (tb + u * G < t1)
#pragma unroll
                            for (int k = 0; k < KMAX; k += 4)
                                *reinterpret_cast<float4 *>(&s_v[((size_t)(tb + u * G - t0) * R + r) * KMAX + k]) = *reinterpret_cast<const float4 *>(&lv[u][k]);
                } else {
#pragma unroll
                    for (int u = 0; u < WALK_U; u++)
#pragma unroll
                        for (int k = 0; k < KMAX; k++) lv[u][k] = cleaf[(size_t)at[u] * K + (k < K ? k : 0)];
#pragma unroll
                    for (int u = 0; u < WALK_U; u++)
                        if (tb + u * G < t1)
#pragma unroll
                            for (int k = 0; k < KMAX; k++) s_v[((size_t)(tb + u * G - t0) * R + r) * KMAX + k] = lv[u][k];
                }
            }
        }
        if (LEAF) continue;
        __syncthreads();
        if constexpr (WIDE) {
            if (tid < L) add_trees_lane<KMAX, P>(acc, s_v + tid, R * KMAX, L, t1 - t0, tid % KMAX, K, loss, t0 == 0);
        } else {
            if (tid < R) add_trees<KMAX>(acc, s_v + tid * KMAX, R * KMAX, t1 - t0, K, loss);
        }
        __syncthreads();
    }
    if constexpr (WIDE && !LEAF) { // the row's outputs meet in one lane, for the link
        if (tid < L)
#pragma unroll
            for (int p = 0; p < P; p++) s_v[tid + p * L] = acc[p];
        __syncthreads();
        if (link) {
            if (tid < R) {
                float o[KMAX];
#pragma unroll
                for (int k = 0; k < KMAX; k++) o[k] = s_v[tid * KMAX + k];
                apply_link<KMAX>(o, K, loss);
#pragma unroll
                for (int k = 0; k < KMAX; k++) s_v[tid * KMAX + k] = o[k];
            }
            __syncthreads();
        }
        // over the bus in whole runs
        const int rows = n - i0 < R ? (int)(n - i0) : R;
        for (int e = tid; e < rows * K; e += 256) out[(size_t)K * i0 + e] = s_v[e / K * KMAX + e % K];
    } else if (!LEAF && tid < R && i0 + tid < n) {
        if (link) apply_link<KMAX>(acc, K, loss);
#pragma unroll
        for (int k = 0; k < KMAX; k++)
            if (k < K) out[(size_t)K * (i0 + tid) + k] = acc[k];
    }
}

template <int KMAX, int R, bool LEAF, int LB>
static int launch_walk(hipStream_t s, const uint32_t *cnodes, int stride, const void *meta, const float *cleaf, const uint32_t *cid, int ntrees,
                       const uint8_t *x, int64_t ldx, int64_t n, int F, int wide, int K, int loss, int link, float *out, void *leaf_out, int64_t leaf_ld) {
    static EvtDevOnce once;
    const int dev = EvtDevOnce::current();
    if (once.pending(dev)) {
        HIPCHK(hipFuncSetAttribute(reinterpret_cast<const void *>(k_walk_rows<KMAX, R, LEAF, LB>), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        once.mark(dev);
    }
    const int G = 256 / R;
    // trees whose values fit 32 KB of LDS
    const int run = LEAF ? ntrees : std::min(ntrees, std::max(G, 8192 / (R * KMAX) / G * G));
    const size_t lds = (size_t)F * R + (LEAF ? 0 : (size_t)run * R * KMAX * 4);
    hipLaunchKernelGGL((k_walk_rows<KMAX, R, LEAF, LB>), dim3((unsigned)((n + R - 1) / R)), dim3(256), lds, s, cnodes, stride,
                       static_cast<const ModelTree *>(meta), cleaf, cid, ntrees, run, x, ldx, n, F, wide, K, loss, link, out, leaf_out, leaf_ld);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

int launch_walk_rows(hipStream_t s, const uint32_t *cnodes, int stride, const void *meta, const float *cleaf, const uint32_t *cid, int ntrees,
                     const uint8_t *x, int64_t ldx, int64_t n, int F, int wide, int K, int loss, int apply_link, float *out, void *leaf_out, int leaf_bytes,
                     int64_t leaf_ld) {
    // rows per block: as few as fill the chip (1024 blocks of four wavefronts, eight of which share a compute unit), and no more than
    // 64 KB of bins
    // (leaf ids go out R to a line, tree after tree: more rows a block for the same number of rows).  Whole calls on bins beside set values of R, 60 to
    // 200 trees of depth 6 to 8, one to twelve outputs, 1 to 200 000 rows: within 12 % of the best, mostly within 5.
    int R = n <= 1024 ? 1 : n <= 8192 ? 4 : n <= 32768 ? 16 : 64;
    if (leaf_out) R = n <= 4 ? 1 : n <= 192 ? 4 : n <= 3072 ? 16 : 64; // us, 1 | 4 | 16 | 64 rows a block: 1024 rows 184 | 73 | 59 | 65, 4096 rows 622 | 185 | 113 | 119
    while (R > 1 && (size_t)R * F > 65536) R /= 4;
#define EVT_WALK(KM_, LEAF_, LB_)                                                                                                                    \
    switch (R) {                                                                                                                                     \
        case 1: return launch_walk<KM_, 1, LEAF_, LB_>(s, cnodes, stride, meta, cleaf, cid, ntrees, x, ldx, n, F, wide, K, loss, apply_link, out, leaf_out, leaf_ld); \
        case 4: return launch_walk<KM_, 4, LEAF_, LB_>(s, cnodes, stride, meta, cleaf, cid, ntrees, x, ldx, n, F, wide, K, loss, apply_link, out, leaf_out, leaf_ld); \
        case 16: return launch_walk<KM_, 16, LEAF_, LB_>(s, cnodes, stride, meta, cleaf, cid, ntrees, x, ldx, n, F, wide, K, loss, apply_link, out, leaf_out, leaf_ld); \
        default: return launch_walk<KM_, 64, LEAF_, LB_>(s, cnodes, stride, meta, cleaf, cid, ntrees, x, ldx, n, F, wide, K, loss, apply_link, out, leaf_out, leaf_ld); \
    }
    if (leaf_out) {
        if (leaf_bytes == 1) { EVT_WALK(1, true, 1) }
        if (leaf_bytes == 2) { EVT_WALK(1, true, 2) }
        EVT_WALK(1, true, 4)
    }
    if (K == 1) { EVT_WALK(1, false, 0) }
    if (K == 2) { EVT_WALK(2, false, 0) }
    if (K <= 4) { EVT_WALK(4, false, 0) }
    if (K <= 8) { EVT_WALK(8, false, 0) }
    EVT_WALK(EVT_MAX_K, false, 0)
#undef EVT_WALK
}
