// Trees of small inputs (thousands to a few hundred thousand rows): one kernel per level, or two where nodes are many, instead of a histogram, a search and a partition.
//
// At these sizes a level is a chain of short dependent kernels - 20 launches of 3 to 9 us for a tree of depth 6 on 2000 rows, whatever they
// do.  Here a block owns one sampled feature and walks ALL rows: it takes the decisions of the level above (every block the same
// ones, from the candidates all blocks left), moves every row's node id on, adds the rows into its feature's histograms in LDS - one
// per active node, built outright: adding all rows costs less than subtracting siblings would save - searches them, and leaves its
// best candidate per node.  The blocks meet only at the kernel boundary.  Rows keep their place: a node id per row stands for the row lists,
// so rows outside the sample walk along (flagged) and the prediction needs no pass of its own over the tree.
// The sums are the same integers and the gains the same expressions as in the kernels of larger inputs: same trees, bit for bit.
#include "grad_math.h"
#include "pool.h"
#include "split_math.h"
#include <algorithm>

#define SMALL_OUT 0x80000000u // the row is not in the sample
#define SMALL_MAX_NODES 256   // nodes of the deepest level that splits

struct SmallHead { // a block's candidate for a node
    double gain;
    int bin;  // NO_BIN: none
    int feat; // 1-based, negative when categorical
    long long left[EVT_MAX_NA + 1]; // totals left of it; more channels go to SmallArgs::left_out
};
static_assert(sizeof(SmallHead) == 64, "one candidate per 64-byte line");

struct SmallArgs {
    const uint8_t *xcm;
    unsigned long long *gq;
    uint8_t *mask;
    const uint32_t *nid_in; // the rows' node ids as the level above left them
    uint32_t *nid_out;
    const SmallHead *head_in; // [node of the level above][block]
    SmallHead *head_out;
    const long long *left_in; // [node][block][NAg]: totals left of the candidate
    long long *left_out;
    long long *hist;
    int64_t node_stride;
    uint32_t *js;
    const uint32_t *js_src; // the column sample where it is new (pinned host memory), or js
    uint32_t *map_dst;
    const uint32_t *map_src;
    int map_words;
    int32_t *status;
    long long *node_sum;
    double *qscale;
    // the root: the gradients; fresh ones are still to be quantised, of their maxima, and leave the tables
    const float *raw;
    int fresh;
    const uint32_t *absmax;
    uint32_t *absmax_next;
    const int32_t *qbits;
    int32_t *qexp;
    TreeDev tree;
    int64_t *stats;
    BlobOut blob; // final kernel: the tree's arrays and their pinned destination
    uint32_t *nidx;
    // final kernel, where it computes the next round's gradients (k_grads)
    float *pred;
    const float *y;
    float *grad;
    uint32_t *maxima;
    double eta, lambda, L2, gamma, min_weight;
    unsigned long long seed;
    int N, F, B, K, NK, NAg, NA, loss, level, D, nnodes, nfs, bagging;
    int slots;     // histograms the block's LDS holds
    int slices;    // blocks that share a feature's rows
    long long *acc; // slices > 1: [node][block][NAg][B], their histograms added up; zero between two levels
    int *counts;    // ... and their rows, [level][slice]
    int *done;      // ... and how many of a feature's blocks have added theirs, zero between two levels
    int apart;      // ... and whether k_small_scan searches their sums instead of the last of those blocks
    int batch;      // ... and the nodes whose sums its last block's LDS holds at a time
    int oblivious, sampled, draw, cond;
    int unit_w;
    int wide;      // channel 0 staged as a 64-bit packed word (more channels than EVT_MAX_NA)
    // the blocks' features, in the launch's arguments: a block need not wait for them.  0-based id | numeric << 16 | (constraint + 1) << 17
    uint32_t feat[256];
};
#define SMALL_NUMERIC (1u << 16)
#define SMALL_ABSENT 1u // no split

__device__ __forceinline__ long long shfl_i64(long long v, int src) {
    const int lo = __shfl((int)(v & 0xffffffffll), src), hi = __shfl((int)(v >> 32), src);
    return ((long long)hi << 32) | (unsigned int)lo;
}
__device__ __forceinline__ double shfl_f64(double v, int src) { return __longlong_as_double(shfl_i64(__double_as_longlong(v), src)); }

// lane i's statistic i (of 2K+1) from lane-held channel sums (decode_vals, a statistic per lane); sc: the lane's scale
__device__ __forceinline__ int lane_channel(const SmallArgs &A, int lane) {
    return EVT_TWO_CHAN(A.loss, A.K) ? (lane == 0 ? 0 : 1) : (lane < A.NAg ? lane : 0);
}
__device__ __forceinline__ double lane_stat(const SmallArgs &A, long long q, double sc, int lane) {
    const bool two = EVT_TWO_CHAN(A.loss, A.K);
    double v = (double)shfl_i64(q, lane_channel(A, lane)) * sc;
    if (two && lane == 1) v = (A.loss == EVT_LOSS_MSE) ? 2.0 * v : 0.0;
    return v;
}
// a node's weight and, for a leaf, its values (leaf_value, an output per lane)
__device__ __forceinline__ void write_node(const SmallArgs &A, int n, long long q, double sc, int lane, bool leaf) {
    const double S = lane_stat(A, q, sc, lane);
    double v[3] = {shfl_f64(S, lane < A.K ? lane : 0), shfl_f64(S, A.K + (lane < A.K ? lane : 0)), shfl_f64(S, 2 * A.K)};
    if (lane == 0) A.tree.w[n - 1] = (float)v[2];
    if (leaf && lane < A.K) A.tree.pred[(int64_t)A.K * (n - 1) + lane] = (float)leaf_value(A.loss, v, 0, 1, A.eta, A.bagging, A.lambda, A.L2);
}

// The decision for node p of the level above `A.level`, by one wavefront: the best of the blocks' candidates (highest gain, then
// earliest feature; its bin is already the lowest).  Leaves the packed split in s_dec[p] (0: none) and the children's totals in
// s_tot; the writer block also writes the Tree arrays and the children's state.  s_own: the nodes' own totals are left there instead of their
// weight and values in the tree's arrays, and SMALL_ABSENT in s_dec[p] where the level did not reach the node (small_leaves).
__device__ __forceinline__ void small_decide(const SmallArgs &A, int p, uint32_t *s_dec, long long *s_tot, bool writer, int lane, long long *s_own = nullptr) {
    const int n = (1 << (A.level - 2)) + p, nag = A.NAg, nwg = A.nfs;
    const int st = A.status[n];
    const long long qn = A.node_sum[(int64_t)n * nag + (lane < nag ? lane : 0)];
    const double sc = A.qscale[lane_channel(A, lane)];
    // Up to 64 candidates: every lane reads a whole one (one line), so that the winner's feature and totals are at hand.  More: their first 16 bytes, and the
    // winner's totals in a second trip - every block of the launch reads all of a level's candidates, and whole ones are what its reads took longest for
    // (rounds, us, whole | first bytes: 1350 rows x 229 features, depth 10 275 | 218, 13k x 156, oblivious of depth 9 173 | 151, 985 x 100 and 250, depth 5 42.4 | 41.8, 46.9 | 44.7).
    const SmallHead *hp = A.head_in + (int64_t)p * nwg;
    union Words {
        SmallHead h;
        uint4 v[4];
    } mine;
    mine.h.gain = -INFINITY;
    mine.h.bin = NO_BIN;
    mine.h.feat = 0;
    int bj = NO_BIN;
    const bool whole = nwg <= 64;
    if (whole) {
        Words c;
        const uint4 *cp = reinterpret_cast<const uint4 *>(hp + (lane < nwg ? lane : nwg - 1));
#pragma unroll
        for (int k = 0; k < 4; k++) c.v[k] = cp[k];
#pragma unroll
        for (int k = 0; k < 4; k++) // all of it now: the compiler fetches the totals behind the comparison of the gains, a second trip to memory
            asm volatile("" : "+v"(c.v[k].x), "+v"(c.v[k].y), "+v"(c.v[k].z), "+v"(c.v[k].w));
        if (lane < nwg && c.h.gain > mine.h.gain) {
            mine = c;
            bj = lane;
        }
    } else {
        for (int w0 = lane; w0 < nwg; w0 += 128) { // two of a lane under way at a time
            Words c[2];
#pragma unroll
            for (int u = 0; u < 2; u++) c[u].v[0] = *reinterpret_cast<const uint4 *>(hp + (w0 + 64 * u < nwg ? w0 + 64 * u : nwg - 1));
#pragma unroll
            for (int u = 0; u < 2; u++)
                if (w0 + 64 * u < nwg && c[u].h.gain > mine.h.gain) {
                    mine.v[0] = c[u].v[0];
                    bj = w0 + 64 * u;
                }
        }
    }
    double bg = mine.h.gain;
    int wj = bj;
    wave_argmax(bg, wj);
    // the writer block may have set the state to SPLIT or LEAF by now: anything but INACTIVE means the level reached the node
    const bool active = st != ST_INACTIVE;
    const bool found = active && wj != NO_BIN && bg > A.gamma;
    uint32_t packed = 0;
    long long ql = 0;
    int feat = 0, bin = 0;
    if (found) {
        const int owner = wj & 63;
        const long long own_left = !whole && nag <= EVT_MAX_NA && lane < nag ? hp[wj].left[lane] : 0;
        bin = __shfl(mine.h.bin, owner);
        feat = __shfl(mine.h.feat, owner);
        const bool numeric = feat > 0;
        feat = numeric ? feat : -feat;
        packed = evt_pack_node(feat, bin, numeric);
        if (!whole && nag <= EVT_MAX_NA) {
            ql = own_left;
        } else if (nag <= EVT_MAX_NA) {
#pragma unroll
            for (int ag = 0; ag < EVT_MAX_NA; ag++) {
                const long long v = shfl_i64(mine.h.left[ag], owner);
                ql = lane == ag ? v : ql;
            }
        } else {
            ql = lane < nag ? A.left_in[((int64_t)p * nwg + wj) * nag + lane] : 0;
        }
    }
    if (lane == 0) s_dec[p] = s_own && !active ? SMALL_ABSENT : packed;
    if (lane < nag) {
        s_tot[(2 * p) * nag + lane] = ql;
        s_tot[(2 * p + 1) * nag + lane] = qn - ql;
        if (s_own) s_own[p * nag + lane] = qn;
    }
    if (!active || !writer) return;
    if (!s_own) write_node(A, n, qn, sc, lane, !found);
    if (lane == 0) {
        A.status[n] = found ? ST_SPLIT : ST_LEAF;
        if (found) {
            A.tree.feat[n - 1] = feat;
            A.tree.cond_bin[n - 1] = (uint8_t)bin;
            A.tree.gain[n - 1] = (float)bg;
            A.tree.split[n - 1] = 1;
            A.tree.packed[n - 1] = packed;
        }
    }
    if (!found) return;
    for (int child = 0; child < 2; child++) {
        const int cn = 2 * n + child;
        const long long qc = child ? qn - ql : ql;
        if (lane < nag) A.node_sum[(int64_t)cn * nag + lane] = qc;
        if (lane == 0) A.status[cn] = A.level < A.D ? ST_BUILD : ST_LEAF;
        if (A.level == A.D && !s_own) write_node(A, cn, qc, sc, lane, true);
    }
}

// Weights and leaf values of the last two levels, behind the decisions that left their totals in LDS: a thread per node, where a wavefront that wrote three
// nodes behind each of its decisions paid their divisions one after the other in every block (rounds, us: 21k rows x 19 features, depth 10 196 -> 183, 9.5k x 7,
// depth 8 174 -> 170, 27k x 65 of two outputs, depth 8 176 -> 172).  s_leaf: the leaves' values, from node np on.
template <int K>
__device__ __forceinline__ void small_leaves(const SmallArgs &A, const uint32_t *s_dec, const long long *s_own, const long long *s_tot, int np, bool writer, const double *sc, float *s_leaf) {
    for (int i = threadIdx.x; i < 3 * np; i += 1024) {
        const bool child = i >= np;
        const uint32_t d = s_dec[child ? (i - np) >> 1 : i];
        const bool split = (d & EVT_NODE_SPLIT) != 0;
        if (child ? !split : d == SMALL_ABSENT) continue;
        double S[2 * K + 1];
        decode_vals(child ? s_tot + (i - np) * A.NAg : s_own + i * A.NAg, sc, A.loss, 2 * K + 1, S);
        const int n = np + i;
        if (writer) A.tree.w[n - 1] = (float)S[2 * K];
        if (split && !child) continue;
#pragma unroll
        for (int k = 0; k < K; k++) {
            const float v = (float)leaf_value(A.loss, S, k, K, A.eta, A.bagging, A.lambda, A.L2);
            if (writer) A.tree.pred[(int64_t)K * (n - 1) + k] = v;
            s_leaf[K * i + k] = v;
        }
    }
}

// a value that is the same in every lane, in scalar registers
__device__ __forceinline__ double uniform_f64(double v) { return __longlong_as_double(readlane_i64(__double_as_longlong(v), 0)); }

// where a row of the level above goes: the decision its node took (0: none, a leaf further up stays), the bin byte that decides, the
// node it moves to
__device__ __forceinline__ uint32_t row_decision(const SmallArgs &A, uint32_t nid, const uint32_t *s_dec) {
    const int p = (int)(nid & ~SMALL_OUT) - (1 << (A.level - 2));
    const uint32_t d = s_dec[p >= 0 ? p : 0];
    return p >= 0 ? d : 0u;
}
__device__ __forceinline__ uint32_t decision_bin(const SmallArgs &A, uint32_t d, int row) {
    const uint32_t f = d & 0xFFFFu;
    return A.xcm[(size_t)(f ? f - 1 : 0) * A.N + row];
}
__device__ __forceinline__ uint32_t row_moves(uint32_t nid, uint32_t d, uint32_t xb) {
    const uint32_t cb = (d >> 16) & 0xFFu;
    const bool left = (d & EVT_NODE_NUMERIC) ? xb <= cb : xb == cb;
    const uint32_t child = (nid & SMALL_OUT) | ((nid & ~SMALL_OUT) * 2 + (left ? 0u : 1u));
    return (d & EVT_NODE_SPLIT) ? child : nid;
}

// 4 and 16 bytes from any 1-, or 4-byte aligned address
__device__ __forceinline__ uint32_t load4(const uint8_t *p) {
    uint32_t v;
    __builtin_memcpy(&v, p, 4);
    return v;
}
__device__ __forceinline__ uint4 load16(const uint32_t *p) {
    uint4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

// a channel's value of one LDS histogram word: the first channel shares its word with the row count
template <bool PACK>
__device__ __forceinline__ long long channel_of(const unsigned long long *H, int B, int NAG, int ag, int b) {
    if (!PACK) return (long long)H[ag * B + b];
    if (ag == NAG - 1) return (long long)(H[b] & ((1ull << EVT_PACK_CNT_BITS) - 1ull));
    const unsigned long long w = H[ag * B + b];
    return ag == 0 ? (long long)w >> EVT_PACK_CNT_BITS : (long long)w;
}

// Searches of this many channels (0: a run-time count) and bins to a lane (1, 2 or 4) hold too many registers to sit in a level's kernel (small_scan_apart).  Compiled
// into it and never run, they still spilt its registers (108 to 340 bytes a lane, now none; rounds of two outputs: 42k rows x 44 features, 255 bins,
// depth 5 147.0 -> 145.0 us, 20k x 6, depth 9 332 -> 327).
constexpr bool small_search_large(int channels, int bins) { return channels * bins >= 10; }
static int bins_per_lane(int B) { return B <= 64 ? 1 : B <= 128 ? 2 : 4; }

// The search of one (node, feature) by one wavefront.  NAG: global channels (2, 3, 5), or 0 when their number is known at run time
// only.  on_gain(b, ok, gain, left) is called for every bin of the lane; left: the totals left of it (NAG channels; NAG == 0: null).
// Returns the node's totals in q (NAG != 0).
// FEW: the node's totals and the scales are kept in scalar registers.  In a level's kernel a large search (small_search_large) spills less by it; elsewhere the moves cost
// more than they give (rounds, us, without | with: two outputs, 3005 rows x 41 features x 100 bins, depth 9 206 | 177, 955 x 93 x 255, depth 7 188 | 177; of 64 bins, 5306 x 36,
// depth 10 236 | 241; in k_small_scan, 429 x 105 x 160 bins, oblivious of depth 9 188 | 200).
template <int NAG, int BPL, bool PACK, bool FEW, typename GAIN>
__device__ __forceinline__ void small_scan(const SmallArgs &A, const double *qs, const unsigned long long *H, const long long *tot, bool numeric, int constraint, int lane,
                                           long long *hist_out, long long *q, GAIN on_gain) {
    const int B = A.B, nag = NAG ? NAG : A.NAg;
    const int bmax = numeric ? B - 1 : B;
    if constexpr (NAG != 0) {
        constexpr int K = NAG == 5 ? 2 : 1, NK = 2 * K + 1;
        long long left[NAG][BPL];
        double sc[NAG], S[NK];
#pragma unroll
        for (int ag = 0; ag < NAG; ag++) {
            sc[ag] = FEW ? uniform_f64(qs[ag]) : qs[ag];
            long long val[BPL], run = 0;
#pragma unroll
            for (int t = 0; t < BPL; t++) {
                const int b = lane * BPL + t;
                val[t] = b < B ? channel_of<PACK>(H, B, NAG, ag, b) : 0;
                if (b < B) hist_out[ag * B + b] = val[t];
                run += val[t];
                left[ag][t] = run;
            }
            const long long incl = wave_incl_scan_i64(run), excl = incl - run;
            // the root's totals are the sums over any feature's bins
            if (FEW) q[ag] = tot ? readlane_i64(tot[ag], 0) : readlane_i64(incl, 63);
            else q[ag] = tot ? tot[ag] : shfl_i64(incl, 63);
#pragma unroll
            for (int t = 0; t < BPL; t++) left[ag][t] = numeric ? left[ag][t] + excl : val[t];
        }
        decode_vals(q, sc, A.loss, NK, S);
        double gain_p = 0.0;
        for (int k = 0; k < K; k++) gain_p += node_gain_k(A.loss, S[k], S[K + k], S[2 * K], A.lambda, A.L2);
        const double w_p = S[NK - 1];
#pragma unroll
        for (int t = 0; t < BPL; t++) {
            const int b = lane * BPL + t;
            long long ql[NAG];
#pragma unroll
            for (int ag = 0; ag < NAG; ag++) ql[ag] = left[ag][t];
            double SL[NK];
            decode_vals(ql, sc, A.loss, NK, SL);
            const double w_l = SL[NK - 1], w_r = w_p - w_l;
            bool ok = b < B && b + 1 <= bmax && w_l > A.min_weight && w_r > A.min_weight;
            if (ok && constraint != 0) {
                double SR[NK];
                for (int k = 0; k < NK; k++) SR[k] = S[k] - SL[k];
                const double predL = leaf_value(A.loss, SL, 0, K, A.eta, A.bagging, A.lambda, A.L2);
                const double predR = leaf_value(A.loss, SR, 0, K, A.eta, A.bagging, A.lambda, A.L2);
                ok = (constraint == -1 && predL > predR) || (constraint == 1 && predL < predR);
            }
            double gain = 0.0;
            if (ok) {
                double sg = 0.0;
                for (int k = 0; k < K; k++) sg += split_gain_k(A.loss, S[k], S[K + k], w_p, SL[k], SL[K + k], w_l, w_r, A.lambda, A.L2);
                gain = sg - gain_p;
            }
            on_gain(b, ok, gain, ql);
        }
    } else {
        const int K = A.K;
        auto lefts = [&](int ag, long long *left, long long &total) {
            long long val[BPL], run = 0;
#pragma unroll
            for (int t = 0; t < BPL; t++) {
                const int b = lane * BPL + t;
                val[t] = b < B ? channel_of<PACK>(H, B, nag, ag, b) : 0;
                if (b < B) hist_out[ag * B + b] = val[t];
                run += val[t];
                left[t] = run;
            }
            const long long incl = wave_incl_scan_i64(run), excl = incl - run;
            total = tot ? tot[ag] : shfl_i64(incl, 63);
#pragma unroll
            for (int t = 0; t < BPL; t++) left[t] = numeric ? left[t] + excl : val[t];
        };
        long long lq[BPL], tq;
        lefts(nag - 1, lq, tq);
        const double w_p = (double)tq * qs[nag - 1];
        double w_l[BPL], w_r[BPL], sg[BPL], gain_p = 0.0;
        bool ok[BPL];
#pragma unroll
        for (int t = 0; t < BPL; t++) {
            const int b = lane * BPL + t;
            w_l[t] = (double)lq[t] * qs[nag - 1];
            w_r[t] = w_p - w_l[t];
            ok[t] = b < B && b + 1 <= bmax && w_l[t] > A.min_weight && w_r[t] > A.min_weight;
            sg[t] = 0.0;
        }
        for (int k = 0; k < K; k++) {
            long long gq[BPL], hq[BPL], tg, th;
            lefts(k, gq, tg);
            lefts(K + k, hq, th);
            const double scg = qs[k], sch = qs[K + k];
            const double Sg = (double)tg * scg, Sh = (double)th * sch;
            gain_p += node_gain_k(A.loss, Sg, Sh, w_p, A.lambda, A.L2);
#pragma unroll
            for (int t = 0; t < BPL; t++)
                sg[t] += split_gain_k(A.loss, Sg, Sh, w_p, (double)gq[t] * scg, (double)hq[t] * sch, w_l[t], w_r[t], A.lambda, A.L2);
        }
#pragma unroll
        for (int t = 0; t < BPL; t++) on_gain(lane * BPL + t, ok[t], ok[t] ? sg[t] - gain_p : 0.0, static_cast<const long long *>(nullptr));
    }
}

// totals left of bin lb (numeric: the bins up to it, categorical: it alone), a channel at a time.  SUMS: Hs lies in memory, where other blocks
// have added to it in this launch
template <bool PACK, bool SUMS>
__device__ __forceinline__ void small_left(const SmallArgs &A, const unsigned long long *Hs, int nag, bool numeric, int lb, int lane, SmallHead *out, long long *left) {
    for (int ag = 0; ag < nag; ag++) {
        long long t = 0;
        for (int b = lane; b < lb && b < A.B; b += 64)
            if (numeric || b + 1 == lb) {
                if (SUMS) t += (long long)__hip_atomic_load(Hs + ag * A.B + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                else t += channel_of<PACK>(Hs, A.B, nag, ag, b);
            }
        t = wave_sum_i64(t);
        if (lane == 0) {
            if (nag <= EVT_MAX_NA) out->left[ag] = t;
            else left[ag] = t;
        }
    }
}

// The search of one (node, feature) and what it leaves: the node's histogram of the feature, the candidate - or, for an oblivious
// level, the gains of all bins in s_gain - and at the root the node's totals.
template <int NAG, int BPL, bool PACK, bool FEW>
__device__ __forceinline__ void small_search(const SmallArgs &A, const double *qs, const unsigned long long *Hs, int q, int jp, int nwg, uint32_t fw, const long long *tot,
                                             bool writer, double *s_gain, int lane) {
    const int B = A.B, nag = NAG ? NAG : A.NAg, n = (1 << (A.level - 1)) + q;
    const bool numeric = (fw & SMALL_NUMERIC) != 0;
    const int feat = numeric ? (int)(fw & 0xFFFFu) + 1 : -((int)(fw & 0xFFFFu) + 1);
    long long *hout = A.hist + (int64_t)(n - 1) * A.node_stride + (int64_t)jp * nag * B;
    double lg = -INFINITY;
    int lb = NO_BIN;
    constexpr int QA = NAG ? NAG : 1;
    long long tq[QA], lq[QA];
#pragma unroll
    for (int ag = 0; ag < QA; ag++) lq[ag] = 0;
    small_scan<NAG, BPL, PACK, FEW>(A, qs, Hs, tot, numeric, (int)(fw >> 17) - 1, lane, hout, tq, [&](int b, bool ok, double gain, const long long *left) {
        if (A.oblivious) {
            if (b < B) s_gain[b] = gain; // update_gains!
        } else if (ok && gain > lg) {
            lg = gain;
            lb = b + 1;
            if constexpr (NAG != 0) {
#pragma unroll
                for (int ag = 0; ag < QA; ag++) lq[ag] = left[ag];
            }
        }
    });
    if (A.level == 1 && writer) { // for the kernels below
        if constexpr (NAG != 0) {
            if (lane == 0)
#pragma unroll
                for (int ag = 0; ag < QA; ag++) A.node_sum[(int64_t)n * nag + ag] = tq[ag];
        } else {
            for (int ag = 0; ag < nag; ag++) {
                long long t = 0;
                for (int b = lane; b < B; b += 64) t += channel_of<PACK>(Hs, B, nag, ag, b);
                t = wave_sum_i64(t);
                if (lane == 0) A.node_sum[(int64_t)n * nag + ag] = t;
            }
        }
    }
    if (A.oblivious) return;
    wave_argmax(lg, lb);
    SmallHead *out = A.head_out + (int64_t)q * nwg + jp;
    if constexpr (NAG != 0) { // the lane that holds the winning bin has the totals left of it
        if (lane == (lb != NO_BIN ? (lb - 1) / BPL : 0)) {
            SmallHead h;
            h.gain = lg;
            h.bin = lb;
            h.feat = feat;
#pragma unroll
            for (int ag = 0; ag < EVT_MAX_NA + 1; ag++) h.left[ag] = ag < QA ? lq[ag < QA ? ag : 0] : 0;
            *out = h;
        }
    } else {
        if (lane == 0) {
            out->gain = lg;
            out->bin = lb;
            out->feat = feat;
        }
        if (lb != NO_BIN) small_left<PACK, false>(A, Hs, nag, numeric, lb, lane, out, A.left_out + ((int64_t)q * nwg + jp) * nag);
    }
}

// Requests the arguments at once, but for the features, of which a block needs its own: read where each is needed, they were ten trips one after the other.  us a round,
// with nine fields named by hand before | this: one block a feature, 30k rows x 10 of two outputs, depth 6 135.6 | 134.4, 8k x 30 72.4 | 70.8; shared rows, the same
// 79.3 | 77.9, 74.9 | 73.2; weighted, two outputs of 192 bins, 21k x 16 198 | 170 (the search of five channels spills less: 87 -> 71 registers of its 256 bins).
__device__ __forceinline__ void touch_small_args() { touch_kernarg_bytes<offsetof(SmallArgs, feat)>(); }

// An oblivious level's row of one feature (grow_otree!, src/fit.jl:190-217), by one wavefront: the gains of the level's nodes added in
// node order, zero where one of them is not positive, and the first maximum over the bins.
__device__ __forceinline__ int small_obliv_best(const SmallArgs &A, const double *s_gain, int nact, int lane, double *gain) {
    double bg = -INFINITY;
    int bb = NO_BIN;
    for (int b = lane; b < A.B; b += 64) {
        double acc = 0.0;
        bool allpos = true;
        for (int s = 0; s < nact; s++) {
            const double g = s_gain[s * A.B + b];
            acc += g;
            if (A.level > 1) allpos = allpos && g > 0.0;
        }
        const double v = allpos ? acc : 0.0;
        if (v > bg) {
            bg = v;
            bb = b + 1;
        }
    }
    wave_argmax(bg, bb);
    *gain = bg;
    return bb;
}

// ROOT: the tree's first level, which also quantises the gradients (no k_quantize: 3.1 us and a launch of a round of 60 at 2000 rows x 10).  A level is a
// chain of trips to memory in few blocks (2000 rows: 9.7 us below the root with its loads behind branches and its arguments read one by one, 8.7
// now; the root 6.5 with the quantisation beside it, 7.0 with it inside).  Whole fits: 2000 x 10, 100 rounds 7.5 -> 6.9 ms, 100k x 10, 200 rounds
// with an eval set 21.1 -> 20.2.
// SMALL_ROOT_WORDS: any number of outputs, quantised ahead (small_root_quantises).
// SPLIT: a feature's rows are shared by `slices` blocks, which add their histograms into A.acc; the last of them to do so reads the sums and
// searches them (100k rows x 10 features: 8.3 us a level and 5.2 for a kernel of its own that searched -> 13.9, and a round of five levels
// 101 -> 92 us).  What passes between the blocks goes by agent-scope atomics, past the caches that are not shared, and is complete before its
// block is counted (as in k_scan).  For inputs of
// few features, whose blocks would fill a part of the chip with long walks: 10 features in 25 slices take 0.4 us per 25k rows and channel pair
// where one block per feature takes 0.4 us per 1k, for 5 us more of flush and hand-over.
enum SmallForm { SMALL_BELOW, SMALL_ROOT, SMALL_ROOT_WORDS };
template <int NAG, int BPL, bool PACK, bool SPLIT, SmallForm FORM>
__global__ __launch_bounds__(1024) void k_small_level(SmallArgs A) {
    extern __shared__ unsigned long long s_dyn[];
    __shared__ uint32_t s_dec[SMALL_MAX_NODES];
    __shared__ uint16_t s_slot[SMALL_MAX_NODES];  // node of the level -> slot among the active ones (0xFFFF: not active)
    __shared__ uint16_t s_node[SMALL_MAX_NODES];  // and back
    __shared__ int s_nact, s_cnt, s_best;
    __shared__ double s_qs[EVT_MC_MAX_NK], s_qmul[EVT_MC_MAX_NK]; // scales of the channels; multipliers of the gradient rows (raw)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    touch_small_args();
    constexpr bool ROOT = FORM != SMALL_BELOW, QUANT = FORM == SMALL_ROOT;
    const int B = A.B, N = A.N, level = ROOT ? 1 : A.level;
    __builtin_assume(ROOT || level > 1);
    const int nag = NAG ? NAG : A.NAg, na = NAG ? NAG - (PACK ? 1 : 0) : A.NA;
    int jp = blockIdx.x, slice = 0;
    if (SPLIT) { // blocks go to the 8 XCDs in turn: each takes a run of slices with all their features, whose rows' gradients then share its L2
        const int L = (int)(blockIdx.y * gridDim.x + blockIdx.x), T = (int)(gridDim.x * gridDim.y), xcd = L & 7, rest = T & 7;
        const int at = xcd * (T >> 3) + (xcd < rest ? xcd : rest) + (L >> 3);
        slice = at / (int)gridDim.x;
        jp = at - slice * (int)gridDim.x;
    }
    const bool writer = jp == 0 && slice == 0;
    const int first = 1 << (level - 1), nlev = first;
    long long *s_tot = reinterpret_cast<long long *>(s_dyn);                         // [nlev][nag]
    double *s_gain = reinterpret_cast<double *>(s_tot + (level > 1 ? nlev * nag : 0)); // oblivious: [slots][B]
    unsigned long long *H = reinterpret_cast<unsigned long long *>(s_gain + (A.oblivious && !SPLIT ? A.slots * B : 0)); // [slots][na][B]
    const uint32_t fw = A.feat[jp];
    const int f = (int)(fw & 0xFFFFu);
    const bool numeric = (fw & SMALL_NUMERIC) != 0;
    if (tid == 0) s_cnt = 0;
    const uint8_t *col = A.xcm + (size_t)f * N;
    // A thread takes U groups of 4 neighbouring rows at a time (the last group of all starts at N - 4 and leaves out what others
    // have); what the first of them need is requested before the decisions, in straight-line code: with the root's loads and the other levels' behind
    // branches each load was waited for before the next (six trips to memory before the first decision).
    constexpr int U = (NAG == 2 && PACK && BPL < 4) ? 2 : 1, GA = NAG ? NAG - (PACK ? 1 : 0) : 1;
    const int allgroups = (N + 3) >> 2, per = SPLIT ? (allgroups + A.slices - 1) / A.slices : allgroups;
    const int gfirst = SPLIT ? slice * per : 0, ngroups = SPLIT && gfirst + per < allgroups ? gfirst + per : allgroups; // the block's: gfirst .. ngroups
    // a row's channel is a word of A.gq, or at the root its gradient, quantised on the way (as k_quantize does, whose launch this saves: A.fresh)
    uint32_t nid[U][4], xb[U], g0[U][4]; // g0: channel 0 where it is 32 bits wide, or at the root the gradient
    unsigned long long g[GA][U][4];
    constexpr bool NARROW = NAG != 0 && PACK; // channel 0 is staged as a 32-bit word
    const uint8_t *const mask = A.sampled && !A.draw ? A.mask : col;
    auto request = [&](int k0) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = k0 + u * 1024 < ngroups ? k0 + u * 1024 : ngroups - 1, r = 4 * k < N - 4 ? 4 * k : N - 4;
            xb[u] = load4(col + r);
            if constexpr (ROOT) {
                nid[u][0] = load4(mask + r); // the rows' mask bytes
            } else {
                const uint4 v = load16(A.nid_in + r);
                nid[u][0] = v.x; nid[u][1] = v.y; nid[u][2] = v.z; nid[u][3] = v.w;
            }
            if constexpr (NAG != 0) {
#pragma unroll
                for (int a = 0; a < GA; a++) {
                    if constexpr (ROOT) {
                        const float *q = A.raw + (size_t)r * A.NK + (NAG == 2 && a == 1 ? 2 : a);
#pragma unroll
                        for (int i = 0; i < 4; i++) g[a][u][i] = __float_as_uint(q[i * A.NK]);
                    } else if (NARROW && a == 0) {
                        const uint4 v = load16(reinterpret_cast<const uint32_t *>(A.gq) + r);
                        g0[u][0] = v.x; g0[u][1] = v.y; g0[u][2] = v.z; g0[u][3] = v.w;
                    } else {
                        const uint32_t *q = reinterpret_cast<const uint32_t *>(A.gq + (size_t)a * N + r);
                        const uint4 v0 = load16(q), v1 = load16(q + 4);
                        g[a][u][0] = ((unsigned long long)v0.y << 32) | v0.x;
                        g[a][u][1] = ((unsigned long long)v0.w << 32) | v0.z;
                        g[a][u][2] = ((unsigned long long)v1.y << 32) | v1.x;
                        g[a][u][3] = ((unsigned long long)v1.w << 32) | v1.z;
                    }
                }
            }
        }
    };
    // the word of a gradient v of channel a, left for the levels below by the block that has the row's share
    auto quantise = [&](float v, int a, int row, bool keep) {
        const long long w = __double2ll_rn((double)v * s_qmul[quant_row(A.loss, A.K, a)]);
        const unsigned long long packed = ((unsigned long long)w << EVT_PACK_CNT_BITS) + 1ull;
        if (PACK && a == 0 && !(NAG == 0 && A.wide)) {
            if (keep) reinterpret_cast<int32_t *>(A.gq)[row] = (int32_t)w;
            return packed;
        }
        const unsigned long long out = PACK && a == 0 ? packed : (unsigned long long)w;
        if (keep) A.gq[(size_t)a * N + row] = out;
        return out;
    };
    request(gfirst + tid);
    if constexpr (ROOT) { // the tables: made here of fresh gradients, or those the words in A.gq were made with
        if constexpr (!QUANT) {
            if (tid < nag) s_qs[tid] = A.qscale[tid];
        } else if (tid < A.NK) {
            const double *mul = A.qscale + EVT_MC_MAX_NK;
            if (A.fresh) {
                const int e = quant_exponent(A.absmax, tid), qb = A.qbits[tid];
                const double m = scalbn(1.0, qb - e);
                s_qmul[tid] = m;
                for (int ag = 0; ag < nag; ag++)
                    if (quant_row(A.loss, A.K, ag) == tid) {
                        const double sc = PACK && ag == nag - 1 ? 1.0 : scalbn(1.0, e - qb);
                        s_qs[ag] = sc;
                        if (writer) A.qscale[ag] = sc;
                    }
                if (writer) {
                    A.qexp[tid] = e;
                    A.qscale[EVT_MC_MAX_NK + tid] = m;
                    if (tid < A.NK - 1)
                        for (int st = 0; st < EVT_ABSMAX_STRIPES; st++) A.absmax_next[st * EVT_MC_MAX_NK + tid] = 0u;
                }
            } else {
                s_qmul[tid] = mul[tid];
                if (tid < nag) s_qs[tid] = A.qscale[tid];
            }
        }
    }
    const double my_scale = A.qscale[tid < nag ? tid : 0];
    // the histograms of the first nodes, cleared while the loads are under way
    for (int i = tid; i < (nlev < A.slots ? nlev : A.slots) * na * B; i += 1024) H[i] = 0ull;
    if constexpr (!ROOT) {
        const int np = nlev >> 1;
        // the first outside the loop: in front of a loop that reads memory the compiler waits for what is under way
        if (wave < np) small_decide(A, wave, s_dec, s_tot, writer, lane);
        for (int p = wave + 16; p < np; p += 16) small_decide(A, p, s_dec, s_tot, writer, lane);
        if (tid < nag) s_qs[tid] = my_scale;
        __syncthreads();
        if (wave == 0) { // the children of split nodes are the level's active nodes
            int base = 0;
            for (int p0 = 0; p0 < np; p0 += 64) {
                const int p = p0 + lane;
                const bool split = p < np && (s_dec[p] & EVT_NODE_SPLIT);
                const unsigned long long m = __ballot(split);
                const int at = base + 2 * __popcll(m & ((1ull << lane) - 1ull));
                if (p < np) {
                    s_slot[2 * p] = split ? (uint16_t)at : 0xFFFFu;
                    s_slot[2 * p + 1] = split ? (uint16_t)(at + 1) : 0xFFFFu;
                    if (split) {
                        s_node[at] = (uint16_t)(2 * p);
                        s_node[at + 1] = (uint16_t)(2 * p + 1);
                    }
                }
                base += 2 * __popcll(m);
            }
            if (lane == 0) s_nact = base;
        }
    } else {
        if (tid == 0) {
            s_slot[0] = 0;
            s_node[0] = 0;
            s_nact = 1;
        }
        if (writer) { // a new tree
            for (int n = tid; n < A.nnodes; n += 1024) {
                A.tree.feat[n] = 0;
                A.tree.cond_bin[n] = 0;
                A.tree.w[n] = 0.0f;
                A.tree.gain[n] = 0.0f;
                A.tree.split[n] = 0;
                A.tree.packed[n] = 0u;
                for (int k = 0; k < A.K; k++) A.tree.pred[(int64_t)A.K * n + k] = 0.0f;
            }
            for (int n = tid; n < A.nnodes + 2; n += 1024) A.status[n] = n == 1 ? ST_BUILD : ST_INACTIVE;
            for (int d = tid; d <= A.D; d += 1024) A.stats[d] = 0;
            if (A.js_src != A.js)
                for (int i = tid; i < A.nfs; i += 1024) A.js[i] = A.js_src[i];
            for (int i = tid; i < A.map_words; i += 1024) A.map_dst[i] = A.map_src[i];
        }
    }
    __syncthreads();
    const int nact = s_nact;
    int counted = 0;
    auto take = [&](int k0, int base, int ns) { // the groups requested at k0, for the nodes in slots base .. base + ns
        uint32_t d[U][4], b[U][4];
        if constexpr (!ROOT) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int k = k0 + u * 1024 < ngroups ? k0 + u * 1024 : ngroups - 1, r = 4 * k < N - 4 ? 4 * k : N - 4;
#pragma unroll
                for (int i = 0; i < 4; i++) d[u][i] = row_decision(A, nid[u][i], s_dec);
#pragma unroll
                for (int i = 0; i < 4; i++) b[u][i] = decision_bin(A, d[u][i], r + i);
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = k0 + u * 1024, r = 4 * k < N - 4 ? 4 * k : N - 4;
            if (k >= ngroups) continue;
            if constexpr (ROOT) {
                const uint32_t mb = nid[u][0];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    uint32_t m = (mb >> (8 * i)) & 0xFFu;
                    if (A.draw) {
                        unsigned long long z = A.seed + (unsigned long long)(((r + i) >> 3) + 1) * 0x9E3779B97F4A7C15ull; // SplitMix64, as mask_flags
                        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
                        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
                        z ^= z >> 31;
                        m = (uint32_t)(z >> (8 * ((r + i) & 7))) & 0xFFu;
                        if (jp == 0) A.mask[r + i] = (uint8_t)m;
                    }
                    nid[u][i] = (A.sampled && m > (uint32_t)A.cond) ? 1u | SMALL_OUT : 1u;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++) nid[u][i] = row_moves(nid[u][i], d[u][i], b[u][i]);
            }
            // every block has the same ids: each writes a share (a wavefront's 256 rows; rows of the last group twice, alike)
            const bool share = base == 0 && (k >> 6) % (int)gridDim.x == jp;
            if (share)
#pragma unroll
                for (int i = 0; i < 4; i++) A.nid_out[r + i] = nid[u][i];
            if constexpr (QUANT) {
                const bool keep = share && A.fresh;
                if constexpr (NAG != 0) {
#pragma unroll
                    for (int a = 0; a < GA; a++)
#pragma unroll
                        for (int i = 0; i < 4; i++) g[a][u][i] = quantise(__uint_as_float((uint32_t)g[a][u][i]), a, r + i, keep);
                } else if (keep) {
                    for (int i = 0; i < 4; i++)
                        for (int a = 0; a < na; a++) quantise(A.raw[(size_t)(r + i) * A.NK + a], a, r + i, true);
                }
            } else if constexpr (NARROW && !ROOT) {
#pragma unroll
                for (int i = 0; i < 4; i++) g[0][u][i] = ((unsigned long long)(long long)(int32_t)g0[u][i] << EVT_PACK_CNT_BITS) + 1ull;
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int q = (int)(nid[u][i] & ~SMALL_OUT) - first;
                if (r + i < 4 * k || (nid[u][i] & SMALL_OUT) || q < 0) continue;
                const int slot = (int)s_slot[q] - base;
                if (slot < 0 || slot >= ns) continue;
                counted++;
                unsigned long long *h = H + (size_t)slot * na * B + ((xb[u] >> (8 * i)) & 0xFFu) - 1;
                if constexpr (NAG != 0) {
#pragma unroll
                    for (int a = 0; a < GA; a++) atomicAdd(h + a * B, g[a][u][i]);
                } else {
                    for (int a = 0; a < na; a++) {
                        unsigned long long v;
                        if (QUANT) v = quantise(A.raw[(size_t)(r + i) * A.NK + a], a, r + i, false);
                        else if (PACK && a == 0 && !A.wide) v = evt_load_narrow(A.gq, (uint32_t)(r + i));
                        else v = A.gq[(size_t)a * N + r + i];
                        atomicAdd(h + a * B, v);
                    }
                }
            }
        }
    };
    int ns = nact < A.slots ? nact : A.slots;
    take(gfirst + tid, 0, ns);
    for (int base = 0; base == 0 || base < nact; base += A.slots) {
        if (base > 0) {
            ns = nact - base < A.slots ? nact - base : A.slots;
            for (int i = tid; i < ns * na * B; i += 1024) H[i] = 0ull;
            __syncthreads();
        }
        for (int k0 = gfirst + tid + (base > 0 ? 0 : 1024 * U); k0 < ngroups; k0 += 1024 * U) {
            request(k0);
            take(k0, base, ns);
        }
        __syncthreads();
        if constexpr (SPLIT) {
            for (int i = tid; i < ns * na * B; i += 1024) {
                const unsigned long long w = H[i];
                if (w == 0ull) continue;
                const int s = i / (na * B), rest = i - s * na * B, a = rest / B, b = rest - a * B;
                unsigned long long *to = reinterpret_cast<unsigned long long *>(A.acc) + ((size_t)s_node[base + s] * A.nfs + jp) * nag * B + b;
                if (PACK && a == 0) {
                    const long long sum = (long long)w >> EVT_PACK_CNT_BITS;
                    if (sum != 0) atomicAdd(to, (unsigned long long)sum);
                    atomicAdd(to + (size_t)(nag - 1) * B, w & ((1ull << EVT_PACK_CNT_BITS) - 1ull));
                } else {
                    atomicAdd(to + (size_t)a * B, w);
                }
            }
        } else
        for (int s = wave; s < ns; s += 16) {
            const int q = s_node[base + s];
            small_search<NAG, BPL, PACK, small_search_large(NAG, BPL)>(A, s_qs, H + (size_t)s * na * B, q, jp, A.nfs, fw, level > 1 ? s_tot + q * nag : nullptr, writer,
                                         A.oblivious ? s_gain + s * B : nullptr, lane);
        }
        __syncthreads();
    }
    if (A.oblivious && !SPLIT) { // all active nodes are in LDS: the feature's row of the level matrix, then its first maximum (grow_otree!, src/fit.jl:190-217)
        if (wave == 0) {
            double bg;
            const int bb = small_obliv_best(A, s_gain, nact, lane, &bg);
            if (lane == 0) s_best = bb;
            for (int s = lane; s < nact; s += 64) {
                SmallHead *out = A.head_out + (int64_t)s_node[s] * gridDim.x + jp;
                out->gain = bg;
                out->bin = bb;
                out->feat = numeric ? f + 1 : -(f + 1);
            }
        }
        __syncthreads();
        const int lb = s_best;
        for (int s = wave; s < nact; s += 16) {
            const int64_t at = (int64_t)s_node[s] * gridDim.x + jp;
            small_left<PACK, false>(A, H + (size_t)s * na * B, nag, numeric, lb, lane, A.head_out + at, A.left_out + at * nag);
        }
    }
    if (jp == 0) { // rows of the level: the root's is the size of the sample
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) counted += __shfl_xor(counted, o);
        if (lane == 0) atomicAdd(&s_cnt, counted);
        __syncthreads();
        if (tid == 0 && SPLIT) A.counts[level * 256 + slice] = s_cnt; // added up by k_small_final
        if (tid == 0 && !SPLIT) {
            A.stats[level] = s_cnt;
            if (level == 1) A.stats[0] = s_cnt;
        }
    }
    if constexpr (SPLIT && !small_search_large(NAG, BPL)) { // instances whose levels are all searched apart end here
        if (A.apart) return;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the block's sums are in memory before it is counted
        __syncthreads();
        if (tid == 0) s_best = __hip_atomic_fetch_add(A.done + jp, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == A.slices - 1;
        __syncthreads();
        if (!s_best) return;
        if (tid == 0) A.done[jp] = 0;
        double *gains = s_gain; // oblivious: [active nodes][B]
        unsigned long long *S = reinterpret_cast<unsigned long long *>(s_gain + (A.oblivious ? nact * B : 0)); // [batch][nag][B]
        const int words = nag * B;
        auto sums = [&](int q) { return reinterpret_cast<unsigned long long *>(A.acc) + ((size_t)q * A.nfs + jp) * words; };
        for (int base = 0; base < nact; base += A.batch) {
            const int nb = nact - base < A.batch ? nact - base : A.batch;
            for (int i0 = tid; i0 < nb * words; i0 += 4096) { // four words of a thread under way at a time
                unsigned long long v[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int i = i0 + 1024 * u < nb * words ? i0 + 1024 * u : i0, k = i / words;
                    v[u] = __hip_atomic_load(sums(s_node[base + k]) + (i - k * words), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
#pragma unroll
                for (int u = 0; u < 4; u++)
                    if (i0 + 1024 * u < nb * words) S[i0 + 1024 * u] = v[u];
            }
            __syncthreads();
            for (int k = wave; k < nb; k += 16) {
                const int q = s_node[base + k];
                small_search<NAG, BPL, false, false>(A, s_qs, S + (size_t)k * words, q, jp, A.nfs, fw, level > 1 ? s_tot + q * nag : nullptr, jp == 0,
                                              A.oblivious ? gains + (base + k) * B : nullptr, lane);
            }
            __syncthreads();
        }
        if (A.oblivious) {
            if (wave == 0) {
                double bg;
                const int bb = small_obliv_best(A, gains, nact, lane, &bg);
                if (lane == 0) s_best = bb;
                for (int k = lane; k < nact; k += 64) {
                    SmallHead *out = A.head_out + (int64_t)s_node[k] * A.nfs + jp;
                    out->gain = bg;
                    out->bin = bb;
                    out->feat = numeric ? f + 1 : -(f + 1);
                }
            }
            __syncthreads();
            const int lb = s_best;
            for (int k = wave; k < nact; k += 16) {
                const int64_t at = (int64_t)s_node[k] * A.nfs + jp;
                small_left<false, true>(A, sums(s_node[k]), nag, numeric, lb, lane, A.head_out + at, A.left_out + at * nag);
            }
            __syncthreads();
        }
        for (int i = tid; i < nact * words; i += 1024) {
            const int k = i / words;
            sums(s_node[k])[i - k * words] = 0;
        }
    }
}

// The searches of a level that the last of a feature's blocks does not take (small_scan_apart): a wavefront per (node, feature), 16 nodes of one
// feature to a block - all of them for an oblivious level, whose nodes' gains meet in LDS.
template <int NAG, int BPL>
__global__ __launch_bounds__(1024) void k_small_scan(SmallArgs A) {
    extern __shared__ double s_gain[]; // oblivious: [active nodes][B]
    __shared__ double s_qs[EVT_MC_MAX_NK];
    __shared__ uint16_t s_node[SMALL_MAX_NODES];
    __shared__ int s_nact, s_best;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    touch_small_args();
    const int nag = NAG ? NAG : A.NAg, jp = blockIdx.x, first = 1 << (A.level - 1), words = nag * A.B;
    const int mine = (int)blockIdx.y * 16 + wave;
    const int st = A.status[first + (mine < first ? mine : 0)];
    const uint32_t fw = A.feat[jp];
    if (tid < nag) s_qs[tid] = A.qscale[tid];
    auto sums = [&](int q) { return A.acc + ((size_t)q * A.nfs + jp) * words; };
    auto search = [&](int q, double *gain) {
        small_search<NAG, BPL, false, false>(A, s_qs, reinterpret_cast<const unsigned long long *>(sums(q)), q, jp, A.nfs, fw,
                                      A.level > 1 ? A.node_sum + (int64_t)(first + q) * nag : nullptr, jp == 0, gain, lane);
    };
    auto clear = [&](int q) {
        for (int i = lane; i < words; i += 64) sums(q)[i] = 0;
    };
    if (!A.oblivious) {
        __syncthreads();
        if (mine >= first || st != ST_BUILD) return;
        search(mine, nullptr);
        clear(mine);
        return;
    }
    if (wave == 0) {
        int base = 0;
        for (int q0 = 0; q0 < first; q0 += 64) {
            const bool on = q0 + lane < first && A.status[first + q0 + lane] == ST_BUILD;
            const unsigned long long m = __ballot(on);
            if (on) s_node[base + __popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)(q0 + lane);
            base += __popcll(m);
        }
        if (lane == 0) s_nact = base;
    }
    __syncthreads();
    const int nact = s_nact;
    for (int s = wave; s < nact; s += 16) search(s_node[s], s_gain + s * A.B);
    __syncthreads();
    const bool numeric = (fw & SMALL_NUMERIC) != 0;
    if (wave == 0) {
        double bg;
        const int bb = small_obliv_best(A, s_gain, nact, lane, &bg);
        if (lane == 0) s_best = bb;
        for (int s = lane; s < nact; s += 64) {
            SmallHead *out = A.head_out + (int64_t)s_node[s] * A.nfs + jp;
            out->gain = bg;
            out->bin = bb;
            out->feat = numeric ? (int)(fw & 0xFFFFu) + 1 : -((int)(fw & 0xFFFFu) + 1);
        }
    }
    __syncthreads();
    const int lb = s_best;
    for (int s = wave; s < nact; s += 16) {
        const int q = s_node[s];
        const int64_t at = (int64_t)q * A.nfs + jp;
        small_left<false, false>(A, reinterpret_cast<const unsigned long long *>(sums(q)), nag, numeric, lb, lane, A.head_out + at, A.left_out + at * nag);
        clear(q);
    }
}

// The last decisions, the leaves, and every row's leaf.  The first block also sends the finished tree to the host's pinned buffer.
// LOSS >= 0: the rows' leaf values are added and the next round's gradients computed here, as k_grads<LOSS> would (whose launch and trip through
// the node ids this saves); otherwise the next pass over the rows adds them, as for larger inputs.
// 2000 rows x 10: 6.0 + 3.4 us and the gap between two launches -> 6.9; 308k rows of two outputs 11.2 + 7.7 -> 16.4.  Whole fits: 100 rounds of the first
// 6.9 -> 6.6 ms, 200 rounds of 100k x 10 with an eval set 20.0 -> 19.3, 138 of the last 24.7 -> 24.1 (with more blocks than are resident at once 25.5).
template <int LOSS>
__global__ __launch_bounds__(1024) void k_small_final(SmallArgs A) {
    extern __shared__ unsigned long long s_dyn[];
    __shared__ uint32_t s_dec[SMALL_MAX_NODES];
    constexpr bool GRADS = LOSS >= 0;
    constexpr int K = LOSS == 2 || LOSS == 7 ? 2 : 1, NK = 2 * K + 1;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool writer = blockIdx.x == 0;
    touch_small_args();
    const int np = 1 << (A.level - 2);
    long long *s_tot = reinterpret_cast<long long *>(s_dyn);
    long long *s_own = GRADS ? s_tot + 2 * np * A.NAg : nullptr;
    float *s_leaf = GRADS ? reinterpret_cast<float *>(s_own + np * A.NAg) : nullptr;
    double sc[NK];
#pragma unroll
    for (int a = 0; a < NK; a++) sc[a] = A.qscale[a];
    // the block's first rows are requested before the decisions; a block has more where there are more than 256 x 1024 of them
    uint32_t nid;
    float pr[K], y = 0.0f, w = 1.0f, mx[2 * K];
#pragma unroll
    for (int k = 0; k < 2 * K; k++) mx[k] = 0.0f;
    auto request = [&](int r) {
        const int row = r < A.N ? r : A.N - 1;
        nid = A.nid_in[row];
        if constexpr (GRADS) {
#pragma unroll
            for (int k = 0; k < K; k++) pr[k] = A.pred[(size_t)K * row + k];
            y = A.y[row];
            if (!A.unit_w) w = A.grad[(size_t)NK * row + NK - 1];
        }
    };
    auto finish = [&](int r) {
        const uint32_t d = row_decision(A, nid, s_dec);
        const uint32_t leaf = row_moves(nid, d, decision_bin(A, d, r < A.N ? r : A.N - 1)) & ~SMALL_OUT;
        if (r < A.N) A.nidx[r] = leaf;
        if constexpr (GRADS) {
            float l[K], out[2 * K];
            const int at = (int)leaf - np; // nodes of the last two levels; leaves above them were written by an earlier kernel
#pragma unroll
            for (int k = 0; k < K; k++) l[k] = at >= 0 ? s_leaf[K * at + k] : A.tree.pred[(size_t)K * (leaf - 1) + k];
            evt_add_leaf(pr, l, K, LOSS);
            grad_row<LOSS>(pr, y, w, out);
            if (r < A.N) {
#pragma unroll
                for (int k = 0; k < K; k++) A.pred[(size_t)K * r + k] = pr[k];
#pragma unroll
                for (int k = 0; k < 2 * K; k++) {
                    A.grad[(size_t)NK * r + k] = out[k];
                    mx[k] = fmaxf(mx[k], fabsf(out[k]));
                }
            }
        }
    };
    const int r0 = (int)blockIdx.x * 1024 + tid;
    request(r0);
    if (wave < np) small_decide(A, wave, s_dec, s_tot, writer, lane, s_own);
    for (int p = wave + 16; p < np; p += 16) small_decide(A, p, s_dec, s_tot, writer, lane, s_own);
    __syncthreads();
    if constexpr (GRADS) {
        small_leaves<K>(A, s_dec, s_own, s_tot, np, writer, sc, s_leaf);
        __syncthreads();
    }
    finish(r0);
    for (int r = r0 + (int)gridDim.x * 1024; r < A.N; r += (int)gridDim.x * 1024) {
        request(r);
        finish(r);
    }
    if constexpr (GRADS) {
        __shared__ float s_m[16][2 * K];
        absmax_raise_block<2 * K>(mx, s_m, A.maxima);
    }
    if (!writer) return;
    if (A.slices > 1) {
        for (int l = 1 + wave; l < A.level; l += 16) {
            int t = 0;
            for (int y = lane; y < A.slices; y += 64) t += A.counts[l * 256 + y];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o);
            if (lane == 0) {
                A.stats[l] = t;
                if (l == 1) A.stats[0] = t;
            }
        }
        __syncthreads();
    }
    blob_send(A.blob, 0);
}

static size_t small_lds(const evt_ctx *c, int level, int slots, bool split) {
    const size_t tot = level > 1 ? (size_t)(1 << (level - 1)) * c->NAg * 8 : 0;
    const size_t gain = c->tree_type == EVT_TREE_OBLIVIOUS && !split ? (size_t)slots * c->B * 8 : 0;
    return tot + gain + (size_t)slots * c->NA * c->B * 8;
}
// of the last of a feature's blocks: the nodes' gains (oblivious) and the sums of `batch` nodes, in the place of its histograms
static size_t small_lds_search(const evt_ctx *c, int level, int batch) {
    const size_t nodes = (size_t)1 << (level - 1), tot = level > 1 ? nodes * c->NAg * 8 : 0;
    return tot + (c->tree_type == EVT_TREE_OBLIVIOUS ? nodes * c->B * 8 : 0) + (size_t)batch * c->NAg * c->B * 8;
}
// Whether a level's searches take a kernel of their own.  The last of a feature's blocks reads its nodes' sums, 1024 words at a time, and its 16 wavefronts search
// them, where that kernel spreads them over the chip for a launch more: apart from the first level on whose sums are 1024 words, which is where rounds of 4 to 128
// features are best as a fit queues them (in the last block up to 512 | 1023 | 5120 words, us: one output of 64 bins, 30k rows x 8, depth 9 156 | 157 | 160, 15k x 60,
// depth 8 126 | 125 | 127; of 128 bins 30k x 10, depth 9 174 | 174 | 178; two outputs of 64 bins 30k x 14, depth 9 208 | 208 | 214, 15k x 20, depth 8 151 | 151 | 155).
// A block searches the many channels of several outputs at once longer: there up to 5120 words (3 classes, 64 bins, 15k x 30, depth 6 in it to 1023 | 5120 words: 1.02 | 1.00).
// The search of two outputs of more than 64 bins, or of one output of three channels and more than 128, holds too many registers to sit in the level's kernel
// (42k rows x 44, 255 bins, depth 5, 64 rounds: in it 13.4 ms, apart 11.9; 4837 x 18, oblivious of depth 8, 133 rounds 35.5 | 27.1; a round of three
// channels x 192 bins, 74k x 3, depth 5 105 | 88 us, of 160 bins, 11k x 206, oblivious of depth 8 310 | 224).  More blocks than compute units (one to each): a
// block that searches holds back those that have yet to walk (20k rows and fewer x 220 features, depth 9, every level in the last block | apart: two outputs of
// 32 bins 405 | 333 us a round, one of 64 bins 354 | 273, oblivious 215 | 190; of 128 features, 256 blocks, oblivious 125 | 132).  An oblivious level is decided
// over all its nodes, whose sums its block holds 16 nodes at a time: apart from two channels of more than 224 bins on (255 bins, depth 8, 20k x 60 175 | 155 us a
// round, 30k x 8 145 | 136; 160 bins, 15k x 60 equal), of several outputs where LDS holds the sums of fewer than 16 nodes.
static bool small_scan_apart(const evt_ctx *c, int nodes, int blocks) {
    if (blocks > 256) return true;
    if (!c->mc && small_search_large(c->NAg, bins_per_lane(c->B))) return true;
    if (c->tree_type == EVT_TREE_OBLIVIOUS) return (size_t)std::min(16, nodes) * c->NAg * c->B * 8 > (c->mc ? 72 : 56) * 1024;
    return nodes > 16 || (int64_t)nodes * c->NAg * c->B > (c->mc ? 5120 : 1023);
}
// histograms a block's LDS holds at the deepest level that splits
static int small_slots(const evt_ctx *c, bool split) {
    const int nodes = 1 << std::max(0, c->D - 2);
    const size_t fixed = small_lds(c, c->D - 1, 0, split), one = small_lds(c, c->D - 1, 1, split) - fixed;
    const size_t budget = 144 * 1024;
    if (fixed > 32 * 1024) return 0;
    return (int)std::min<size_t>((size_t)nodes, (budget - fixed) / one);
}

static size_t small_acc_bytes(const evt_ctx *c) { return (size_t)(1 << (c->D - 2)) * std::min(c->F, 256) * c->NAg * c->B * 8; }

static int small_tree_buffers(evt_ctx *c, bool split) {
    const size_t cand = (size_t)(1 << (c->D - 2)) * std::min(c->F, 256);
    for (int k = 0; k < 2 && !c->small_nid[1]; k++) {
        c->small_head[k] = dev_take(sizeof(SmallHead) * cand);
        if (c->NK > EVT_MAX_NA) c->small_left[k] = static_cast<long long *>(dev_take(sizeof(long long) * cand * c->NK));
        c->small_nid[k] = static_cast<uint32_t *>(dev_take(sizeof(uint32_t) * (size_t)c->N));
        if (!c->small_head[k] || !c->small_nid[k] || (c->NK > EVT_MAX_NA && !c->small_left[k])) return EVT_ERR_NOMEM;
    }
    if (split && !c->small_acc) {
        // the counts of the slices' rows, then the sums, for the larger of the weight modes
        const size_t bytes = 17 * 256 * sizeof(int) + small_acc_bytes(c) / c->NAg * c->NK; // the blocks' counts behind the rows'
        c->small_acc = static_cast<uint8_t *>(dev_take(bytes));
        if (!c->small_acc) return EVT_ERR_NOMEM;
        const int r = launch_fill_bytes(c, c->small_acc, (int64_t)bytes);
        if (r != EVT_OK) return r;
    }
    return EVT_OK;
}

// Which form a tree takes: 0 the kernels of larger inputs, SMALL_PATH one launch (small_path_takes), 1 a block per feature, S > 1 a feature's rows
// shared by S blocks.  A block walks its rows once per level (and once more for every `slots` nodes), so a level grows with
// rows / S, the channels and - through the candidates every block reads and the searches its 16 wavefronts share - the nodes; slices
// add the words they flush and, where a level is searched apart, a launch.  The other path spreads rows of any number over the chip and pays for its launches.
// Estimates in microseconds, fitted to rounds of an earlier state of these kernels and checked on the present ones (500 to 300k rows, 3 to 250 features, depths 3 to
// 10): of 364 shapes of one or two outputs 313 take a form within 4 % of the best and 334 within 10, the worst 1.44 times the best; of 186 of several outputs 141
// and 154, the worst 1.92, where the other path, which has since become faster than its estimate, is not taken (profiles/rule_small_tree.txt).
// What a further walk of all channels costs whatever its rows was added for those: 16 classes, 192 bins, 893 rows x 3, depth 6 906 -> 244 us, 14 classes, 160 bins,
// 1558 x 4, depth 9 1209 -> 337; of 1658 shapes one takes more than 3 % longer by it.
// A round of depth 6, 64 bins and 8 features as a fit queues it, microseconds for the other path, S = 1 and S > 1: mse 82, 48, 64 at 2k rows (31 in one launch), 91, 101, 66 at
// 30k, 104, -, 79 at 250k; 3 classes 125, 122, 113 at 8k, 147, 482, 129 at 60k, 173, -, 187 at 250k; 7 classes 129, 147, 170 at 2k, 181, -, 254 at 120k, 220, -, 341 at 250k.
int small_tree_form(const evt_ctx *c, int nfs, bool all_rows) {
    if (!c->small_tree || c->D < 2 || c->D > 10 || nfs > 256 || c->N < 4 || c->N > (1 << 24) || !c->defer_pred || EVT_IS_QUANTILE(c->loss)) return 0;
    if (c->record_nidx && !all_rows) return 0;
    if ((c->small_tree == 1 || c->small_tree == 4) && small_path_takes(c, nfs, c->small_tree == 4)) return SMALL_PATH;
    if (c->small_tree == 4) return 0;
    const bool obliv = c->tree_type == EVT_TREE_OBLIVIOUS;
    const int nodes = 1 << (c->D - 2), slots = small_slots(c, false), slots_split = small_slots(c, true);
    const int S = std::max(2, 256 / nfs);
    const bool can1 = c->N <= 65535 && slots >= 1 && (!obliv || slots == nodes);
    const bool canS = slots_split >= 1 && c->N / S < 65000 && small_acc_bytes(c) <= ((size_t)64 << 20) && small_lds_search(c, c->D - 1, 1) <= 144 * 1024;
    if (c->small_tree == 2) return can1 ? 1 : 0;
    if (c->small_tree == 3) return canS ? S : 0;
    const double k = 1e-3 * c->N, per_1k = c->mc ? 0.3 + 0.2 * c->NA : 0.35 + 0.058 * c->NA, per_1k_s = c->mc ? 0.3 + 0.3 * c->NA : per_1k;
    double one = 0.0, split = 0.0;
    for (int l = 1; l < c->D; l++) {
        const int n = (int)std::min<int64_t>(1 << (l - 1), c->N), searches = (n + 15) / 16;
        const int walks = (n + slots - 1) / std::max(1, slots), walks_split = (n + slots_split - 1) / std::max(1, slots_split);
        const double again = c->mc ? 0.5 * c->NA : 0.0; // a walk more clears and flushes the histograms of all channels, however few its rows
        one += 5.0 + 3.5 * searches + per_1k * k * walks + again * (walks - 1);
        split += (c->mc ? 6.0 + 0.8 * c->NA : 11.0) + 2.5 * searches + per_1k_s * k / S * walks_split + again * (walks_split - 1) +
                 (double)std::min<int64_t>((int64_t)n * c->B, c->N / S) * c->NA * nfs * S / 141e3; // words flushed: no more than rows
    }
    const double launches = c->mc ? 16.0 + 0.8 * c->NA + (nfs > 16 ? 2.0 + 0.008 * c->NA * std::max(0, nfs - 20) : std::max(0.0, 8.0 - 0.35 * c->NA))
                                  : 18.0 + 3.0 * std::min(c->NA, 8) + (nfs > 16 ? 8.0 : 0.0);
    const double other = (c->D - 1) * (launches + (obliv ? 5.0 : 0.0) + 0.0068 * c->NA * k);
    if (can1 && one < other && (!canS || one <= split)) return 1;
    return canS && split < other ? S : 0;
}

// Whether the root's kernel of a tree of this form (small_tree_form) quantises the gradients, or k_quantize does ahead of it.  Of any number of
// outputs every block converts all channels of its rows, where a word made ahead is one load: there only blocks of few rows save by it.  Rounds of depth 5,
// 64 bins, us, in the root | ahead: one block a feature, 7 outputs x 6 features 400 rows 131 | 130, 3000 145 | 134, 12k 297 | 209; several, 3 outputs
// x 6 features (42 blocks each) 6k rows 105 | 109, 25k 109 | 111, 50k 114 | 115, x 30 (8) 6k 108 | 110, 12k 113 | 111, 25k 127 | 118; 7 x 100 (2) 2k 164 | 163, 6k 184 | 175.
bool small_root_quantises(const evt_ctx *c, int form) { return !c->mc || (form > 1 && c->N <= (int64_t)1500 * form); }

int launch_small_tree(evt_ctx *c, const evt_params *p, bool draw, int slices) {
    const bool split = slices > 1;
    int r = small_tree_buffers(c, split);
    if (r != EVT_OK) return r;
    SmallArgs A;
    memset((void *)&A, 0, sizeof(A));
    A.xcm = c->xcm;
    A.gq = c->gq;
    A.mask = c->mask;
    A.hist = c->hist;
    A.node_stride = (int64_t)c->F * c->NAg * c->B;
    A.js = c->js;
    A.js_src = c->js;
    if (c->js_staged) { // read from the pinned buffer by the first kernel
        A.js_src = reinterpret_cast<const uint32_t *>(c->h_stage_dev + c->blob_bytes);
        A.map_src = reinterpret_cast<const uint32_t *>(c->h_stage_dev + c->blob_bytes + (size_t)c->F * 4);
        A.map_dst = reinterpret_cast<uint32_t *>(c->jsmap);
        A.map_words = c->RS / 2;
        c->js_staged = false;
    }
    A.status = c->status;
    A.node_sum = c->node_sum;
    A.qscale = c->qscale;
    A.tree = c->tree;
    A.stats = c->stats;
    A.nidx = c->nidx;
    A.eta = p->eta; A.lambda = p->lambda; A.L2 = p->L2; A.gamma = p->gamma; A.min_weight = p->min_weight;
    A.bagging = p->bagging_size;
    A.seed = c->mask_seed;
    A.N = (int)c->N; A.F = c->F; A.B = c->B; A.K = c->K; A.NK = c->NK; A.NAg = c->NAg; A.NA = c->NA; A.loss = c->loss; A.D = c->D; A.nnodes = c->nnodes;
    A.nfs = c->n_js_last;
    A.slots = small_slots(c, split);
    A.slices = slices;
    A.counts = reinterpret_cast<int *>(c->small_acc);
    A.done = A.counts + 16 * 256;
    A.acc = reinterpret_cast<long long *>(c->small_acc + 17 * 256 * sizeof(int));
    A.oblivious = c->tree_type == EVT_TREE_OBLIVIOUS ? 1 : 0;
    A.sampled = c->step.all_rows ? 0 : 1;
    A.draw = draw ? 1 : 0;
    A.cond = c->last_cond;
    A.wide = c->NA > EVT_MAX_NA ? 1 : 0;
    for (int j = 0; j < A.nfs; j++) {
        const int f = (int)c->js_last[j] - 1;
        A.feat[j] = (uint32_t)f | (c->h_feattypes[f] ? SMALL_NUMERIC : 0u) | ((uint32_t)(c->h_mono[f] + 1) << 17);
    }
    const int bpl = bins_per_lane(c->B);
    A.raw = c->grad;
    if (c->quant_pending) {
        A.fresh = 1;
        A.absmax = absmax_set(c, c->absmax_cur);
        A.absmax_next = absmax_set(c, c->absmax_other);
        A.qbits = c->qbits;
        A.qexp = c->qexp;
    }
    for (int level = 1; level <= c->D; level++) {
        A.level = level;
        const int in = (level & 1) ^ 1, out = level & 1;
        A.nid_in = c->small_nid[in]; A.nid_out = c->small_nid[out];
        A.head_in = static_cast<const SmallHead *>(c->small_head[in]); A.head_out = static_cast<SmallHead *>(c->small_head[out]);
        A.left_in = c->small_left[in]; A.left_out = c->small_left[out];
        if (level == c->D) {
            prof_begin(c, EVT_K_PARTITION, level);
            blob_out(c, A.blob);
            A.blob.blocks = 1; // the one that writes the tree
            c->step.grads_done = grads_with_tree(c, p);
            A.pred = c->pred;
            A.y = c->y;
            A.grad = c->grad;
            A.maxima = absmax_set(c, c->absmax_cur);
            A.unit_w = c->unit_w ? 1 : 0;
            const size_t lds = (size_t)(1 << (level - 1)) * c->NAg * 8 + (c->step.grads_done ? (size_t)(1 << (level - 2)) * (c->NAg * 8 + 3 * c->K * 4) : 0);
            // no more blocks than are resident at once: a second generation would take the decisions again
#define FINAL(L_) hipLaunchKernelGGL(k_small_final<L_>, dim3((unsigned)std::min<int64_t>(256, (c->N + 1023) / 1024)), dim3(1024), lds, c->stream, A)
            if (!c->step.grads_done) FINAL(-1);
            else EVT_GRAD_ROW_CASES(c, FINAL)
#undef FINAL
            prof_end(c);
            break;
        }
        const int nodes = 1 << (level - 1), slots = std::min(A.slots, nodes);
        const int most = A.slots;
        A.slots = slots;
        size_t lds = small_lds(c, level, slots, split);
        if (split) { // a wavefront per node at a time, as far as they fit
            A.batch = std::min(16, nodes);
            while (A.batch > 1 && small_lds_search(c, level, A.batch) > std::max<size_t>(lds, 72 * 1024)) A.batch >>= 1;
            A.apart = small_scan_apart(c, nodes, c->n_js_last * slices) ? 1 : 0;
            if (!A.apart) lds = std::max(lds, small_lds_search(c, level, A.batch));
        }
        prof_begin(c, level == 1 ? EVT_K_HIST : EVT_K_PARTITION, level); // below the root it moves rows, builds and searches at once
#define SMALL4(NAG_, BPL_, PACK_, SPLIT_, FORM_)                                                                                          \
    {                                                                                                                                     \
        static EvtDevOnce once;                                                                                                           \
        if (once.pending(c->device)) {                                                                                                    \
            HIPCHK(hipFuncSetAttribute(reinterpret_cast<const void *>(k_small_level<NAG_, BPL_, PACK_, SPLIT_, FORM_>),                    \
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024));                                          \
            once.mark(c->device);                                                                                                         \
        }                                                                                                                                 \
        hipLaunchKernelGGL((k_small_level<NAG_, BPL_, PACK_, SPLIT_, FORM_>), dim3((unsigned)c->n_js_last, split ? (unsigned)slices : 1u), \
                           dim3(1024), lds, c->stream, A);                                                                                \
    }
#define SMALL3(NAG_, BPL_, PACK_)                                    \
    if (split) {                                                     \
        if (level > 1) SMALL4(NAG_, BPL_, PACK_, true, SMALL_BELOW) \
        else if (A.fresh) SMALL4(NAG_, BPL_, PACK_, true, SMALL_ROOT) \
        else SMALL4(NAG_, BPL_, PACK_, true, (NAG_ ? SMALL_ROOT : SMALL_ROOT_WORDS)) \
        if (A.apart) {                                               \
            static EvtDevOnce once;                                  \
            if (once.pending(c->device)) {                           \
                HIPCHK(hipFuncSetAttribute(reinterpret_cast<const void *>(k_small_scan<NAG_, BPL_>), hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024)); \
                once.mark(c->device);                                \
            }                                                        \
            const size_t gain = A.oblivious ? (size_t)nodes * c->B * 8 : 0; \
            prof_end(c);                                             \
            prof_begin(c, EVT_K_SCAN, level);                        \
            hipLaunchKernelGGL((k_small_scan<NAG_, BPL_>), dim3((unsigned)c->n_js_last, A.oblivious ? 1u : (unsigned)((nodes + 15) / 16)), dim3(1024), gain, c->stream, A); \
        }                                                            \
    } else {                                                         \
        if (level > 1) SMALL4(NAG_, BPL_, PACK_, false, SMALL_BELOW) \
        else SMALL4(NAG_, BPL_, PACK_, false, (NAG_ ? SMALL_ROOT : SMALL_ROOT_WORDS)) \
    }
#define SMALL2(NAG_, PACK_)             \
    if (bpl == 1) { SMALL3(NAG_, 1, PACK_) } \
    else if (bpl == 2) { SMALL3(NAG_, 2, PACK_) } \
    else { SMALL3(NAG_, 4, PACK_) }
#define SMALL1(NAG_)            \
    if (c->unit_w) { SMALL2(NAG_, true) } \
    else { SMALL2(NAG_, false) }
        if (c->mc) { SMALL1(0) }
        else if (c->NAg == 2) { SMALL1(2) }
        else if (c->NAg == 3) { SMALL1(3) }
        else { SMALL1(5) }
#undef SMALL1
#undef SMALL2
#undef SMALL3
#undef SMALL4
        A.slots = most;
        prof_end(c);
        HIPCHK(hipGetLastError());
        if (c->quant_pending) { // made by the root's kernel, which cleared the set that the next gradient pass raises
            quant_taken(c);
        }
    }
    HIPCHK(hipGetLastError());
    c->step.blob_sent = true;
    return EVT_OK;
}
