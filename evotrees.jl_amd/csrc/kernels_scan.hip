// Split search: subtract_hist! + _scan_node!/get_best_split + _child_sums! + leaf values
// (src/fit-utils.jl:321-332, :403-486; src/split.jl:1, :58-66, :108-117; src/predict.jl:198-234).
//
// One block per node of the level; each wave takes sampled features round-robin; lanes are bins.
// The left sums of all bins of one (node, feature) come from one wavefront inclusive prefix scan
// of the int64 histogram (DPP row shifts + row broadcasts), the candidate gains are evaluated in
// Float64 with the reference's expression order, and the best candidate is found with a
// cross-lane arg-max whose ties go to the lowest bin, then the earliest feature of js — the
// reference's "first maximum wins" (strict '>' at src/fit-utils.jl:447).
#include "obliv_rule.h"
#include "split_math.h"
#include <algorithm>

struct ScanBest {
    double gain;
    int jp, bin;
};
// The candidate as the one- and two-output kernels hand it over: with the feature (1-based id, negative when categorical)
// and the fixed-point totals left of the split, so that the pass that decides needs neither the feature tables nor the
// histogram again.
struct ScanBestQ {
    double gain;
    int jp, bin;
    int feat, pad;
    long long qL[EVT_MAX_NA];
};
static_assert(sizeof(ScanBestQ) == 64, "one candidate per 64-byte line");

struct ScanArgs {
    ScanBest *sbest; // ScanBestQ entries for k_scan / k_scan_fin (same buffer)
    long long *hist;
    int64_t node_stride;
    const uint32_t *js;
    const uint8_t *feattypes;
    const int32_t *mono;
    int32_t *status;
    long long *node_sum;
    const double *qscale;
    TreeDev tree;
    double *ogains;
    double eta, lambda, L2, gamma, min_weight;
    int bagging;
    int nfs, B, F, K, NK, NAg, loss, level, leaf_level, oblivious, zero_children;
    int32_t *counts; // last_decides: blocks of each node of the level that have handed in their candidate, zero between launches
    int last_decides;
    int fold_leaves; // the level's children are leaves: their weight and values are written along with the split (no pass of their own)
};

// The root's totals -> Float64 statistics: the bin sums of its first sampled feature (exact in integers: every feature's bins sum to the same total); other nodes
// carry the totals their parent's split gave them.
template <int NAG>
__device__ __forceinline__ void root_totals(const ScanArgs &A, int n, const long long *hn, long long *s_Sq, double *s_S, double *s_sc) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid < NAG) s_sc[tid] = A.qscale[tid];
    if (wave == 0) {
        for (int ag = 0; ag < NAG; ag++) {
            long long s = 0;
            for (int b = lane; b < A.B; b += 64) s += hn[(int64_t)ag * A.B + b];
            s = wave_sum_i64(s);
            if (lane == 0) {
                s_Sq[ag] = s;
                A.node_sum[(int64_t)n * NAG + ag] = s;
            }
        }
    }
    __syncthreads();
    if (tid == 0) {
        double v[EVT_MAX_NK];
        long long q[NAG];
        for (int ag = 0; ag < NAG; ag++) q[ag] = s_Sq[ag];
        decode_vals(q, s_sc, A.loss, A.NK, v);
        for (int k = 0; k < A.NK; k++) s_S[k] = v[k];
    }
    __syncthreads();
}

// The decision for one node (get_best_split's threshold, src/fit-utils.jl:444-450; the Tree arrays, src/fit.jl:96-103;
// a node without a split becomes a leaf, src/predict.jl:198-262): thread 0 holds the node's best candidate (bg, bj, bb)
// and its feature (1-based id, type); S: the node's statistics (in shared memory).  Leaves {found, bj, bb} in s_dec.
template <int NAG>
__device__ __forceinline__ void scan_decide(const ScanArgs &A, int n, const double *S, int *s_dec, double bg, int bj, int bb, int feat, bool numeric) {
    constexpr int K = NAG == 5 ? 2 : 1; // the channel layout names the outputs
    const int found = (bb != NO_BIN && bg > A.gamma) ? 1 : 0;
    s_dec[0] = found; s_dec[1] = bj; s_dec[2] = bb;
    if (found) {
        A.tree.feat[n - 1] = feat;
        A.tree.cond_bin[n - 1] = (uint8_t)bb;
        A.tree.gain[n - 1] = (float)bg;
        A.tree.split[n - 1] = 1;
        A.tree.packed[n - 1] = evt_pack_node(feat, bb, numeric);
        A.status[n] = ST_SPLIT;
    } else {
        for (int k = 0; k < K; k++) A.tree.pred[(int64_t)K * (n - 1) + k] = (float)leaf_value(A.loss, S, k, K, A.eta, A.bagging, A.lambda, A.L2);
        A.status[n] = ST_LEAF;
    }
}

// Totals of the two children from the left child's (qL; right = parent - left, exact in integers; _child_sums!,
// src/fit-utils.jl:472-486), by one lane.  With fold_leaves the children are leaves of the last level: their weight, values
// and state are written here too - what the leaf-level pass would compute from node_sum (same integers, same expressions).
template <int NAG>
__device__ __forceinline__ void write_children(const ScanArgs &A, int n, const long long *qL, const long long *s_Sq, const double *s_sc) {
    constexpr int K = NAG == 5 ? 2 : 1, NK = 2 * K + 1;
#pragma unroll
    for (int child = 0; child < 2; child++) {
        const int cn = 2 * n + child;
        long long qc[NAG];
#pragma unroll
        for (int ag = 0; ag < NAG; ag++) {
            qc[ag] = child ? s_Sq[ag] - qL[ag] : qL[ag];
            A.node_sum[(int64_t)cn * NAG + ag] = qc[ag];
        }
        if (A.fold_leaves) {
            double v[NK];
            decode_vals(qc, s_sc, A.loss, NK, v);
            A.tree.w[cn - 1] = (float)v[NK - 1];
            for (int k = 0; k < K; k++) A.tree.pred[(int64_t)K * (cn - 1) + k] = (float)leaf_value(A.loss, v, k, K, A.eta, A.bagging, A.lambda, A.L2);
            A.status[cn] = ST_LEAF;
        }
    }
}

// the children's histogram slices start from zero (the build child accumulates into its own)
template <int NAG>
__device__ __forceinline__ void zero_children_slices(const ScanArgs &A, int n) {
    long long *hc = A.hist + (int64_t)(2 * n - 1) * A.node_stride;
    const int64_t used = (int64_t)A.nfs * NAG * A.B;
    for (int64_t i = threadIdx.x; i < used; i += blockDim.x) {
        hc[i] = 0;
        hc[A.node_stride + i] = 0;
    }
}

// Pass 1: grid (nodes of the level, feature groups); one wave per (node, sampled feature).
// Writes the group's best candidate to sbest[node][group] (or the gain matrix for oblivious trees)
// and, for subtract nodes, materialises h[n] = h[parent] - h[sibling].
// FUSED: one block of 16 waves per node covers every sampled feature (at most 16) and finishes the node itself
// (scan_finish): one launch per level instead of two where a level is a chain of small kernels.
// What the first requests are made from comes as arguments of its own, ahead of the rest: these are in scalar registers when a wavefront starts (a struct's fields are not), and the
// rest is on its way beside the feature id and the node's state, which are now one trip (the id was waited for before the state was asked for, and the block's size was a trip of
// its own).  us a launch: 500k x 100 of 64 bins, half the features, 6.14 -> 5.8 (5.7 to 5.9; without the registers 6.0), 800k x 28 of 128 bins 8.6 -> 8.1 (8.3), 10M x 100 14.1 -> 13.4.
template <int NAG, int BPL, bool FUSED>
__global__ __launch_bounds__(FUSED ? 1024 : 256) void k_scan(const uint32_t *js, const int32_t *status, long long *hist, int64_t node_stride, int level, int nfs, int B,
                                                             ScanArgs A) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int nwaves = FUSED ? 16 : 4;
    const int n = (1 << (level - 1)) + blockIdx.x; // 1-based node id
    // The block's time is a chain of round trips to memory, so requests go out in as few dependent steps as the data
    // allows: node state and feature id first; then, in one batch of unconditional loads, the histogram slices, the
    // feature's type and constraint, the node totals and the decode scales.
    const int jp = blockIdx.y * nwaves + wave;
    const bool have = jp < nfs; // wave-uniform; a wave past the last feature loads the last one's data and drops it
    const int jpc = have ? jp : nfs - 1;
    int f = (int)js[jpc], st = status[n];
    touch_kernargs<decltype(k_scan<NAG, BPL, FUSED>)>();
    asm volatile("" : "+s"(f), "+s"(st)); // both are requested before either is waited for, and ahead of the branch on the state
    if (st != ST_BUILD && st != ST_SUBTRACT) return;
    f -= 1;
    const bool is_sub = (st == ST_SUBTRACT);
    // the channel layout fixes the outputs: two-output MLE losses have five channels, every other shape here one output
    constexpr int K = (NAG == 5) ? 2 : 1, NK = 2 * K + 1;
    // BPL = bins per lane = ceil(nbins / 64), a template parameter so that nbins <= 64 keeps one bin per lane in registers
    long long *hn = hist + (int64_t)(n - 1) * node_stride;
    const long long *hp = hist + (int64_t)((n >> 1) - 1) * node_stride;
    const long long *hs = hist + (int64_t)((n ^ 1) - 1) * node_stride;

    __shared__ long long s_Sq[EVT_MAX_NA];
    __shared__ double s_S[EVT_MAX_NK];
    __shared__ double s_sc[EVT_MAX_NA];
    __shared__ double s_wg[16];
    __shared__ int s_wjp[16], s_wbin[16];
    __shared__ int s_wfeat[16]; // feature of each wave (1-based id, negative when categorical)
    __shared__ long long s_wq[FUSED ? 1 : 4][NAG]; // two-pass search: left totals of each wave's best candidate
    __shared__ int s_dec[3];

    long long pre[NAG][BPL];
    long long vb[NAG][BPL];
    long long excl[NAG];
    const int64_t o0 = (int64_t)jpc * NAG * B;
    if (is_sub) {
#pragma unroll
        for (int ag = 0; ag < NAG; ag++) {
#pragma unroll
            for (int t = 0; t < BPL; t++) {
                const int b = lane * BPL + t;
                const int64_t o = o0 + (int64_t)ag * B + (b < B ? b : B - 1);
                pre[ag][t] = hp[o];
                vb[ag][t] = hs[o];
            }
        }
    } else {
#pragma unroll
        for (int ag = 0; ag < NAG; ag++) {
#pragma unroll
            for (int t = 0; t < BPL; t++) {
                const int b = lane * BPL + t;
                pre[ag][t] = hn[o0 + (int64_t)ag * B + (b < B ? b : B - 1)];
                vb[ag][t] = 0;
            }
        }
    }
    const bool numeric = A.feattypes[f] != 0;
    const int constraint = A.mono[f];
    // node totals and decode scales: the same few words for every thread of the block (scalar loads), so that below the
    // root no thread waits at a barrier for another to decode them
    long long nsq[NAG];
    double sc[NAG];
#pragma unroll
    for (int ag = 0; ag < NAG; ag++) {
        sc[ag] = A.qscale[ag];
        nsq[ag] = A.node_sum[(int64_t)n * NAG + ag]; // not yet written at level 1, and not used there
    }

#pragma unroll
    for (int ag = 0; ag < NAG; ag++) {
#pragma unroll
        for (int t = 0; t < BPL; t++) {
            const int b = lane * BPL + t;
            const long long v = (have && b < B) ? pre[ag][t] - vb[ag][t] : 0;
            if (is_sub && have && b < B) hn[o0 + (int64_t)ag * B + b] = v; // subtract_hist!: h[n] = h[parent] - h[sibling]
            pre[ag][t] = v;
        }
    }

    // node totals -> Float64 statistics
    if (level == 1) { // the root's totals are any sampled feature's sums over its bins: the wavefront's own (a wavefront past the last feature has none, and no use for them).
        // Read again by one wavefront, with two barriers behind it, they took the root's search from 6.5 to 7.8 us (50 features x 64 bins), from 8.9 to 11.4 (28 x 128).
#pragma unroll
        for (int ag = 0; ag < NAG; ag++) {
            long long sum = 0;
#pragma unroll
            for (int t = 0; t < BPL; t++) sum += pre[ag][t];
            nsq[ag] = wave_sum_i64(sum);
            if (blockIdx.y == 0 && tid == 0) A.node_sum[(int64_t)n * NAG + ag] = nsq[ag];
        }
    }
    double S[NK];
    decode_vals(nsq, sc, A.loss, NK, S);
    if (FUSED && tid == 0) { // the block's last step reads them from shared memory, behind the barriers below
#pragma unroll
        for (int ag = 0; ag < NAG; ag++) {
            s_sc[ag] = sc[ag];
            s_Sq[ag] = nsq[ag];
        }
        for (int k = 0; k < NK; k++) s_S[k] = S[k];
    }

    double gain_p = 0.0;
    for (int k = 0; k < K; k++) gain_p += node_gain_k(A.loss, S[k], S[K + k], S[2 * K], A.lambda, A.L2);
    const double w_p = S[NK - 1];

    double wbest = -INFINITY;
    int wjp = NO_BIN, wbin = NO_BIN;
    const int nodeidx = blockIdx.x;

    if (have) {
        const int bmax = numeric ? B - 1 : B;
        // inclusive prefix over the bins: within the lane, then across the wavefront
#pragma unroll
        for (int ag = 0; ag < NAG; ag++) {
            long long run = 0;
#pragma unroll
            for (int t = 0; t < BPL; t++) {
                run += pre[ag][t];
                pre[ag][t] = run;
            }
            const long long incl = wave_incl_scan_i64(run);
            excl[ag] = incl - run;
#pragma unroll
            for (int t = 0; t < BPL; t++) pre[ag][t] += excl[ag];
        }
        double lg = -INFINITY;
        int lb = NO_BIN;
        long long lq[NAG]; // fixed-point totals left of this lane's best candidate
#pragma unroll
        for (int ag = 0; ag < NAG; ag++) lq[ag] = 0;
#pragma unroll
        for (int t = 0; t < BPL; t++) {
            const int b = lane * BPL + t;
            if (b < B) {
                double gain = 0.0;
                bool ok = false;
                long long q[NAG];
#pragma unroll
                for (int ag = 0; ag < NAG; ag++) q[ag] = 0;
                if (b + 1 <= bmax) {
#pragma unroll
                    for (int ag = 0; ag < NAG; ag++) {
                        const long long prev = (t == 0) ? excl[ag] : pre[ag][t > 0 ? t - 1 : 0];
                        q[ag] = numeric ? pre[ag][t] : (pre[ag][t] - prev); // _acc_left!: accumulate vs single bin
                    }
                    double SL[NK];
                    decode_vals(q, sc, A.loss, NK, SL);
                    const double w_l = SL[NK - 1];
                    const double w_r = w_p - w_l;
                    if (w_l > A.min_weight && w_r > A.min_weight) {
                        ok = true;
                        if (constraint != 0) {
                            double SR[NK];
                            for (int k = 0; k < NK; k++) SR[k] = S[k] - SL[k];
                            const double predL = leaf_value(A.loss, SL, 0, K, A.eta, A.bagging, A.lambda, A.L2);
                            const double predR = leaf_value(A.loss, SR, 0, K, A.eta, A.bagging, A.lambda, A.L2);
                            ok = (constraint == -1 && predL > predR) || (constraint == 1 && predL < predR);
                        }
                        if (ok) {
                            double sg = 0.0;
                            for (int k = 0; k < K; k++) {
                                sg += split_gain_k(A.loss, S[k], S[K + k], w_p, SL[k], SL[K + k], w_l, w_r, A.lambda, A.L2);
                            }
                            gain = sg - gain_p;
                        }
                    }
                }
                if (A.oblivious) {
                    A.ogains[((int64_t)nodeidx * nfs + jp) * B + b] = ok ? gain : 0.0; // update_gains!
                } else if (ok && gain > lg) {
                    lg = gain;
                    lb = b + 1;
#pragma unroll
                    for (int ag = 0; ag < NAG; ag++) lq[ag] = q[ag];
                }
            }
        }
        if (!A.oblivious) {
            wave_argmax(lg, lb);
            if (lg > wbest) { wbest = lg; wjp = jp; wbin = lb; }
            if constexpr (!FUSED) {
                // the lane that holds the winning bin hands its left totals over
                if (lane == (lb != NO_BIN ? (lb - 1) / BPL : 0)) {
#pragma unroll
                    for (int ag = 0; ag < NAG; ag++) s_wq[wave][ag] = lq[ag];
                }
            }
        }
    }
    if (A.oblivious) return; // decision is taken for the whole level by k_obliv_max and k_obliv_apply

    if (lane == 0) {
        s_wg[wave] = wbest; s_wjp[wave] = wjp; s_wbin[wave] = wbin;
        s_wfeat[wave] = numeric ? f + 1 : -(f + 1);
    }
    __syncthreads();
    double bg = -INFINITY;
    int bj = NO_BIN, bb = NO_BIN, bw = 0;
    if (tid == 0) { // the waves' features ascend: only a strictly larger gain replaces an earlier one
        constexpr int NW = FUSED ? 16 : 4;
        double g[NW]; // all of them in one trip to LDS
#pragma unroll
        for (int w = 0; w < NW; w++) g[w] = s_wg[w];
#pragma unroll
        for (int w = 0; w < NW; w++)
            if (g[w] > bg) { bg = g[w]; bw = w; }
        if (bg > -INFINITY) { bj = s_wjp[bw]; bb = s_wbin[bw]; }
    }
    if constexpr (FUSED) {
        // the node is finished here: wave jp scanned sampled feature jp, so the winner's left totals are still in the
        // registers of the lane that holds the winning bin - no second read of the histogram
        if (tid == 0) {
            A.tree.w[n - 1] = (float)S[NK - 1];
            const int wf = (bb != NO_BIN) ? s_wfeat[bj] : 1;
            scan_decide<NAG>(A, n, s_S, s_dec, bg, bj, bb, wf < 0 ? -wf : wf, wf > 0);
        }
        __syncthreads();
        if (!s_dec[0]) return;
        if (have && jp == s_dec[1]) {
            const int b0 = s_dec[2] - 1; // 0-based winning bin: lane b0 / BPL, position b0 % BPL
            long long qL[NAG];
#pragma unroll
            for (int ag = 0; ag < NAG; ag++) {
                long long v = 0;
#pragma unroll
                for (int t = 0; t < BPL; t++) {
                    const long long prev = (t == 0) ? excl[ag] : pre[ag][t > 0 ? t - 1 : 0];
                    const long long q = numeric ? pre[ag][t] : (pre[ag][t] - prev);
                    if (t == b0 % BPL) v = q;
                }
                qL[ag] = v;
            }
            if (lane == b0 / BPL) write_children<NAG>(A, n, qL, s_Sq, s_sc);
        }
        if (A.zero_children) zero_children_slices<NAG>(A, n);
    } else if (A.last_decides) {
        // The node's blocks meet at a counter: each hands in its candidate with stores that go past its XCD's cache, and the one that
        // comes last reads them all the same way and decides.  No block waits for another.  Bound by that chain (2 to 3 us: store, count,
        // read) where a level has few nodes, by the histograms it reads and clears where it has many.  A second launch
        // for the decision took 5 to 7 us and its gap: 100 features x 64 bins, two kernels -> one: 1 node 5.7 + 5.1 -> 7.4 us, 32 nodes
        // 6.6 + 10.4 -> 9.4, 256 nodes 23.1 + 11.5 -> 28.7, 512 nodes 41.6 + 6.5 -> 46.1; 28 features x 128 bins 6.0 + 5.6 -> 7.8, 26.6 + 7.5 -> 31.0.
        // (Counters side by side, 32 to a line: 500 features and 16 nodes 31 us, 14 with a line each.)
        // Order: every word handed over is stored and loaded by agent-scope atomics, which go past the caches that are not shared, so that
        // what a release adds to them is only the wait for the stores' completion, written out here, and what an acquire adds is only
        // that the loads come behind the count, which the branch on it and the barrier for the compiler see to.  The language's own
        // release also writes back the histograms that lie dirty in L2, and an acquire throws L2 away: a count with both 1318 us a tree, with
        // the release and an acquire by the last block alone 1175, as it is 648 (100 features x 64 bins, 1M rows, depth 11).
        constexpr int CW = 3 + NAG; // words of a candidate: gain, position and bin, feature, totals
        unsigned long long *cand = reinterpret_cast<unsigned long long *>(reinterpret_cast<ScanBestQ *>(A.sbest) + (int64_t)nodeidx * gridDim.y);
        int last = 0;
        if (tid == 0) {
            unsigned long long w[CW];
            w[0] = (unsigned long long)__double_as_longlong(bg);
            w[1] = (unsigned int)bj | ((unsigned long long)(unsigned int)bb << 32);
            w[2] = (unsigned int)s_wfeat[bw];
#pragma unroll
            for (int ag = 0; ag < NAG; ag++) w[3 + ag] = (unsigned long long)s_wq[bw][ag];
#pragma unroll
            for (int k = 0; k < CW; k++) __hip_atomic_store(cand + (size_t)blockIdx.y * 8 + k, w[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the candidate is in memory before it is counted
            last = __hip_atomic_fetch_add(A.counts + (size_t)nodeidx * EVT_SCAN_COUNT_STEP, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.y - 1;
        }
        // the children's slices start from zero: a wave clears its feature's bins in both, whatever the node turns out to be
        if (A.zero_children && have) {
            long long *hc = hist + (int64_t)(2 * n - 1) * node_stride + o0;
            for (int i = lane; i < NAG * B; i += 64) {
                hc[i] = 0;
                hc[node_stride + i] = 0;
            }
        }
        if (wave != 0 || !__builtin_amdgcn_readfirstlane(last)) return;
        asm volatile("" ::: "memory");
        ScanBestQ mine;
        mine.gain = -INFINITY; mine.jp = NO_BIN; mine.bin = NO_BIN; mine.feat = 1;
        for (int g = lane; g < (int)gridDim.y; g += 64) { // ascending positions: only a strictly larger gain replaces an earlier one
            unsigned long long w[CW];
#pragma unroll
            for (int k = 0; k < CW; k++) w[k] = __hip_atomic_load(cand + (size_t)g * 8 + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const double gg = __longlong_as_double((long long)w[0]);
            if (gg > mine.gain) {
                mine.gain = gg;
                mine.jp = (int)(w[1] & 0xffffffffull);
                mine.bin = (int)(w[1] >> 32);
                mine.feat = (int)w[2];
#pragma unroll
                for (int ag = 0; ag < NAG; ag++) mine.qL[ag] = (long long)w[3 + ag];
            }
        }
        double g = mine.gain;
        int j = mine.jp;
        wave_argmax(g, j); // highest gain, then the earliest feature, whose bin is already the lowest
        const bool found = j != NO_BIN && g > A.gamma;
        if (found ? (mine.jp == j) : (lane == 0)) {
            A.counts[(size_t)nodeidx * EVT_SCAN_COUNT_STEP] = 0;
            A.tree.w[n - 1] = (float)S[NK - 1];
            const int feat = found ? (mine.feat < 0 ? -mine.feat : mine.feat) : 1;
            scan_decide<NAG>(A, n, S, s_dec, g, j, found ? mine.bin : NO_BIN, feat, found ? mine.feat > 0 : true);
            if (found) {
                write_children<NAG>(A, n, mine.qL, nsq, sc);
            }
        }
    } else if (tid == 0) {
        ScanBestQ r;
        r.gain = bg; r.jp = bj; r.bin = bb;
        r.feat = s_wfeat[bw]; r.pad = 0;
#pragma unroll
        for (int ag = 0; ag < EVT_MAX_NA; ag++) r.qL[ag] = (ag < NAG) ? s_wq[bw][ag < NAG ? ag : 0] : 0;
        reinterpret_cast<ScanBestQ *>(A.sbest)[(int64_t)nodeidx * gridDim.y + blockIdx.y] = r;
    }
}

// Pass 2 (leaf levels, and the search as two kernels): one block per node.  Leaf level: leaf value only.  Otherwise: arg-max over the feature
// groups (first maximum: highest gain, then earliest feature, whose bin is already the lowest),
// split iff gain > gamma; writes the Tree arrays, the children's totals (_child_sums!: left = bins
// 1..bin of the parent histogram, or that bin alone for categorical features; right = parent - left,
// exact in integers) and zeroes the children's histogram slices.
template <int NAG>
__global__ __launch_bounds__(256) void k_scan_fin(ScanArgs A, int ngroups) {
    const int tid = threadIdx.x;
    const int n = (1 << (A.level - 1)) + blockIdx.x;
    if (blockIdx.y > 0) {
        // Blocks beyond the first of a node only clear the children's histogram slices (the build child accumulates
        // into its own; a level with few nodes would otherwise leave 200 KB per node to one block).  They do not wait
        // for the decision: the slices of a node that turns out a leaf are never read.  The node's state may already
        // read SPLIT or LEAF here (the first block sets it), anything but INACTIVE means the level reached it.
        if (A.status[n] == ST_INACTIVE) return;
        long long *hc = A.hist + (int64_t)(2 * n - 1) * A.node_stride;
        const int64_t used = (int64_t)A.nfs * NAG * A.B;
        const int64_t zb = gridDim.y - 1, per = (used + zb - 1) / zb;
        const int64_t i0 = (int64_t)(blockIdx.y - 1) * per, i1 = i0 + per < used ? i0 + per : used;
        for (int64_t i = i0 + tid; i < i1; i += blockDim.x) {
            hc[i] = 0;
            hc[A.node_stride + i] = 0;
        }
        return;
    }
    // Everything the block needs is requested in one batch of unconditional loads, ahead of the branch on the node's
    // state: the state itself, the node's totals and decode scales, and this thread's candidate (group tid, clamped).
    const int tq = tid < NAG ? tid : 0;
    double qs = A.qscale[tq];
    long long nsq = A.node_sum[(int64_t)n * NAG + tq]; // not yet written at level 1, and not used there
    union CandWords {
        ScanBestQ q;
        uint4 v[4];
    };
    CandWords cw;
    {
        const uint4 *cp = reinterpret_cast<const uint4 *>(reinterpret_cast<const ScanBestQ *>(A.sbest) + (int64_t)blockIdx.x * ngroups + (tid < ngroups ? tid : 0));
#pragma unroll
        for (int k = 0; k < 4; k++) cw.v[k] = cp[k];
    }
    // nodes of the last level are the children of the split nodes above them (the root when max_depth == 1)
    int st = A.leaf_level ? (n > 1 ? A.status[n >> 1] : ST_SPLIT) : A.status[n];
    asm volatile("" : "+v"(st), "+v"(qs), "+v"(nsq));
#pragma unroll
    for (int k = 0; k < 4; k++) asm volatile("" : "+v"(cw.v[k].x), "+v"(cw.v[k].y), "+v"(cw.v[k].z), "+v"(cw.v[k].w));
    if (A.leaf_level) {
        if (st != ST_SPLIT) return;
    } else {
        if (st != ST_BUILD && st != ST_SUBTRACT) return;
    }
    const int NK = A.NK, K = A.K;
    long long *hn = A.hist + (int64_t)(n - 1) * A.node_stride;

    __shared__ long long s_Sq[EVT_MAX_NA];
    __shared__ double s_S[EVT_MAX_NK];
    __shared__ double s_sc[EVT_MAX_NA];
    __shared__ double s_g[256];
    __shared__ int s_j[256], s_b[256];
    __shared__ int s_dec[3];

    if (A.level == 1) {
        root_totals<NAG>(A, n, hn, s_Sq, s_S, s_sc);
    } else {
        if (tid < NAG) {
            s_sc[tid] = qs;
            s_Sq[tid] = nsq;
        }
        __syncthreads();
        if (tid == 0) {
            double v[EVT_MAX_NK];
            long long q[NAG];
            for (int ag = 0; ag < NAG; ag++) q[ag] = s_Sq[ag];
            decode_vals(q, s_sc, A.loss, NK, v);
            for (int k = 0; k < NK; k++) s_S[k] = v[k];
        }
        __syncthreads();
    }
    double S[EVT_MAX_NK];
    for (int k = 0; k < NK; k++) S[k] = s_S[k];
    if (tid == 0) A.tree.w[n - 1] = (float)S[NK - 1];

    if (A.leaf_level) {
        if (tid < K) A.tree.pred[(int64_t)K * (n - 1) + tid] = (float)leaf_value(A.loss, S, tid, K, A.eta, A.bagging, A.lambda, A.L2);
        if (tid == 0) A.status[n] = ST_LEAF;
        return;
    }
    // a thread takes the groups tid, tid + 256, ... (more than 1024 sampled features): ascending feature positions, so
    // only a strictly larger gain replaces an earlier one.  It keeps the whole candidate: the thread whose candidate wins
    // decides the node and writes the children's totals from its own registers - no feature table, no histogram read.
    ScanBestQ mine = cw.q;
    if (tid >= ngroups) {
        mine.gain = -INFINITY; mine.jp = NO_BIN; mine.bin = NO_BIN;
    }
    const ScanBestQ *cand = reinterpret_cast<const ScanBestQ *>(A.sbest) + (int64_t)blockIdx.x * ngroups;
    for (int g = tid + 256; g < ngroups; g += 256) {
        const ScanBestQ r = cand[g];
        if (r.gain > mine.gain) mine = r;
    }
    s_g[tid] = mine.gain; s_j[tid] = mine.jp; s_b[tid] = mine.bin;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) {
            if (s_g[tid + o] > s_g[tid] || (s_g[tid + o] == s_g[tid] && s_j[tid + o] < s_j[tid])) {
                s_g[tid] = s_g[tid + o]; s_j[tid] = s_j[tid + o]; s_b[tid] = s_b[tid + o];
            }
        }
        __syncthreads();
    }
    const double bg = s_g[0];
    const int bj = s_j[0], bb = s_b[0];
    // every sampled feature belongs to one group and every group to one thread: exactly one thread holds the winner;
    // without any candidate the first thread turns the node into a leaf
    const bool found = (bb != NO_BIN && bg > A.gamma);
    const bool owner = found ? (mine.jp == bj && mine.bin != NO_BIN) : (tid == 0);
    if (owner) {
        const int feat = found ? (mine.feat < 0 ? -mine.feat : mine.feat) : 1;
        scan_decide<NAG>(A, n, s_S, s_dec, bg, bj, bb, feat, found ? mine.feat > 0 : true);
        if (found) {
            long long qL[NAG];
#pragma unroll
            for (int ag = 0; ag < NAG; ag++) qL[ag] = mine.qL[ag];
            write_children<NAG>(A, n, qL, s_Sq, s_sc);
        }
    }
    if (!found) return;
    // with one block per node this block clears the children's slices, otherwise the node's other blocks have
    if (A.zero_children && gridDim.y == 1) zero_children_slices<NAG>(A, n);
}

// Oblivious trees (grow_otree!, src/fit.jl:190-257): per-level decision from the sum of the
// nodes' gain matrices, masked where any node's gain is not positive; first maximum in
// (feature position, bin) order; all nodes of the level split on it iff it exceeds gamma.
struct OblivArgs {
    long long *hist;
    int64_t node_stride;
    const uint32_t *js;
    const uint8_t *feattypes;
    int32_t *status;
    long long *node_sum;
    const double *qscale;
    TreeDev tree;
    const double *ogains;
    const int64_t *hdr;
    const int32_t *act_node;
    double eta, lambda, L2, gamma;
    int bagging, nfs, B, K, NK, NAg, loss, level, zero_children;
    ScanBest *best; // first maximum (gain, cell) of each block of k_obliv_max
    int nbest;
};

// The level matrix and its first maximum: a block takes a share of the (feature position, bin) cells, a thread a cell at a time; the
// nodes' gains are added in node order, eight requested ahead of their use.  One block of the whole level took 5 to 20 us per
// level for this (50 features x 64 bins, up to 32 nodes), waiting for one load after the other.
__global__ __launch_bounds__(256) void k_obliv_max(OblivArgs A) {
    const int tid = threadIdx.x;
    const int n_act = (int)A.hdr[LH_N_ACT];
    if (n_act <= 0) return;
    const int first = 1 << (A.level - 1);
    const int cells = A.nfs * A.B;
    __shared__ double s_g[256];
    __shared__ int s_i[256];
    double bg = -INFINITY;
    int bi = NO_BIN;
    for (int c = (int)blockIdx.x * 256 + tid; c < cells; c += (int)gridDim.x * 256) {
        double acc = 0.0;
        bool allpos = true;
        for (int i0 = 0; i0 < n_act; i0 += 8) {
            double g[8];
            int n[8];
#pragma unroll
            for (int j = 0; j < 8; j++) n[j] = A.act_node[i0 + j < n_act ? i0 + j : n_act - 1];
#pragma unroll
            for (int j = 0; j < 8; j++) g[j] = A.ogains[(int64_t)(n[j] - first) * cells + c];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                if (i0 + j >= n_act) continue;
                acc += g[j];
                if (n[j] > 1) allpos = allpos && (g[j] > 0.0);
            }
        }
        const double v = allpos ? acc : 0.0;
        if (v > bg) { bg = v; bi = c; } // c ascending per thread: first maximum kept
    }
    s_g[tid] = bg;
    s_i[tid] = bi;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o && (s_g[tid + o] > s_g[tid] || (s_g[tid + o] == s_g[tid] && s_i[tid + o] < s_i[tid]))) {
            s_g[tid] = s_g[tid + o];
            s_i[tid] = s_i[tid + o];
        }
        __syncthreads();
    }
    if (tid == 0) {
        A.best[blockIdx.x].gain = s_g[0];
        A.best[blockIdx.x].jp = s_i[0];
    }
}

// One node per block column (nodes of the level that are not active return): its first block takes the maximum of k_obliv_max's
// blocks and writes the node's part of the level's decision, the others clear the children's histogram slices (whatever the
// decision: the slices of a leaf are never read).
__global__ __launch_bounds__(256) void k_obliv_apply(OblivArgs A) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwaves = 4;
    const int B = A.B, K = A.K, NK = A.NK, NAG = A.NAg;
    const int n_act = (int)A.hdr[LH_N_ACT];
    if ((int)blockIdx.x >= n_act) return;
    const int n = A.act_node[blockIdx.x];
    if (blockIdx.y > 0) {
        long long *hc = A.hist + (int64_t)(2 * n - 1) * A.node_stride;
        const int64_t used = (int64_t)A.nfs * NAG * B;
        const int64_t zb = gridDim.y - 1, per = (used + zb - 1) / zb;
        const int64_t i0 = (int64_t)(blockIdx.y - 1) * per, i1 = i0 + per < used ? i0 + per : used;
        for (int64_t i = i0 + tid; i < i1; i += 256) {
            hc[i] = 0;
            hc[A.node_stride + i] = 0;
        }
        return;
    }
    __shared__ double s_g[256];
    __shared__ int s_i[256];
    __shared__ double s_sc[EVT_MC_MAX_NK], s_S[EVT_MC_MAX_NK];
    __shared__ long long s_Sq[EVT_MC_MAX_NK];
    double bg = -INFINITY;
    int bi = NO_BIN;
    for (int k = tid; k < A.nbest; k += 256) { // blocks' cells interleave: ties go to the lowest cell
        const ScanBest r = A.best[k];
        if (r.gain > bg || (r.gain == bg && r.jp < bi)) { bg = r.gain; bi = r.jp; }
    }
    s_g[tid] = bg;
    s_i[tid] = bi;
    if (tid < NAG) {
        s_sc[tid] = A.qscale[tid];
        s_Sq[tid] = A.node_sum[(int64_t)n * NAG + tid];
    }
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o && (s_g[tid + o] > s_g[tid] || (s_g[tid + o] == s_g[tid] && s_i[tid + o] < s_i[tid]))) {
            s_g[tid] = s_g[tid + o];
            s_i[tid] = s_i[tid + o];
        }
        __syncthreads();
    }
    if (tid == 0) decode_vals(s_Sq, s_sc, A.loss, NK, s_S);
    __syncthreads();
    const bool found = s_i[0] != NO_BIN && s_g[0] > A.gamma;
    if (tid == 0) A.tree.w[n - 1] = (float)s_S[NK - 1];
    if (!found) {
        if (tid < K) A.tree.pred[(int64_t)K * (n - 1) + tid] = (float)leaf_value(A.loss, s_S, tid, K, A.eta, A.bagging, A.lambda, A.L2);
        if (tid == 0) A.status[n] = ST_LEAF;
        return;
    }
    const int bj = s_i[0] / B, bb = s_i[0] % B + 1;
    const int feat = (int)A.js[bj];
    const bool numeric = A.feattypes[feat - 1] != 0;
    const long long *hn = A.hist + (int64_t)(n - 1) * A.node_stride;
    for (int ag = wave; ag < NAG; ag += nwaves) {
        const int64_t o = ((int64_t)bj * NAG + ag) * B;
        long long s = 0;
        for (int b = lane; b < B; b += 64) {
            const bool in = numeric ? (b + 1 <= bb) : (b + 1 == bb);
            if (in) s += hn[o + b];
        }
        s = wave_sum_i64(s);
        if (lane == 0) {
            A.node_sum[(int64_t)(2 * n) * NAG + ag] = s;
            A.node_sum[(int64_t)(2 * n + 1) * NAG + ag] = s_Sq[ag] - s;
        }
    }
    if (tid == 0) {
        A.tree.feat[n - 1] = feat;
        A.tree.cond_bin[n - 1] = (uint8_t)bb;
        A.tree.gain[n - 1] = (float)s_g[0];
        A.tree.split[n - 1] = 1;
        A.tree.packed[n - 1] = evt_pack_node(feat, bb, numeric);
        A.status[n] = ST_SPLIT;
    }
}

// A whole oblivious level in one launch: a block owns a sampled feature and searches all nodes of the level, a wavefront one or two of them, as
// k_scan; adds their gains in node order in LDS, and hands in its first maximum with the nodes' totals left of it; the last block to do
// so takes the best and writes the level's decision, the children's totals and, on the last level that splits, their leaves.  The hand-over is
// k_scan's.  Bound by that chain and, from 16 nodes on, by the divisions of a block's searches (nodes spread over several blocks need one
// more hand-over, which cost more than it gave: 16 nodes 14.7 -> 16.2 us).  In three launches (k_scan, k_obliv_max, k_obliv_apply) and one for
// the leaves the chain was cut by kernel boundaries: 500k rows x 50 features x 64 bins of two outputs, 1, 4, 16 and 32 nodes and the leaves,
// 18.7, 15.5, 16.2 and 23.0 -> 8.8, 9.0, 12.5 and 15.6 us.
struct OblivLevelArgs {
    OblivArgs o;
    const int32_t *mono;
    int32_t *counts;
    double min_weight;
    int fold_leaves;
    unsigned long long *lefts; // [feature][node][NAG]: totals left of the feature's candidate
};

// NPW: nodes of a wavefront
template <int NAG, int BPL, int NPW>
__global__ __launch_bounds__(NAG * BPL > 12 ? 512 : 1024) void k_obliv_level(OblivLevelArgs L) {
    extern __shared__ double s_gain[]; // [nodes][B]
    __shared__ long long s_tot[OBLIV_LEVEL_NODES * NAG], s_left[OBLIV_LEVEL_NODES * NAG];
    __shared__ int s_last, s_bin, s_cell;
    __shared__ double s_best;
    const OblivArgs &A = L.o;
    touch_kernargs<decltype(k_obliv_level<NAG, BPL, NPW>)>();
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwaves = blockDim.x >> 6;
    constexpr int K = (NAG == 5) ? 2 : 1, NK = 2 * K + 1;
    const int B = A.B, jp = blockIdx.x;
    // all nodes of a level split on the same feature or none does: the level's nodes are all active, or none is
    const int first = 1 << (A.level - 1), nodes = first;
    const bool any = A.hdr[LH_N_ACT] > 0;
    const int f = (int)A.js[jp] - 1;
    int st[NPW];
#pragma unroll
    for (int j = 0; j < NPW; j++) st[j] = A.status[first + (wave + j * nwaves < nodes ? wave + j * nwaves : 0)];
    double sc[NAG];
#pragma unroll
    for (int ag = 0; ag < NAG; ag++) sc[ag] = A.qscale[ag];
#pragma unroll
    for (int j = 0; j < NPW; j++) asm volatile("" : "+v"(st[j])); // requested ahead of the branch
    if (!any) return; // every block alike
    const bool numeric = A.feattypes[f] != 0;
    const int constraint = L.mono[f];
    const int64_t o0 = (int64_t)jp * NAG * B;
    const int bmax = numeric ? B - 1 : B;

    long long left[NPW][NAG][BPL]; // the words of the wavefront's nodes, requested together, then the sums left of every bin
    {
        long long vb[NPW][NAG][BPL], nsq[NPW][NAG];
#pragma unroll
        for (int j = 0; j < NPW; j++) {
            const int n = first + (wave + j * nwaves < nodes ? wave + j * nwaves : 0);
            const bool is_sub = st[j] == ST_SUBTRACT;
            const long long *pa = A.hist + (int64_t)((is_sub ? n >> 1 : n) - 1) * A.node_stride + o0, *pb = A.hist + (int64_t)((n ^ 1) - 1) * A.node_stride + o0;
#pragma unroll
            for (int ag = 0; ag < NAG; ag++) {
                nsq[j][ag] = A.node_sum[(int64_t)n * NAG + ag]; // not yet written at level 1, and not used there
#pragma unroll
                for (int t = 0; t < BPL; t++) {
                    const int o = ag * B + (lane * BPL + t < B ? lane * BPL + t : B - 1);
                    left[j][ag][t] = pa[o];
                    vb[j][ag][t] = is_sub ? pb[o] : 0;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < NPW; j++) {
            const int s = wave + j * nwaves, n = first + s;
            if (s >= nodes) continue;
            const bool is_sub = st[j] == ST_SUBTRACT;
            long long *hn = A.hist + (int64_t)(n - 1) * A.node_stride + o0;
#pragma unroll
            for (int ag = 0; ag < NAG; ag++) {
                long long run = 0, val[BPL];
#pragma unroll
                for (int t = 0; t < BPL; t++) {
                    const int b = lane * BPL + t;
                    val[t] = b < B ? left[j][ag][t] - vb[j][ag][t] : 0;
                    if (is_sub && b < B) hn[ag * B + b] = val[t]; // subtract_hist!
                    run += val[t];
                    left[j][ag][t] = run;
                }
                const long long incl = wave_incl_scan_i64(run), excl = incl - run;
                if (A.level == 1) { // the root's totals are any feature's sums over its bins
                    nsq[j][ag] = readlane_i64(incl, 63);
                    if (jp == 0 && lane == 0) A.node_sum[(int64_t)n * NAG + ag] = nsq[j][ag];
                }
                if (lane == 0) s_tot[s * NAG + ag] = nsq[j][ag];
#pragma unroll
                for (int t = 0; t < BPL; t++) left[j][ag][t] = numeric ? left[j][ag][t] + excl : val[t];
            }
            double S[NK];
            decode_vals(nsq[j], sc, A.loss, NK, S);
            double gain_p = 0.0;
            for (int k = 0; k < K; k++) gain_p += node_gain_k(A.loss, S[k], S[K + k], S[2 * K], A.lambda, A.L2);
            const double w_p = S[NK - 1];
#pragma unroll
            for (int t = 0; t < BPL; t++) {
                const int b = lane * BPL + t;
                long long q[NAG];
#pragma unroll
                for (int ag = 0; ag < NAG; ag++) q[ag] = left[j][ag][t];
                double SL[NK];
                decode_vals(q, sc, A.loss, NK, SL);
                const double w_l = SL[NK - 1], w_r = w_p - w_l;
                bool ok = b < B && b + 1 <= bmax && w_l > L.min_weight && w_r > L.min_weight;
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
                if (b < B) s_gain[s * B + b] = gain; // update_gains!
            }
        }
    }
    __syncthreads();
    if (wave == 0) { // the feature's row of the level matrix and its first maximum
        double bg = -INFINITY;
        int bi = NO_BIN;
        for (int b = lane; b < B; b += 64) {
            double acc = 0.0;
            bool allpos = true;
#pragma unroll 8
            for (int s = 0; s < nodes; s++) {
                const double g = s_gain[s * B + b];
                acc += g;
                if (A.level > 1) allpos = allpos && g > 0.0;
            }
            const double v = allpos ? acc : 0.0;
            if (v > bg) {
                bg = v;
                bi = b;
            }
        }
        wave_argmax(bg, bi);
        if (lane == 0) {
            s_bin = bi;
            s_best = bg;
        }
    }
    __syncthreads();
    const int bi = s_bin;
    if (bi != NO_BIN) { // the totals left of it, from the lane that holds the bin
#pragma unroll
        for (int j = 0; j < NPW; j++) {
            const int s = wave + j * nwaves;
            if (s < nodes && lane == bi / BPL) {
#pragma unroll
                for (int ag = 0; ag < NAG; ag++) {
                    long long v = left[j][ag][0];
#pragma unroll
                    for (int t = 1; t < BPL; t++) v = bi % BPL == t ? left[j][ag][t] : v;
                    __hip_atomic_store(L.lefts + ((size_t)jp * nodes + s) * NAG + ag, (unsigned long long)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
    }
    if (tid == 0) {
        unsigned long long *mine = reinterpret_cast<unsigned long long *>(A.best + jp);
        __hip_atomic_store(mine, (unsigned long long)__double_as_longlong(s_best), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(mine + 1, (unsigned long long)(unsigned int)bi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // every wavefront's part of the candidate is in memory before it is counted
    __syncthreads();
    if (tid == 0) s_last = __hip_atomic_fetch_add(L.counts, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1;
    if (A.zero_children && wave > 0) { // meanwhile, whatever the decision: the slices of a leaf are never read
        for (int s = wave - 1; s < nodes; s += nwaves - 1) {
            long long *hc = A.hist + (int64_t)(2 * (first + s) - 1) * A.node_stride + o0;
            for (int i = lane; i < NAG * B; i += 64) {
                hc[i] = 0;
                hc[A.node_stride + i] = 0;
            }
        }
    }
    __syncthreads();
    if (!s_last) return;
    if (wave == 0) {
        double g = -INFINITY;
        int j = NO_BIN, b = 0;
        const unsigned long long *cand = reinterpret_cast<const unsigned long long *>(A.best);
        for (int q = lane; q < (int)gridDim.x; q += 64) { // ascending features: only a strictly larger gain replaces an earlier one
            const double gg = __longlong_as_double((long long)__hip_atomic_load(cand + 2 * q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            const int c = (int)__hip_atomic_load(cand + 2 * q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (gg > g) {
                g = gg;
                j = q;
                b = c;
            }
        }
        const int own = j;
        wave_argmax(g, j); // highest gain, then the earliest feature, whose bin is already the lowest
        if (j != NO_BIN ? own == j : lane == 0) {
            s_best = g;
            s_cell = j != NO_BIN && g > A.gamma ? j : NO_BIN;
            s_bin = b;
            *L.counts = 0;
        }
    }
    __syncthreads();
    const bool found = s_cell != NO_BIN;
    const int bj = found ? s_cell : 0, bb = s_bin + 1;
    if (found && tid < nodes * NAG)
        s_left[tid] = (long long)__hip_atomic_load(L.lefts + (size_t)bj * nodes * NAG + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int feat = (int)A.js[bj];
    const bool num = A.feattypes[feat - 1] != 0;
    __syncthreads();
    // a thread writes a node, or a child
    const int who = tid / nodes, s = tid % nodes, n = first + s;
    double S[EVT_MAX_NK];
    if (who == 0) {
        decode_vals(s_tot + s * NAG, sc, A.loss, NK, S);
        A.tree.w[n - 1] = (float)S[NK - 1];
        A.status[n] = found ? ST_SPLIT : ST_LEAF;
        if (found) {
            A.tree.feat[n - 1] = feat;
            A.tree.cond_bin[n - 1] = (uint8_t)bb;
            A.tree.gain[n - 1] = (float)s_best;
            A.tree.split[n - 1] = 1;
            A.tree.packed[n - 1] = evt_pack_node(feat, bb, num);
        } else {
            for (int k = 0; k < K; k++) A.tree.pred[(int64_t)K * (n - 1) + k] = (float)leaf_value(A.loss, S, k, K, A.eta, A.bagging, A.lambda, A.L2);
        }
    } else if (found && who <= 2) {
        const int cn = 2 * n + who - 1;
        long long qc[NAG];
#pragma unroll
        for (int ag = 0; ag < NAG; ag++) {
            const long long l = s_left[s * NAG + ag];
            qc[ag] = who == 2 ? s_tot[s * NAG + ag] - l : l;
            A.node_sum[(int64_t)cn * NAG + ag] = qc[ag];
        }
        if (L.fold_leaves) { // as the pass over the last level would (write_children)
            decode_vals(qc, sc, A.loss, NK, S);
            A.tree.w[cn - 1] = (float)S[NK - 1];
            for (int k = 0; k < K; k++) A.tree.pred[(int64_t)K * (cn - 1) + k] = (float)leaf_value(A.loss, S, k, K, A.eta, A.bagging, A.lambda, A.L2);
            A.status[cn] = ST_LEAF;
        }
    }
}

// ---- any number of outputs (multi-class log loss) ------------------------------------------------
// Same search as k_scan / k_scan_fin with the channel count a run-time value: the node statistics live in shared
// memory and the candidate gain is the sum of term(left_k) + term(right_k) over the outputs, added in the
// reference's order (split_gain, src/split.jl:108-117), from one prefix scan per channel.
__device__ __forceinline__ void node_totals_mc(const ScanArgs &A, int n, const long long *hn, long long *s_Sq, double *s_S, double *s_sc) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int NAG = A.NAg;
    if (tid < NAG) s_sc[tid] = A.qscale[tid];
    if (A.level == 1) {
        for (int ag = wave; ag < NAG; ag += (blockDim.x >> 6)) {
            long long s = 0;
            for (int b = lane; b < A.B; b += 64) s += hn[(int64_t)ag * A.B + b];
            s = wave_sum_i64(s);
            if (lane == 0) {
                s_Sq[ag] = s;
                A.node_sum[(int64_t)n * NAG + ag] = s;
            }
        }
    } else if (tid < NAG) {
        s_Sq[tid] = A.node_sum[(int64_t)n * NAG + tid];
    }
    __syncthreads();
    if (tid < NAG) s_S[tid] = (double)s_Sq[tid] * s_sc[tid];
    __syncthreads();
}

// one channel's histogram words for this lane's BPL bins, requested (fetch) well before they are summed (left_sums): a node's own, or
// its parent's and its sibling's
template <int BPL>
struct ChannelWords {
    long long a[BPL], b[BPL];
    __device__ __forceinline__ void fetch(const ScanArgs &A, const long long *hn, const long long *hp, const long long *hs, int64_t o, bool is_sub, int lane) {
#pragma unroll
        for (int t = 0; t < BPL; t++) {
            const int bin = lane * BPL + t < A.B ? lane * BPL + t : A.B - 1;
            a[t] = is_sub ? hp[o + bin] : hn[o + bin];
            b[t] = is_sub ? hs[o + bin] : 0;
        }
    }
    // left-side sums (numeric: inclusive prefix; categorical: the bin alone), and the sum of all bins; store: subtract nodes
    // materialise h[n] = h[parent] - h[sibling] on the way
    __device__ __forceinline__ long long left_sums(const ScanArgs &A, long long *hn, int64_t o, bool store, bool numeric, int lane, long long *left) const {
        long long val[BPL];
        long long run = 0;
#pragma unroll
        for (int t = 0; t < BPL; t++) {
            const int bin = lane * BPL + t;
            const long long v = bin < A.B ? a[t] - b[t] : 0;
            if (store && bin < A.B) hn[o + bin] = v;
            val[t] = v;
            run += v;
            left[t] = run;
        }
        const long long incl = wave_incl_scan_i64(run), excl = incl - run;
#pragma unroll
        for (int t = 0; t < BPL; t++) left[t] = numeric ? left[t] + excl : val[t];
        return readlane_i64(incl, 63);
    }
};

// One block per (node, sampled feature), a wavefront per two outputs: a wavefront sums the weight's bins and its outputs' four channels
// and leaves its outputs' terms of every bin's gain in LDS, where the first adds them in the outputs' order.  Bound by that chain - one
// trip for all of a wavefront's channels, two scans' and two divisions' length - where one wavefront per feature went through the
// outputs one pair after the other: 60k rows x 30 features x 64 bins of 7 classes 16.2 -> 10.2 us a level.
// LOOP: a wavefront takes one pair of outputs after the other.
template <int BPL, bool LOOP>
__global__ __launch_bounds__(64 * (EVT_MAX_K / 2)) void k_scan_mc(ScanArgs A) {
    extern __shared__ double s_term[]; // [K][B]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwaves = blockDim.x >> 6;
    touch_kernargs<decltype(k_scan_mc<BPL, LOOP>)>();
    const int nodeidx = blockIdx.x, n = (1 << (A.level - 1)) + nodeidx, jp = blockIdx.y;
    int f = (int)A.js[jp] - 1;
    const int st = A.status[n];
    asm volatile("" : "+v"(f)); // requested ahead of the branch on the node's state
    if (st != ST_BUILD && st != ST_SUBTRACT) return;
    const bool is_sub = (st == ST_SUBTRACT);
    const int B = A.B, K = A.K, NAG = A.NAg;
    long long *hn = A.hist + (int64_t)(n - 1) * A.node_stride;
    const long long *hp = A.hist + (int64_t)((n >> 1) - 1) * A.node_stride;
    const long long *hs = A.hist + (int64_t)((n ^ 1) - 1) * A.node_stride;

    __shared__ long long s_Sq[EVT_MC_MAX_NK];
    __shared__ double s_S[EVT_MC_MAX_NK];
    __shared__ double s_sc[EVT_MC_MAX_NK];
    __shared__ double s_gp[EVT_MAX_K];
    __shared__ int s_last, s_jp, s_bin;

    const int64_t of = (int64_t)jp * NAG * B, ow = of + (int64_t)(NAG - 1) * B; // the feature's slice; its weights
    int k0 = 2 * wave, k1 = k0 + 1 < K ? k0 + 1 : k0;
    ChannelWords<BPL> cw, cg[2], ch[2];
    cw.fetch(A, hn, hp, hs, ow, is_sub, lane);
    auto fetch = [&]() {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            cg[j].fetch(A, hn, hp, hs, of + (int64_t)(j ? k1 : k0) * B, is_sub, lane);
            ch[j].fetch(A, hn, hp, hs, of + (int64_t)(K + (j ? k1 : k0)) * B, is_sub, lane);
        }
    };
    fetch();
    const bool numeric = A.feattypes[f] != 0;
    if (tid < NAG) {
        s_sc[tid] = A.qscale[tid];
        if (A.level > 1) s_Sq[tid] = A.node_sum[(int64_t)n * NAG + tid];
    }
    long long lq[BPL], gq[2][BPL], hq[2][BPL];
    const long long tw = cw.left_sums(A, hn, ow, is_sub && wave == 0, numeric, lane, lq);
    auto sums = [&]() {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int k = j ? k1 : k0;
            const long long tg = cg[j].left_sums(A, hn, of + (int64_t)k * B, is_sub, numeric, lane, gq[j]);
            const long long th = ch[j].left_sums(A, hn, of + (int64_t)(K + k) * B, is_sub, numeric, lane, hq[j]);
            if (!LOOP && A.level == 1 && lane == 0) { // the root's totals are any feature's sums over its bins
                s_Sq[k] = tg;
                s_Sq[K + k] = th;
                s_Sq[2 * K] = tw; // every wavefront the same
            }
        }
    };
    sums();
    __syncthreads();
    if (tid < NAG) {
        s_S[tid] = (double)s_Sq[tid] * s_sc[tid];
        if (A.level == 1 && jp == 0) A.node_sum[(int64_t)n * NAG + tid] = s_Sq[tid];
    }
    const double scw = s_sc[NAG - 1], w_p = (double)s_Sq[NAG - 1] * scw;
    if (tid < K) s_gp[tid] = node_gain_k(A.loss, (double)s_Sq[tid] * s_sc[tid], (double)s_Sq[K + tid] * s_sc[K + tid], w_p, A.lambda, A.L2);
    for (;;) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int k = j ? k1 : k0;
            const double scg = s_sc[k], sch = s_sc[K + k], Sg = (double)s_Sq[k] * scg, Sh = (double)s_Sq[K + k] * sch;
#pragma unroll
            for (int t = 0; t < BPL; t++) {
                const int b = lane * BPL + t;
                const double w_l = (double)lq[t] * scw;
                const double term = split_gain_k(A.loss, Sg, Sh, w_p, (double)gq[j][t] * scg, (double)hq[j][t] * sch, w_l, w_p - w_l, A.lambda, A.L2);
                if (b < B) s_term[k * B + b] = term;
            }
        }
        if (!LOOP) break;
        k0 += 2 * nwaves;
        if (k0 >= K) break;
        k1 = k0 + 1 < K ? k0 + 1 : k0;
        fetch();
        sums();
    }
    __syncthreads();
    if (wave == 0) {
        double gain_p = 0.0, sg[BPL];
#pragma unroll
        for (int t = 0; t < BPL; t++) sg[t] = 0.0;
        for (int k = 0; k < K; k++) {
            gain_p += s_gp[k];
#pragma unroll
            for (int t = 0; t < BPL; t++) sg[t] += s_term[k * B + (lane * BPL + t < B ? lane * BPL + t : B - 1)];
        }
        const int bmax = numeric ? B - 1 : B;
        double lg = -INFINITY;
        int lb = NO_BIN;
#pragma unroll
        for (int t = 0; t < BPL; t++) {
            const int b = lane * BPL + t;
            const double w_l = (double)lq[t] * scw, w_r = w_p - w_l, gain = sg[t] - gain_p;
            const bool ok = b < B && b + 1 <= bmax && w_l > A.min_weight && w_r > A.min_weight;
            if (A.oblivious) {
                if (b < B) A.ogains[((int64_t)nodeidx * A.nfs + jp) * B + b] = ok ? gain : 0.0;
            } else if (ok && gain > lg) {
                lg = gain;
                lb = b + 1;
            }
        }
        if (!A.oblivious) {
            wave_argmax(lg, lb);
            if (lane == 0) {
                const int bj = lb != NO_BIN ? jp : NO_BIN;
                ScanBest *mine = A.sbest + (int64_t)nodeidx * gridDim.y + jp;
                if (!A.last_decides) {
                    mine->gain = lg; mine->jp = bj; mine->bin = lb;
                } else { // the last of the node's blocks decides, as in k_scan
                    unsigned long long *to = reinterpret_cast<unsigned long long *>(mine);
                    __hip_atomic_store(to, (unsigned long long)__double_as_longlong(lg), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(to + 1, (unsigned int)bj | ((unsigned long long)(unsigned int)lb << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the candidate is in memory before it is counted
                    s_last = __hip_atomic_fetch_add(A.counts + (size_t)nodeidx * EVT_SCAN_COUNT_STEP, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                             (int)gridDim.y - 1;
                }
            }
        }
    }
    if (A.oblivious || !A.last_decides) return;
    if (A.zero_children) { // the children's slices start from zero, whatever the node turns out to be
        long long *hc = A.hist + (int64_t)(2 * n - 1) * A.node_stride + of;
        for (int i = tid; i < NAG * B; i += blockDim.x) {
            hc[i] = 0;
            hc[A.node_stride + i] = 0;
        }
    }
    __syncthreads();
    if (!s_last) return;
    if (wave == 0) {
        double g = -INFINITY;
        int j = NO_BIN, b = NO_BIN;
        const unsigned long long *cand = reinterpret_cast<const unsigned long long *>(A.sbest + (int64_t)nodeidx * gridDim.y);
        for (int q = lane; q < (int)gridDim.y; q += 64) { // ascending positions: only a strictly larger gain replaces an earlier one
            const double gg = __longlong_as_double((long long)__hip_atomic_load(cand + 2 * q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            const unsigned long long w = __hip_atomic_load(cand + 2 * q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (gg > g) { g = gg; j = (int)(w & 0xffffffffull); b = (int)(w >> 32); }
        }
        const int own = j;
        wave_argmax(g, j);
        const bool found = j != NO_BIN && g > A.gamma;
        if (found ? own == j : lane == 0) {
            A.counts[(size_t)nodeidx * EVT_SCAN_COUNT_STEP] = 0;
            A.tree.w[n - 1] = (float)w_p;
            s_jp = found ? j : NO_BIN;
            s_bin = b;
            if (found) {
                const int feat = (int)A.js[j];
                A.tree.feat[n - 1] = feat;
                A.tree.cond_bin[n - 1] = (uint8_t)b;
                A.tree.gain[n - 1] = (float)g;
                A.tree.split[n - 1] = 1;
                A.tree.packed[n - 1] = evt_pack_node(feat, b, A.feattypes[feat - 1] != 0);
            }
            A.status[n] = found ? ST_SPLIT : ST_LEAF;
        }
    }
    __syncthreads();
    const int bj = s_jp, bb = s_bin;
    if (bj == NO_BIN) {
        if (tid < K) A.tree.pred[(int64_t)K * (n - 1) + tid] = (float)leaf_value(A.loss, s_S, tid, K, A.eta, A.bagging, A.lambda, A.L2);
        return;
    }
    // the children's totals, five of a wavefront's channels (all of them where it has two outputs) requested at once; a subtract node's own slice was
    // written by other blocks, so it is its parent's less its sibling's here too
    const bool num = A.feattypes[A.js[bj] - 1] != 0;
    for (int ag0 = wave; ag0 < NAG; ag0 += 5 * nwaves) {
        ChannelWords<BPL> cc[5];
#pragma unroll
        for (int j = 0; j < 5; j++) {
            const int ag = ag0 + j * nwaves < NAG ? ag0 + j * nwaves : NAG - 1;
            cc[j].fetch(A, hn, hp, hs, ((int64_t)bj * NAG + ag) * B, is_sub, lane);
        }
#pragma unroll
        for (int j = 0; j < 5; j++) {
            const int ag = ag0 + j * nwaves;
            long long s = 0;
#pragma unroll
            for (int t = 0; t < BPL; t++) {
                const int b = lane * BPL + t;
                if (b < B && (num ? b + 1 <= bb : b + 1 == bb)) s += cc[j].a[t] - cc[j].b[t];
            }
            s = wave_sum_i64(s);
            if (lane == 0 && ag < NAG) {
                A.node_sum[(int64_t)(2 * n) * NAG + ag] = s;
                A.node_sum[(int64_t)(2 * n + 1) * NAG + ag] = s_Sq[ag] - s;
            }
        }
        if (!LOOP) break;
    }
}

__global__ __launch_bounds__(256) void k_scan_fin_mc(ScanArgs A, int ngroups) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = (1 << (A.level - 1)) + blockIdx.x;
    const int B = A.B, NK = A.NK, K = A.K, NAG = A.NAg;
    if (blockIdx.y > 0) { // the blocks beyond a node's first only clear the children's slices, whatever the decision (as in k_scan_fin)
        if (A.status[n] == ST_INACTIVE) return;
        long long *hc = A.hist + (int64_t)(2 * n - 1) * A.node_stride;
        const int64_t used = (int64_t)A.nfs * NAG * B;
        const int64_t zb = gridDim.y - 1, per = (used + zb - 1) / zb;
        const int64_t i0 = (int64_t)(blockIdx.y - 1) * per, i1 = i0 + per < used ? i0 + per : used;
        for (int64_t i = i0 + tid; i < i1; i += 256) {
            hc[i] = 0;
            hc[A.node_stride + i] = 0;
        }
        return;
    }
    if (A.leaf_level) {
        if (n > 1 && A.status[n >> 1] != ST_SPLIT) return;
    } else {
        const int st = A.status[n];
        if (st != ST_BUILD && st != ST_SUBTRACT) return;
    }
    long long *hn = A.hist + (int64_t)(n - 1) * A.node_stride;
    __shared__ long long s_Sq[EVT_MC_MAX_NK];
    __shared__ double s_S[EVT_MC_MAX_NK];
    __shared__ double s_sc[EVT_MC_MAX_NK];
    __shared__ double s_g[256];
    __shared__ int s_j[256], s_b[256];
    __shared__ int s_dec[3];
    node_totals_mc(A, n, hn, s_Sq, s_S, s_sc);
    if (tid == 0) A.tree.w[n - 1] = (float)s_S[NK - 1];
    if (A.leaf_level) {
        if (tid < K) A.tree.pred[(int64_t)K * (n - 1) + tid] = (float)leaf_value(A.loss, s_S, tid, K, A.eta, A.bagging, A.lambda, A.L2);
        if (tid == 0) A.status[n] = ST_LEAF;
        return;
    }
    double bg = -INFINITY;
    int bj = NO_BIN, bb = NO_BIN;
    // a thread takes the groups tid, tid + 256, ... (more than 1024 sampled features): ascending feature positions, so
    // only a strictly larger gain replaces an earlier one
    for (int g = tid; g < ngroups; g += 256) {
        const ScanBest r = A.sbest[(int64_t)blockIdx.x * ngroups + g];
        if (r.gain > bg) { bg = r.gain; bj = r.jp; bb = r.bin; }
    }
    s_g[tid] = bg; s_j[tid] = bj; s_b[tid] = bb;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) {
            if (s_g[tid + o] > s_g[tid] || (s_g[tid + o] == s_g[tid] && s_j[tid + o] < s_j[tid])) {
                s_g[tid] = s_g[tid + o]; s_j[tid] = s_j[tid + o]; s_b[tid] = s_b[tid + o];
            }
        }
        __syncthreads();
    }
    if (tid == 0) {
        bg = s_g[0]; bj = s_j[0]; bb = s_b[0];
        const int found = (bb != NO_BIN && bg > A.gamma) ? 1 : 0;
        s_dec[0] = found; s_dec[1] = bj; s_dec[2] = bb;
        if (found) {
            const int feat = (int)A.js[bj];
            A.tree.feat[n - 1] = feat;
            A.tree.cond_bin[n - 1] = (uint8_t)bb;
            A.tree.gain[n - 1] = (float)bg;
            A.tree.split[n - 1] = 1;
            A.tree.packed[n - 1] = evt_pack_node(feat, bb, A.feattypes[feat - 1] != 0);
            A.status[n] = ST_SPLIT;
        } else {
            A.status[n] = ST_LEAF;
        }
    }
    __syncthreads();
    if (!s_dec[0]) {
        if (tid < K) A.tree.pred[(int64_t)K * (n - 1) + tid] = (float)leaf_value(A.loss, s_S, tid, K, A.eta, A.bagging, A.lambda, A.L2);
        return;
    }
    bj = s_dec[1]; bb = s_dec[2];
    {
        const int f = (int)A.js[bj] - 1;
        const bool numeric = A.feattypes[f] != 0;
        for (int ag = wave; ag < NAG; ag += (blockDim.x >> 6)) {
            const int64_t o = ((int64_t)bj * NAG + ag) * B;
            long long s = 0;
            for (int b = lane; b < B; b += 64) {
                const bool in = numeric ? (b + 1 <= bb) : (b + 1 == bb);
                if (in) s += hn[o + b];
            }
            s = wave_sum_i64(s);
            if (lane == 0) {
                A.node_sum[(int64_t)(2 * n) * NAG + ag] = s;
                A.node_sum[(int64_t)(2 * n + 1) * NAG + ag] = s_Sq[ag] - s;
            }
        }
    }
}

// Blocks per node that clear the children's histogram slices beside the block that decides: about 512 in all, so that neither a level
// of one node nor one of wide slices (16 channels x 100 features: 1.6 MB per node) leaves them to few blocks.
static unsigned zero_blocks_per_node(unsigned nodes) { return nodes >= 512 ? 1u : (512u / nodes < 64u ? 512u / nodes : 64u); }

// An oblivious level in one launch
static bool obliv_one_launch(const evt_ctx *c, int level) {
    return c->tree_type == EVT_TREE_OBLIVIOUS && !c->mc && c->scan_fused && obliv_level_fits(c->NAg, c->B, 1 << (level - 1));
}

// The pass over the last split level also writes its children's leaf values (the fixed channel layouts).
bool scan_folds_leaves(const evt_ctx *c) { return !c->mc && c->D > 1 && (c->tree_type != EVT_TREE_OBLIVIOUS || obliv_one_launch(c, c->D - 1)); }

static int launch_obliv_level(evt_ctx *c, int level, const evt_params *p);

// Whether two wavefronts take a block's pairs of outputs one after the other: blocks of five to seven wavefronts leave a compute unit places for too few of them
// when a level is generations of blocks (rounds of depth 9, 3000 rows x 250 features, us, a wavefront to each pair | two: 10 classes 64 bins 1121 | 1021, 128 1722 |
// 1607, 160 2740 | 2477, 255 3499 | 3204, 13 classes 1457 | 1287, 2166 | 2087, 3224 | 3201, 4483 | 4279; 7 classes, four wavefronts, 753 | 753, 1183 | 1184,
// 1782 | 1883; 16 classes, eight, 160 bins 3596 | 3660; levels of at most 2560 blocks, 13 classes x 160 bins, depth 9, 479 | 488).
static bool scan_mc_loops(const evt_ctx *c, int level) { return level > 1 && c->K > 8 && c->K < 15 && ((int64_t)c->n_js_last << (level - 1)) >= 8192; }

int launch_scan(evt_ctx *c, int level, const evt_params *p, bool leaf_level) {
    if (!leaf_level && obliv_one_launch(c, level)) return launch_obliv_level(c, level, p);
    ScanArgs A;
    A.sbest = reinterpret_cast<ScanBest *>(c->sbest);
    A.hist = c->hist;
    A.node_stride = (int64_t)c->F * c->NAg * c->B;
    A.js = c->js;
    A.feattypes = c->feattypes;
    A.mono = c->mono;
    A.status = c->status;
    A.node_sum = c->node_sum;
    A.qscale = c->qscale;
    A.tree = c->tree;
    A.ogains = c->ogains;
    A.eta = p->eta; A.lambda = p->lambda; A.L2 = p->L2; A.gamma = p->gamma; A.min_weight = p->min_weight;
    A.bagging = p->bagging_size;
    A.nfs = c->n_js_last; A.B = c->B; A.F = c->F; A.K = c->K; A.NK = c->NK; A.NAg = c->NAg; A.loss = c->loss;
    A.level = level;
    A.leaf_level = leaf_level ? 1 : 0;
    A.oblivious = (c->tree_type == EVT_TREE_OBLIVIOUS) ? 1 : 0;
    A.zero_children = (level + 1 < c->D) ? 1 : 0; // children at the last level never get a histogram
    A.fold_leaves = (!leaf_level && scan_folds_leaves(c) && level + 1 == c->D) ? 1 : 0;
    A.counts = c->scan_count;
    A.last_decides = 0;
    const unsigned nodes = 1u << (level - 1);
    const int ngroups = (A.nfs + 3) / 4; // 4 waves per block, one sampled feature each
    dim3 grid(nodes, (unsigned)ngroups);
    const int bpl = (c->B + 63) / 64;
    // extra blocks per node that only clear the children's histogram slices, while a level has few nodes
    unsigned zero_blocks = 0;
    if (!leaf_level && A.zero_children && !A.oblivious && nodes < 64) zero_blocks = 64 / nodes < 16 ? 64 / nodes : 16;
    A.last_decides = !leaf_level && !A.oblivious && c->scan_fused ? 1 : 0;
    if (c->mc) { // any number of outputs: multi-class, several targets
        if (!leaf_level) { // a block per node and feature; two outputs to a wavefront
            const unsigned pairs = ((unsigned)c->K + 1) / 2;
            const bool loop = scan_mc_loops(c, level);
            const dim3 per_feature(nodes, (unsigned)A.nfs), block(64u * (loop ? 2 : pairs));
            const size_t lds = (size_t)c->K * c->B * sizeof(double);
#define MCCASE(BPL_)                                                                                             \
    if (loop) hipLaunchKernelGGL((k_scan_mc<BPL_, true>), per_feature, block, lds, c->stream, A);                \
    else hipLaunchKernelGGL((k_scan_mc<BPL_, false>), per_feature, block, lds, c->stream, A);
            if (bpl == 1) { MCCASE(1) }
            else if (bpl == 2) { MCCASE(2) }
            else { MCCASE(4) }
#undef MCCASE
        }
        if (leaf_level || (!A.oblivious && !A.last_decides))
            hipLaunchKernelGGL(k_scan_fin_mc, dim3(nodes, !leaf_level && A.zero_children ? 1 + zero_blocks_per_node(nodes) : 1), dim3(256), 0, c->stream, A, A.nfs);
        HIPCHK(hipGetLastError());
        return EVT_OK;
    }
    // few sampled features: one block of 16 waves scans a node's features and finishes the node, no second launch
    const bool fused = !leaf_level && !A.oblivious && A.nfs <= 16 && c->scan_fused;
    if (fused) A.last_decides = 0;
#define SCAN_FIRST A.js, A.status, A.hist, A.node_stride, A.level, A.nfs, A.B
#define SCASE(NAG_)                                                                                     \
    case NAG_:                                                                                          \
        if (fused) {                                                                                    \
            if (bpl == 1) hipLaunchKernelGGL((k_scan<NAG_, 1, true>), dim3(nodes), dim3(1024), 0, c->stream, SCAN_FIRST, A);      \
            else if (bpl == 2) hipLaunchKernelGGL((k_scan<NAG_, 2, true>), dim3(nodes), dim3(1024), 0, c->stream, SCAN_FIRST, A); \
            else hipLaunchKernelGGL((k_scan<NAG_, 4, true>), dim3(nodes), dim3(1024), 0, c->stream, SCAN_FIRST, A);               \
            break;                                                                                      \
        }                                                                                               \
        if (!leaf_level) {                                                                              \
            if (bpl == 1) hipLaunchKernelGGL((k_scan<NAG_, 1, false>), grid, dim3(256), 0, c->stream, SCAN_FIRST, A);      \
            else if (bpl == 2) hipLaunchKernelGGL((k_scan<NAG_, 2, false>), grid, dim3(256), 0, c->stream, SCAN_FIRST, A); \
            else hipLaunchKernelGGL((k_scan<NAG_, 4, false>), grid, dim3(256), 0, c->stream, SCAN_FIRST, A);               \
        }                                                                                               \
        if (leaf_level || (!A.oblivious && !A.last_decides)) hipLaunchKernelGGL(k_scan_fin<NAG_>, dim3(nodes, 1 + zero_blocks), dim3(256), 0, c->stream, A, ngroups); \
        break;
    switch (c->NAg) {
        SCASE(2)
        SCASE(3)
        SCASE(5)
    default: evt_set_error("unsupported global channel count %d", c->NAg); return EVT_ERR_ARG;
    }
#undef SCASE
#undef SCAN_FIRST
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

static void fill_obliv_args(evt_ctx *c, int level, const evt_params *p, OblivArgs &A) {
    const LevelTab &L = c->lvl[level & 1];
    A.hist = c->hist;
    A.node_stride = (int64_t)c->F * c->NAg * c->B;
    A.js = c->js;
    A.feattypes = c->feattypes;
    A.status = c->status;
    A.node_sum = c->node_sum;
    A.qscale = c->qscale;
    A.tree = c->tree;
    A.ogains = c->ogains;
    A.hdr = L.hdr;
    A.act_node = L.act_node;
    A.eta = p->eta; A.lambda = p->lambda; A.L2 = p->L2; A.gamma = p->gamma;
    A.bagging = p->bagging_size;
    A.nfs = c->n_js_last; A.B = c->B; A.K = c->K; A.NK = c->NK; A.NAg = c->NAg; A.loss = c->loss; A.level = level;
    A.zero_children = (level + 1 < c->D) ? 1 : 0;
    A.best = reinterpret_cast<ScanBest *>(c->sbest);
    A.nbest = (int)std::min<int64_t>(EVT_OBLIV_BLOCKS, ((int64_t)A.nfs * A.B + 255) / 256);
}

static int launch_obliv_level(evt_ctx *c, int level, const evt_params *p) {
    OblivLevelArgs A;
    fill_obliv_args(c, level, p, A.o);
    A.mono = c->mono;
    A.counts = c->scan_count;
    A.min_weight = p->min_weight;
    A.fold_leaves = level + 1 == c->D ? 1 : 0;
    A.lefts = reinterpret_cast<unsigned long long *>(c->ogains); // nodes x features x bins words, unused in this form
    const int nodes = 1 << (level - 1);
    const dim3 grid((unsigned)A.o.nfs), block(64u * std::min(16, std::max(4, nodes)));
    const size_t lds = (size_t)nodes * c->B * sizeof(double);
#define OLCASE(NAG_, BPL_, NPW_)                                                                                     \
    if (c->NAg == NAG_ && obliv_lane_bins(c->B) == BPL_ && obliv_wave_nodes(nodes) == NPW_) {                        \
        hipLaunchKernelGGL((k_obliv_level<NAG_, BPL_, NPW_>), grid, block, lds, c->stream, A);                       \
        HIPCHK(hipGetLastError());                                                                                   \
        return EVT_OK;                                                                                               \
    }
    EVT_OBLIV_LEVELS(OLCASE)
#undef OLCASE
    evt_set_error("internal: no kernel for an oblivious level of %d nodes, %d channels, %d bins", nodes, c->NAg, c->B);
    return EVT_ERR_ARG;
}

int launch_obliv_select(evt_ctx *c, int level, const evt_params *p) {
    if (obliv_one_launch(c, level)) return EVT_OK; // decided by launch_obliv_level
    OblivArgs A;
    fill_obliv_args(c, level, p, A);
    hipLaunchKernelGGL(k_obliv_max, dim3((unsigned)A.nbest), dim3(256), 0, c->stream, A);
    const unsigned nodes = 1u << (level - 1);
    hipLaunchKernelGGL(k_obliv_apply, dim3(nodes, A.zero_children ? 1 + zero_blocks_per_node(nodes) : 1), dim3(256), 0, c->stream, A);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}
