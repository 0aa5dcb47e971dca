// Trees of few rows and features: the whole tree in one launch.
//
// A level of such a tree is a launch and four trips to memory in a handful of blocks (kernels_small.hip), ten microseconds for work of one.  Here a block follows
// ONE path from the root to a node of the last level that splits - 2^(D-2) blocks for a tree of depth D - and takes every decision on it by itself: it adds the
// rows of the path's node into LDS histograms of all sampled features, searches them, and goes on with the rows of the child its number names.  Blocks whose
// paths share a node repeat its work on compute units that would have nothing to do otherwise, so no block waits for another and none need be resident
// together; all of them add the same integers and so decide alike.  The first block under a node is the node's owner: it writes the node's part of the tree, its
// histogram, and, of a leaf, its rows.
// What a block uses of other blocks' rows (bins, gradients, mask) nobody writes in this launch: the next gradients go to a second array, their maxima to a third set.
// Predictions alone are read and written in one array: a block requests those of all rows, and by then a block that has finished may have added its leaves' values
// to its own.  It uses only those of the rows it finishes itself, which no other block writes (each row ends in one leaf, and a leaf's rows are its owner's).
// The sums are the same integers and the gains the same expressions as in the other kernels: same trees, bit for bit.
#include "grad_math.h"
#include "pool.h"
#include "split_math.h"
#include <algorithm>

#define PATH_MAX_ROWS 32767 // a row and its mark are 16 bits of a list
#define PATH_MAX_FEATS 64
#define PATH_OUT 0x8000u    // the row is not in the sample
#define PATH_NUMERIC (1u << 16)
#define PATH_LDS (148 * 1024)

struct PathArgs {
    const uint8_t *xcm;
    const float *raw; // the gradients the tree is grown on
    unsigned long long *gq;
    uint8_t *mask;
    long long *hist;
    int64_t node_stride;
    uint32_t *js;
    const uint32_t *js_src;
    uint32_t *map_dst;
    const uint32_t *map_src;
    int map_words;
    int32_t *status;
    long long *node_sum;
    double *qscale;
    // fresh gradients: of their maxima are made the tables and the words that other kernels would read
    int fresh;
    const uint32_t *absmax;
    uint32_t *absmax_next;
    const int32_t *qbits;
    int32_t *qexp;
    TreeDev tree;
    unsigned long long *host;  // the tree's nodes in pinned memory (PathNode)
    unsigned long long *flags; // ... and a word per block, which becomes seq when the block's nodes are there
    unsigned long long seq;
    uint32_t *nidx;
    // where the next round's gradients are computed (grad_loss >= 0, as k_grads): another array than raw
    float *pred;
    const float *y;
    float *grad;
    uint32_t *maxima;
    double eta, lambda, L2, gamma, min_weight;
    unsigned long long seed;
    int N, F, B, K, NAg, loss, grad_loss, D, nnodes, nfs, bagging;
    int sampled, draw, cond;
    uint32_t feat[PATH_MAX_FEATS]; // as SmallArgs::feat, the last again behind them
};

struct PathCand { // a wavefront's best split of a node
    double gain;
    int order; // of equal gains the lowest wins: the feature's place in the sample << 8 | bin
    int pad;
    long long left[EVT_MAX_NA];
};

// Nodes of the tree, one to each of a wavefront's first lanes (n: its number, 0 none), to the device's arrays and to the host.  A node's three words go out by three
// lanes in one instruction: each store on its own is a write of part of a line over the bus (1000 rows x 10, depth 10: a round 85 us, with them together 45).
template <int K>
__device__ __forceinline__ void path_put_nodes(const PathArgs &A, int lane, int n, int rows, float w, uint32_t packed, float gain, const float *pred) {
    const uint32_t feat = packed & 0xFFFFu, bin = (packed >> 16) & 0xFFu, split = packed ? 1u : 0u;
    if (n) {
        A.tree.w[n - 1] = w;
        A.tree.feat[n - 1] = (int32_t)feat;
        A.tree.cond_bin[n - 1] = (uint8_t)bin;
        A.tree.gain[n - 1] = gain;
        A.tree.split[n - 1] = (uint8_t)split;
        A.tree.packed[n - 1] = packed;
#pragma unroll
        for (int k = 0; k < K; k++) A.tree.pred[(int64_t)K * (n - 1) + k] = pred[k];
    }
    const uint32_t lo[3] = {feat | bin << 16 | split << 24, __float_as_uint(w), __float_as_uint(pred[0])};
    const uint32_t hi[3] = {(uint32_t)rows, __float_as_uint(gain), K > 1 ? __float_as_uint(pred[K - 1]) : 0u};
    const int from = lane / 3, word = lane - 3 * from, m = __shfl(n, from);
    uint32_t l = 0, h = 0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const uint32_t vl = (uint32_t)__shfl((int)lo[i], from), vh = (uint32_t)__shfl((int)hi[i], from);
        l = word == i ? vl : l;
        h = word == i ? vh : h;
    }
    if (m) __hip_atomic_store(A.host + (size_t)3 * (m - 1) + word, ((unsigned long long)h << 32) | l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <int K>
__device__ __forceinline__ void path_grads(int loss, float *pr, float y, float w, const float *leaf, float *out) {
#define PATH_GRAD(L_)                       \
    case L_:                                \
        evt_add_leaf(pr, leaf, K, L_);      \
        grad_row<L_>(pr, y, w, out);        \
        break
    if constexpr (K == 2) {
        switch (loss) {
            PATH_GRAD(2);
            PATH_GRAD(7);
        }
    } else {
        switch (loss) {
            PATH_GRAD(0);
            PATH_GRAD(1);
            PATH_GRAD(3);
            PATH_GRAD(4);
            PATH_GRAD(5);
            PATH_GRAD(8);
            PATH_GRAD(9);
        }
    }
#undef PATH_GRAD
}

// What bounds it: chains, not bytes.  Everything of a row that the levels need - the sampled features' bins side by side, its words - is brought to LDS once, so that a
// level is two barriers and what lies between: list, record and words out of LDS and into the histograms, the sums and gains of a wavefront, two maxima.
template <int NAG, int BPL, bool PACK>
__global__ __launch_bounds__(1024) void k_small_path(PathArgs A) {
    extern __shared__ __align__(16) unsigned long long s_dyn[]; // [2][feature][channel][bin] histograms of two levels, then the rows
    constexpr int NA = NAG - (PACK ? 1 : 0), K = NAG == 5 ? 2 : 1, NK = 2 * K + 1;
    constexpr int WIDE = PACK ? NA - 1 : NA; // channels of 64 bits a row; with PACK the first takes 32
    __shared__ double s_qs[NAG], s_qmul[NK];
    __shared__ PathCand s_cand[16];
    __shared__ long long s_root[NAG];     // totals of the root
    __shared__ double s_S[NK], s_gain_p;  // statistics and gain of the path's node, below the root
    __shared__ int s_len[2], s_in[2];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    touch_kernargs<decltype(k_small_path<NAG, BPL, PACK>)>();
    const int b = blockIdx.x, B = A.B, N = A.N, nfs = A.nfs, splits = A.D - 1, words = nfs * NA * B, pieces = (nfs + 15) >> 4;
    // [row][piece] of 16 bytes.  A record starts with another feature of the sample from row to row (byte t: feature (row + t) % nfs), so that lanes that add the
    // same byte of their rows add to different features: lanes that add to one bin wait for each other, and of one feature's 64 bins 64 lanes share many (4000 rows x
    // 10 features, depth 6, a round 52.8 -> 48.2 us).
    uint4 *const s_rec = reinterpret_cast<uint4 *>(s_dyn + ((2 * words + 1) & ~1));
    unsigned long long *const s_wide = reinterpret_cast<unsigned long long *>(s_rec + (size_t)N * pieces); // [channel][row]
    int32_t *const s_narrow = reinterpret_cast<int32_t *>(s_wide + (size_t)WIDE * N);     // [row]
    float *const s_pred = reinterpret_cast<float *>(s_narrow + (PACK ? N : 0));           // [row][output]: predictions; then targets and weights
    float *const s_y = s_pred + (size_t)K * N, *const s_w = s_y + N;
    uint16_t *const s_lists = reinterpret_cast<uint16_t *>(s_w + (PACK ? 0 : N));         // the rows of a level's node and of the one above
    auto record_byte = [&](uint32_t j, uint32_t turn) { // (j - turn) mod nfs, both below it
        const uint32_t d = j - turn;
        return min(d, d + (uint32_t)nfs);
    };
    auto owns = [&](int level) { return (b & ((1 << (splits - level)) - 1)) == 0; };

    // ---- the rows to LDS.  What a thread's first two rows need is requested before the tables are made.
    struct Row {
        uint32_t x[16], m;
        float g[NA], pr[K], y, w;
    };
    auto request = [&](int k, int piece) {
        Row r;
        const int row = k < N ? k : N - 1;
#pragma unroll
        for (int t = 0; t < 16; t++) r.x[t] = A.xcm[(size_t)(A.feat[piece * 16 + t] & 0xFFFFu) * N + row]; // past the last feature: that one again
        if (piece == 0) {
            r.m = A.sampled && !A.draw ? A.mask[row] : 0;
#pragma unroll
            for (int a = 0; a < NA; a++) r.g[a] = A.raw[(size_t)row * NK + (NAG == 2 && a == 1 ? 2 : a)];
            if (A.grad_loss >= 0) { // for the next gradients: a trip to memory less at the end; old or new, of rows that another block finishes, and then not used
#pragma unroll
                for (int k = 0; k < K; k++) r.pr[k] = A.pred[(size_t)K * row + k];
                r.y = A.y[row];
                if (!PACK) r.w = A.raw[(size_t)row * NK + NK - 1];
            }
        }
        return r;
    };
    auto store = [&](const Row &r, int row, int piece) {
        const bool valid = row < N;
        if (valid) {
            uint8_t *rec = reinterpret_cast<uint8_t *>(s_rec + row * pieces);
            const uint32_t turn = (uint32_t)row % (uint32_t)nfs;
#pragma unroll
            for (int t = 0; t < 16; t++) {
                if (piece * 16 + t >= nfs) break;
                rec[record_byte(piece * 16 + t, turn)] = (uint8_t)r.x[t];
            }
        }
        if (piece != 0) return;
        uint32_t m = r.m;
        if (A.draw) {
            unsigned long long z = A.seed + (unsigned long long)((row >> 3) + 1) * 0x9E3779B97F4A7C15ull; // SplitMix64, as mask_flags
            z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
            z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
            z ^= z >> 31;
            m = (uint32_t)(z >> (8 * (row & 7))) & 0xFFu;
            if (b == 0 && valid) A.mask[row] = (uint8_t)m;
        }
        const bool out = A.sampled && m > (uint32_t)A.cond;
        if (!PACK) {
            const int c = __popcll(__ballot(valid && !out));
            if (lane == 0 && c) atomicAdd(&s_in[0], c);
        }
        if (!valid) return;
        s_lists[row] = (uint16_t)(row | (out ? PATH_OUT : 0u));
        if (A.grad_loss >= 0) {
#pragma unroll
            for (int k = 0; k < K; k++) s_pred[K * row + k] = r.pr[k];
            s_y[row] = r.y;
            if (!PACK) s_w[row] = r.w;
        }
        const bool keep = A.fresh && (row >> 6) % (int)gridDim.x == b; // the words that other kernels would read, a share of the rows
#pragma unroll
        for (int a = 0; a < NA; a++) {
            const long long q = __double2ll_rn((double)r.g[a] * s_qmul[quant_row(A.loss, K, a)]);
            if (PACK && a == 0) s_narrow[row] = (int32_t)q;
            else s_wide[(size_t)(a - (PACK ? 1 : 0)) * N + row] = (unsigned long long)q;
            if (keep) {
                if (PACK && a == 0) reinterpret_cast<int32_t *>(A.gq)[row] = (int32_t)q;
                else A.gq[(size_t)a * N + row] = (unsigned long long)q;
            }
        }
    };
    Row r0 = request(tid, 0), r1 = request(tid + 1024, 0);
    if (tid < NK) {
        if (A.fresh) {
            const int e = quant_exponent(A.absmax, tid), qb = A.qbits[tid];
            const double m = scalbn(1.0, qb - e);
            s_qmul[tid] = m;
            for (int ag = 0; ag < NAG; ag++)
                if (quant_row(A.loss, K, ag) == tid) {
                    const double sc = PACK && ag == NAG - 1 ? 1.0 : scalbn(1.0, e - qb);
                    s_qs[ag] = sc;
                    if (b == 0) A.qscale[ag] = sc;
                }
            if (b == 0) {
                A.qexp[tid] = e;
                A.qscale[EVT_MC_MAX_NK + tid] = m;
                // the set that the next pass raises but one starts from zero; the one raised here keeps the weights' maximum
                for (int st = 0; st < EVT_ABSMAX_STRIPES; st++) {
                    if (tid < NK - 1) A.absmax_next[st * EVT_MC_MAX_NK + tid] = 0u;
                    else if (A.grad_loss >= 0) A.maxima[st * EVT_MC_MAX_NK + tid] = A.absmax[st * EVT_MC_MAX_NK + tid];
                }
            }
        } else {
            s_qmul[tid] = A.qscale[EVT_MC_MAX_NK + tid];
        }
    }
    if (!A.fresh && tid < NAG) s_qs[tid] = A.qscale[tid];
    if (tid < 2) s_len[tid] = s_in[tid] = 0;
    for (int i = tid; i < words; i += 1024) s_dyn[i] = 0ull;
    if (b == 0) { // a new tree
        if (A.js_src != A.js)
            for (int i = tid; i < nfs; i += 1024) A.js[i] = A.js_src[i];
        for (int i = tid; i < A.map_words; i += 1024) A.map_dst[i] = A.map_src[i];
        if (tid == 0) A.status[0] = A.status[A.nnodes + 1] = ST_INACTIVE;
    }
    __syncthreads();
    for (int k = tid;;) {
        store(r0, k, 0);
        if (k - tid + 1024 < N) store(r1, k + 1024, 0);
        k += 2048;
        if (k - tid >= N) break;
        r0 = request(k, 0);
        r1 = request(k + 1024, 0);
    }
    for (int p = 1; p < pieces; p++)
        for (int k = tid; k < N; k += 2048) {
            r0 = request(k, p);
            r1 = request(k + 1024, p);
            store(r0, k, p);
            store(r1, k + 1024, p);
        }
    __syncthreads();

    // ---- down the path
    long long qn[NAG], ql[NAG]; // totals of the node, of the left child
    int level = 1, n = N;
    bool found = false, right = false, less = false;
    int buf = 0; // the histograms' half of LDS
    uint32_t fw = 0, bin = 0;
    int jw = 0;
    for (;; level++) {
        // the rows of the level above that come here: into the node's list and, of the sample, its histograms
        const int cur = (level - 1) & 1, nxt = level & 1;
        const uint16_t *src = s_lists + (level == 1 ? 0 : nxt) * N;
        uint16_t *dst = s_lists + cur * N;
        unsigned long long *H = s_dyn + buf * words;
        for (int k0 = wave * 64; k0 < n; k0 += 1024) {
            const int k = k0 + lane;
            const uint32_t e = src[k < n ? k : n - 1], row = e & ~PATH_OUT;
            uint4 rec = s_rec[row * pieces];
            const uint32_t turn = row % (uint32_t)nfs;
            unsigned long long g[NA];
#pragma unroll
            for (int a = 0; a < NA; a++) {
                if (PACK && a == 0) g[0] = ((unsigned long long)(long long)s_narrow[row] << EVT_PACK_CNT_BITS) + 1ull;
                else g[a] = s_wide[(size_t)(a - (PACK ? 1 : 0)) * N + row];
            }
            bool goes = k < n;
            if (level > 1) {
                const uint32_t x = reinterpret_cast<const uint8_t *>(s_rec + row * pieces)[record_byte(jw, turn)];
                goes = goes && ((fw & PATH_NUMERIC) ? x <= bin : x == bin) != right;
                const unsigned long long m = __ballot(goes);
                int base = 0;
                if (lane == 0) base = atomicAdd(&s_len[cur], __popcll(m));
                base = __builtin_amdgcn_readfirstlane(base);
                if (goes) dst[base + __popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)e;
                if (!PACK) {
                    const int c = __popcll(__ballot(goes && !(e & PATH_OUT)));
                    if (lane == 0 && c) atomicAdd(&s_in[cur], c);
                }
            }
            if (less ? k >= n || goes : !goes) continue;
            if (e & PATH_OUT) continue;
            if (less)
#pragma unroll
                for (int a = 0; a < NA; a++) g[a] = 0ull - g[a];
            uint32_t at = turn * (uint32_t)(NA * B); // the feature's histogram
            for (int p = 0;;) {
                const uint32_t v[4] = {rec.x, rec.y, rec.z, rec.w};
#pragma unroll
                for (int t = 0; t < 16; t++) {
                    if (p * 16 + t >= nfs) break;
                    unsigned long long *h = H + (at + ((v[t >> 2] >> (8 * (t & 3))) & 0xFFu) - 1u);
#pragma unroll
                    for (int a = 0; a < NA; a++) atomicAdd(h + a * B, g[a]);
                    at += NA * B;
                    at = min(at, at - (uint32_t)words); // past the last feature: the first
                }
                if (++p >= pieces) break;
                rec = s_rec[row * pieces + p];
            }
        }
        __syncthreads();
        const int node = (1 << (level - 1)) + (b >> (splits - level));
        const bool own = owns(level);
        if (level > 1) n = s_len[cur];
        int rows_in = PACK ? 0 : s_in[cur];
        if (tid == 0) s_len[nxt] = s_in[nxt] = 0; // of the level above: read by all
        if (level < splits)
            for (int i = tid; i < words; i += 1024) s_dyn[(buf ^ 1) * words + i] = 0ull;
        // the search: a wavefront per feature, 16 at a time (the expressions of small_scan)
        double lg = -INFINITY;
        int lo = NO_BIN;
        long long lq[NAG];
#pragma unroll
        for (int a = 0; a < NAG; a++) lq[a] = 0;
        for (int j = wave; j < nfs; j += 16) {
            const uint32_t fj = A.feat[j];
            const bool numeric = (fj & PATH_NUMERIC) != 0;
            const int constraint = (int)(fj >> 17) - 1, bmax = numeric ? B - 1 : B;
            const unsigned long long *Hj = H + j * NA * B;
            long long *keep = A.hist + (int64_t)(node - 1) * A.node_stride + (int64_t)j * NAG * B;
            long long left[NAG][BPL], total[NAG];
#pragma unroll
            for (int a = 0; a < NA; a++) { // a word that holds the count too is added up as it is: its low bits are the rows', at most PATH_MAX_ROWS
                long long val[BPL], run = 0, at[BPL];
#pragma unroll
                for (int t = 0; t < BPL; t++) {
                    const int i = lane * BPL + t;
                    val[t] = i < B ? (long long)Hj[a * B + i] : 0;
                    run += val[t];
                    at[t] = run;
                }
                const long long incl = wave_incl_scan_i64(run), excl = incl - run, all = level == 1 ? readlane_i64(incl, 63) : 0;
#pragma unroll
                for (int t = 0; t < BPL; t++) at[t] = numeric ? at[t] + excl : val[t];
                const bool both = PACK && a == 0;
                total[a] = both ? all >> EVT_PACK_CNT_BITS : all;
                if (both) total[NAG - 1] = all & ((1ll << EVT_PACK_CNT_BITS) - 1);
#pragma unroll
                for (int t = 0; t < BPL; t++) {
                    left[a][t] = both ? at[t] >> EVT_PACK_CNT_BITS : at[t];
                    if (both) left[NAG - 1][t] = at[t] & ((1ll << EVT_PACK_CNT_BITS) - 1);
                    const int i = lane * BPL + t;
                    if (own && i < B) {
                        keep[a * B + i] = both ? val[t] >> EVT_PACK_CNT_BITS : val[t];
                        if (both) keep[(NAG - 1) * B + i] = val[t] & ((1ll << EVT_PACK_CNT_BITS) - 1);
                    }
                }
            }
            double S[NK], gain_p = 0.0;
            if (level == 1) {
                if (j == 0 && lane == 0)
#pragma unroll
                    for (int a = 0; a < NAG; a++) s_root[a] = total[a];
                decode_vals(total, s_qs, A.loss, NK, S);
                for (int k = 0; k < K; k++) gain_p += node_gain_k(A.loss, S[k], S[K + k], S[2 * K], A.lambda, A.L2);
            } else {
#pragma unroll
                for (int k = 0; k < NK; k++) S[k] = s_S[k];
                gain_p = s_gain_p;
            }
            const double w_p = S[NK - 1];
#pragma unroll
            for (int t = 0; t < BPL; t++) {
                const int i = lane * BPL + t;
                long long q[NAG];
                double SL[NK];
#pragma unroll
                for (int a = 0; a < NAG; a++) q[a] = left[a][t];
                decode_vals(q, s_qs, A.loss, NK, SL);
                const double w_l = SL[NK - 1], w_r = w_p - w_l;
                bool ok = i < B && i + 1 <= bmax && w_l > A.min_weight && w_r > A.min_weight;
                if (ok && constraint != 0) {
                    double SR[NK];
                    for (int k = 0; k < NK; k++) SR[k] = S[k] - SL[k];
                    const double predL = leaf_value(A.loss, SL, 0, K, A.eta, A.bagging, A.lambda, A.L2);
                    const double predR = leaf_value(A.loss, SR, 0, K, A.eta, A.bagging, A.lambda, A.L2);
                    ok = (constraint == -1 && predL > predR) || (constraint == 1 && predL < predR);
                }
                if (ok) {
                    double gain = 0.0;
                    for (int k = 0; k < K; k++) gain += split_gain_k(A.loss, S[k], S[K + k], w_p, SL[k], SL[K + k], w_l, w_r, A.lambda, A.L2);
                    gain -= gain_p;
                    if (gain > lg) {
                        lg = gain;
                        lo = j << 8 | (i + 1);
#pragma unroll
                        for (int a = 0; a < NAG; a++) lq[a] = q[a];
                    }
                }
            }
        }
        double bg = lg;
        int order = lo;
        wave_argmax(bg, order);
        if (order == NO_BIN ? lane == 0 : lo == order) { // an order names one lane
            s_cand[wave].gain = order == NO_BIN ? -INFINITY : bg;
            s_cand[wave].order = order;
#pragma unroll
            for (int a = 0; a < NAG; a++) s_cand[wave].left[a] = lq[a];
        }
        __syncthreads();
        bg = s_cand[lane & 15].gain;
        order = s_cand[lane & 15].order;
        wave_argmax<true>(bg, order);
        found = order != NO_BIN && bg > A.gamma;
        jw = found ? order >> 8 : 0;
        fw = A.feat[jw];
        bin = (uint32_t)order & 0xFFu;
        right = level < splits && ((b >> (splits - 1 - level)) & 1);
#pragma unroll
        for (int a = 0; a < NAG; a++) {
            if (level == 1) qn[a] = s_root[a];
            ql[a] = s_cand[jw & 15].left[a];
        }
        if (PACK) rows_in = (int)qn[NAG - 1];
        if (own && wave == 15) { // the node and, of the last level that splits, its children: a lane each
            const bool leaves = found && level == splits;
            const int m = lane == 0 ? node : leaves && lane < 3 ? 2 * node + lane - 1 : 0;
            const bool split = found && lane == 0;
            long long q[NAG];
            double S[NK];
            float v[K];
#pragma unroll
            for (int a = 0; a < NAG; a++) {
                q[a] = lane == 0 ? qn[a] : lane == 1 ? ql[a] : qn[a] - ql[a];
                if (m) A.node_sum[(int64_t)m * NAG + a] = q[a];
            }
            decode_vals(q, s_qs, A.loss, NK, S);
#pragma unroll
            for (int k = 0; k < K; k++) v[k] = split ? 0.0f : (float)leaf_value(A.loss, S, k, K, A.eta, A.bagging, A.lambda, A.L2);
            path_put_nodes<K>(A, lane, m, lane == 0 ? rows_in : 0, (float)S[2 * K], split ? evt_pack_node((int)(fw & 0xFFFFu) + 1, (int)bin, (fw & PATH_NUMERIC) != 0) : 0u,
                              split ? (float)bg : 0.0f, v);
            if (m) A.status[m] = split ? ST_SPLIT : ST_LEAF;
        }
        if (!found || level == splits) break;
        const long long all_w = qn[NAG - 1];
#pragma unroll
        for (int a = 0; a < NAG; a++) qn[a] = right ? qn[a] - ql[a] : ql[a];
        // the child's histograms: its rows', or its parent's less the rows that do not come along, whichever are fewer (or weigh less)
        less = qn[NAG - 1] > all_w - qn[NAG - 1];
        if (!less) buf ^= 1;
        if (wave == 14) { // once for the next level's wavefronts
            double S[NK], gain_p = 0.0;
            decode_vals(qn, s_qs, A.loss, NK, S);
            for (int k = 0; k < K; k++) gain_p += node_gain_k(A.loss, S[k], S[K + k], S[2 * K], A.lambda, A.L2);
            if (lane == 0) {
#pragma unroll
                for (int k = 0; k < NK; k++) s_S[k] = S[k];
                s_gain_p = gain_p;
            }
        }
    }

    const int node = (1 << (level - 1)) + (b >> (splits - level));
    if (wave < 15) { // ---- the rows of the path's last node, in its leaf or in the two below it
        if (!found && !owns(level)) return;
        float mx[2 * K], lv[2][K];
#pragma unroll
        for (int k = 0; k < 2 * K; k++) mx[k] = 0.0f;
        const uint16_t *list = s_lists + ((level - 1) & 1) * N;
        if (wave * 64 >= n) return;
#pragma unroll
        for (int side = 0; side < 2; side++) {
            long long q[NAG];
            double S[NK];
#pragma unroll
            for (int a = 0; a < NAG; a++) q[a] = !found ? qn[a] : side ? qn[a] - ql[a] : ql[a];
            decode_vals(q, s_qs, A.loss, NK, S);
#pragma unroll
            for (int k = 0; k < K; k++) lv[side][k] = (float)leaf_value(A.loss, S, k, K, A.eta, A.bagging, A.lambda, A.L2);
        }
        for (int k0 = tid; k0 < n; k0 += 960) {
            const int row = (int)(list[k0] & ~PATH_OUT);
            const uint32_t x = reinterpret_cast<const uint8_t *>(s_rec + row * pieces)[record_byte(jw, (uint32_t)row % (uint32_t)nfs)];
            const bool second = found && !((fw & PATH_NUMERIC) ? x <= bin : x == bin);
            A.nidx[row] = (uint32_t)(found ? 2 * node + (second ? 1 : 0) : node);
            if (A.grad_loss >= 0) {
                float l[K], pr[K], out[2 * K];
                const float w = PACK ? 1.0f : s_w[row];
#pragma unroll
                for (int k = 0; k < K; k++) {
                    l[k] = second ? lv[1][k] : lv[0][k];
                    pr[k] = s_pred[K * row + k];
                }
                path_grads<K>(A.grad_loss, pr, s_y[row], w, l, out);
#pragma unroll
                for (int k = 0; k < K; k++) A.pred[(size_t)K * row + k] = pr[k];
#pragma unroll
                for (int k = 0; k < 2 * K; k++) {
                    A.grad[(size_t)NK * row + k] = out[k];
                    mx[k] = fmaxf(mx[k], fabsf(out[k]));
                }
                A.grad[(size_t)NK * row + NK - 1] = w;
            }
        }
        if (A.grad_loss >= 0) {
#pragma unroll
            for (int k = 0; k < 2 * K; k++) {
                const float m = wave_max_f32(mx[k]);
                if (lane == 0 && m > 0.0f) atomicMax(A.maxima + (b % EVT_ABSMAX_STRIPES) * EVT_MC_MAX_NK + k, __float_as_uint(m));
            }
        }
        return;
    }
    // ---- meanwhile one wavefront, which has written the nodes: those of this block that the tree does not reach
    {
        const int l = level + 1 + lane;
        const bool leaves = !(found && level == splits); // lanes behind the levels': the two leaves below the path's end
        const int m = l <= splits ? (owns(l) ? (1 << (l - 1)) + (b >> (splits - l)) : 0) : leaves && l <= A.D + 1 ? (1 << splits) + 2 * b + (l - A.D) : 0;
        const float none[K] = {};
        path_put_nodes<K>(A, lane, m, 0, 0.0f, 0u, 0.0f, none);
        if (m) A.status[m] = ST_INACTIVE;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the block's nodes have arrived
    if (lane == 0) __hip_atomic_store(A.flags + b, A.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// of a block: histograms of two levels, then per row its record, words and place in two lists
static size_t path_lds(const evt_ctx *c, int nfs) {
    const size_t words = (size_t)nfs * c->NA * c->B, row = (size_t)((nfs + 15) / 16) * 16 + (size_t)8 * c->NA - (c->unit_w ? 4 : 0) + 4 * c->K + 4 + (c->unit_w ? 0 : 4) + 4;
    return ((2 * words + 1) & ~(size_t)1) * 8 + (size_t)c->N * row;
}

// What the kernel takes at all
static bool path_can(const evt_ctx *c, int nfs) {
    return c->path_off && nfs <= PATH_MAX_FEATS && c->N >= 4 && c->N <= PATH_MAX_ROWS && path_lds(c, nfs) <= PATH_LDS;
}

// Whether a tree takes it.  A level costs a round of the searches for every 16 features, by channels and bins, and every path adds all rows of the root; the kernels of
// one level each (kernels_small.hip) spread the features over blocks and pay a launch and four trips to memory a level.  Both in microseconds a round, fitted to 500
// rounds of an earlier state of the kernel and checked on 1535 shapes that the present one can hold: 30 to 4735 rows (the most, of one feature and two bins), 1 to 64
// features, 2 to 255 bins, depths 2 to 10.  1201 of them take it, whose rounds take 0.61 of the time in the mean; 33 of these take more than 3 % longer, 12 more than
// 10, the worst 1.21 (29 to 43 features of two bins; few rows of 255).  Of the 334 others 38 would gain more than 3 %, the most 37; all together 1.005 of the better form.
// Fitted again to 1035 of them it lost 6 shapes for 33, but 15 of the other 500 took 3 to 37 % longer than by these figures.
// 10 features, 64 bins, depth 6, us a round in one launch | one a level: 500 rows 26 | 44, 2000 34 | 47, 4000 43 | 50;
// 1000 rows, depth 2 16 | 13, 10 43 | 123; 1000 rows of 20 features 38 | 46, of 32 49 | 46.
bool small_path_takes(const evt_ctx *c, int nfs, bool wherever) {
    if (!path_can(c, nfs)) return false;
    if (wherever) return true;
    const double k = 1e-3 * c->N, levels = c->D - 1, weight = (c->NAg - 1) * (c->B <= 64 ? 1 : c->B <= 128 ? 2 : 4);
    double searches = 0.0;
    for (int l = 1; l < c->D; l++) searches += ((int)std::min<int64_t>(1 << (l - 1), c->N) + 15) / 16;
    const double path = 13.5 + levels * (0.2 + (nfs + 15) / 16 * (1.15 + 0.26 * weight) + 0.62 * k + 5.3e-4 * nfs * c->NA * c->B) + 0.21 * k * nfs * c->NA;
    const double other = 8.1 + levels * (4.5 + 0.6 * weight + 0.8 * k) + 2.2 * searches;
    return path < 0.9 * other;
}

int launch_small_path(evt_ctx *c, const evt_params *p, bool draw) {
    PathArgs A;
    memset((void *)&A, 0, sizeof(A));
    A.grad_loss = grads_with_tree(c, p) ? grad_row_loss(c) : -1;
    if (A.grad_loss >= 0 && !c->grad_next) {
        c->grad_next = static_cast<float *>(dev_take(sizeof(float) * (size_t)c->N * c->NK));
        if (!c->grad_next) return EVT_ERR_NOMEM;
    }
    A.xcm = c->xcm;
    A.raw = c->grad;
    A.gq = c->gq;
    A.mask = c->mask;
    A.hist = c->hist;
    A.node_stride = (int64_t)c->F * c->NAg * c->B;
    A.js = c->js;
    A.js_src = c->js;
    if (c->js_staged) { // read from the pinned buffer
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
    A.host = reinterpret_cast<unsigned long long *>(c->h_stage_dev + c->path_off);
    A.flags = A.host + (size_t)3 * c->nnodes;
    A.seq = (unsigned long long)c->tree_seq;
    A.nidx = c->nidx;
    A.pred = c->pred;
    A.y = c->y;
    A.grad = c->grad_next;
    A.maxima = absmax_set(c, c->quant_pending ? c->absmax_spare : c->absmax_cur);
    if (c->quant_pending) {
        A.fresh = 1;
        A.absmax = absmax_set(c, c->absmax_cur);
        A.absmax_next = absmax_set(c, c->absmax_other);
        A.qbits = c->qbits;
        A.qexp = c->qexp;
    }
    A.eta = p->eta; A.lambda = p->lambda; A.L2 = p->L2; A.gamma = p->gamma; A.min_weight = p->min_weight;
    A.bagging = p->bagging_size;
    A.seed = c->mask_seed;
    A.N = (int)c->N; A.F = c->F; A.B = c->B; A.K = c->K; A.NAg = c->NAg; A.loss = c->loss; A.D = c->D; A.nnodes = c->nnodes;
    A.nfs = c->n_js_last;
    A.sampled = c->step.all_rows ? 0 : 1;
    A.draw = draw ? 1 : 0;
    A.cond = c->last_cond;
    for (int j = 0; j < PATH_MAX_FEATS; j++) {
        const int f = (int)c->js_last[std::min(j, A.nfs - 1)] - 1;
        A.feat[j] = (uint32_t)f | (c->h_feattypes[f] ? PATH_NUMERIC : 0u) | ((uint32_t)(c->h_mono[f] + 1) << 17);
    }
    const size_t lds = path_lds(c, A.nfs);
    const unsigned blocks = 1u << (c->D - 2); // at most EVT_PATH_BLOCKS: path_off
    prof_begin(c, EVT_K_PARTITION, 1);
#define PATH3(NAG_, BPL_, PACK_)                                                                                                                                  \
    {                                                                                                                                                             \
        static EvtDevOnce once;                                                                                                                                   \
        if (once.pending(c->device)) {                                                                                                                            \
            HIPCHK(hipFuncSetAttribute(reinterpret_cast<const void *>(k_small_path<NAG_, BPL_, PACK_>), hipFuncAttributeMaxDynamicSharedMemorySize, PATH_LDS));   \
            once.mark(c->device);                                                                                                                                 \
        }                                                                                                                                                         \
        hipLaunchKernelGGL((k_small_path<NAG_, BPL_, PACK_>), dim3(blocks), dim3(1024), lds, c->stream, A);                                                       \
    }
#define PATH2(NAG_, BPL_)                     \
    if (c->unit_w) PATH3(NAG_, BPL_, true)    \
    else PATH3(NAG_, BPL_, false)
#define PATH1(NAG_)                             \
    if (c->B <= 64) { PATH2(NAG_, 1) } \
    else if (c->B <= 128) { PATH2(NAG_, 2) } \
    else { PATH2(NAG_, 4) }
    if (c->NAg == 2) { PATH1(2) }
    else if (c->NAg == 3) { PATH1(3) }
    else { PATH1(5) }
#undef PATH1
#undef PATH2
#undef PATH3
    prof_end(c);
    HIPCHK(hipGetLastError());
    const bool fresh = c->quant_pending, grads = A.grad_loss >= 0;
    if (fresh && grads) { // the set raised here is the next to be read, the one cleared the next spare
        const int raised = c->absmax_spare;
        c->absmax_spare = c->absmax_other;
        c->absmax_other = c->absmax_cur;
        c->absmax_cur = raised;
        c->quant_pending = false;
    } else if (fresh) {
        quant_taken(c);
    }
    if (grads) std::swap(c->grad, c->grad_next);
    c->step.grads_done = grads;
    c->step.blob_sent = true;
    return EVT_OK;
}
