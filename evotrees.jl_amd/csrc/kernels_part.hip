// Row partitioning and level bookkeeping, all device resident.
//
// split_set! (src/fit-utils.jl:93-312) is a stable partition of each split node's row-id segment, whose order is free here (all sums are of integers);
// update_nodes_idx_kernel! (ext/EvoTreesKernelAbstractionsExt/fit-utils.jl:9-31) is the same
// decision written per row.  Here every node owns a contiguous segment [seg_start, seg_start+seg_len)
// of the row-id list; a split rewrites the segment (lefts first) into the other list buffer, so children are again
// contiguous segments.  Segments are cut into chunks that never cross a node boundary.  Two forms:
//  one pass (k_part_move, unit weights): the split search left the children's row counts in the count channel of their
//  totals, so a block decides its chunk, claims places in both children with one atomic addition and moves the rows;
//  two passes (weights, whose totals hold no counts, and histograms built on the way):
//   count   : one block per chunk evaluates x_bin[row, feat] <= cond_bin, keeps the ballots,
//             counts lefts;
//   scatter : one block per chunk moves row ids to their stable destination (ascending ids on both sides where the node's are: in a tree on every row).
// In both, chunks of nodes that became leaves record the node id per row (and add the leaf value to the prediction), and one
// block sets the children's segments, picks which child is built (fewer rows; tie -> left, src/fit.jl:123-129) and writes
// the next level's tables (active nodes, chunk prefix, build list).  It rides in the kernel that moves the rows; two passes
// over thousands of chunks scan the counts in a kernel of its own before the scatter.
// No host round trip is needed between levels.
#include "grad_math.h"
#include <algorithm>
#include <type_traits>

// largest i in [0, n) with pre[i] <= v   (pre ascending, pre[0] <= v): the number of such entries, less one.  Every
// wavefront counts them for itself, 64 entries per step, all loads independent: one trip to memory where a binary
// search makes log2(n) dependent ones - these blocks are short, so their chain of dependent loads is their run time.
__device__ __forceinline__ int find_owner(const int64_t *__restrict__ pre, int n, int64_t v) {
    const int lane = threadIdx.x & 63;
    int cnt = 0;
    for (int k0 = 0; k0 < n; k0 += 64) {
        const int k = k0 + lane;
        const bool hit = (k < n) && (pre[k < n ? k : 0] <= v);
        cnt += __popcll(__ballot(hit));
    }
    return cnt - 1;
}

struct PartArgs {
    const int64_t *hdr;
    const uint4 *cdesc; // per chunk: {node, first position, end of the node's segment, first chunk of the node}
    const int32_t *act_node;
    const int64_t *cprefix;
    const int32_t *status;
    const int64_t *seg_start;
    const int64_t *seg_len;
    const uint32_t *t_packed; // split nodes as one word: feature | cond_bin << 16 | split << 24 | numeric << 25
    const uint8_t *xcm;
    int64_t N;
    const uint32_t *is_cur;
    uint32_t *is_next;
    unsigned long long *flagw;
    int32_t *chunk_nleft;
    const int64_t *chunk_lpre;
    // leaf finalisation
    uint32_t *nidx;
    float *pred;
    const float *t_pred;
    int K, loss, fuse_pred, write_nidx;
    int stream_hint; // the binned matrix does not fit the last-level cache
    int fold;        // scatter: the level's bookkeeping block rides along and the blocks add up chunk counts themselves
    // threshold bit planes (nullptr: none): numeric splits read one bit of plane (feature, cond_bin) per row
    const uint32_t *planes;
    int64_t plane_words;
    int B;
    // scatter pass that also builds the next level's histograms (16-byte records)
    const uint8_t *xrm;
    const unsigned long long *gq;
    int gq_stride;
    const uint16_t *jsmap;
    long long *hist;
    int64_t node_stride;
    int F, nfs, NAg;
    BlobOut blob; // last pass of a tree: its arrays go to the host in blob.blocks extra blocks
    // one-pass form: rows the node's chunks have placed so far, and the nodes' totals, whose last channel counts rows
    unsigned long long *cursor;
    const long long *node_sum;
};

// The word of the decision source that holds row `rid`: its bin byte, or - for a numeric split with bit planes - the
// plane word whose bit (rid & 31) says x_bin[rid, f] <= cond_bin.
template <bool NT>
__device__ __forceinline__ uint32_t load_decision(const uint8_t *__restrict__ col, const uint32_t *__restrict__ plane, uint32_t rid) {
    if (plane) {
        const uint32_t *p = plane + (rid >> 5);
        return NT ? __builtin_nontemporal_load(p) : *p;
    }
    const uint8_t *p = col + rid;
    return (uint32_t)(NT ? __builtin_nontemporal_load(p) : *p);
}
__device__ __forceinline__ bool decide_left(uint32_t v, bool use_plane, uint32_t rid, bool numeric, uint32_t cb) {
    if (use_plane) return (v >> (rid & 31u)) & 1u;
    return numeric ? (v <= cb) : (v == cb);
}

// NT: the streaming hint on the gathered bin bytes (a template parameter: a run-time branch between two otherwise
// identical loads is merged by the compiler, which drops the hint)
template <bool NT>
__global__ __launch_bounds__(256) void k_part_count(PartArgs A) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // the first descriptor is requested together with the level's chunk count (the grid never exceeds the table)
    touch_kernargs<decltype(k_part_count<NT>)>();
    uint4 cd = A.cdesc[blockIdx.x];
    const int64_t n_chunks = A.hdr[LH_N_CHUNKS];
    asm volatile("" : "+v"(cd.x), "+v"(cd.y), "+v"(cd.z), "+v"(cd.w));
    __shared__ int s_cnt[4];
    for (int64_t c = blockIdx.x; c < n_chunks; c += gridDim.x, cd = A.cdesc[c < n_chunks ? c : 0]) {
        // the chunk's descriptor names its node and its positions: the row ids are requested together with the node's
        // state, one trip to memory after the descriptor
        const int n = (int)cd.x;
        const int64_t p0 = cd.y, pend = cd.z;
        constexpr int NI = EVT_CHUNK / 256;
        uint32_t rid[NI], xbv[NI];
#pragma unroll
        for (int it = 0; it < NI; it++) {
            const int64_t p = p0 + it * 256 + tid;
            rid[it] = A.is_cur[p < pend ? p : pend - 1];
        }
        // the node's split word is requested together with its state (and the row ids), not one trip later behind the
        // branch on the state: a node without a split holds 0 there, which is not used
        const int st = A.status[n];
        uint32_t nd = A.t_packed[n - 1];
        asm volatile("" : "+v"(nd));
        if (st != ST_SPLIT) {
            if (tid == 0) A.chunk_nleft[c] = 0;
            continue;
        }
        const int f = (int)(nd & 0xFFFFu) - 1;
        const uint32_t cb = (nd >> 16) & 0xFFu;
        const bool numeric = (nd & EVT_NODE_NUMERIC) != 0;
        const uint8_t *col = A.xcm + (size_t)f * A.N;
        const uint32_t *plane = (A.planes && numeric && cb >= 1u && cb < (uint32_t)A.B) ? A.planes + ((size_t)f * (A.B - 1) + (cb - 1)) * A.plane_words : nullptr;
        int cnt = 0;
        // a binned matrix larger than the last-level cache is gathered with the streaming hint: each byte's line would
        // displace data that is read again (row lists, gradient words) and is rarely hit a second time itself
#pragma unroll
        for (int it = 0; it < NI; it++) xbv[it] = load_decision<NT>(col, plane, rid[it]);
#pragma unroll
        for (int it = 0; it < NI; it++) {
            const int64_t p = p0 + it * 256 + tid;
            const bool flag = (p < pend) && decide_left(xbv[it], plane != nullptr, rid[it], numeric, cb);
            const unsigned long long bal = __ballot(flag);
            if (lane == 0) A.flagw[c * EVT_CHUNK_WORDS + it * 4 + wave] = bal;
            cnt += __popcll(bal);
        }
        if (lane == 0) s_cnt[wave] = cnt;
        __syncthreads();
        if (tid == 0) A.chunk_nleft[c] = s_cnt[0] + s_cnt[1] + s_cnt[2] + s_cnt[3];
        __syncthreads();
    }
}

// ---- single-block scans -----------------------------------------------------------------------
// Exclusive prefix over the threads of the block (up to 1024); returns the prefix, *total gets the sum.
__device__ long long block_excl_scan(long long v, long long *total, long long *s_tmp /* [17] */) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    long long x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int lo = __shfl_up((int)(x & 0xffffffffll), o), hi = __shfl_up((int)(x >> 32), o);
        long long y = ((long long)hi << 32) | (unsigned int)lo;
        if (lane >= o) x += y;
    }
    __syncthreads(); // s_tmp may still be read from a previous call
    if (lane == 63) s_tmp[wave] = x;
    __syncthreads();
    if (tid == 0) {
        long long run = 0;
        const int nw = blockDim.x >> 6;
        for (int w = 0; w < nw; w++) { long long t = s_tmp[w]; s_tmp[w] = run; run += t; }
        s_tmp[16] = run;
    }
    __syncthreads();
    *total = s_tmp[16];
    return s_tmp[wave] + x - v;
}

struct NextArgs {
    const int64_t *hdr;
    const int32_t *act_node;
    const int64_t *cprefix;
    int32_t *status;
    int64_t *seg_start;
    int64_t *seg_len;
    const int32_t *chunk_nleft;
    int64_t *chunk_lpre;
    // next level
    int64_t *n_hdr;
    int32_t *n_act_node;
    int64_t *n_cprefix;
    int32_t *n_bnode;
    int64_t *n_bstart;
    int64_t *n_bprefix;
    int64_t *n_stats; // rows the next level builds (the level's slot of the per-tree counts; the histogram kernel writes the same figure when it runs)
    int64_t seg_cost; // cost units added per build node in the histogram kernel's span space
    uint4 *n_cdesc;
    int n_chunk_sh;   // rows of a chunk of the next level, a power of two (64-bit divisions by a number of it took 1 us of the chain)
    // one-pass form: a child's rows are its count channel, and its cursor starts from zero
    const long long *node_sum;
    int NAg;
    unsigned long long *cursor;
};

// Two exclusive prefixes in one pass (same shape as block_excl_scan); s_tmp holds 34 values.
__device__ void block_excl_scan2(long long va, long long vb, long long *pa, long long *pb, long long *ta, long long *tb, long long *s_tmp) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    long long xa = va, xb = vb;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int al = __shfl_up((int)(xa & 0xffffffffll), o), ah = __shfl_up((int)(xa >> 32), o);
        const int bl = __shfl_up((int)(xb & 0xffffffffll), o), bh = __shfl_up((int)(xb >> 32), o);
        if (lane >= o) {
            xa += ((long long)ah << 32) | (unsigned int)al;
            xb += ((long long)bh << 32) | (unsigned int)bl;
        }
    }
    __syncthreads(); // s_tmp may still be read from a previous call
    if (lane == 63) {
        s_tmp[wave] = xa;
        s_tmp[17 + wave] = xb;
    }
    __syncthreads();
    if (tid < 2) {
        long long *t = s_tmp + 17 * tid;
        long long run = 0;
        const int nw = blockDim.x >> 6;
        for (int w = 0; w < nw; w++) { long long x = t[w]; t[w] = run; run += x; }
        t[16] = run;
    }
    __syncthreads();
    *ta = s_tmp[16];
    *tb = s_tmp[33];
    *pa = s_tmp[wave] + xa - va;
    *pb = s_tmp[17 + wave] + xb - vb;
}

// One block turns the chunk counts of a level into the next level's tables (children's segments, which child is
// built, active nodes, chunk prefix, build list), in two halves: the scan of the chunk counts (A) and the tables (B).  It
// rides along as the last block of the scatter kernel, whose other blocks need nothing from it: they add up the chunk
// counts of their own node themselves - or, with thousands of chunks per level, read the counts scanned by half A in a
// kernel of its own just before, while half B runs beside them.  Loads that do not depend on each other are issued
// together (fixed-trip loops over clamped indices instead of data-dependent ones).
// A: exclusive scan of the chunks' left counts (chunk_lpre[c] = lefts in the chunks before c, chunk_lpre[n_chunks] = all)
__device__ void chunk_scan_block(const NextArgs &A, long long *s_tmp /* [34] */) {
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int64_t n_chunks = A.hdr[LH_N_CHUNKS];
    long long total;
    {
        constexpr int SP = 8;
        const int64_t span = (n_chunks + nthr - 1) >> __builtin_ctz(nthr);
        const int64_t c0 = (int64_t)tid * span, c1 = (c0 + span < n_chunks) ? c0 + span : n_chunks;
        if (span <= SP) {
            int v[SP];
#pragma unroll
            for (int k = 0; k < SP; k++) {
                const int64_t c = c0 + k;
                const int x = A.chunk_nleft[c < c1 ? c : 0];
                v[k] = c < c1 ? x : 0;
            }
            long long s = 0;
#pragma unroll
            for (int k = 0; k < SP; k++) s += v[k];
            long long pre = block_excl_scan(s, &total, s_tmp);
#pragma unroll
            for (int k = 0; k < SP; k++) {
                if (c0 + k < c1) A.chunk_lpre[c0 + k] = pre;
                pre += v[k];
            }
        } else {
            long long s = 0;
            for (int64_t c = c0; c < c1; c++) s += A.chunk_nleft[c];
            long long pre = block_excl_scan(s, &total, s_tmp);
            for (int64_t c = c0; c < c1; c++) { A.chunk_lpre[c] = pre; pre += A.chunk_nleft[c]; }
        }
        if (tid == 0) A.chunk_lpre[n_chunks] = total;
    }
}

// B: children segments + three scans over the active nodes (children count, chunks, build rows) -> the next level's tables
// SCAN: half A as well.  Of up to LEVEL_LPRE chunks its sums stay in LDS, and the nodes are read while they are added up: two trips to memory
// less, 0.3 us of a scatter kernel of 7 (500k rows).
#define LEVEL_LPRE 1024
struct NextNode {
    int n, st;
    int64_t cp0, cp1, len, start;
};
template <bool SCAN>
__device__ void level_tables_block(const NextArgs &A, long long *s_tmp /* [34] */, uint4 *s_child /* [512] */, int *s_lpre /* SCAN: [LEVEL_LPRE + 1] */) {
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int n_act = (int)A.hdr[LH_N_ACT];
    const int64_t n_chunks = SCAN ? A.hdr[LH_N_CHUNKS] : 0;
    const int span = (n_act + nthr - 1) >> __builtin_ctz(nthr); // threads of a block: a power of two
    const int64_t whole = ((int64_t)1 << A.n_chunk_sh) - 1;
    const int i0 = tid * span, i1 = (i0 + span < n_act) ? i0 + span : n_act;
    long long s_pos = 0, s_chunks = 0, s_brows = 0;
    int n1 = 0; // a thread's only node, where no thread has more: what the second half needs of it stays in registers
    int64_t nl1 = 0, nr1 = 0, start1 = 0;
    NextNode first = {0, 0, 0, 0, 0, 0};
    if (i0 < i1) {
        first.n = A.act_node[i0];
        first.cp0 = A.cprefix[i0];
        first.cp1 = A.cprefix[i0 + 1];
    }
    const bool near = SCAN && n_chunks <= LEVEL_LPRE;
    if constexpr (SCAN) {
        if (near) {
            constexpr int SP = LEVEL_LPRE / 256;
            const int sp = ((int)n_chunks + nthr - 1) >> __builtin_ctz(nthr), c0 = tid * sp, c1 = min(c0 + sp, (int)n_chunks);
            int v[SP], sum = 0;
#pragma unroll
            for (int k = 0; k < SP; k++) v[k] = A.chunk_nleft[c0 + k < c1 ? c0 + k : 0];
            if (i0 < i1) {
                first.st = A.status[first.n];
                first.len = A.seg_len[first.n];
                first.start = A.seg_start[first.n];
            }
#pragma unroll
            for (int k = 0; k < SP; k++) sum += v[k] = c0 + k < c1 ? v[k] : 0;
            long long total;
            int pre = (int)block_excl_scan(sum, &total, s_tmp);
#pragma unroll
            for (int k = 0; k < SP; k++) {
                if (c0 + k < c1) s_lpre[c0 + k] = pre;
                pre += v[k];
            }
            if (tid == 0) s_lpre[n_chunks] = (int)total;
        } else {
            chunk_scan_block(A, s_tmp);
        }
        __syncthreads();
    }
    if (!near && i0 < i1) {
        first.st = A.status[first.n];
        first.len = A.seg_len[first.n];
        first.start = A.seg_start[first.n];
    }
    for (int i = i0; i < i1; i++) {
        NextNode q = first;
        if (i > i0) {
            q.n = A.act_node[i];
            q.cp0 = A.cprefix[i];
            q.cp1 = A.cprefix[i + 1];
            q.st = A.status[q.n];
            q.len = A.seg_len[q.n];
            q.start = A.seg_start[q.n];
        }
        const int n = q.n;
        const int64_t len = q.len, start = q.start;
        const int64_t nl = A.node_sum ? A.node_sum[(int64_t)(2 * n) * A.NAg + A.NAg - 1] : near ? s_lpre[q.cp1] - s_lpre[q.cp0] : A.chunk_lpre[q.cp1] - A.chunk_lpre[q.cp0];
        if (q.st != ST_SPLIT) continue;
        const int64_t nr = len - nl;
        A.seg_start[2 * n] = start;
        A.seg_len[2 * n] = nl;
        A.seg_start[2 * n + 1] = start + nl;
        A.seg_len[2 * n + 1] = nr;
        const bool build_left = nr >= nl; // the smaller child is built, tie -> left (src/fit.jl:123-129)
        A.status[2 * n] = build_left ? ST_BUILD : ST_SUBTRACT;
        A.status[2 * n + 1] = build_left ? ST_SUBTRACT : ST_BUILD;
        if (A.cursor) {
            A.cursor[EVT_CURSOR_SLOT(2 * n)] = 0ull;
            A.cursor[EVT_CURSOR_SLOT(2 * n + 1)] = 0ull;
        }
        n1 = n;
        nl1 = nl;
        nr1 = nr;
        start1 = start;
        s_pos += 1;
        s_chunks += ((nl + whole) >> A.n_chunk_sh) + ((nr + whole) >> A.n_chunk_sh);
        s_brows += (build_left ? nl : nr) + A.seg_cost;
    }
    // children count (low 24 bits) and chunk count share one scan; the build rows take the other
    long long t_pc, t_brows, p_pc, p_brows;
    block_excl_scan2((s_chunks << 24) | s_pos, s_brows, &p_pc, &p_brows, &t_pc, &t_brows, s_tmp);
    long long p_pos = p_pc & 0xFFFFFF, p_chunks = p_pc >> 24;
    const long long t_pos = t_pc & 0xFFFFFF, t_chunks = t_pc >> 24;
    // the chunks' descriptors: LDS holds the children of 256 nodes at a time, which share the block's lanes; what a child has beyond
    // eight of each of its lanes is written by a whole wavefront (a wavefront for every child of more than four took 1.5 us at 32 children)
    const int lane = tid & 63;
    int i = i0;
    for (int base = 0; base < t_pos; base += 256) { // (positions ascend with the thread, and with i)
        for (; i < i1 && p_pos < base + 256; i++) {
            const bool one = span == 1;
            const int n = one ? n1 : A.act_node[i];
            if (one ? n1 == 0 : A.status[n] != ST_SPLIT) continue;
            const int64_t nl = one ? nl1 : A.seg_len[2 * n], nr = one ? nr1 : A.seg_len[2 * n + 1], start = one ? start1 : A.seg_start[2 * n];
            const bool build_left = nr >= nl;
            const int64_t cl = (nl + whole) >> A.n_chunk_sh, cr = (nr + whole) >> A.n_chunk_sh;
            A.n_act_node[2 * p_pos] = 2 * n;
            A.n_act_node[2 * p_pos + 1] = 2 * n + 1;
            A.n_cprefix[2 * p_pos] = p_chunks;
            A.n_cprefix[2 * p_pos + 1] = p_chunks + cl;
            A.n_bnode[p_pos] = build_left ? 2 * n : 2 * n + 1;
            A.n_bstart[p_pos] = build_left ? start : start + nl;
            A.n_bprefix[p_pos] = p_brows;
            s_child[2 * (p_pos - base)] = make_uint4(2 * n, (uint32_t)start, (uint32_t)(start + nl), (uint32_t)p_chunks);
            s_child[2 * (p_pos - base) + 1] = make_uint4(2 * n + 1, (uint32_t)(start + nl), (uint32_t)(start + nl + nr), (uint32_t)(p_chunks + cl));
            p_pos += 1;
            p_chunks += cl + cr;
            p_brows += (build_left ? nl : nr) + A.seg_cost;
        }
        __syncthreads();
        const int kids = t_pos - base < 256 ? 2 * (int)(t_pos - base) : 512;
        const uint32_t chunk = 1u << A.n_chunk_sh;
        const int gs = kids < nthr ? __clz(kids - 1) - __clz(nthr - 1) : 0, g = 1 << gs, sub = tid & (g - 1); // g lanes to a child
        for (int q0 = 0; q0 < kids; q0 += nthr >> gs) {
            const int q = q0 + (tid >> gs);
            const uint4 d = q < kids ? s_child[q] : make_uint4(0, 0, 0, 0);
            const uint32_t chunks = (uint32_t)((d.z - d.y + (uint64_t)chunk - 1) >> A.n_chunk_sh);
#pragma unroll 1
            for (uint32_t c = sub; c < min(chunks, 8u * g); c += g) A.n_cdesc[d.w + c] = make_uint4(d.x, d.y + c * chunk, d.z, d.w);
            for (unsigned long long many = __ballot(chunks > 8u * g && (lane & (g - 1)) == 0); many; many &= many - 1) {
                const int l = __ffsll((long long)many) - 1;
                const uint4 e = make_uint4(__builtin_amdgcn_readlane(d.x, l), __builtin_amdgcn_readlane(d.y, l), __builtin_amdgcn_readlane(d.z, l), __builtin_amdgcn_readlane(d.w, l));
                for (uint32_t c = 8 * g + lane; (int64_t)c * chunk < (int64_t)(e.z - e.y); c += 64) A.n_cdesc[e.w + c] = make_uint4(e.x, e.y + c * chunk, e.z, e.w);
            }
        }
        __syncthreads();
    }
    if (tid == 0) {
        A.n_cprefix[2 * t_pos] = t_chunks;
        A.n_bprefix[t_pos] = t_brows;
        A.n_hdr[LH_N_ACT] = 2 * t_pos;
        A.n_hdr[LH_N_CHUNKS] = t_chunks;
        A.n_hdr[LH_N_BUILD] = t_pos;
        A.n_hdr[LH_TOTAL_BUILD] = t_brows;
        if (A.n_stats) *A.n_stats = t_brows - t_pos * A.seg_cost;
    }
}

// Inputs with thousands of chunks per level: the scan of the chunk counts is a kernel of its own (one block of 1024 threads)
// between the count and the scatter pass - every scatter block adding up its node's chunk counts would cost more than this
// launch - and only the next level's tables, which no scatter block reads, ride along in the scatter kernel.
__global__ __launch_bounds__(1024) void k_chunk_scan(NextArgs A) {
    __shared__ long long s_tmp[34];
    chunk_scan_block(A, s_tmp);
}

// HNA > 0: the pass also builds the next level's histograms (update_hist!, src/fit-utils.jl:345-394) for inputs whose
// levels are chains of short kernels: 16-byte records (at most 16 features, one lane per row) and few chunks.  A block
// knows its node's left and right sizes, hence which child is built (the smaller, tie -> left, src/fit.jl:123-129); the rows
// of its chunk that go there are added into an LDS histogram of HNA channels (PACK: gradient and row count share channel
// 0's word) and the chunk's partial histogram is added to the child's zero-initialised slice with global atomics.  No
// histogram kernel runs below the root then.
template <int HNA, bool PACK>
__global__ __launch_bounds__(256) void k_part_scatter(PartArgs A, NextArgs NX) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    __shared__ long long s_tmp[34];
    extern __shared__ unsigned long long s_H[]; // HNA > 0: [HNA][sampled features][bins]
    // fold 1: the level's bookkeeping rides along whole and the blocks add up their node's chunk counts themselves;
    // fold 2: the chunk counts were scanned by k_chunk_scan, only the next level's tables ride along
    touch_kernargs<decltype(k_part_scatter<HNA, PACK>)>();
    const bool fold = A.fold == 1;
    if (blockIdx.x == gridDim.x - 1) { // the level's bookkeeping, beside the blocks that move the rows
        __shared__ uint4 s_child[512];
        __shared__ int s_lpre[LEVEL_LPRE + 1];
        // both halves for inputs of up to a thousand chunks per level
        if (fold) level_tables_block<true>(NX, s_tmp, s_child, s_lpre);
        else level_tables_block<false>(NX, s_tmp, s_child, nullptr);
        return;
    }
    // the 16 features of a record -> LDS word of their first bin (bins are 1-based); vmask bit t: feature t is sampled
    int off[16];
    unsigned vmask = 0;
    const int plane = (HNA > 0) ? A.nfs * A.B : 0;
    if constexpr (HNA > 0) {
#pragma unroll
        for (int t = 0; t < 16; t++) {
            const int sl = (t < A.F) ? (int)A.jsmap[t] : 0xFFFF;
            const bool ok = sl != 0xFFFF;
            off[t] = ok ? sl * A.B - 1 : 0;
            vmask |= ok ? (1u << t) : 0u;
        }
        for (int i = tid; i < HNA * plane; i += 256) s_H[i] = 0ull;
    }
    const int64_t G = gridDim.x - 1;
    uint4 cd = A.cdesc[blockIdx.x];
    const int64_t n_chunks = A.hdr[LH_N_CHUNKS];
    asm volatile("" : "+v"(cd.x), "+v"(cd.y), "+v"(cd.z), "+v"(cd.w)); // with the chunk count
    __shared__ unsigned long long s_w[EVT_CHUNK_WORDS];
    __shared__ int s_pre[EVT_CHUNK_WORDS];
    for (int64_t c = blockIdx.x; c < n_chunks; c += G, cd = A.cdesc[c < n_chunks ? c : 0]) {
        const int n = (int)cd.x;
        const int64_t p0 = cd.y, pend = cd.z, c0 = cd.w;
        const int64_t cl = c - c0;
        const int64_t seg = p0 - cl * EVT_CHUNK;
        // everything the chunk needs is requested at once, behind the descriptor: node state, the count pass's ballots
        // and prefixes, the left child's size and the row ids (positions past the end read the segment's last row)
        const int st = A.status[n];
        const unsigned long long fw = A.flagw[c * EVT_CHUNK_WORDS + (tid & (EVT_CHUNK_WORDS - 1))];
        // lefts of this node before this chunk, and in all of the node: the block adds up the node's chunk counts itself
        // (a node's chunks are few, or the sums are spread over the 256 threads)
        const int64_t c1 = c0 + (pend - seg + EVT_CHUNK - 1) / EVT_CHUNK;
        long long sum_before = 0, sum_node = 0;
        if (fold) {
            for (int64_t k = c0 + tid; k < c1; k += 256) {
                const int v = A.chunk_nleft[k];
                sum_node += v;
                sum_before += (k < c) ? v : 0;
            }
        } else { // the chunk counts were scanned before this kernel (the children's sizes are being written beside it)
            const long long l0 = A.chunk_lpre[c0];
            sum_before = A.chunk_lpre[c] - l0;
            sum_node = A.chunk_lpre[c1] - l0;
        }
        constexpr int NI = EVT_CHUNK / 256;
        uint32_t rid[NI];
#pragma unroll
        for (int it = 0; it < NI; it++) {
            const int64_t p = p0 + it * 256 + tid;
            rid[it] = A.is_cur[p < pend ? p : pend - 1];
        }
        // HNA > 0: the record and the gradient words of every row are requested along with everything else, before it is
        // known which child is built and which rows go there (16 + 4..8 bytes per row, off the block's chain of dependent loads)
        uint4 rec[HNA > 0 ? NI : 1];
        unsigned long long gw[HNA > 0 ? NI : 1][HNA > 0 ? HNA : 1];
        if constexpr (HNA > 0) {
#pragma unroll
            for (int it = 0; it < NI; it++) {
                rec[it] = *reinterpret_cast<const uint4 *>(A.xrm + (size_t)rid[it] * 16);
                evt_load_words<HNA, PACK>(A.gq, A.gq_stride, 0, rid[it], gw[it]);
            }
        }
        if (st == ST_SPLIT) {
            if (fold) {
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) {
                    sum_before += __shfl_xor(sum_before, o);
                    sum_node += __shfl_xor(sum_node, o);
                }
                if (lane == 0) { s_tmp[wave] = sum_before; s_tmp[4 + wave] = sum_node; }
            }
            if (tid < EVT_CHUNK_WORDS) s_w[tid] = fw;
            __syncthreads();
            if (tid == 0) {
                int run = 0;
                for (int t = 0; t < EVT_CHUNK_WORDS; t++) { s_pre[t] = run; run += __popcll(s_w[t]); }
            }
            __syncthreads();
            const int64_t lbase = fold ? s_tmp[0] + s_tmp[1] + s_tmp[2] + s_tmp[3] : sum_before; // lefts of this node before this chunk
            const int64_t nl_node = fold ? s_tmp[4] + s_tmp[5] + s_tmp[6] + s_tmp[7] : sum_node;
            const int64_t dstL = seg + lbase;
            const int64_t dstR = seg + nl_node + (cl * EVT_CHUNK - lbase);
            unsigned onmask = 0; // rows of this thread that go to the built child
            bool build_left = false;
            if constexpr (HNA > 0) {
                build_left = (pend - seg) - nl_node >= nl_node;
#pragma unroll
                for (int it = 0; it < NI; it++) {
                    const int64_t p = p0 + it * 256 + tid;
                    const bool flag = (s_w[it * 4 + wave] >> lane) & 1ull;
                    if (p < pend && flag == build_left) onmask |= 1u << it;
                }
            }
#pragma unroll
            for (int it = 0; it < NI; it++) {
                const int64_t p = p0 + it * 256 + tid;
                if (p < pend) {
                    const int wi = it * 4 + wave;
                    const unsigned long long word = s_w[wi];
                    const int lrank = s_pre[wi] + __popcll(word & ((1ull << lane) - 1ull));
                    const bool flag = (word >> lane) & 1ull;
                    const int within = it * 256 + tid;
                    const int64_t d = flag ? (dstL + lrank) : (dstR + (within - lrank));
                    A.is_next[d] = rid[it];
                }
            }
            if constexpr (HNA > 0) {
#pragma unroll
                for (int it = 0; it < NI; it++) {
                    if (onmask & (1u << it)) {
                        const uint32_t wds[4] = {rec[it].x, rec[it].y, rec[it].z, rec[it].w};
#pragma unroll
                        for (int t = 0; t < 16; t++) {
                            if (vmask & (1u << t)) {
                                const int idx = off[t] + (int)((wds[t >> 2] >> (8 * (t & 3))) & 0xFFu);
#pragma unroll
                                for (int a = 0; a < HNA; a++) atomicAdd(&s_H[a * plane + idx], gw[it][a]);
                            }
                        }
                    }
                }
                __syncthreads();
                // the chunk's partial histogram joins the built child's slice hist[node][slot][channel][bin]; chunks start
                // at different words so that concurrent flushes of one node do not queue on the same addresses
                unsigned long long *hn = reinterpret_cast<unsigned long long *>(A.hist) + (int64_t)(2 * n + (build_left ? 0 : 1) - 1) * A.node_stride;
                const int nwords = HNA * plane;
                const int rot = (int)((c * 1021) % nwords);
                for (int k = tid; k < nwords; k += 256) {
                    int idx = k + rot;
                    if (idx >= nwords) idx -= nwords;
                    const unsigned long long w = s_H[idx];
                    if (w != 0ull) {
                        s_H[idx] = 0ull;
                        const int a = idx / plane;
                        const int rem = idx - a * plane;
                        const int sl = rem / A.B;
                        const int bin = rem - sl * A.B;
                        unsigned long long *base = hn + ((int64_t)sl * A.NAg) * A.B + bin;
                        if (PACK && a == 0) {
                            const long long gsum = (long long)w >> EVT_PACK_CNT_BITS;
                            const unsigned long long cnt = w & ((1ull << EVT_PACK_CNT_BITS) - 1ull);
                            if (gsum != 0) atomicAdd(base, (unsigned long long)gsum);
                            atomicAdd(base + (int64_t)(A.NAg - 1) * A.B, cnt);
                        } else {
                            atomicAdd(base + (int64_t)a * A.B, w);
                        }
                    }
                }
            }
            __syncthreads();
        } else if (st == ST_LEAF && (A.write_nidx || A.fuse_pred)) {
            // rows of a node that stops here: record the node id; add the leaf value
            // (predict!, src/predict.jl:1-46: plain add / clamp(-15,15) / floor -15 on scale rows)
            const int K = A.K;
#pragma unroll
            for (int it = 0; it < EVT_CHUNK / 256; it++) {
                const int64_t p = p0 + it * 256 + tid;
                if (p < pend) {
                    const uint32_t row = rid[it];
                    if (A.write_nidx) A.nidx[row] = (uint32_t)n;
                    if (A.fuse_pred) {
                        float *pr = A.pred + (size_t)K * row;
                        const float *lp = A.t_pred + (size_t)K * (n - 1);
                        evt_add_leaf(pr, lp, K, A.loss);
                    }
                }
            }
        }
    }
}

// p's element at a byte offset
template <typename V>
__device__ __forceinline__ V &at_offset(V *p, uint32_t bytes) {
    return *reinterpret_cast<V *>(reinterpret_cast<char *>(const_cast<std::remove_const_t<V> *>(p)) + bytes);
}

// The partition of a level in one pass: a block decides its chunk's rows, claims as many places of either child with one addition to the
// node's cursor, and writes the row ids there.  A chunk's rows keep their order; the chunks of a node follow each other in the order of
// their claims, which nothing depends on: sums are integers, leaves are recorded by row id.  A wavefront owns NI * 64 neighbouring
// positions, so that one total per wavefront is all that is exchanged.
// Bound by its chain of trips to memory (descriptor, row ids and node, decision words, claim, stores) below a million rows; above, by the claims of a node of
// many chunks, by the lists and, deeper, the decision words' lines.  A chunk's numbers are in scalar registers and a lane's addresses offsets from them, which takes
// a third of the registers (97 -> 64 for 16 rows a thread) and twice the wavefronts.  us a level, count + scan of the counts + scatter -> one pass -> this: 800k
// rows x 28 features, depth 8 5.2 + 6.5 -> 7.4 -> 7.1; 500k of 100 4.7 + 5.9 -> 6.3 -> 6.2; 10M x 100, depth 11, root 17 + 5 + 19 -> 32 -> 26, level 5 18 + 5 + 18 -> 36 -> 35, level 9 33 + 5 +
// 19 -> 45 -> 43.
template <bool NT, int T, int NI>
__global__ __launch_bounds__(T, 8) void k_part_move(PartArgs A, NextArgs NX) {
    constexpr int W = T / 64, CHUNK = NI * T;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    __shared__ long long s_tmp[34];
    __shared__ int s_cnt[W];
    __shared__ unsigned long long s_claim;
    touch_kernargs<decltype(k_part_move<NT, T, NI>)>();
    const int64_t G = (int64_t)gridDim.x - 1;
    if (blockIdx.x == 0) { // the next level's tables, beside the blocks that move the rows
        __shared__ uint4 s_child[512];
        level_tables_block<false>(NX, s_tmp, s_child, nullptr);
        return;
    }
    uint4 cd = A.cdesc[blockIdx.x - 1];
    const int64_t n_chunks = A.hdr[LH_N_CHUNKS];
    asm volatile("" : "+v"(cd.x), "+v"(cd.y), "+v"(cd.z), "+v"(cd.w)); // requested with the level's chunk count, not behind the branch on it
    for (int64_t c = blockIdx.x - 1; c < n_chunks; c += G, cd = A.cdesc[c < n_chunks ? c : 0]) {
        // a chunk's numbers are the block's, in scalar registers: a lane's addresses are 32-bit offsets from them
        const int n = __builtin_amdgcn_readfirstlane((int)cd.x);
        const uint32_t p0 = __builtin_amdgcn_readfirstlane((int)cd.y), pend = __builtin_amdgcn_readfirstlane((int)cd.z), c0 = __builtin_amdgcn_readfirstlane((int)cd.w);
        const uint32_t seg = p0 - (uint32_t)(c - c0) * CHUNK;                             // positions are 32-bit numbers, as the row ids
        const uint32_t left_of = pend - p0, wofs = wave * (NI * 64) + lane;               // rows from the chunk's first on; this lane's first
        const uint32_t *isp = A.is_cur + p0;
        uint32_t rid[NI], xbv[NI];
#pragma unroll
        for (int it = 0; it < NI; it++) rid[it] = at_offset(isp, 4u * (wofs + it * 64 < left_of ? wofs + it * 64 : left_of - 1));
        int stv = A.status[n];
        uint32_t ndv = A.t_packed[n - 1]; // requested with the state, not behind the branch on it
        uint32_t nlv = (uint32_t)A.node_sum[(int64_t)(2 * n) * A.NAg + A.NAg - 1];
        asm volatile("" : "+v"(stv), "+v"(ndv), "+v"(nlv));
        const int st = __builtin_amdgcn_readfirstlane(stv);
        const uint32_t nd = __builtin_amdgcn_readfirstlane((int)ndv), nl = __builtin_amdgcn_readfirstlane((int)nlv);
        if (st == ST_SPLIT) {
            const int f = (int)(nd & 0xFFFFu) - 1;
            const uint32_t cb = (nd >> 16) & 0xFFu;
            const bool numeric = (nd & EVT_NODE_NUMERIC) != 0;
            const uint8_t *col = A.xcm + (size_t)f * A.N;
            const bool plane = A.planes && numeric && cb >= 1u && cb < (uint32_t)A.B;
            uint32_t lefts_of = 0; // bit it: the lane's row of step it goes left
            if (plane) {
                const uint32_t *words = A.planes + ((size_t)f * (A.B - 1) + (cb - 1)) * A.plane_words;
#pragma unroll
                for (int it = 0; it < NI; it++) xbv[it] = NT ? __builtin_nontemporal_load(&at_offset(words, (rid[it] >> 5) * 4u)) : at_offset(words, (rid[it] >> 5) * 4u);
#pragma unroll
                for (int it = 0; it < NI; it++) lefts_of |= (wofs + it * 64 < left_of ? (xbv[it] >> (rid[it] & 31u)) & 1u : 0u) << it;
            } else {
#pragma unroll
                for (int it = 0; it < NI; it++) xbv[it] = NT ? __builtin_nontemporal_load(&at_offset(col, rid[it])) : at_offset(col, rid[it]);
#pragma unroll
                for (int it = 0; it < NI; it++) lefts_of |= (uint32_t)(wofs + it * 64 < left_of && (numeric ? xbv[it] <= cb : xbv[it] == cb)) << it;
            }
            int cnt = 0;
#pragma unroll
            for (int it = 0; it < NI; it++) cnt += __popcll(__ballot((lefts_of >> it) & 1u));
            if (lane == 0) s_cnt[wave] = cnt;
            __syncthreads();
            int lefts = 0, before = 0; // of the chunk, of the wavefronts before this one
#pragma unroll
            for (int w = 0; w < W; w++) {
                const int v = s_cnt[w];
                lefts += v;
                before += w < wave ? v : 0;
            }
            const int rows = (int)(left_of < (uint32_t)CHUNK ? left_of : (uint32_t)CHUNK);
            if (tid == 0) s_claim = atomicAdd(A.cursor + EVT_CURSOR_SLOT(n), (unsigned long long)lefts | ((unsigned long long)(rows - lefts) << 32));
            __syncthreads();
            before = __builtin_amdgcn_readfirstlane(before);
            const uint32_t claim_l = __builtin_amdgcn_readfirstlane((int)(uint32_t)s_claim), claim_r = __builtin_amdgcn_readfirstlane((int)(uint32_t)(s_claim >> 32));
            uint32_t *out_l = A.is_next + (seg + claim_l + before), *out_r = A.is_next + (seg + nl + claim_r + (wave * (NI * 64) - before));
#pragma unroll
            for (int it = 0; it < NI; it++) {
                const bool left = (lefts_of >> it) & 1u;
                const unsigned long long bal = __ballot(left);
                const uint32_t lrank = __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
                if (left) at_offset(out_l, 4u * lrank) = rid[it];
                asm volatile(""); // two stores from scalar addresses, not one from an address chosen by the lane
                if (!left && wofs + it * 64 < left_of) at_offset(out_r, 4u * (lane - lrank)) = rid[it];
                const int k = __popcll(bal);
                out_l += k;
                out_r += 64 - k;
            }
        } else if (st == ST_LEAF && (A.write_nidx || A.fuse_pred)) { // rows of a node that stops here, as in k_part_scatter
            for (uint32_t k = tid; k < (uint32_t)CHUNK && k < left_of; k += T) {
                const uint32_t row = isp[k];
                if (A.write_nidx) A.nidx[row] = (uint32_t)n;
                if (A.fuse_pred) evt_add_leaf(A.pred + (size_t)A.K * row, A.t_pred + (size_t)A.K * (n - 1), A.K, A.loss);
            }
        }
    }
}

// Last pass of a tree: rows of the deepest split level go straight to their leaf.  For a node that split,
// the child is decided from x_bin[row, feat] exactly as the partition would (left iff <= cond_bin, or ==
// for a categorical feature) but the row list is not rewritten: nothing reads it afterwards.  Each row
// gets its leaf's value added to the prediction (predict!, src/predict.jl:1-46) and, on request, its
// node id recorded.
template <bool NT>
__global__ __launch_bounds__(256) void k_final_fused(PartArgs A) {
    const int tid = threadIdx.x;
    touch_kernargs<decltype(k_final_fused<NT>)>();
    const int64_t G = (int64_t)gridDim.x - A.blob.blocks;
    if ((int64_t)blockIdx.x >= G) {
        // the tree's arrays are complete (this is the tree's last kernel and writes none of them): their way back to the
        // host rides along instead of taking a launch of its own
        blob_send(A.blob, (int)(blockIdx.x - G));
        return;
    }
    uint4 cd = A.cdesc[blockIdx.x];
    const int64_t n_chunks = A.hdr[LH_N_CHUNKS];
    asm volatile("" : "+v"(cd.x), "+v"(cd.y), "+v"(cd.z), "+v"(cd.w)); // with the chunk count
    const int K = A.K;
    for (int64_t c = blockIdx.x; c < n_chunks; c += G, cd = A.cdesc[c < n_chunks ? c : 0]) {
        const int n = (int)cd.x;
        const int64_t p0 = cd.y, pend = cd.z;
        constexpr int NI = EVT_CHUNK / 256;
        uint32_t rid[NI], xbv[NI];
        float prv[NI];
#pragma unroll
        for (int it = 0; it < NI; it++) {
            const int64_t p = p0 + it * 256 + tid;
            rid[it] = A.is_cur[p < pend ? p : pend - 1];
        }
        const int st = A.status[n];
        uint32_t nd = A.t_packed[n - 1]; // requested with the state, not behind the branch on it
        asm volatile("" : "+v"(nd));
        if (st != ST_SPLIT && st != ST_LEAF) continue;
        const bool is_split = (st == ST_SPLIT);
        int f = 0;
        uint32_t cb = 0;
        bool numeric = true;
        if (is_split) {
            f = (int)(nd & 0xFFFFu) - 1;
            cb = (nd >> 16) & 0xFFu;
            numeric = (nd & EVT_NODE_NUMERIC) != 0;
        }
        const uint8_t *col = A.xcm + (size_t)f * A.N;
        const uint32_t *plane = (A.planes && is_split && numeric && cb >= 1u && cb < (uint32_t)A.B) ? A.planes + ((size_t)f * (A.B - 1) + (cb - 1)) * A.plane_words : nullptr;
        // every request of the chunk goes out before the first result is used: row ids (above), then bin bytes or plane
        // words, then (one output) the predictions; positions past the end read the segment's last row and are not written
#pragma unroll
        for (int it = 0; it < NI; it++) xbv[it] = is_split ? load_decision<NT>(col, plane, rid[it]) : 0u;
        const bool fast1 = A.fuse_pred && K == 1;
        if (fast1) {
#pragma unroll
            for (int it = 0; it < NI; it++) prv[it] = A.pred[rid[it]];
        }
#pragma unroll
        for (int it = 0; it < NI; it++) {
            const int64_t p = p0 + it * 256 + tid;
            if (p < pend) {
                const uint32_t row = rid[it];
                int leaf = n;
                if (is_split) {
                    const bool left = decide_left(xbv[it], plane != nullptr, row, numeric, cb);
                    leaf = 2 * n + (left ? 0 : 1);
                }
                if (A.write_nidx) A.nidx[row] = (uint32_t)leaf;
                if (fast1) {
                    const float s = prv[it] + A.t_pred[leaf - 1];
                    A.pred[row] = (A.loss == EVT_LOSS_LOGLOSS) ? fminf(fmaxf(s, -15.0f), 15.0f) : s;
                    continue;
                }
                if (A.fuse_pred) {
                    float *pr = A.pred + (size_t)K * row;
                    const float *lp = A.t_pred + (size_t)K * (leaf - 1);
                    evt_add_leaf(pr, lp, K, A.loss);
                }
            }
        }
    }
}

// Start of a tree: zero the Tree arrays (Tree{L,K}(depth), src/structs.jl:97-106) and node states,
// make the root the only active (build) node over rows [0, n_is), zero its histogram slice.
struct BeginArgs {
    TreeDev tree;
    int32_t *status;
    int64_t *seg_start;
    int64_t *seg_len;
    int64_t *hdr;
    int32_t *act_node;
    int64_t *cprefix;
    int32_t *bnode;
    int64_t *bstart;
    int64_t *bprefix;
    long long *hist;
    int64_t *stats;
    int64_t n_is; // rows of a tree on every row
    int64_t seg_cost;
    int64_t root_words;
    int nnodes, K, D;
    int chunk_sh; // rows of a chunk of the root, a power of two
    uint4 *cdesc;
    unsigned long long *cursor;
    // the tree's column sample and its inverse map, from the pinned staging buffer to the device copies (0 words: unchanged)
    const uint32_t *js_src, *map_src;
    uint32_t *js_dst, *map_dst;
    int js_words, map_words;
};

// One block prepares a tree: empty Tree arrays, node states, the column sample; and, once the number of its rows is known, the first level's tables.
// A kernel of its own for a tree on every row; with a row sample they ride in the kernel that
// lists the sampled rows (k_mask_sample), which counts them.
__device__ void tree_begin_arrays(const BeginArgs &A) {
    const int tid = threadIdx.x, nthr = blockDim.x; // 256 or 1024; each of four wavefronts starts another of the short lists
    for (int n = tid; n < A.nnodes; n += nthr) {
        A.tree.feat[n] = 0;
        A.tree.cond_bin[n] = 0;
        A.tree.w[n] = 0.0f;
        A.tree.gain[n] = 0.0f;
        A.tree.split[n] = 0;
        A.tree.packed[n] = 0u;
        for (int k = 0; k < A.K; k++) A.tree.pred[(int64_t)A.K * n + k] = 0.0f;
    }
    for (int n = tid ^ 64; n < A.nnodes + 2; n += nthr) A.status[n] = n == 1 ? ST_BUILD : ST_INACTIVE;
    for (int d = tid ^ 128; d <= A.D; d += nthr)
        if (d) A.stats[d] = 0;
    for (int i = tid; i < A.js_words; i += nthr) A.js_dst[i] = A.js_src[i];
    for (int i = tid; i < A.map_words; i += nthr) A.map_dst[i] = A.map_src[i];
}
__device__ void tree_begin_rows(const BeginArgs &A, int64_t n_is) {
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int64_t n_chunks = (n_is + ((int64_t)1 << A.chunk_sh) - 1) >> A.chunk_sh;
    for (int64_t c = tid ^ 192; c < n_chunks; c += nthr) A.cdesc[c] = make_uint4(1, (uint32_t)(c << A.chunk_sh), (uint32_t)n_is, 0);
    if (tid == 128) {
        A.stats[0] = n_is; // read back with the tree: the host learns how many rows the mask kept
        A.seg_start[1] = 0;
        A.seg_len[1] = n_is;
        A.hdr[LH_N_ACT] = 1;
        A.hdr[LH_N_CHUNKS] = n_chunks;
        A.hdr[LH_N_BUILD] = 1;
        A.hdr[LH_TOTAL_BUILD] = n_is + A.seg_cost;
        A.act_node[0] = 1;
        A.cprefix[0] = 0;
        A.cprefix[1] = n_chunks;
        A.cursor[EVT_CURSOR_SLOT(1)] = 0ull;
        A.bnode[0] = 1;
        A.bstart[0] = 0;
        A.bprefix[0] = 0;
        A.bprefix[1] = n_is + A.seg_cost;
    }
}

// The root's slice, shared by the kernel's blocks: one block took 26 us for 212 000 words (166 features, five channels, 255 bins).
__device__ void tree_begin_root(const BeginArgs &A, int blocks) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < A.root_words; i += (int64_t)blocks * blockDim.x) A.hist[i] = 0;
}
// Blocks from `blocks` on quantise the gradients, which have nothing to do with the set-up: side by side in one launch where the gradients' words are
// still to be made: set-up + quantisation, us, 500k rows of four channels 4.2 + 6.9 -> 7.0, 60k of 14 channels 3.0 + 7.9 -> 9.3 - and a launch each.
__global__ __launch_bounds__(1024) void k_tree_begin(BeginArgs A, QuantArgs Q, int blocks) {
    touch_kernargs<decltype(k_tree_begin)>();
    if ((int)blockIdx.x >= blocks) {
        quant_rows(Q, (int)blockIdx.x - blocks, (int)gridDim.x - blocks);
        return;
    }
    tree_begin_root(A, blocks);
    if (blockIdx.x == 0) {
        tree_begin_arrays(A);
        tree_begin_rows(A, A.n_is);
    }
}

// ---- row subsampling: is = rows with mask <= cond (src/subsample.jl:6-38) -----------
// Which of the rows p0 .. p0 + 7 (p0 a multiple of 8) the mask keeps, row p0 in the lowest bit.
// DRAW: the bytes are not read but drawn here and written to `mask` on the way: the mask's 8-byte word w is output w of
// SplitMix64 (Steele, Lea, Flood 2014: a Weyl sequence with increment 0x9E3779B97F4A7C15 passed through two
// multiply-xorshift rounds) started at state `seed`, stored little end first - byte i of the mask is bits 8*(i%8).. of output
// i/8.  Stands in for rand!(rng, mask) of src/subsample.jl:7 when the caller accepts a counter-based stream keyed by one 64-bit
// draw of its own generator per tree.
template <bool DRAW>
__device__ __forceinline__ unsigned mask_flags(uint8_t *mask, uint8_t cond, int64_t N, int64_t p0, unsigned long long seed) {
    unsigned long long v = ~0ull; // bytes past the end read as 255
    if (DRAW) {
        unsigned long long z = seed + (unsigned long long)((p0 >> 3) + 1) * 0x9E3779B97F4A7C15ull;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        v = z;
        if (p0 + 8 <= N) {
            *reinterpret_cast<unsigned long long *>(mask + p0) = z;
        } else {
            for (int j = 0; p0 + j < N; j++) mask[p0 + j] = (uint8_t)(z >> (8 * j));
        }
    } else if (p0 + 8 <= N) {
        v = *reinterpret_cast<const unsigned long long *>(mask + p0);
    } else {
        for (int j = 0; j < 8; j++)
            if (p0 + j < N) v = (v & ~(0xFFull << (8 * j))) | ((unsigned long long)mask[p0 + j] << (8 * j));
    }
    unsigned flags = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const bool keep = (p0 + j < N) && ((uint8_t)(v >> (8 * j)) <= cond);
        flags |= keep ? (1u << j) : 0u;
    }
    return flags;
}

// The sample's rows, and the tree's set-up, in one kernel: a block flags its 8192 rows, claims as many places of the
// list by one addition and writes their ids there.  A block's rows stay in order, the blocks follow each other in the order of their
// claims, which nothing depends on (k_part_move's chunks do the same).  The block that claims last knows the number of rows and writes the first
// level's tables; block 0 prepares the rest of the tree.  Blocks behind the sample's help it clear the root's slice where that has more words than the
// sample's blocks write in a few stores each (30k rows x 120 features of 255 bins and 15 channels, 459k words: 6.8 us; 18.3 by the 4 blocks of the sample), those behind them quantise.  Bound by its chain (draw, count, claim, stores) and the
// quantisation beside it: 1M rows 7.9 us with one word a row, 10.0 with two (a block's rows by 1024 threads: 9.1, 12.4: quantisation gets its blocks later).  In two kernels, a
// count and a scatter that added the counts up, 5.9 + 5.1 and 8.9 + 4.7; where a scan ran between them, from 2M rows on, and the quantisation is a kernel of its own, 6M rows
// 15.8 us for 6.2 + 4.7 + 7.6, 10M 23.1 for 7.4 + 5.4 + 10.9.
template <bool DRAW>
__global__ __launch_bounds__(256) void k_mask_sample(uint8_t *mask, uint8_t cond, int64_t N, unsigned long long seed, uint32_t *is_out,
                                                     unsigned long long *claims, BeginArgs B, QuantArgs Q, int blocks, int clear) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    touch_kernargs<decltype(k_mask_sample<DRAW>)>();
    const int own_block = (int)blockIdx.x - 1, set_up = blocks + clear;
    if (own_block >= set_up) { // as k_tree_begin
        quant_rows(Q, own_block - set_up, (int)gridDim.x - 1 - set_up);
        return;
    }
    if (own_block < 0) {
        tree_begin_arrays(B);
        return;
    }
    auto clear_root = [&]() {
        for (int64_t i = (int64_t)own_block * 256 + tid; i < B.root_words; i += (int64_t)set_up * 256) B.hist[i] = 0;
    };
    if (own_block >= blocks) {
        clear_root();
        return;
    }
    static_assert(EVT_SAMPLE_ROWS == 256 * 32, "32 rows to a thread");
    __shared__ uint16_t s_row[EVT_SAMPLE_ROWS]; // the rows kept, from the block's first
    __shared__ int s_cnt[4];
    __shared__ unsigned long long s_claim;
    const int64_t b0 = (int64_t)own_block * EVT_SAMPLE_ROWS;
    uint32_t flags = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) flags |= mask_flags<DRAW>(mask, cond, N, b0 + tid * 32 + 8 * j, seed) << (8 * j);
    const int own = __popc(flags);
    int incl = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int x = __shfl_up(incl, o);
        if (lane >= o) incl += x;
    }
    if (lane == 63) s_cnt[wave] = incl;
    __syncthreads();
    int total = 0, at = incl - own;
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const int v = s_cnt[w];
        total += v;
        at += w < wave ? v : 0;
    }
    // rows claimed so far, blocks that have claimed in the upper half
    if (tid == 0) s_claim = atomicAdd(claims, (unsigned long long)total | (1ull << 40));
    for (uint32_t f = flags; f; f &= f - 1) s_row[at++] = (uint16_t)(tid * 32 + __ffs(f) - 1);
    clear_root();
    __syncthreads();
    const unsigned long long claim = s_claim;
    const int64_t base = (int64_t)(claim & ((1ull << 40) - 1));
    for (int i = tid; i < total; i += 256) is_out[base + i] = (uint32_t)b0 + s_row[i];
    if ((int)(claim >> 40) == blocks - 1) {
        if (tid == 0) *claims = 0ull; // for the next launch
        tree_begin_rows(B, base + total);
    }
}

static unsigned grid_for_chunks(int64_t max_chunks) {
    int64_t g = max_chunks;
    if (g > 4096) g = 4096;
    if (g < 1) g = 1;
    return (unsigned)g;
}

static void fill_begin_args(evt_ctx *c, BeginArgs &A) {
    const LevelTab &L = c->lvl[1];
    A.tree = c->tree;
    A.status = c->status;
    A.seg_start = c->seg_start;
    A.seg_len = c->seg_len;
    A.hdr = L.hdr;
    A.act_node = L.act_node;
    A.cprefix = L.cprefix;
    A.bnode = L.bnode;
    A.bstart = L.bstart;
    A.bprefix = L.bprefix;
    A.hist = c->hist;
    A.stats = c->stats;
    A.n_is = c->N;
    A.seg_cost = c->hist_seg_cost;
    A.root_words = (int64_t)c->n_js_last * c->NAg * c->B;
    A.nnodes = c->nnodes;
    A.K = c->K;
    A.D = c->D;
    A.chunk_sh = __builtin_ctz(part_chunk_rows(c, 1));
    A.cdesc = L.cdesc;
    A.cursor = c->cursor;
    A.js_words = A.map_words = 0;
    A.js_src = A.map_src = nullptr;
    A.js_dst = A.map_dst = nullptr;
    if (c->js_staged) { // read from the pinned buffer by the kernel (no trip through the copy engine, no launch of its own)
        const size_t o_js = c->blob_bytes, o_map = c->blob_bytes + (size_t)c->F * 4;
        A.js_src = reinterpret_cast<const uint32_t *>(c->h_stage_dev + o_js);
        A.js_dst = c->js;
        A.js_words = c->n_js_last;
        A.map_src = reinterpret_cast<const uint32_t *>(c->h_stage_dev + o_map);
        A.map_dst = reinterpret_cast<uint32_t *>(c->jsmap);
        A.map_words = c->RS / 2;
    }
}

// a tree on every row: the set-up block as a kernel of its own
int launch_tree_begin(evt_ctx *c) {
    BeginArgs A;
    fill_begin_args(c, A);
    QuantArgs Q = {};
    const unsigned blocks = (unsigned)std::min<int64_t>(1 + A.root_words / 4096, 64);
    unsigned quant = 0;
    if (c->quant_pending) {
        quant_args(c, Q);
        quant = quant_blocks(c, 1024);
    }
    hipLaunchKernelGGL(k_tree_begin, dim3(blocks + quant), dim3(1024), 0, c->stream, A, Q, (int)blocks);
    HIPCHK(hipGetLastError());
    if (quant) quant_taken(c);
    c->js_staged = false;
    return EVT_OK;
}

// Subsampling of a tree and its set-up.  draw: the mask's bytes are drawn from `seed` on the way (and written to
// c->mask) instead of read.
int launch_compact_mask(evt_ctx *c, uint8_t cond, bool draw, unsigned long long seed) {
    BeginArgs B;
    fill_begin_args(c, B);
    QuantArgs Q = {};
    unsigned quant = 0;
    const int64_t blocks = (c->N + EVT_SAMPLE_ROWS - 1) / EVT_SAMPLE_ROWS;
    if (c->quant_pending) {
        quant_args(c, Q);
        quant = quant_blocks(c, 256);
    }
    const int64_t clear = std::max<int64_t>(0, std::min<int64_t>(256, B.root_words / 4096) - blocks); // 16 words a thread, up to a block to a compute unit
    const dim3 grid((unsigned)(1 + blocks + clear) + quant);
    if (draw) hipLaunchKernelGGL(k_mask_sample<true>, grid, dim3(256), 0, c->stream, c->mask, cond, c->N, seed, c->is_a, c->sample_claims, B, Q, (int)blocks, (int)clear);
    else hipLaunchKernelGGL(k_mask_sample<false>, grid, dim3(256), 0, c->stream, c->mask, cond, c->N, 0ull, c->is_a, c->sample_claims, B, Q, (int)blocks, (int)clear);
    HIPCHK(hipGetLastError());
    if (quant) quant_taken(c);
    c->js_staged = false;
    return EVT_OK;
}

static void fill_part_args(evt_ctx *c, int level, const uint32_t *is_cur, uint32_t *is_next, bool fuse_pred, PartArgs &A) {
    const LevelTab &L = c->lvl[level & 1];
    A.hdr = L.hdr;
    A.cdesc = L.cdesc;
    A.act_node = L.act_node;
    A.cprefix = L.cprefix;
    A.status = c->status;
    A.seg_start = c->seg_start;
    A.seg_len = c->seg_len;
    A.t_packed = c->tree.packed;
    A.xcm = c->xcm;
    A.N = c->N;
    A.is_cur = is_cur;
    A.is_next = is_next;
    A.flagw = c->flagw;
    A.chunk_nleft = c->chunk_nleft;
    A.chunk_lpre = c->chunk_lpre;
    A.nidx = c->nidx;
    A.pred = c->pred;
    A.t_pred = c->tree.pred;
    A.K = c->K;
    A.loss = c->loss; // selects the leaf-add rule
    A.fuse_pred = fuse_pred ? 1 : 0;
    A.write_nidx = c->write_nidx ? 1 : 0;
    A.stream_hint = ((size_t)c->N * c->F > ((size_t)256 << 20)) ? 1 : 0;
    A.fold = 0;
    A.planes = c->planes_ready ? c->planes : nullptr;
    A.plane_words = c->plane_words;
    A.B = c->B;
    A.xrm = nullptr;
    A.gq = nullptr;
    A.jsmap = nullptr;
    A.hist = nullptr;
    A.node_stride = 0;
    A.F = A.nfs = 0;
    A.NAg = c->NAg;
    A.blob.blocks = 0;
    A.cursor = c->cursor;
    A.node_sum = c->node_sum;
}

// One pass where the children's sizes are in the totals (unit weights) and no histogram is built on the way.
static bool part_in_one_pass(const evt_ctx *c) { return c->part_one_pass && c->unit_w && !c->step.hist_fused; }

// Rows of a chunk of the level.  A node's chunks queue at its cursor, ~20 ns each: where a node has more than 128 of them they grow (us a level of
// 1M rows, 2048 | 4096 | 8192 rows a chunk: root 11.7 | 8.9 | 9.0, two nodes 9.0 | 7.6 | 8.4, eight 6.8 | 6.8 | 8.3; 10M: 67 | 39 | 28, 62 | 36 | 28,
// 34 | 28 | 23; 8192 | 16384, blocks of 1024: one to four nodes 31 | 26, 29 | 24, 29 | 26, eight 30 | 34, whose nodes of 1.25M rows keep the narrower;
// whole rounds of 10 to 40 features: 2.2M to 6M rows level within 0.7 % either way, 7M 290 | 285, 8M 317 | 311, 9M 352 | 346, 20M 1447 | 1439).  They grow too where the level is more blocks than the chip holds at once and nodes are many chunks (10M rows, 64 nodes 44 | - | 40).
int part_chunk_rows(const evt_ctx *c, int level) {
    int rows = EVT_CHUNK;
    if (!part_in_one_pass(c) || level >= c->D - 1) return rows;
    const int64_t per_node = (c->last_all_rows ? c->N : c->N * (c->last_cond + 1) / 256) >> (level - 1);
    const int64_t all = per_node << (level - 1);
    while (rows < EVT_CHUNK_MAX / 2 && (per_node > (int64_t)rows * 128 || (all > (int64_t)rows * 2048 && per_node >= (int64_t)rows * 16))) rows *= 2;
    if (rows == EVT_CHUNK_MAX / 2 && per_node > (int64_t)rows * 256) rows = EVT_CHUNK_MAX;
    return rows;
}

int launch_part_count(evt_ctx *c, int level, const uint32_t *is_cur) {
    if (part_in_one_pass(c)) return EVT_OK;
    PartArgs A;
    fill_part_args(c, level, is_cur, nullptr, false, A);
    if (A.stream_hint) hipLaunchKernelGGL(k_part_count<true>, dim3(grid_for_chunks(c->max_chunks)), dim3(256), 0, c->stream, A);
    else hipLaunchKernelGGL(k_part_count<false>, dim3(grid_for_chunks(c->max_chunks)), dim3(256), 0, c->stream, A);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

static void fill_next_args(evt_ctx *c, int level, NextArgs &A) {
    const LevelTab &L = c->lvl[level & 1];
    const LevelTab &Nx = c->lvl[(level + 1) & 1];
    A.hdr = L.hdr;
    A.act_node = L.act_node;
    A.cprefix = L.cprefix;
    A.status = c->status;
    A.seg_start = c->seg_start;
    A.seg_len = c->seg_len;
    A.chunk_nleft = c->chunk_nleft;
    A.chunk_lpre = c->chunk_lpre;
    A.n_hdr = Nx.hdr;
    A.n_act_node = Nx.act_node;
    A.n_cprefix = Nx.cprefix;
    A.n_bnode = Nx.bnode;
    A.n_bstart = Nx.bstart;
    A.n_bprefix = Nx.bprefix;
    A.n_cdesc = Nx.cdesc;
    A.n_stats = (level + 1 <= c->D) ? c->stats + level + 1 : nullptr;
    A.seg_cost = c->hist_seg_cost;
    A.n_chunk_sh = __builtin_ctz(part_chunk_rows(c, level + 1));
    A.node_sum = nullptr;
    A.NAg = c->NAg;
    A.cursor = nullptr;
}

// Moves the rows of the level's split nodes to their children and, in one extra block, writes the next level's tables.
int launch_part_scatter(evt_ctx *c, int level, const uint32_t *is_cur, uint32_t *is_next, bool fuse_pred) {
    PartArgs A;
    fill_part_args(c, level, is_cur, is_next, fuse_pred, A);
    NextArgs NX;
    fill_next_args(c, level, NX);
    if (part_in_one_pass(c)) {
        NX.node_sum = c->node_sum;
        NX.cursor = c->cursor;
        const int chunk = part_chunk_rows(c, level);
        const dim3 grid((unsigned)std::min<int64_t>(c->N / chunk + (1 << (level - 1)) + 1, 4096) + 1);
#define PMCASE(T_, NI_)                                                                                              \
    if (chunk == T_ * NI_) {                                                                                         \
        if (A.stream_hint) hipLaunchKernelGGL((k_part_move<true, T_, NI_>), grid, dim3(T_), 0, c->stream, A, NX);    \
        else hipLaunchKernelGGL((k_part_move<false, T_, NI_>), grid, dim3(T_), 0, c->stream, A, NX);                 \
    }
        PMCASE(256, 8) PMCASE(512, 8) PMCASE(512, 16) PMCASE(1024, 16)
#undef PMCASE
        HIPCHK(hipGetLastError());
        return EVT_OK;
    }
    // up to a thousand chunks per level the bookkeeping rides along in the scatter kernel (one launch less per level)
    A.fold = c->max_chunks <= 1024 + c->maxlvl ? 1 : 2;
    if (A.fold == 2) {
        hipLaunchKernelGGL(k_chunk_scan, dim3(1), dim3(1024), 0, c->stream, NX);
        HIPCHK(hipGetLastError());
    }
    const dim3 grid(grid_for_chunks(c->max_chunks) + 1);
    if (c->step.hist_fused) {
        // the next level's histograms are built here: no histogram kernel runs at that level
        A.xrm = c->xrm;
        A.gq = c->gq;
        A.gq_stride = EVT_GQ_STRIDE(c->NA);
        A.jsmap = c->jsmap;
        A.hist = c->hist;
        A.node_stride = (int64_t)c->F * c->NAg * c->B;
        A.F = c->F;
        A.nfs = c->n_js_last;
        const size_t lds = (size_t)c->NA * c->n_js_last * c->B * 8;
        if (A.fold != 1 || !scatter_can_build_hist(c, c->n_js_last)) {
            evt_set_error("internal: scatter pass cannot build histograms for this shape");
            return EVT_ERR_STATE;
        }
#define PSCASE(NA_)                                                                                                        \
    case NA_:                                                                                                              \
        if (c->unit_w) hipLaunchKernelGGL((k_part_scatter<NA_, true>), grid, dim3(256), lds, c->stream, A, NX);          \
        else hipLaunchKernelGGL((k_part_scatter<NA_, false>), grid, dim3(256), lds, c->stream, A, NX);                   \
        break;
        switch (c->NA) {
            PSCASE(1)
            PSCASE(2)
            PSCASE(3)
            PSCASE(4)
            PSCASE(5)
        default: evt_set_error("unsupported channel count %d", c->NA); return EVT_ERR_ARG;
        }
#undef PSCASE
    } else {
        hipLaunchKernelGGL((k_part_scatter<0, false>), grid, dim3(256), 0, c->stream, A, NX);
    }
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

// The scatter pass can build the next level's histograms: 16-byte records, one launch's worth of channels in at most
// 32 KB of LDS, the split search of one block per node (k_scan's fused form) and at most 128 chunks per level (a quarter of a million rows), where a level is a chain of
// kernels of a few microseconds each and one of them less is worth more than the histogram kernel's better use of the
// machine: at 100k rows x 10 features the pass takes 12 us against 5 + 10 us for the two kernels, at 1M rows 22 against 6 + 12.
bool scatter_can_build_hist(const evt_ctx *c, int nfs) {
    return c->hist_in_scatter && c->RS == 16 && !c->mc && c->tree_type != EVT_TREE_OBLIVIOUS && c->scan_fused && nfs <= 16 &&
           c->NA <= EVT_MAX_NA && c->max_chunks <= 128 + c->maxlvl && (size_t)c->NA * nfs * c->B * 8 <= 32 * 1024;
}

int launch_final_fused(evt_ctx *c, int level, const uint32_t *is_cur, bool fuse_pred, bool send_blob) {
    if (!fuse_pred && !c->write_nidx) return EVT_OK;
    PartArgs A;
    fill_part_args(c, level, is_cur, nullptr, fuse_pred, A);
    if (send_blob) {
        blob_out(c, A.blob);
        c->step.blob_sent = true;
    }
    const dim3 grid(grid_for_chunks(c->max_chunks) + (unsigned)A.blob.blocks);
    if (A.stream_hint) hipLaunchKernelGGL(k_final_fused<true>, grid, dim3(256), 0, c->stream, A);
    else hipLaunchKernelGGL(k_final_fused<false>, grid, dim3(256), 0, c->stream, A);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

// Node of every row that is still on its way down, read off the row lists: node n of the level owns
// is[seg_start[n] .. +seg_len[n]).  Read-back for a tree grown in stages (rows that reached a leaf above this level
// had their node recorded when they got there).
__global__ __launch_bounds__(256) void k_nidx_from_segments(const uint32_t *__restrict__ is, const int64_t *__restrict__ seg_start,
                                                           const int64_t *__restrict__ seg_len, const int32_t *__restrict__ status,
                                                           int first_node, uint32_t *__restrict__ nidx) {
    const int n = first_node + blockIdx.x;
    if (status[n] == ST_INACTIVE) return;
    const int64_t start = seg_start[n], len = seg_len[n];
    for (int64_t i = (int64_t)blockIdx.y * 256 + threadIdx.x; i < len; i += (int64_t)gridDim.y * 256) nidx[is[start + i]] = (uint32_t)n;
}

int launch_nidx_from_segments(evt_ctx *c, int level, const uint32_t *is_cur) {
    const int first = 1 << (level - 1), count = first; // nodes first .. 2 * first - 1
    hipLaunchKernelGGL(k_nidx_from_segments, dim3((unsigned)count, 64), dim3(256), 0, c->stream, is_cur, c->seg_start, c->seg_len, c->status,
                       first, c->nidx);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

