// A model kept on the device between predictions: _predict(m, data) (src/predict.jl:118-136) and predict_leaf_idx (:138-185) for a program
// that calls them again and again.  The host arrays of the trees stay the caller's; a copy of them is kept beside the packed device
// form, and every call compares before it uses the latter.
#include "upload.h"

#include <math.h>
#include <string.h>

#include <algorithm>
#include <list>
#include <memory>
#include <mutex>

int predict_lds_shape(int F, int max_int, int K, int hint);
int launch_predict_model_lds(hipStream_t s, const uint32_t *cnodes, const float *cleaf, const void *meta, int ntrees, const uint8_t *xcm, int64_t N,
                             int F, int max_int, int K, int ks, int loss, int apply_link, int all_numeric, int shape, float *out);
int walk_leaf_stride(int K);
int launch_walk_rows(hipStream_t s, const uint32_t *cnodes, int stride, const void *meta, const float *cleaf, const uint32_t *cid, int ntrees,
                     const uint8_t *x, int64_t ldx, int64_t n, int F, int wide, int K, int loss, int apply_link, float *out, void *leaf_out, int leaf_bytes,
                     int64_t leaf_ld);

namespace {

struct CompletedTree { // as k_predict_model_lds and k_walk_rows read it
    int32_t node_off, leaf_off, levels, n_int;
};

struct Model {
    std::mutex mu;
    int loss = 0, K = 0;
    // the caller's arrays as they were when the device form was built
    std::vector<int32_t> nn;
    std::vector<int64_t> feat;
    std::vector<uint8_t> cond_bin, split, feattypes;
    std::vector<float> pred;
    std::vector<double> edges;
    std::vector<int32_t> edge_off;
    // device form: trees completed to their depth, `stride` node words each, padded to a multiple of four trees; on the device that
    // was current in the call that built it
    bool built = false;
    int device = -1;
    int ntrees = 0, max_int = 0, max_feat = 0, max_nodes = 0;
    bool all_numeric = true, wide = false;
    uint32_t *d_nodes = nullptr, *d_cid = nullptr;
    float *d_leaf = nullptr;
    CompletedTree *d_meta = nullptr;
    uint8_t *d_form = nullptr; // the four of them, one after the other
    size_t cap_form = 0;
    std::vector<CompletedTree> meta;
    std::unique_ptr<HbPlan> plan[2]; // by source type
    size_t kept = 0;                 // bytes it is counted with in Kept; under Kept::mu, as the place in its list
    std::list<Model *>::iterator at;

    size_t bytes() const {
        size_t n = cap_form + 4 * nn.capacity() + 8 * feat.capacity() + cond_bin.capacity() + split.capacity() + feattypes.capacity() +
                   4 * pred.capacity() + 8 * edges.capacity() + 4 * edge_off.capacity() + sizeof(CompletedTree) * meta.capacity();
        for (const auto &p : plan)
            if (p) n += sizeof(HbFeature) * p->feat.capacity() + 8 * p->edges.capacity() + 4 * p->heap_store.capacity();
        return n;
    }
    void drop() { // all that a call can make again; no call is running, and each has waited for its stream
        built = false;
        dev_give(d_form);
        d_form = nullptr;
        cap_form = 0;
        std::vector<int32_t>().swap(nn);
        std::vector<int64_t>().swap(feat);
        std::vector<float>().swap(pred);
        std::vector<double>().swap(edges);
        std::vector<int32_t>().swap(edge_off);
        std::vector<CompletedTree>().swap(meta);
        for (auto *v : {&cond_bin, &split, &feattypes}) std::vector<uint8_t>().swap(*v);
        for (auto &p : plan) p.reset();
    }
    ~Model() { drop(); }
};

// All models, the last used first.  What they keep on the device and beside it is bounded together; beyond it those not used for longest
// are packed anew by their next call (0.6 ms for 100 trees of depth 6, 1.3 ms for 200 of depth 8).
struct Kept {
    static const size_t MOST = (size_t)1 << 30; // bytes: some 800 models of 200 trees of depth 8
    std::mutex mu;
    std::list<Model *> models;
    size_t bytes = 0;
    static Kept &get() { // never destroyed: models outlive main
        static Kept *k = new Kept();
        return *k;
    }
    void count(Model *m, size_t n) {
        bytes += n - m->kept;
        m->kept = n;
    }
    void add(Model *m) {
        std::lock_guard<std::mutex> lk(mu);
        m->at = models.insert(models.end(), m);
    }
    void remove(Model *m) {
        std::lock_guard<std::mutex> lk(mu);
        count(m, 0);
        models.erase(m->at);
    }
    void used(Model *m) { // by a call that holds its lock and is about to end
        std::lock_guard<std::mutex> lk(mu);
        count(m, m->bytes());
        models.splice(models.begin(), models, m->at);
        shrink(MOST, m);
    }
    void shrink(size_t most, Model *mine) {
        for (auto it = models.rbegin(); it != models.rend() && bytes > most; ++it) {
            Model *o = *it;
            if (!o->kept) continue;
            std::unique_lock<std::mutex> lk(o->mu, std::defer_lock);
            if (o != mine && !lk.try_lock()) continue; // in a call: it comes by here at its end
            o->drop();
            count(o, 0);
        }
    }
};

// A stream for one call, on the current device.
struct CallStream {
    hipStream_t s = nullptr;
    int device = 0;
    bool idle = false; // the call has waited for all it queued
    ~CallStream() {
        if (!s) return;
        if (!idle) (void)hipStreamSynchronize(s);
        stream_give(s, true, device);
    }
};
// Device memory for one call, given back when nothing uses it any more: declared before what waits for the stream.
struct CallBuffer {
    uint8_t *p = nullptr;
    ~CallBuffer() { dev_give(p); }
};

struct TreePtrs {
    int32_t n;
    const int64_t *nn;
    const int64_t *const *feat;
    const uint8_t *const *cond_bin;
    const uint8_t *const *split;
    const float *const *pred;
};

bool same_shape(const Model &m, const TreePtrs &t) {
    if (!m.built || (size_t)t.n != m.nn.size()) return false;
    for (int i = 0; i < t.n; i++)
        if (m.nn[i] != t.nn[i]) return false;
    return true;
}
bool same_trees(const Model &m, const TreePtrs &t) { // of trees of the same shape
    size_t o = 0;
    for (int i = 0; i < t.n; i++) {
        const size_t n = (size_t)m.nn[i];
        if (memcmp(m.feat.data() + o, t.feat[i], 8 * n) || memcmp(m.cond_bin.data() + o, t.cond_bin[i], n) ||
            memcmp(m.split.data() + o, t.split[i], n) || memcmp(m.pred.data() + o * m.K, t.pred[i], 4 * n * m.K))
            return false;
        o += n;
    }
    return true;
}

// Copies the caller's arrays, checks them by the rules of evt_predict, completes the trees and uploads them.
int build(Model &m, const TreePtrs &t, const uint8_t *feattypes, int nft, hipStream_t s) {
    m.built = false;
    size_t total = 0, leaves = 0;
    int levels_max = 0;
    for (int i = 0; i < t.n; i++) {
        ARGCHK(t.nn[i] >= 1 && t.nn[i] <= ((int64_t)1 << 20) - 1, "a kept model takes trees of up to 2^20 - 1 nodes");
        total += (size_t)t.nn[i];
        int d = 0;
        while (((int64_t)1 << d) - 1 < t.nn[i]) d++;
        levels_max = std::max(levels_max, d - 1);
        leaves += (size_t)1 << (d - 1);
    }
    const int npad = (t.n + 3) / 4 * 4;
    m.max_int = (1 << levels_max) - 1;
    const int stride = std::max(1, m.max_int);
    ARGCHK((size_t)npad * stride <= ((size_t)1 << 28), "the completed trees of a kept model exceed 2^28 nodes");
    m.nn.resize(t.n);
    m.feat.resize(total);
    m.cond_bin.resize(total);
    m.split.resize(total);
    m.pred.resize(total * m.K);
    m.feattypes.assign(feattypes ? feattypes : nullptr, feattypes ? feattypes + nft : nullptr);
    size_t o = 0;
    m.max_feat = m.max_nodes = 0;
    for (int i = 0; i < t.n; i++) {
        const int64_t n = t.nn[i];
        m.nn[i] = (int32_t)n;
        m.max_nodes = std::max(m.max_nodes, (int)n);
        memcpy(m.feat.data() + o, t.feat[i], 8 * n);
        memcpy(m.cond_bin.data() + o, t.cond_bin[i], n);
        memcpy(m.split.data() + o, t.split[i], n);
        memcpy(m.pred.data() + o * m.K, t.pred[i], 4 * n * m.K);
        for (int64_t k = 0; k < n; k++)
            if (m.split[o + k]) {
                ARGCHK(2 * k + 3 <= n, "split node without children inside the tree arrays");
                ARGCHK(m.feat[o + k] >= 1 && m.feat[o + k] <= EVT_MAX_FEATS && (!feattypes || m.feat[o + k] <= nft), "tree feature id outside 1..nfeats");
                m.max_feat = std::max(m.max_feat, (int)m.feat[o + k]);
            }
        o += (size_t)n;
    }
    m.wide = m.max_feat > 1024;
    m.all_numeric = true;
    m.ntrees = t.n;
    const int ks = walk_leaf_stride(m.K);
    ARGCHK(leaves * m.K < ((size_t)1 << 31), "the leaves of a kept model exceed 2^31 values");
    std::vector<uint32_t> nodes((size_t)npad * stride, 0u), cid(leaves);
    std::vector<float> leaf(leaves * ks, 0.0f); // (one by one they took a tenth of a small model's first call)
    leaves = 0;
    m.meta.assign(npad, CompletedTree{0, 0, 0, 0});
    std::vector<int32_t> src; // 0: a split node of the tree; otherwise the leaf whose value the node carries
    const uint32_t always_left = (255u << 16) | EVT_NODE_NUMERIC; // feature 1, bin <= 255
    o = 0;
    for (int i = 0; i < t.n; i++) {
        const int n = m.nn[i];
        int d = 0;
        while ((1 << d) - 1 < n) d++;
        const int full = (1 << d) - 1, n_int = full / 2, n_leaf = n_int + 1;
        m.meta[i] = {(int32_t)((size_t)i * stride), (int32_t)leaves, d - 1, n_int};
        src.assign(full + 1, 0);
        for (int k = 1; k <= full; k++) {
            const int32_t up = k == 1 ? 0 : src[k >> 1];
            src[k] = up ? up : (m.split[o + k - 1] ? 0 : k); // a split node's children lie inside the arrays: k <= n here
        }
        uint32_t *cn = nodes.data() + (size_t)i * stride;
        for (int k = 1; k <= n_int; k++) {
            uint32_t w = always_left;
            if (src[k] == 0) {
                const int f0 = (int)m.feat[o + k - 1] - 1;
                const bool numeric = m.feattypes.empty() || m.feattypes[f0] != 0;
                m.all_numeric = m.all_numeric && numeric;
                w = (m.wide ? (uint32_t)f0 : (uint32_t)(((f0 >> 2) << 8) | (f0 & 3))) | ((uint32_t)m.cond_bin[o + k - 1] << 16) | (numeric ? EVT_NODE_NUMERIC : 0u);
            }
            cn[k - 1] = w;
        }
        for (int q = 0; q < n_leaf; q++, leaves++) {
            const int32_t at = src[n_int + 1 + q];
            cid[leaves] = (uint32_t)at;
            for (int k = 0; k < m.K; k++) leaf[leaves * ks + k] = m.pred[m.K * (o + at - 1) + k];
        }
        o += (size_t)n;
    }
    // one block on the device, one copy: meta | nodes | leaf ids | leaf values, each from a 256-byte boundary on
    auto up = [](size_t n) { return (n + 255) / 256 * 256; };
    const size_t o_nodes = up(sizeof(CompletedTree) * m.meta.size()), o_cid = o_nodes + up(4 * nodes.size()), o_leaf = o_cid + up(4 * cid.size());
    const size_t bytes = o_leaf + up(4 * leaf.size());
    if (m.cap_form < bytes) { // no walk of the old form is running: each has been waited for
        dev_give(m.d_form);
        m.cap_form = 0;
        m.d_form = static_cast<uint8_t *>(dev_take(bytes));
        if (!m.d_form) return EVT_ERR_NOMEM;
        m.cap_form = bytes;
    }
    struct Staged { // pinned, and given back whichever way the call ends
        void *p;
        ~Staged() { pinned_give(p); }
    } stage{bytes <= PINNED_BYTES ? pinned_take(PINNED_BYTES) : nullptr};
    std::vector<uint8_t> plain(stage.p ? 0 : bytes);
    uint8_t *h = stage.p ? static_cast<uint8_t *>(stage.p) : plain.data();
    memcpy(h, m.meta.data(), sizeof(CompletedTree) * m.meta.size());
    memcpy(h + o_nodes, nodes.data(), 4 * nodes.size());
    memcpy(h + o_cid, cid.data(), 4 * cid.size());
    memcpy(h + o_leaf, leaf.data(), 4 * leaf.size());
    const hipError_t e = hipMemcpyAsync(m.d_form, h, bytes, hipMemcpyHostToDevice, s);
    const hipError_t e2 = hipStreamSynchronize(s);
    HIPCHK(e);
    HIPCHK(e2);
    m.d_meta = reinterpret_cast<CompletedTree *>(m.d_form);
    m.d_nodes = reinterpret_cast<uint32_t *>(m.d_form + o_nodes);
    m.d_cid = reinterpret_cast<uint32_t *>(m.d_form + o_cid);
    m.d_leaf = reinterpret_cast<float *>(m.d_form + o_leaf);
    m.built = true;
    return EVT_OK;
}

// Rows from this many on in one launch take the kernel that walks 1024 rows per block from LDS (k_predict_model_lds), fewer the one
// that spreads a row's trees over lanes: below it the former leaves compute units without a block.
const int64_t WALK_LDS_MIN_ROWS = 131072;

struct Request {
    const HbPlan *plan; // null: `bins` are the host's, column-major with N rows
    HbSource src;
    const uint8_t *bins;
    int64_t N;
    int F, ntrees, link;
    float *out;
    uint32_t *leaf_out;
    const TreePtrs *check; // compare the caller's trees with the device form once the device is at work (null: known to be the same)
    bool differ;           // they are not the same: the results are those of the old trees
};

int walk(Model &m, hipStream_t s, const Request &q, const uint8_t *x, int64_t n, void *out, int leaf_bytes) {
    if (q.leaf_out)
        return launch_walk_rows(s, m.d_nodes, std::max(1, m.max_int), m.d_meta, m.d_leaf, m.d_cid, q.ntrees, x, n, n, q.F, m.wide, m.K, m.loss, 0, nullptr, out,
                                leaf_bytes, n);
    const int shape = n >= WALK_LDS_MIN_ROWS ? predict_lds_shape(q.F, m.max_int, m.K, 0) : 0;
    if (shape > 0)
        return launch_predict_model_lds(s, m.d_nodes, m.d_leaf, m.d_meta, q.ntrees, x, n, q.F, m.max_int, m.K, walk_leaf_stride(m.K), m.loss, q.link,
                                        m.all_numeric ? 1 : 0, shape, static_cast<float *>(out));
    return launch_walk_rows(s, m.d_nodes, std::max(1, m.max_int), m.d_meta, m.d_leaf, m.d_cid, q.ntrees, x, n, n, q.F, m.wide, m.K, m.loss, q.link,
                            static_cast<float *>(out), nullptr, 0, 0);
}

template <typename T>
void widen(const T *src, uint32_t *dst, int64_t n) {
    for (int64_t i = 0; i < n; i++) dst[i] = src[i];
}

int run(Model &m, hipStream_t s, Request &q) {
    const int leaf_bytes = !q.leaf_out ? 0 : m.max_nodes <= 255 ? 1 : m.max_nodes <= 65535 ? 2 : 4;
    const int64_t back = q.leaf_out ? (int64_t)q.ntrees * leaf_bytes : (int64_t)m.K * 4; // bytes a row sends back
    const bool raw = q.plan && 64 * ((int64_t)q.src.esize() * q.F + back) <= (int64_t)PINNED_BYTES - 4096 && bins_by_device(q.src.dtype, q.N * q.F);
    const int64_t cell = raw ? (int64_t)q.src.esize() : 1, per_row = q.F * cell + back;
    // pieces of a twelfth of the whole, so that binning, copies and kernels overlap; 256 KB at least, a buffer at most.  Leaf ids: of a
    // fourth, so that as many as fit the buffers are spread out into the caller's words (most of the work) together at the end
    const int64_t goal = std::min<int64_t>((int64_t)PINNED_BYTES - 4096, std::max<int64_t>(256 << 10, q.N * per_row / (q.leaf_out ? 4 : 12)));
    ARGCHK(64 * per_row <= (int64_t)PINNED_BYTES - 4096, "too many trees for one piece");
    const int64_t rows_most = std::max<int64_t>(64, goal / per_row / 64 * 64);
    const bool rowwise = q.plan && q.src.rows_contiguous();
    const BinPieces B(q.N, q.F, rowwise, true, rows_most, 0);
    const int NS = (int)std::min<int64_t>(PinnedSlots::NS, B.np);
    const size_t xd = ((size_t)B.rows * q.F + 255) / 256 * 256;        // a piece's bins on the device
    const size_t xs = ((size_t)B.rows * q.F * cell + 255) / 256 * 256; // a pinned buffer holds them (or the values), then what comes back
    CallBuffer d_x; // bins of the pieces in flight
    DeviceBins D;
    PinnedSlots U(s);
    int r = U.init(NS);
    if (r != EVT_OK) return r;
    const bool direct = !raw && B.np == 1 && (int64_t)q.N * q.F <= 65536; // a few bins are read over the bus by the kernel itself
    if (!direct) {
        d_x.p = static_cast<uint8_t *>(dev_take(xd * NS));
        if (!d_x.p) return EVT_ERR_NOMEM;
        if (raw) r = D.init(s, *q.plan, xs, NS);
        if (r != EVT_OK) return r;
    }
    auto piece = [&](int64_t p, int64_t *r0, int64_t *n) {
        int f0, f1;
        B.at(p, r0, n, &f0, &f1);
    };
    auto fill = [&](int64_t p, int t) {
        uint8_t *h = static_cast<uint8_t *>(U.host[p % NS]);
        if (raw) {
            B.copy(q.src, p, t, h);
        } else if (q.plan) {
            B.bin(*q.plan, q.src, p, t, h);
        } else {
            int64_t r0, n;
            piece(p, &r0, &n);
            const int64_t b0 = (int64_t)(t % B.row_blocks) * B.block;
            const int f = t / B.row_blocks;
            if (b0 < n) memcpy(h + (size_t)f * n + b0, q.bins + (size_t)f * q.N + r0 + b0, (size_t)std::min(B.block, n - b0));
        }
    };
    auto send = [&](int64_t p) -> int {
        int64_t r0, n;
        piece(p, &r0, &n);
        uint8_t *h = static_cast<uint8_t *>(U.host[p % NS]);
        const uint8_t *x = h;
        if (!direct) {
            uint8_t *d = d_x.p + (p % NS) * xd;
            if (raw) {
                const int rb = D.send(s, (int)(p % NS), h, q.src, n, 0, q.F, d, n);
                if (rb != EVT_OK) return rb;
            } else {
                HIPCHK(hipMemcpyAsync(d, h, (size_t)n * q.F, hipMemcpyHostToDevice, s));
            }
            x = d;
        }
        const int rw = walk(m, s, q, x, n, h + xs, leaf_bytes); // the kernel writes what comes back over the bus itself
        if (rw != EVT_OK) return rw;
        if (!direct) HIPCHK(hipEventRecord(U.ev[p % NS], s));
        if (p == 0 && q.check) q.differ = !same_trees(m, *q.check);
        return EVT_OK;
    };
    auto retire = [&](int64_t p) {
        int64_t r0, n;
        piece(p, &r0, &n);
        const uint8_t *h = static_cast<const uint8_t *>(U.host[p % NS]) + xs;
        if (q.leaf_out) {
            hb_parallel(q.ntrees, hb_workers(n * q.ntrees / 2), [&](int t) {
                uint32_t *d = q.leaf_out + (size_t)t * q.N + r0;
                const size_t at = (size_t)t * n;
                if (leaf_bytes == 1) widen(h + at, d, n);
                else if (leaf_bytes == 2) widen(reinterpret_cast<const uint16_t *>(h) + at, d, n);
                else widen(reinterpret_cast<const uint32_t *>(h) + at, d, n);
            });
        } else {
            memcpy(q.out + (size_t)r0 * m.K, h, (size_t)n * m.K * 4);
        }
    };
    if (direct) {
        for (int t = 0; t < B.per_piece; t++) fill(0, t);
        r = send(0);
        if (r != EVT_OK) return r;
        HIPCHK(hipStreamSynchronize(s));
        U.idle = true;
        retire(0);
        return EVT_OK;
    }
    return run_pieces(U, NS, B.np, B.per_piece, hb_workers(q.plan ? q.N * q.F : q.N * q.F / 8), fill, send, retire);
}

} // namespace

extern "C" int evt_model_create(int32_t loss, int32_t K, void **out) {
    return guarded([&]() -> int {
    ARGCHK(out, "out is NULL");
    *out = nullptr;
    ARGCHK(K >= 1 && K <= EVT_MAX_K && loss >= 0 && loss <= EVT_LOSS_LAST, "invalid loss or number of outputs");
    int ndev = 0;
    const int r = evt_device_count(&ndev);
    if (r != EVT_OK) return r;
    std::unique_ptr<Model> m(new Model());
    m->loss = loss;
    m->K = K;
    Kept::get().add(m.get());
    *out = m.release();
    return EVT_OK;
    });
}
extern "C" int evt_model_destroy(void *model) {
    return guarded([&]() -> int {
    if (!model) return EVT_OK;
    Kept::get().remove(static_cast<Model *>(model));
    delete static_cast<Model *>(model);
    return EVT_OK;
    });
}

void models_trim() {
    Kept &k = Kept::get();
    std::lock_guard<std::mutex> lk(k.mu);
    k.shrink(0, nullptr);
}

extern "C" int evt_model_predict(void *model, int32_t n_model, const int64_t *nnodes, const int64_t *const *feat, const uint8_t *const *cond_bin,
                                 const float *const *pred, const uint8_t *const *split, const uint8_t *feattypes, int32_t nfeattypes,
                                 const double *const *edges, const int32_t *n_edges, const void *x, int32_t dtype, int64_t row_stride, int64_t col_stride,
                                 int64_t nobs, int32_t nfeats, int32_t ntrees, int32_t apply_link, float *out, uint32_t *leaf_out) {
    return guarded([&]() -> int {
    ARGCHK(model && nnodes && feat && cond_bin && pred && split && x, "NULL argument");
    ARGCHK(n_model >= 1 && ntrees >= 1 && ntrees <= n_model && nobs >= 1 && nfeats >= 1 && nfeats <= EVT_MAX_FEATS, "nobs, nfeats, ntrees must be >= 1");
    ARGCHK((out != nullptr) != (leaf_out != nullptr), "one of out and leaf_out");
    Model &m = *static_cast<Model *>(model);
    std::lock_guard<std::mutex> lock(m.mu);
    struct Used {
        Model *m;
        ~Used() { Kept::get().used(m); }
    } on_return{&m};
    CallStream call;
    HIPCHK(hipGetDevice(&call.device)); // the caller's, as for the whole-model calls
    if (m.device != call.device) m.drop();
    m.device = call.device;
    HIPCHK(stream_take(&call.s, true));
    const hipStream_t s = call.s;
    const TreePtrs t{n_model, nnodes, feat, cond_bin, split, pred};
    const size_t nft = feattypes ? (size_t)nfeattypes : 0;
    // The trees are compared with the device form while the device already walks it (20 us for 700 KB of trees); if they turn out to
    // have changed, the new ones are packed and the call runs again.
    bool known = m.feattypes.size() == nft && (!nft || !memcmp(m.feattypes.data(), feattypes, nft)) && same_shape(m, t) && m.max_feat <= nfeats;
    if (!known) {
        const int r = build(m, t, feattypes, nfeattypes, s);
        if (r != EVT_OK) return r;
    }
    auto walk_all = [&](Request &q) -> int {
        q.check = known ? &t : nullptr;
        q.differ = false;
        int r = run(m, s, q);
        if (r == EVT_OK && q.differ) {
            r = build(m, t, feattypes, nfeattypes, s);
            if (r != EVT_OK) return r;
            ARGCHK(m.max_feat <= nfeats, "tree feature id outside 1..nfeats");
            q.check = nullptr;
            r = run(m, s, q);
        }
        call.idle = r == EVT_OK;
        return r;
    };
    ARGCHK(m.max_feat <= nfeats, "tree feature id outside 1..nfeats");
    Request q{nullptr, {}, nullptr, nobs, nfeats, ntrees, apply_link, out, leaf_out, nullptr, false};
    if (!edges) {
        ARGCHK(dtype == EVT_U8, "a matrix of bins is EVT_U8");
        q.bins = static_cast<const uint8_t *>(x);
        return walk_all(q);
    }
    ARGCHK((dtype == EVT_F32 || dtype == EVT_F64) && (row_stride == 1 || col_stride == 1), "dtype must be EVT_F32 or EVT_F64 and one of the two strides 1");
    bool same = m.edge_off.size() == (size_t)nfeats + 1;
    for (int j = 0; j < nfeats; j++) {
        ARGCHK(edges[j] && n_edges[j] >= 1 && n_edges[j] <= 254, "each feature needs 1..254 edges");
        same = same && m.edge_off[j + 1] - m.edge_off[j] == n_edges[j] && !memcmp(m.edges.data() + m.edge_off[j], edges[j], 8 * (size_t)n_edges[j]);
    }
    if (!same) {
        m.plan[0].reset();
        m.plan[1].reset();
        m.edges.clear();
        m.edge_off.assign(1, 0);
        for (int j = 0; j < nfeats; j++) {
            m.edges.insert(m.edges.end(), edges[j], edges[j] + n_edges[j]);
            m.edge_off.push_back((int32_t)m.edges.size());
        }
    }
    std::unique_ptr<HbPlan> &plan = m.plan[dtype];
    if (!plan) {
        plan.reset(new HbPlan());
        plan->build(m.edges.data(), m.edge_off.data(), nfeats, dtype);
    }
    q.plan = plan.get();
    q.src = HbSource{x, dtype, row_stride, col_stride};
    return walk_all(q);
    });
}
