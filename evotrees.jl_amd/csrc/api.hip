// C ABI of libevotrees_hip.so: handle lifecycle, uploads, the per-tree level loop, read-back.
#include "grad_math.h"
#include "upload.h"
#include "walk_rule.h"

#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <memory>
#include <new>
#include <thread>

int launch_absmax_rows(evt_ctx *c, int k0, int k1);
int launch_check_unit_weight(evt_ctx *c);
int launch_predict_tree_nodes(evt_ctx *c, const uint32_t *nodes_dev, int nnodes, const float *leaf_pred_dev);
int launch_predict_model(hipStream_t s, const uint32_t *nodes, const float *leaf_pred, const int64_t *off, int ntrees, const uint8_t *xcm, int64_t N,
                         int K, int loss, int apply_link, float *out, const int32_t *skip_flag);
int predict_lds_shape(int F, int max_int, int K, int hint);
int launch_predict_model_lds(hipStream_t s, const uint32_t *cnodes, const float *cleaf, const void *meta, int ntrees, const uint8_t *xcm, int64_t N,
                             int F, int max_int, int K, int ks, int loss, int apply_link, int all_numeric, int shape, float *out);
int launch_leaf_idx_model(hipStream_t s, const uint32_t *nodes, const int64_t *off, int ntrees, const uint8_t *xcm, int64_t N, uint32_t *out);

static thread_local char g_err[512] = "";

void evt_set_error(const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

extern "C" const char *evt_last_error(void) { return g_err; }

extern "C" int evt_device_count(int32_t *count) {
    return guarded([&]() -> int {
    ARGCHK(count, "count is NULL");
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n <= 0) {
        *count = 0;
        evt_set_error("no HIP device: %s", hipGetErrorString(e));
        return EVT_ERR_HIP;
    }
    *count = n;
    return EVT_OK;
    });
}

// ---- profiling ------------------------------------------------------------------------------
void prof_begin(evt_ctx *c, int cls, int level) {
    c->prof_open = false;
    if (!((c->profiling >> cls) & 1)) return;
    c->prof_open = true;
    ProfRec r;
    r.cls = cls;
    r.level = level;
    r.seq = c->tree_seq;
    auto get = [&]() {
        hipEvent_t e;
        if (!c->free_events.empty()) {
            e = c->free_events.back();
            c->free_events.pop_back();
        } else {
            (void)hipEventCreateWithFlags(&e, hipEventDisableSystemFence);
        }
        return e;
    };
    r.e0 = get();
    r.e1 = get();
    (void)hipEventRecord(r.e0, c->stream);
    c->recs.push_back(r);
}
// Histogram launches carry their events themselves (hipExtLaunchKernelGGL: the timestamps of the kernel's own dispatch)
// instead of being bracketed by two event-record packets, which cost the stream about 5 us on each side of the kernel.
// The launcher takes c->launch_e0 / launch_e1 and records them one way or the other.
void prof_begin_launch(evt_ctx *c, int cls, int level) {
    c->launch_e0 = c->launch_e1 = nullptr;
    c->prof_open = false;
    if (!((c->profiling >> cls) & 1)) return;
    ProfRec r;
    r.cls = cls;
    r.level = level;
    r.seq = c->tree_seq;
    for (hipEvent_t *e : {&r.e0, &r.e1}) {
        if (!c->free_events.empty()) {
            *e = c->free_events.back();
            c->free_events.pop_back();
        } else {
            (void)hipEventCreateWithFlags(e, hipEventDisableSystemFence);
        }
    }
    c->recs.push_back(r);
    c->launch_e0 = r.e0;
    c->launch_e1 = r.e1;
}
void prof_end(evt_ctx *c) {
    if (!c->prof_open || c->recs.empty()) return;
    c->prof_open = false;
    (void)hipEventRecord(c->recs.back().e1, c->stream);
}
// after a stream sync or the arrival of tree `upto_seq`: fold finished event pairs into the per-class totals.  stats_host:
// the rows built per level of that tree, the units of its histogram launches; pairs of a tree queued behind it wait for
// their own tree's counts.
static void prof_collect(evt_ctx *c, const int64_t *stats_host, int64_t upto_seq = INT64_MAX) {
    std::vector<ProfRec> later; // pairs whose kernels are still queued (work placed behind the point the host waited for)
    for (auto &r : c->recs) {
        if (r.seq > upto_seq) {
            later.push_back(r);
            continue;
        }
        float ms = 0.0f;
        const hipError_t e = hipEventElapsedTime(&ms, r.e0, r.e1);
        if (e == hipErrorNotReady) {
            (void)hipGetLastError();
            later.push_back(r);
            continue;
        }
        if (e == hipSuccess) {
            c->prof_launches[r.cls] += 1;
            c->prof_ms[r.cls] += (double)ms;
            if (r.cls == EVT_K_HIST && stats_host && r.level >= 1) c->prof_units[r.cls] += stats_host[r.level];
        } else {
            (void)hipGetLastError();
        }
        c->free_events.push_back(r.e0);
        c->free_events.push_back(r.e1);
    }
    c->recs.swap(later);
}

template <typename T>
static int dev_alloc(T **p, size_t n) {
    *p = static_cast<T *>(dev_take(n * sizeof(T)));
    return *p ? EVT_OK : EVT_ERR_NOMEM;
}
#define ALLOC(ptr, n)                         \
    do {                                      \
        int _r = dev_alloc(&(ptr), (size_t)(n)); \
        if (_r != EVT_OK) {                   \
            evt_destroy(c);                   \
            return _r;                        \
        }                                     \
    } while (0)

static int record_stride(int F) {
    if (F <= 16) return 16;
    if (F <= 32) return 32;
    if (F <= 64) return 64;
    return ((F + 63) / 64) * 64;
}

// Piece layout of a record (evt_ctx::PBL, PU).  The conflict-free histogram kernel gives a row NS lanes, one per piece of
// 8, 4 or 2 bytes, and issues one LDS atomic instruction per byte position of a piece: when the features fill the
// record's last pieces only partly, ceil(F / pieces) features per piece use more of the lanes and take fewer instructions per row
// (100 features: 7 per piece over 15 lanes instead of 8 over 13).  Chosen when one block's LDS histogram takes the whole
// record for the largest channel count the loss can have (weights are only known later); densely packed otherwise.
static void record_layout(int F, int B, int na_max, int RS, int *PBL, int *PU) {
    *PBL = *PU = 1;
    if (RS < 32 || RS > 512) return;
    int tw = 32;
    while (tw < RS) tw <<= 1;
    const int pb = tw >= 128 ? 8 : (tw == 64 ? 4 : 2);
    const int ns = tw / pb;      // lanes per row
    const int pieces = RS / pb;  // of which the record fills this many
    const int pu = (F + pieces - 1) / pieces;
    if (pu >= pb || (size_t)na_max * B * ns * pu * 8 > 128 * 1024) return;
    *PBL = pb;
    *PU = pu;
}

static int ceil_log2_i64(int64_t v) {
    int b = 0;
    while (((int64_t)1 << b) < v) b++;
    return b;
}

extern "C" int evt_destroy(evt_handle c) {
    return guarded([&]() -> int {
    if (!c) return EVT_OK;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    void *ptrs[] = {c->xcm, c->xrm, c->y, c->pred, c->grad, c->grad_next, c->gq, c->is_a, c->is_b, c->nidx, c->mask, c->flagw, c->sample_claims, c->blob_arrived, c->chunk_nleft, c->chunk_lpre, c->cursor,
                    c->hist, c->seg_start, c->seg_len, c->status, c->node_sum, c->tree_blob, c->tree.packed, c->js, c->jsmap, c->feattypes, c->mono, c->absmax, c->qexp_buf[0], c->qexp_buf[1], c->qbits,
                    c->qscale_buf[0], c->qscale_buf[1], c->planes, c->metric_partial, c->errflag, c->ogains, c->sbest, c->scan_count, c->is_id, c->pt_nodes, c->mask_next,
                    c->small_nid[0], c->small_nid[1], c->small_head[0], c->small_head[1], c->small_left[0], c->small_left[1], c->small_acc,
                    c->alphas, c->alphas_f, c->qkeys_a, c->qkeys_b, c->qtemp};
    if (c->copy_stream) (void)hipStreamSynchronize(c->copy_stream);
    for (void *p : ptrs) dev_give(p);
    for (int l = 0; l < 2; l++) {
        LevelTab &L = c->lvl[l];
        void *lp[] = {L.hdr, L.act_node, L.cprefix, L.bnode, L.bstart, L.bprefix, L.cdesc};
        for (void *p : lp) dev_give(p);
    }
    coherent_give(c->h_stage_base);
    for (auto &r : c->recs) {
        (void)hipEventDestroy(r.e0);
        (void)hipEventDestroy(r.e1);
    }
    for (auto e : c->free_events) (void)hipEventDestroy(e);
    for (hipEvent_t e : c->tree_evs)
        if (e) (void)hipEventDestroy(e);
    pinned_give(c->pt_stage);
    if (c->copy_stream) stream_give(c->copy_stream, true, c->device);
    if (c->stream) stream_give(c->stream, false, c->device);
    delete c;
    return EVT_OK;
    });
}

// by way of the end of the pinned staging buffer, past what trees stage there
static hipError_t upload_alphas(evt_ctx *c) {
    double *ad = reinterpret_cast<double *>(c->h_stage_base + c->h_stage_bytes - 512);
    static_assert((sizeof(double) + sizeof(float)) * EVT_MAX_K <= 512, "the levels fit the slack of h_stage_bytes");
    float *af = reinterpret_cast<float *>(ad + EVT_MAX_K);
    for (int k = 0; k < EVT_MAX_K; k++) {
        ad[k] = c->h_alphas[k];
        af[k] = (float)c->h_alphas[k];
    }
    hipError_t e = hipMemcpyAsync(c->alphas, ad, sizeof(double) * EVT_MAX_K, hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(c->alphas_f, af, sizeof(float) * EVT_MAX_K, hipMemcpyHostToDevice, c->stream);
    return e;
}

// LDS channels: rows of the gradient matrix that need their own accumulator
static int n_channels(const evt_ctx *c, bool unit_w) { return (EVT_TWO_CHAN(c->loss, c->K) ? 1 : c->NK - 1) + (unit_w ? 0 : 1); }

extern "C" int evt_create(int64_t nobs, int32_t nfeats, int32_t nbins, int32_t K, int32_t max_depth, int32_t loss, int32_t tree_type,
                          evt_handle *out) {
    return guarded([&]() -> int {
    ARGCHK(out, "out handle is NULL");
    *out = nullptr;
    ARGCHK(nobs >= 1 && nobs <= (int64_t)0xFFFFFFFFll, "nobs must be in [1, 2^32-1]");
    ARGCHK(nfeats >= 1 && nfeats <= EVT_MAX_FEATS, "nfeats must be in [1, 65534]");
    ARGCHK(nbins >= 2 && nbins <= 255, "nbins must be in [2, 255]");
    ARGCHK(max_depth >= 1 && max_depth <= EVT_MAX_DEPTH, "max_depth must be in [1, 16]");
    ARGCHK(loss >= 0 && loss <= EVT_LOSS_LAST,
           "loss must be one of mse (0), logloss (1), gaussian_mle (2), poisson (3), gamma (4), tweedie (5), mlogloss (6), logistic_mle (7), mae (8), "
           "cred_var (9), cred_std (10), quantile (11), multiquantile (12)");
    ARGCHK(tree_type == EVT_TREE_BINARY || tree_type == EVT_TREE_OBLIVIOUS, "tree_type must be binary (0) or oblivious (1)");
    if (loss == EVT_LOSS_MLOGLOSS) ARGCHK(K >= 2 && K <= EVT_MAX_K, "mlogloss needs 2 <= K <= 16 classes");
    else if (EVT_IS_MLE2P(loss)) ARGCHK(K >= 2 && K <= EVT_MAX_K && K % 2 == 0, "gaussian_mle / logistic_mle need K = 2 x targets, 2 <= K <= 16");
    else ARGCHK(K >= 1 && K <= EVT_MAX_K, "K (targets) must be in [1, 16]");
    int ndev = 0;
    {
        int r = evt_device_count(&ndev);
        if (r != EVT_OK) return r;
    }
    evt_ctx *c = new (std::nothrow) evt_ctx();
    if (!c) {
        evt_set_error("out of host memory");
        return EVT_ERR_NOMEM;
    }
    memset((void *)&c->device, 0, sizeof(int));
    c->stream = nullptr;
    c->N = nobs; c->F = nfeats; c->B = nbins; c->K = K; c->NK = 2 * K + 1; c->D = max_depth; c->loss = loss; c->tree_type = tree_type;
    c->T = (loss == EVT_LOSS_MLOGLOSS || loss == EVT_LOSS_MULTIQUANTILE) ? 1 : (EVT_IS_MLE2P(loss) ? K / 2 : K);
    c->mc = (loss == EVT_LOSS_MLOGLOSS) || K > (EVT_IS_MLE2P(loss) ? 2 : 1);
    c->nnodes = (1 << max_depth) - 1;
    c->maxlvl = 1 << (max_depth - 1);
    c->RS = record_stride(nfeats);
    c->LPR = c->RS / 16;
    {
        // accumulator channels of one histogram launch at most: every gradient row and the weights, EVT_HIST_GROUP at a time
        // beyond EVT_MAX_NA (set_channels)
        const int na_all = EVT_TWO_CHAN(loss, K) ? 2 : 2 * K + 1;
        record_layout(nfeats, nbins, na_all <= EVT_MAX_NA ? na_all : EVT_HIST_GROUP, c->RS, &c->PBL, &c->PU);
    }
    c->unit_w = true;
    c->have_xbin = c->have_target = c->have_grads = false;
    c->planes = nullptr; c->plane_words = 0; c->planes_ready = false; c->use_planes = 1;
    c->xcm = nullptr; c->xrm = nullptr; c->y = nullptr; c->pred = nullptr; c->grad = nullptr; c->gq = nullptr; c->gq_words = 0; c->gq_rows = false;
    c->is_a = c->is_b = nullptr; c->nidx = nullptr; c->mask = nullptr; c->flagw = nullptr; c->sample_claims = nullptr; c->blob_arrived = nullptr; c->slot_ev[0] = c->slot_ev[1] = false; c->chunk_nleft = nullptr; c->chunk_lpre = nullptr; c->cursor = nullptr;
    c->hist = nullptr; c->seg_start = c->seg_len = nullptr; c->status = nullptr; c->node_sum = nullptr;
    memset(&c->tree, 0, sizeof(c->tree));
    c->tree_blob = nullptr;
    memset(c->lvl, 0, sizeof(c->lvl));
    c->js = nullptr; c->jsmap = nullptr; c->feattypes = nullptr; c->mono = nullptr; c->absmax = nullptr; c->absmax_cur = 0; c->absmax_other = 1; c->absmax_spare = 2; c->grad_next = nullptr; c->path_off = 0; c->metric_host = nullptr; c->metric_queued = false; c->slot_path[0] = c->slot_path[1] = false; c->qexp = nullptr; c->qbits = nullptr;
    c->alphas = nullptr; c->alphas_f = nullptr; c->qkeys_a = c->qkeys_b = nullptr; c->qtemp = nullptr; c->qtemp_bytes = 0;
    c->n_alphas = 1;
    for (int k = 0; k < EVT_MAX_K; k++) c->h_alphas[k] = 0.5;
    c->qscale = nullptr; c->qexp_buf[0] = c->qexp_buf[1] = nullptr; c->qscale_buf[0] = c->qscale_buf[1] = nullptr; c->q_cur = c->q_tree = 0; c->quant_pending = false;
    c->stats = nullptr; c->errflag = nullptr; c->ogains = nullptr; c->sbest = nullptr; c->scan_count = nullptr;
    c->h_stage = nullptr; c->h_stage_dev = nullptr; c->h_stage_bytes = 0; c->h_stage_base = nullptr; c->h_stage_dev_base = nullptr;
    c->n_js_last = 0;
    c->js_staged = false;
    c->last_all_rows = true;
    // one block of 16 waves per CU: as many waves as two blocks of 8 (the LDS histogram caps a CU at 128 KB), half
    // the flushes per node
    c->hist_blocks = 256;
    c->hist_threads = 1024;
    c->hist_min_rows = 1024;
    c->hist_variant = 0;
    c->hist_tile = 0;
    c->scan_fused = 1;
    c->hist_in_scatter = 1;
    c->part_one_pass = 1;
    c->small_tree = 1;
    c->small_acc = nullptr;
    for (int k = 0; k < 2; k++) {
        c->small_nid[k] = nullptr;
        c->small_head[k] = nullptr;
        c->small_left[k] = nullptr;
    }
    c->hist_seg_cost = 2048;
    c->record_nidx = false;
    c->nidx_valid = false;
    c->defer_pred = 1;
    c->write_nidx = false;
    c->pend_pred = false;
    c->is_id = nullptr;
    c->tree_in_flight = 0;
    c->slot_w = c->slot_r = 0;
    c->tree_seq = 0;
    c->slot_seq[0] = c->slot_seq[1] = 0;
    c->step.phase = 0;
    c->pt_nodes = nullptr; c->pt_stage = nullptr; c->pt_stage_dev = nullptr; c->pt_cap = 0; c->pt_busy = false;
    c->tree_evs[0] = c->tree_evs[1] = nullptr;
    c->mask_next = nullptr;
    c->copy_stream = nullptr;
    c->mask_next_valid = false;
    c->mask_seed_valid = false;
    c->mask_seed = 0;
    c->grads_ahead = false;
    c->grads_ready = false;
    c->last_cond = 255;
    c->profiling = 0;
    c->prof_open = false;
    c->launch_e0 = c->launch_e1 = nullptr;
    memset(c->prof_launches, 0, sizeof(c->prof_launches));
    memset(c->prof_ms, 0, sizeof(c->prof_ms));
    memset(c->prof_units, 0, sizeof(c->prof_units));
    hipError_t e = hipGetDevice(&c->device);
    if (e == hipSuccess) e = stream_take(&c->stream, false);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&c->tree_evs[0], hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&c->tree_evs[1], hipEventDisableTiming);
    if (e != hipSuccess) {
        evt_set_error("stream creation failed: %s", hipGetErrorString(e));
        if (c->stream) stream_give(c->stream, false, c->device);
        delete c;
        return EVT_ERR_HIP;
    }
    const int64_t N = nobs;
    const int NAgmax = c->NK; // upper bound over the weight modes
    c->max_chunks = (N + EVT_CHUNK - 1) / EVT_CHUNK + c->maxlvl + 2;
    ALLOC(c->xcm, (size_t)N * c->F);
    ALLOC(c->xrm, (size_t)N * c->RS);
    ALLOC(c->y, N * c->T);
    ALLOC(c->pred, (size_t)N * K);
    ALLOC(c->grad, (size_t)N * c->NK);
    c->gq_words = EVT_GQ_WORDS(N, n_channels(c, true)); // evt_set_target takes what weights need beside
    ALLOC(c->gq, c->gq_words);
    ALLOC(c->is_a, N);
    ALLOC(c->is_b, N);
    ALLOC(c->is_id, N);
    ALLOC(c->nidx, N);
    ALLOC(c->mask, N);
    ALLOC(c->sample_claims, 1);
    ALLOC(c->blob_arrived, 1);
    ALLOC(c->flagw, (size_t)c->max_chunks * EVT_CHUNK_WORDS);
    ALLOC(c->chunk_nleft, c->max_chunks + 1);
    ALLOC(c->chunk_lpre, c->max_chunks + 1);
    ALLOC(c->cursor, EVT_CURSOR_WORDS(c->nnodes));
    ALLOC(c->hist, (size_t)c->nnodes * c->F * NAgmax * c->B);
    ALLOC(c->seg_start, c->nnodes + 2);
    ALLOC(c->seg_len, c->nnodes + 2);
    ALLOC(c->status, c->nnodes + 2);
    ALLOC(c->node_sum, (size_t)(c->nnodes + 2) * NAgmax);
    {
        // the Tree arrays and the per-level row counts live in one allocation so that a finished tree is
        // read back with a single copy
        const size_t nn = (size_t)c->nnodes;
        c->blob_feat = 0;
        c->blob_w = c->blob_feat + nn * 4;
        c->blob_gain = c->blob_w + nn * 4;
        c->blob_pred = c->blob_gain + nn * 4;
        c->blob_stats = ((c->blob_pred + nn * 4 * K + 7) / 8) * 8;
        c->blob_bin = c->blob_stats + (size_t)(c->D + 2) * 8;
        c->blob_split = c->blob_bin + nn;
        c->blob_bytes = ((c->blob_split + nn + 15) / 16) * 16;
        ALLOC(c->tree_blob, c->blob_bytes);
        c->tree.feat = reinterpret_cast<int32_t *>(c->tree_blob + c->blob_feat);
        c->tree.w = reinterpret_cast<float *>(c->tree_blob + c->blob_w);
        c->tree.gain = reinterpret_cast<float *>(c->tree_blob + c->blob_gain);
        c->tree.pred = reinterpret_cast<float *>(c->tree_blob + c->blob_pred);
        c->stats = reinterpret_cast<int64_t *>(c->tree_blob + c->blob_stats);
        c->tree.cond_bin = c->tree_blob + c->blob_bin;
        c->tree.split = c->tree_blob + c->blob_split;
    }
    ALLOC(c->tree.packed, c->nnodes);
    for (int l = 0; l < 2; l++) {
        ALLOC(c->lvl[l].hdr, LH_SIZE);
        ALLOC(c->lvl[l].act_node, c->maxlvl + 2);
        ALLOC(c->lvl[l].cprefix, c->maxlvl + 2);
        ALLOC(c->lvl[l].bnode, c->maxlvl + 2);
        ALLOC(c->lvl[l].bstart, c->maxlvl + 2);
        ALLOC(c->lvl[l].bprefix, c->maxlvl + 2);
        ALLOC(c->lvl[l].cdesc, c->max_chunks + 1);
    }
    ALLOC(c->js, c->F);
    ALLOC(c->jsmap, c->RS);
    ALLOC(c->feattypes, c->F);
    ALLOC(c->mono, c->F);
    ALLOC(c->absmax, 3 * EVT_ABSMAX_STRIPES * EVT_MC_MAX_NK);
    ALLOC(c->alphas, EVT_MAX_K);
    ALLOC(c->alphas_f, EVT_MAX_K);
    for (int s = 0; s < 2; s++) {
        ALLOC(c->qexp_buf[s], EVT_MC_MAX_NK);
        ALLOC(c->qscale_buf[s], 2 * EVT_MC_MAX_NK);
    }
    c->qexp = c->qexp_buf[0];
    c->qscale = c->qscale_buf[0];
    ALLOC(c->qbits, EVT_MC_MAX_NK);
    ALLOC(c->metric_partial, 2 * EVT_METRIC_BLOCKS + 1);
    ALLOC(c->errflag, 1);
    if (tree_type == EVT_TREE_OBLIVIOUS) ALLOC(c->ogains, (size_t)c->maxlvl * c->F * c->B);
    {
        uint8_t *sb = nullptr;
        // one 64-byte candidate (ScanBestQ, kernels_scan.hip) per node and group of 4 features; oblivious: one of 16 bytes per block
        ALLOC(sb, std::max((size_t)c->maxlvl * ((c->F + 3) / 4) * 64, (size_t)EVT_OBLIV_BLOCKS * 16));
        c->sbest = sb;
        ALLOC(c->scan_count, (size_t)c->maxlvl * EVT_SCAN_COUNT_STEP);
    }
    // pinned staging: tree read-back + small per-tree uploads; coherent: wait_for_tree reads it while the kernel that fills it runs
    c->h_stage_bytes = c->blob_bytes + (size_t)c->F * 4 + (size_t)c->RS * 2 + 1024;
    c->h_stage_bytes = (c->h_stage_bytes + 255) / 256 * 256;
    if (!c->mc && tree_type != EVT_TREE_OBLIVIOUS && c->D >= 2 && c->D <= EVT_PATH_DEPTH) {
        c->path_off = c->h_stage_bytes;
        c->h_stage_bytes += ((size_t)c->nnodes * sizeof(PathNode) + 8 * EVT_PATH_BLOCKS + 255) / 256 * 256;
    }
    c->h_stage_base = c->h_stage_dev_base = static_cast<uint8_t *>(coherent_take(2 * c->h_stage_bytes + 192));
    if (!c->h_stage_base) {
        evt_destroy(c);
        return EVT_ERR_NOMEM;
    }
    for (int k = 0; k < 2; k++) { // behind the slots, a line each; trees count from 1
        c->slot_flag[k] = reinterpret_cast<unsigned long long *>(c->h_stage_base + 2 * c->h_stage_bytes + 64 * k);
        *c->slot_flag[k] = 0;
        if (c->path_off) memset(c->h_stage_base + k * c->h_stage_bytes + c->path_off + (size_t)c->nnodes * sizeof(PathNode), 0, 8 * EVT_PATH_BLOCKS);
    }
    c->metric_host = reinterpret_cast<double *>(c->h_stage_base + 2 * c->h_stage_bytes + 128);
    c->h_stage = c->h_stage_base;
    c->h_stage_dev = c->h_stage_dev_base;
    // defaults: all numeric, no monotone constraint; queued in stream order ahead of whatever reads them
    c->h_feattypes.assign(c->F, 1);
    c->h_mono.assign(c->F, 0);
    hipError_t e2 = hipMemsetAsync(c->feattypes, 1, c->F, c->stream);
    if (e2 == hipSuccess) e2 = hipMemsetAsync(c->mono, 0, sizeof(int32_t) * c->F, c->stream);
    if (e2 == hipSuccess) e2 = hipMemsetAsync(c->absmax, 0, sizeof(uint32_t) * 3 * EVT_ABSMAX_STRIPES * EVT_MC_MAX_NK, c->stream);
    if (e2 == hipSuccess) e2 = hipMemsetAsync(c->nidx, 0, sizeof(uint32_t) * N, c->stream);
    if (e2 == hipSuccess) e2 = hipMemsetAsync(c->errflag, 0, sizeof(int32_t), c->stream);
    if (e2 == hipSuccess) e2 = hipMemsetAsync(c->blob_arrived, 0, sizeof(int), c->stream);
    if (e2 == hipSuccess) e2 = hipMemsetAsync(c->sample_claims, 0, sizeof(unsigned long long), c->stream);
    if (e2 == hipSuccess) e2 = hipMemsetAsync(c->scan_count, 0, sizeof(int32_t) * EVT_SCAN_COUNT_STEP * c->maxlvl, c->stream);
    if (e2 == hipSuccess) e2 = hipMemsetAsync(c->metric_partial + 2 * EVT_METRIC_BLOCKS, 0, sizeof(double), c->stream);
    if (e2 == hipSuccess) e2 = upload_alphas(c);
    int r = EVT_OK;
    if (e2 == hipSuccess) r = launch_iota(c, c->is_id, N);
    if (r != EVT_OK || e2 != hipSuccess) {
        if (r == EVT_OK) evt_set_error("initial fills failed: %s", hipGetErrorString(e2));
        evt_destroy(c);
        return r != EVT_OK ? r : EVT_ERR_HIP;
    }
    *out = c;
    return EVT_OK;
    });
}

// every call on a handle but evt_grow_tree_end, evt_synchronize and evt_destroy waits for a tree begun with
// evt_grow_tree_begin to be collected: its arrays sit in the handle's staging buffer until then
#define CTXCHK(c)                                                                                      \
    do {                                                                                               \
        ARGCHK((c) != nullptr, "handle is NULL");                                                      \
        HIPCHK(hipSetDevice((c)->device));                                                             \
        if ((c)->tree_in_flight) {                                                                     \
            evt_set_error("a tree begun with evt_grow_tree_begin has not been collected (evt_grow_tree_end)"); \
            return EVT_ERR_STATE;                                                                      \
        }                                                                                              \
        if ((c)->step.phase != 0) {                                                                    \
            evt_set_error("a tree opened with evt_tree_open has not been closed (evt_tree_close)");    \
            return EVT_ERR_STATE;                                                                      \
        }                                                                                              \
    } while (0)
// calls that only queue work behind what is already queued (the next tree, the next gradient update, the next mask) are
// also allowed while ONE tree waits to be collected: two trees may be in flight, evt_grow_tree_end collects the older
#define CTXCHK_QUEUE(c)                                                                                \
    do {                                                                                               \
        ARGCHK((c) != nullptr, "handle is NULL");                                                      \
        HIPCHK(hipSetDevice((c)->device));                                                             \
        if ((c)->tree_in_flight > 1) {                                                                 \
            evt_set_error("two trees begun with evt_grow_tree_begin have not been collected (evt_grow_tree_end)"); \
            return EVT_ERR_STATE;                                                                      \
        }                                                                                              \
        if ((c)->step.phase != 0) {                                                                    \
            evt_set_error("a tree opened with evt_tree_open has not been closed (evt_tree_close)");    \
            return EVT_ERR_STATE;                                                                      \
        }                                                                                              \
    } while (0)
// calls that are also allowed between the stages of a tree opened with evt_tree_open
#define CTXCHK_STEP(c)                                                                                 \
    do {                                                                                               \
        ARGCHK((c) != nullptr, "handle is NULL");                                                      \
        HIPCHK(hipSetDevice((c)->device));                                                             \
        if ((c)->tree_in_flight) {                                                                     \
            evt_set_error("a tree begun with evt_grow_tree_begin has not been collected (evt_grow_tree_end)"); \
            return EVT_ERR_STATE;                                                                      \
        }                                                                                              \
    } while (0)

static int check_errflag(evt_ctx *c, const char *what) {
    int32_t f = 0;
    HIPCHK(hipMemcpyAsync(&f, c->errflag, sizeof(int32_t), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    if (f != 0) {
        HIPCHK(hipMemsetAsync(c->errflag, 0, sizeof(int32_t), c->stream));
        HIPCHK(hipStreamSynchronize(c->stream));
        evt_set_error("%s", what);
        return EVT_ERR_ARG;
    }
    return EVT_OK;
}

extern "C" int evt_set_xbin(evt_handle c, const uint8_t *x_bin_colmajor) {
    return guarded([&]() -> int {
    CTXCHK(c);
    ARGCHK(x_bin_colmajor, "x_bin is NULL");
    c->have_xbin = false;
    c->planes_ready = false;
    int ru = upload_bytes(c->stream, x_bin_colmajor, c->xcm, (size_t)c->N * c->F);
    if (ru != EVT_OK) return ru;
    int r = launch_transpose_validate(c);
    if (r != EVT_OK) return r;
    r = check_errflag(c, "x_bin holds values outside 1..nbins");
    if (r != EVT_OK) return r;
    c->have_xbin = true;
    return EVT_OK;
    });
}

// bins are in xcm: the records
static int bins_arrived(evt_ctx *c) {
    int r = launch_transpose_validate(c);
    if (r == EVT_OK) r = check_errflag(c, "binarize produced values outside 1..nbins");
    if (r != EVT_OK) return r;
    c->have_xbin = true;
    return EVT_OK;
}

extern "C" int evt_binarize(evt_handle c, const void *x, int32_t dtype, int64_t row_stride, int64_t col_stride, const double *edges,
                            const int32_t *edge_off) {
    return guarded([&]() -> int {
    CTXCHK(c);
    ARGCHK(x && edges && edge_off, "NULL argument");
    ARGCHK(dtype == EVT_F32 || dtype == EVT_F64, "dtype must be EVT_F32 or EVT_F64");
    ARGCHK(row_stride == 1 || col_stride == 1, "one of the two strides must be 1");
    for (int j = 0; j < c->F; j++) {
        const int ne = edge_off[j + 1] - edge_off[j];
        ARGCHK(ne >= 1 && ne <= c->B - 1 && edge_off[j] >= 0, "each feature needs 1..nbins-1 edges");
    }
    c->have_xbin = false;
    c->planes_ready = false;
    HbPlan P;
    P.build(edges, edge_off, c->F, dtype);
    const int r = upload_bins(c->stream, P, HbSource{x, dtype, row_stride, col_stride}, c->N, c->xcm, c->N);
    return r == EVT_OK ? bins_arrived(c) : r;
    });
}

extern "C" int evt_binarize_f64(evt_handle c, const double *x_colmajor, const double *edges, const int32_t *edge_off) {
    return guarded([&]() -> int {
    CTXCHK(c);
    ARGCHK(x_colmajor && edges && edge_off, "NULL argument");
    hipPointerAttribute_t attr;
    bool on_dev = (hipPointerGetAttributes(&attr, x_colmajor) == hipSuccess) && attr.type == hipMemoryTypeDevice;
    (void)hipGetLastError();
    // edge_off is read on the host to size the edges
    std::vector<int32_t> off(c->F + 1);
    HIPCHK(hipMemcpy(off.data(), edge_off, sizeof(int32_t) * (c->F + 1), hipMemcpyDefault));
    for (int j = 0; j < c->F; j++) {
        int ne = off[j + 1] - off[j];
        ARGCHK(ne >= 1 && ne <= c->B - 1 && off[j] >= 0, "each feature needs 1..nbins-1 edges");
    }
    if (!on_dev) {
        std::vector<double> ev(off[c->F]);
        HIPCHK(hipMemcpy(ev.data(), edges, sizeof(double) * off[c->F], hipMemcpyDefault));
        return evt_binarize(c, x_colmajor, EVT_F64, 1, c->N, ev.data(), off.data());
    }
    c->have_xbin = false;
    c->planes_ready = false;
    double *d_edges = nullptr;
    int32_t *d_off = nullptr;
    HIPCHK(hipMalloc((void **)&d_edges, sizeof(double) * std::max(1, off[c->F])));
    hipError_t e = hipMalloc((void **)&d_off, sizeof(int32_t) * (c->F + 1));
    if (e == hipSuccess) e = hipMemcpyAsync(d_edges, edges, sizeof(double) * off[c->F], hipMemcpyDefault, c->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(d_off, off.data(), sizeof(int32_t) * (c->F + 1), hipMemcpyHostToDevice, c->stream);
    int r = EVT_OK;
    if (e == hipSuccess) {
        r = launch_binarize(c->stream, x_colmajor, EVT_F64, 1, c->N, d_edges, d_off, c->B - 1, c->xcm, c->N, c->F, c->N);
        e = hipStreamSynchronize(c->stream);
    }
    if (d_off) (void)hipFree(d_off);
    if (d_edges) (void)hipFree(d_edges);
    if (r != EVT_OK) return r;
    if (e != hipSuccess) {
        evt_set_error("binarize failed: %s", hipGetErrorString(e));
        return EVT_ERR_HIP;
    }
    return bins_arrived(c);
    });
}

static void set_channels(evt_ctx *c) {
    int na = 0;
    if (EVT_TWO_CHAN(c->loss, c->K)) {
        c->chan_k[na++] = 0;                   // g ; h is derived (mse: 2w, mae: 0)
        if (!c->unit_w) c->chan_k[na++] = 2;   // w
    } else {
        for (int k = 0; k < c->NK - 1; k++) c->chan_k[na++] = k;
        if (!c->unit_w) c->chan_k[na++] = c->NK - 1;
    }
    c->NA = na;
    c->gq_rows = na > 1; // what the first tree most likely reads; no words are there yet
    for (int a = na; a < EVT_MC_MAX_NK; a++) c->chan_k[a] = 0;
    c->NAg = EVT_TWO_CHAN(c->loss, c->K) ? 2 : c->NK;
    int qbg = 62 - ceil_log2_i64(c->N);
    if (qbg > 40) qbg = 40;
    for (int k = 0; k < c->NK; k++) c->h_qbits[k] = qbg;
    if (c->unit_w) c->h_qbits[0] = EVT_PACK_QBITS;
    for (int k = c->NK; k < EVT_MC_MAX_NK; k++) c->h_qbits[k] = 0;
}

// The gradients' fixed-point words, where they were left to a tree that has not come
static int finish_quantize(evt_ctx *c) { return c->quant_pending ? launch_quantize(c) : EVT_OK; }

extern "C" int evt_set_target(evt_handle c, const float *y, const float *w, const float *mu, const float *offset) {
    return guarded([&]() -> int {
    CTXCHK(c);
    ARGCHK(y && mu, "y and mu must not be NULL");
    const int fin = finish_quantize(c); // as the channels stand
    if (fin != EVT_OK) return fin;
    c->have_target = false;
    c->have_grads = false;
    c->pend_pred = false; // the predictions start again from mu
    c->grads_ready = false;
    c->unit_w = (w == nullptr);
    set_channels(c);
    const size_t words = EVT_GQ_WORDS(c->N, c->NA);
    if (words > c->gq_words) { // no target, no tree: nobody reads the words that were there
        HIPCHK(hipStreamSynchronize(c->stream));
        dev_give(c->gq);
        c->gq_words = 0;
        c->gq = static_cast<unsigned long long *>(dev_take(words * sizeof(*c->gq)));
        if (!c->gq) return EVT_ERR_NOMEM;
        c->gq_words = words;
    }
    HIPCHK(hipMemcpyAsync(c->y, y, sizeof(float) * c->N * c->T, hipMemcpyDefault, c->stream));
    if (c->loss == EVT_LOSS_MLOGLOSS) {
        int r = launch_validate_classes(c);
        if (r != EVT_OK) return r;
        r = check_errflag(c, "mlogloss targets must be whole numbers in 1..K");
        if (r != EVT_OK) return r;
    }
    HIPCHK(hipMemcpyAsync(c->qbits, c->h_qbits, sizeof(int32_t) * EVT_MC_MAX_NK, hipMemcpyHostToDevice, c->stream));
    // stage w / offset through the (not yet needed) fixed-point buffer
    float *tmp = reinterpret_cast<float *>(c->gq);
    if (w) {
        HIPCHK(hipMemcpyAsync(tmp, w, sizeof(float) * c->N, hipMemcpyDefault, c->stream));
        int r = launch_set_weight_row(c, tmp);
        if (r != EVT_OK) return r;
    } else {
        int r = launch_set_weight_row(c, nullptr);
        if (r != EVT_OK) return r;
    }
    {
        int r = launch_absmax_rows(c, c->NK - 1, c->NK);
        if (r != EVT_OK) return r;
    }
    float *mu_dev = reinterpret_cast<float *>(c->metric_partial); // small scratch: thousands of doubles, K <= 16 floats needed
    HIPCHK(hipMemcpyAsync(mu_dev, mu, sizeof(float) * c->K, hipMemcpyDefault, c->stream));
    if (offset) {
        HIPCHK(hipStreamSynchronize(c->stream));
        HIPCHK(hipMemcpyAsync(tmp, offset, sizeof(float) * c->N * c->K, hipMemcpyDefault, c->stream));
        int r = launch_init_pred(c, mu_dev, tmp);
        if (r != EVT_OK) return r;
    } else {
        int r = launch_init_pred(c, mu_dev, nullptr);
        if (r != EVT_OK) return r;
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    c->have_target = true;
    return EVT_OK;
    });
}

extern "C" int evt_set_alphas(evt_handle c, const double *alphas, int32_t n) {
    return guarded([&]() -> int {
    CTXCHK(c);
    ARGCHK(alphas != nullptr, "alphas is NULL");
    if (c->loss == EVT_LOSS_MULTIQUANTILE) ARGCHK(n == c->K, "the multiquantile loss takes one level per output (n == K)");
    else ARGCHK(n == 1, "one level (n == 1) unless the loss is multiquantile");
    double a[EVT_MAX_K];
    HIPCHK(hipMemcpy(a, alphas, sizeof(double) * n, hipMemcpyDefault));
    for (int k = 0; k < n; k++) {
        ARGCHK(a[k] >= 0.0 && a[k] <= 1.0, "a quantile level must be in [0, 1]");
        ARGCHK(k == 0 || a[k] > a[k - 1], "quantile levels must be strictly increasing");
    }
    HIPCHK(hipStreamSynchronize(c->stream)); // kernels queued earlier read the old levels
    for (int k = 0; k < EVT_MAX_K; k++) c->h_alphas[k] = (k < n) ? a[k] : a[n - 1];
    c->n_alphas = n;
    HIPCHK(upload_alphas(c));
    HIPCHK(hipStreamSynchronize(c->stream));
    c->have_grads = false; // the gradients of the quantile losses depend on the levels
    c->grads_ready = false;
    return EVT_OK;
    });
}

extern "C" int evt_set_feature_meta(evt_handle c, const uint8_t *feattypes, const int32_t *monotone) {
    return guarded([&]() -> int {
    CTXCHK(c);
    std::vector<uint8_t> ft(c->F, 1);
    std::vector<int32_t> mo(c->F, 0);
    if (feattypes) HIPCHK(hipMemcpy(ft.data(), feattypes, c->F, hipMemcpyDefault));
    if (monotone) HIPCHK(hipMemcpy(mo.data(), monotone, sizeof(int32_t) * c->F, hipMemcpyDefault));
    for (int j = 0; j < c->F; j++) {
        ft[j] = ft[j] ? 1 : 0;
        ARGCHK(mo[j] >= -1 && mo[j] <= 1, "monotone constraints must be -1, 0 or 1");
        // the reference has no pred_scalar method for the multi-class loss (src/predict.jl:205-238): a constraint cannot be evaluated there
        ARGCHK(mo[j] == 0 || c->loss != EVT_LOSS_MLOGLOSS, "monotone constraints are not defined for mlogloss");
        ARGCHK(mo[j] == 0 || !EVT_IS_QUANTILE(c->loss), "monotone constraints are not defined for the quantile losses"); // no pred_scalar either
        // with several targets the reference's pred_scalar (src/predict.jl:205-208, :235-238) still reads the statistics at the
        // one-target positions, i.e. another target's gradient as the hessian: refused rather than reproduced
        ARGCHK(mo[j] == 0 || !c->mc, "monotone constraints are not defined for more than one target");
    }
    HIPCHK(hipMemcpy(c->feattypes, ft.data(), c->F, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(c->mono, mo.data(), sizeof(int32_t) * c->F, hipMemcpyHostToDevice));
    c->h_feattypes = ft;
    c->h_mono = mo;
    return EVT_OK;
    });
}

// Threshold bit planes for the partition, built before the first tree grown on the current x_bin.  They cost
// F * (B - 1) * N / 8 bytes: taken when that is at most 16 GiB and a third of the memory still free, skipped otherwise
// (the partition then gathers bin bytes).  A failed allocation is not an error.
static int ensure_planes(evt_ctx *c) {
    if (c->planes_ready || c->use_planes == 0 || c->D < 2) return EVT_OK;
    if (!c->planes) {
        if (c->use_planes < 0) return EVT_OK; // tried before, did not fit
        const int64_t W = (((c->N + 31) / 32) + 31) / 32 * 32;
        const size_t bytes = (size_t)c->F * (size_t)(c->B - 1) * (size_t)W * 4;
        size_t free_b = 0, total_b = 0;
        if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) free_b = 0;
        (void)hipGetLastError();
        if (bytes <= ((size_t)16 << 30) && bytes <= free_b / 3) c->planes = static_cast<uint32_t *>(dev_take(bytes));
        if (!c->planes) {
            (void)hipGetLastError();
            c->planes = nullptr;
            c->use_planes = -1;
            return EVT_OK;
        }
        c->plane_words = W;
    }
    const int r = launch_build_planes(c);
    if (r != EVT_OK) return r;
    c->planes_ready = true;
    return EVT_OK;
}

static int queue_grads(evt_ctx *c) {
    int r = finish_quantize(c); // the pass raises the maxima that the quantisation before it clears
    if (r != EVT_OK) return r;
    prof_begin(c, EVT_K_GRAD, 0);
    r = launch_grads(c);
    prof_end(c);
    if (r != EVT_OK) return r;
    if (c->profiling) c->prof_units[EVT_K_GRAD] += c->N;
    // a tree quantises on its way: inside its first kernel, or beside its set-up
    c->quant_pending = true;
    if (c->N <= EVT_QUANT_LATER) return EVT_OK;
    prof_begin(c, EVT_K_OTHER, 0);
    r = launch_quantize(c);
    prof_end(c);
    return r;
}

extern "C" int evt_update_grads(evt_handle c) {
    return guarded([&]() -> int {
    CTXCHK_QUEUE(c);
    if (!c->have_target) {
        evt_set_error("evt_set_target must be called before evt_update_grads");
        return EVT_ERR_STATE;
    }
    if (c->grads_ready) { // queued behind the last tree ("grads_ahead"): the predictions have not changed since
        c->grads_ready = false;
        c->have_grads = true;
        return EVT_OK;
    }
    const int r = queue_grads(c);
    if (r != EVT_OK) return r;
    c->have_grads = true;
    return EVT_OK;
    });
}

extern "C" int evt_set_grads(evt_handle c, const float *grad) {
    return guarded([&]() -> int {
    CTXCHK(c);
    ARGCHK(grad, "grad is NULL");
    if (!c->have_target) {
        evt_set_error("evt_set_target must be called before evt_set_grads");
        return EVT_ERR_STATE;
    }
    c->grads_ready = false;
    c->have_grads = false;
    int r = finish_quantize(c);
    if (r != EVT_OK) return r;
    HIPCHK(hipMemcpyAsync(c->grad, grad, sizeof(float) * (size_t)c->N * c->NK, hipMemcpyDefault, c->stream));
    if (c->unit_w) { // the target was set without weights: the row count stands for the weight, the weight row must say so
        r = launch_check_unit_weight(c);
        if (r == EVT_OK) r = check_errflag(c, "evt_set_grads: the weight row must be all ones when evt_set_target was given no weights");
        if (r != EVT_OK) return r;
    }
    r = launch_absmax_rows(c, 0, c->NK);
    if (r != EVT_OK) return r;
    r = launch_quantize(c);
    if (r != EVT_OK) return r;
    HIPCHK(hipStreamSynchronize(c->stream));
    c->have_grads = true;
    return EVT_OK;
    });
}

static int tree_open(evt_ctx *c, const uint8_t *mask, bool mask_staged, uint8_t cond, const uint32_t *js, int32_t n_js, const evt_params *p,
                     bool staged) {
    ARGCHK(js && p, "js and params must not be NULL");
    ARGCHK(n_js >= 1 && n_js <= c->F, "n_js must be in [1, nfeats]");
    ARGCHK(p->bagging_size >= 1, "bagging_size must be >= 1");
    ARGCHK(p->lambda >= 0 && p->gamma >= 0 && p->min_weight >= 0 && p->eta >= 0, "lambda, gamma, min_weight, eta must be >= 0");
    if (!c->have_xbin || !c->have_target || !c->have_grads) {
        evt_set_error("x_bin, target and gradients must be set before evt_grow_tree");
        return EVT_ERR_STATE;
    }
    // js: 1-based, strictly ascending
    std::vector<uint32_t> jsv(n_js);
    {
        hipPointerAttribute_t attr;
        const bool on_dev = (hipPointerGetAttributes(&attr, js) == hipSuccess) && attr.type == hipMemoryTypeDevice;
        (void)hipGetLastError();
        if (on_dev) HIPCHK(hipMemcpy(jsv.data(), js, sizeof(uint32_t) * n_js, hipMemcpyDeviceToHost));
        else memcpy(jsv.data(), js, sizeof(uint32_t) * n_js);
    }
    for (int i = 0; i < n_js; i++) {
        ARGCHK(jsv[i] >= 1 && jsv[i] <= (uint32_t)c->F, "js entries must be in 1..nfeats");
        ARGCHK(i == 0 || jsv[i] > jsv[i - 1], "js must be strictly ascending");
    }
    // LDS budget of one block: the channels of one launch x bins of a single feature must fit (more than EVT_MAX_NA
    // channels go EVT_HIST_GROUP per launch)
    ARGCHK((size_t)(c->NA <= EVT_MAX_NA ? c->NA : EVT_HIST_GROUP) * c->B * 8 <= 64 * 1024, "histogram of one feature exceeds the LDS budget");

    // the arguments are in order: the tree takes its staging slot (the one the tree collected last, or never used,
    // held) and its number in the profile
    c->h_stage = c->h_stage_base + (size_t)c->slot_w * c->h_stage_bytes;
    c->h_stage_dev = c->h_stage_dev_base + (size_t)c->slot_w * c->h_stage_bytes;
    c->tree_seq += 1;

    // rows kept by the mask (the host owns the RNG; src/subsample.jl:7-9).  The threshold, the count and the
    // compaction run on the device; the count comes back with the finished tree.
    const bool all_rows = (mask == nullptr && !mask_staged) || (cond == 255);
    c->grads_ready = false; // this tree changes the predictions
    c->last_all_rows = all_rows;
    c->last_cond = cond;
    const int small = staged ? 0 : small_tree_form(c, n_js, all_rows);
    int r = gq_layout(c, !small);
    if (r != EVT_OK) return r;
    if (c->quant_pending) {
        if (small ? small_root_quantises(c, small) : c->N <= EVT_QUANT_LATER) quant_set(c); // by the tree's first kernel
        else r = launch_quantize(c);
        if (r != EVT_OK) return r;
    }
    c->q_tree = c->q_cur; // this tree is grown on (and decoded with) the tables of the gradients quantised last
    // a tree grown in stages records the node of every row on the way, so that evt_get_nidx can show it after each stage
    // ... and so does a quantile loss: its leaves are valued from the rows they hold once the tree is complete
    const bool rec_nidx = c->record_nidx || staged || EVT_IS_QUANTILE(c->loss);
    c->nidx_valid = rec_nidx;

    // per-tree small uploads through pinned memory
    if (c->n_js_last != n_js || c->js_last != jsv || c->js_staged) { // the column sample changed: refresh the device copies
        uint32_t *h_js = reinterpret_cast<uint32_t *>(c->h_stage + c->blob_bytes);
        uint16_t *h_map = reinterpret_cast<uint16_t *>(c->h_stage + c->blob_bytes + (size_t)c->F * 4);
        for (int f = 0; f < c->RS; f++) h_map[f] = 0xFFFF;
        for (int i = 0; i < n_js; i++) {
            h_js[i] = jsv[i];
            const int f = (int)jsv[i] - 1;
            h_map[(f / c->PU) * c->PBL + f % c->PU] = (uint16_t)i;
        }
        // k_tree_begin reads them from the pinned buffer (this tree's staging slot, not written again before the tree has
        // been collected)
        c->js_staged = true;
        c->n_js_last = n_js;
        c->js_last = jsv;
    }

    // With every row in the tree the leaf of each row is recorded while growing and its value is added later, in row
    // order (fused into the next gradient pass): a scattered 4-byte write per row instead of a scattered read-modify-write.
    // (a quantile loss's leaf values do not exist before the tree is complete: always deferred)
    // ... or, with the next gradients, by walking the tree
    const bool walk = p->update_pred && all_rows && !small && !rec_nidx && (c->defer_pred == 2 || (c->defer_pred == 1 && walk_pays(c->N, c->F, c->n_js_last, c->D, c->tree_type == EVT_TREE_OBLIVIOUS))) && grads_with_tree(c, p);
    const bool defer = p->update_pred && all_rows && !walk && (c->defer_pred || EVT_IS_QUANTILE(c->loss));
    const bool fuse_pred = p->update_pred && all_rows && !walk && !defer;
    c->write_nidx = rec_nidx || defer;

    c->step.hist_fused = !staged && scatter_can_build_hist(c, n_js); // the set-up below cuts the root's chunks by it
    r = small ? EVT_OK : ensure_planes(c);
    if (r != EVT_OK) return r;
    if (EVT_IS_QUANTILE(c->loss)) {
        r = quantile_leaf_buffers(c);
        if (r != EVT_OK) return r;
    }
    prof_begin(c, EVT_K_OTHER, 0);
    r = launch_apply_pending(c); // an earlier tree's values go in before its node ids are overwritten
    if (r != EVT_OK) return r;
    bool draw = false;
    if (mask_staged) {
        if (c->mask_seed_valid) { // evt_draw_mask: the compaction pass below draws the bytes into the mask buffer
            draw = true;
            c->mask_seed_valid = false;
        } else { // uploaded by evt_stage_mask, which waited for the copy: the two buffers change places
            std::swap(c->mask, c->mask_next);
        }
        c->mask_next_valid = false;
    }
    if (!all_rows) {
        if (!mask_staged) {
            HIPCHK(hipMemcpyAsync(c->mask, mask, c->N, hipMemcpyDefault, c->stream));
            HIPCHK(hipStreamSynchronize(c->stream)); // the caller may reuse its mask buffer as soon as this call returns
        }
        if (!small) r = launch_compact_mask(c, cond, draw, c->mask_seed);
        if (r == EVT_OK && rec_nidx) r = launch_fill_u32(c, c->nidx, 0u, c->N);
    }
    if (r == EVT_OK && all_rows && !small) r = launch_tree_begin(c); // with a row sample the compaction above has set the tree up
    prof_end(c);
    if (r != EVT_OK) return r;

    c->step.all_rows = all_rows;
    c->step.defer = defer || (small && p->update_pred); // there rows outside the sample have a leaf too
    c->step.small = small;
    c->step.small_draw = draw;
    c->step.fuse_pred = fuse_pred;
    c->step.walk = walk;
    c->step.blob_sent = false;
    c->step.grads_done = false;
    c->step.p = *p;
    // the root's list is the identity (kept, never written) or what the mask compaction left in is_a; the levels below
    // alternate between is_a and is_b
    c->step.is_cur = all_rows ? c->is_id : c->is_a;
    c->step.is_next = all_rows ? c->is_a : c->is_b;
    c->step.level = 1;
    c->step.phase = 1;
    return EVT_OK;
}

// levels 1 .. D-1 split; the last of them sends its rows straight to the leaves of level D
static inline int tree_last_split(const evt_ctx *c) { return (c->D > 1) ? c->D - 1 : 1; }

// update_hist! for the build nodes of the level (src/fit-utils.jl:345-360)
static int tree_stage_hist(evt_ctx *c) {
    const int level = c->step.level;
    if (level > 1 && c->step.hist_fused) { // built by the scatter pass of the level above
        c->step.phase = 2;
        return EVT_OK;
    }
    prof_begin_launch(c, EVT_K_HIST, level);
    int r = launch_hist_build(c, level, c->step.is_cur);
    c->launch_e0 = c->launch_e1 = nullptr;
    if (r != EVT_OK) return r;
    c->step.phase = 2;
    return EVT_OK;
}

// subtract_hist!, _scan_node!/get_best_split (update_gains! and the level's choice for oblivious trees), child sums and
// leaf values for the active nodes of the level (src/fit-utils.jl:321-332, :403-486; src/fit.jl:190-217)
static int tree_stage_scan(evt_ctx *c) {
    const int level = c->step.level, last_split = tree_last_split(c);
    const evt_params *p = &c->step.p;
    const bool obliv = (c->tree_type == EVT_TREE_OBLIVIOUS);
    int r;
    prof_begin(c, EVT_K_SCAN, level);
    if (c->D == 1) {
        r = launch_scan(c, 1, p, true); // a stump: the root is the only leaf
    } else {
        r = launch_scan(c, level, p, false);
        if (r == EVT_OK && obliv) r = launch_obliv_select(c, level, p);
        if (r == EVT_OK && level == last_split && !scan_folds_leaves(c)) r = launch_scan(c, c->D, p, true); // leaf values of level D
    }
    prof_end(c);
    if (r != EVT_OK) return r;
    c->step.phase = 3;
    return EVT_OK;
}

// split_set! / update_nodes_idx!: the rows of every split node move to its children (src/fit-utils.jl:93-132,
// ext/.../fit-utils.jl:9-31)
static int tree_stage_partition(evt_ctx *c) {
    const int level = c->step.level, last_split = tree_last_split(c);
    uint32_t *is_cur = c->step.is_cur, *is_next = c->step.is_next;
    int r;
    prof_begin(c, EVT_K_PARTITION, level);
    if (level < last_split) {
        r = launch_part_count(c, level, is_cur);
        if (r == EVT_OK) r = launch_part_scatter(c, level, is_cur, is_next, c->step.fuse_pred);
    } else {
        // the tree's last kernel unless its leaves are still to be valued (quantile losses) or the rows outside the sample
        // are still to be predicted: the finished tree's transfer to the host rides along
        const bool last_kernel = !EVT_IS_QUANTILE(c->loss) && !(c->step.p.update_pred && (!c->step.all_rows || c->step.walk));
        r = launch_final_fused(c, level, is_cur, c->step.fuse_pred, last_kernel);
    }
    prof_end(c);
    if (r != EVT_OK) return r;
    if (is_cur == c->is_id) {
        c->step.is_cur = is_next;
        c->step.is_next = c->is_b;
    } else {
        std::swap(c->step.is_cur, c->step.is_next);
    }
    if (level < last_split) {
        c->step.level = level + 1;
        c->step.phase = 1;
    } else {
        c->step.phase = 4;
    }
    return EVT_OK;
}

static int tree_close(evt_ctx *c) {
    const evt_params *p = &c->step.p;
    const bool all_rows = c->step.all_rows, defer = c->step.defer;
    int r;
    c->step.phase = 0;
    if (EVT_IS_QUANTILE(c->loss)) { // pred_leaf_cpu! of the quantile losses: every leaf's value from the residuals of its rows
        prof_begin(c, EVT_K_OTHER, 0);
        r = launch_quantile_leaves(c, p);
        prof_end(c);
        if (r != EVT_OK) return r;
    }
    if (p->update_pred && (!all_rows || c->step.walk) && !c->step.small) {
        // rows outside the sample are predicted too (src/fit.jl:37): walk the new tree for all rows
        prof_begin(c, EVT_K_PREDICT, 0);
        r = launch_predict_tree_cache(c, true, grads_with_tree(c, p)); // with the tree's transfer to the host in its last blocks
        prof_end(c);
        if (r != EVT_OK) return r;
        if (c->profiling) c->prof_units[EVT_K_PREDICT] += c->N;
    }
    if (defer) {
        c->pend_pred = !c->step.grads_done; // the gradient pass adds them
        c->nidx_valid = all_rows; // with a row sample the recorded leaves are those of all rows
    }

    // the tree (and the per-level row counts) comes back in one pinned transfer, queued behind the kernels
    if (!c->step.blob_sent) {
        r = launch_copy_to_host(c, true);
        if (r != EVT_OK) return r;
    }
    c->slot_path[c->slot_w] = c->step.small == SMALL_PATH;
    c->slot_ev[c->slot_w] = c->profiling != 0; // the times of all its kernels are read when it is collected
    if (c->profiling) HIPCHK(hipEventRecord(c->tree_evs[c->slot_w], c->stream));
    c->slot_seq[c->slot_w] = c->tree_seq;
    if (c->grads_ahead && p->update_pred && p->bagging_size == 1) {
        // the next round's gradient update runs while the host collects this tree and prepares the next call.  Not with
        // bagging: the trees of one round are all grown on the same gradients (src/fit.jl:9-11), and the library cannot
        // tell which call is the round's last.
        if (c->step.grads_done) { // by the tree's last kernel
            c->quant_pending = true;
            if (c->N > EVT_QUANT_LATER) r = launch_quantize(c);
        } else {
            r = queue_grads(c);
        }
        if (r != EVT_OK) return r;
        c->grads_ready = true;
    }
    c->tree_in_flight += 1;
    c->slot_w ^= 1;
    return EVT_OK;
}


static int tree_fail(evt_ctx *c, int r) { // a failed stage leaves no tree open
    c->step.phase = 0;
    return r;
}

// every stage of an opened tree, then the close: what evt_grow_tree_begin queues
static int tree_run_stages(evt_ctx *c, int r) {
    if (r == EVT_OK && c->step.small) {
        r = c->step.small == SMALL_PATH ? launch_small_path(c, &c->step.p, c->step.small_draw) : launch_small_tree(c, &c->step.p, c->step.small_draw, c->step.small);
        c->step.phase = 4;
    }
    while (r == EVT_OK && c->step.phase != 4) {
        r = tree_stage_hist(c);
        if (r == EVT_OK) r = tree_stage_scan(c);
        if (r == EVT_OK) r = tree_stage_partition(c);
    }
    if (r != EVT_OK) return tree_fail(c, r);
    return tree_close(c);
}

extern "C" int evt_grow_tree_begin(evt_handle c, const uint8_t *mask, uint8_t cond, const uint32_t *js, int32_t n_js, const evt_params *p) {
    return guarded([&]() -> int {
    CTXCHK_QUEUE(c);
    int r = tree_open(c, mask, false, cond, js, n_js, p, false);
    return tree_run_stages(c, r);
    });
}

// The next tree's mask, uploaded while this one grows: the copy runs on a stream of its own, into the buffer the tree
// in flight does not read.
extern "C" int evt_stage_mask(evt_handle c, const uint8_t *mask) {
    return guarded([&]() -> int {
    ARGCHK(c != nullptr, "handle is NULL");
    ARGCHK(mask != nullptr, "mask is NULL");
    HIPCHK(hipSetDevice(c->device));
    if (c->step.phase != 0) {
        evt_set_error("a tree opened with evt_tree_open has not been closed (evt_tree_close)");
        return EVT_ERR_STATE;
    }
    if (c->tree_in_flight > 1) { // the older tree may still be reading the buffer this copy would overwrite
        evt_set_error("evt_stage_mask with two trees in flight: collect the older one first (evt_grow_tree_end)");
        return EVT_ERR_STATE;
    }
    if (!c->copy_stream) HIPCHK(stream_take(&c->copy_stream, true));
    if (!c->mask_next) {
        int r = dev_alloc(&c->mask_next, (size_t)c->N);
        if (r != EVT_OK) return r;
    }
    c->mask_next_valid = false;
    c->mask_seed_valid = false; // an uploaded mask replaces a seed given before
    HIPCHK(hipMemcpyAsync(c->mask_next, mask, c->N, hipMemcpyDefault, c->copy_stream));
    HIPCHK(hipStreamSynchronize(c->copy_stream)); // the caller may reuse its buffer; the tree in flight keeps running
    c->mask_next_valid = true;
    return EVT_OK;
    });
}

// The next tree's mask drawn by the device from a 64-bit seed (no nobs-byte draw on the host, no upload): written on
// the handle's own stream into the buffer the tree in flight does not read.
extern "C" int evt_draw_mask(evt_handle c, uint64_t seed) {
    return guarded([&]() -> int {
    CTXCHK_QUEUE(c);
    // nothing is queued here: the bytes are drawn by the next staged tree's compaction pass, which writes them into the
    // mask buffer on its way (in stream order behind whatever still reads that buffer)
    c->mask_seed = (unsigned long long)seed;
    c->mask_seed_valid = true;
    c->mask_next_valid = true;
    return EVT_OK;
    });
}

extern "C" int evt_grow_tree_begin_staged(evt_handle c, uint8_t cond, const uint32_t *js, int32_t n_js, const evt_params *p) {
    return guarded([&]() -> int {
    CTXCHK_QUEUE(c);
    if (!c->mask_next_valid) {
        evt_set_error("evt_grow_tree_begin_staged: no mask has been staged since the last tree (evt_stage_mask / evt_draw_mask)");
        return EVT_ERR_STATE;
    }
    int r = tree_open(c, nullptr, true, cond, js, n_js, p, false);
    return tree_run_stages(c, r);
    });
}

extern "C" int evt_tree_open(evt_handle c, const uint8_t *mask, uint8_t cond, const uint32_t *js, int32_t n_js, const evt_params *p) {
    return guarded([&]() -> int {
    CTXCHK(c);
    int r = tree_open(c, mask, false, cond, js, n_js, p, true);
    if (r != EVT_OK) return tree_fail(c, r);
    return EVT_OK;
    });
}

static int stage_check(evt_ctx *c, int phase, int32_t level, const char *name) {
    if (c->step.phase == 0) {
        evt_set_error("%s: no tree is open (evt_tree_open)", name);
        return EVT_ERR_STATE;
    }
    if (c->step.phase != phase || c->step.level != level) {
        static const char *const what[] = {"", "evt_hist_build", "evt_split_scan", "evt_update_nodes_idx", "evt_tree_close"};
        evt_set_error("%s(level %d) out of order: the open tree expects %s%s%d%s", name, (int)level, what[c->step.phase],
                      c->step.phase == 4 ? "" : "(level ", c->step.phase == 4 ? 0 : c->step.level, c->step.phase == 4 ? "" : ")");
        return EVT_ERR_STATE;
    }
    return EVT_OK;
}

extern "C" int evt_hist_build(evt_handle c, int32_t level) {
    return guarded([&]() -> int {
    CTXCHK_STEP(c);
    int r = stage_check(c, 1, level, "evt_hist_build");
    if (r != EVT_OK) return r;
    r = tree_stage_hist(c);
    return r == EVT_OK ? r : tree_fail(c, r);
    });
}

extern "C" int evt_split_scan(evt_handle c, int32_t level) {
    return guarded([&]() -> int {
    CTXCHK_STEP(c);
    int r = stage_check(c, 2, level, "evt_split_scan");
    if (r != EVT_OK) return r;
    r = tree_stage_scan(c);
    return r == EVT_OK ? r : tree_fail(c, r);
    });
}

extern "C" int evt_update_nodes_idx(evt_handle c, int32_t level) {
    return guarded([&]() -> int {
    CTXCHK_STEP(c);
    int r = stage_check(c, 3, level, "evt_update_nodes_idx");
    if (r != EVT_OK) return r;
    r = tree_stage_partition(c);
    return r == EVT_OK ? r : tree_fail(c, r);
    });
}

extern "C" int evt_tree_close(evt_handle c) {
    return guarded([&]() -> int {
    CTXCHK_STEP(c);
    if (c->step.phase != 4) {
        evt_set_error(c->step.phase == 0 ? "evt_tree_close: no tree is open" : "evt_tree_close before the last level was partitioned");
        return EVT_ERR_STATE;
    }
    return tree_close(c);
    });
}

// host copy of the device's tree arrays (in the pinned staging buffer) -> the caller's arrays
static int fill_tree_out(evt_ctx *c, const uint8_t *hs, evt_tree_out *tree) {
    ARGCHK(tree->feat && tree->cond_bin && tree->w && tree->gain && tree->pred && tree->split, "tree output arrays must not be NULL");
    const int nn = c->nnodes, K = c->K;
    const int32_t *f32 = reinterpret_cast<const int32_t *>(hs + c->blob_feat);
    for (int n = 0; n < nn; n++) tree->feat[n] = (int64_t)f32[n];
    memcpy(tree->w, hs + c->blob_w, (size_t)nn * 4);
    memcpy(tree->gain, hs + c->blob_gain, (size_t)nn * 4);
    memcpy(tree->pred, hs + c->blob_pred, (size_t)nn * 4 * K);
    memcpy(tree->cond_bin, hs + c->blob_bin, nn);
    memcpy(tree->split, hs + c->blob_split, nn);
    return EVT_OK;
}

// ... and of a tree of one launch
static int fill_tree_out(evt_ctx *c, const PathNode *nodes, evt_tree_out *tree) {
    ARGCHK(tree->feat && tree->cond_bin && tree->w && tree->gain && tree->pred && tree->split, "tree output arrays must not be NULL");
    for (int n = 0; n < c->nnodes; n++) {
        const PathNode v = nodes[n];
        tree->feat[n] = v.feat;
        tree->cond_bin[n] = (uint8_t)v.cond_bin;
        tree->w[n] = v.w;
        tree->gain[n] = v.gain;
        tree->split[n] = (uint8_t)v.split;
        for (int k = 0; k < c->K; k++) tree->pred[(size_t)c->K * n + k] = v.pred[k];
    }
    return EVT_OK;
}

static inline void spin_pause() {
#if defined(__x86_64__)
    __builtin_ia32_pause();
#endif
}

// Until a slot's tree has arrived; work queued behind it, and what else its last kernel does, may still be running.  The device writes the tree's number
// behind its arrays; a stream that has failed, or run dry without, is found out by asking it now and then.
static int wait_for_tree(evt_ctx *c, int slot) {
    if (c->slot_ev[slot]) {
        HIPCHK(hipEventSynchronize(c->tree_evs[slot]));
        return EVT_OK;
    }
    const unsigned long long seq = (unsigned long long)c->slot_seq[slot];
    const bool path = c->slot_path[slot];
    const unsigned long long *flags =
        path ? reinterpret_cast<const unsigned long long *>(c->h_stage_base + (size_t)slot * c->h_stage_bytes + c->path_off + (size_t)c->nnodes * sizeof(PathNode)) : c->slot_flag[slot];
    int seen = 0;
    const int words = path ? 1 << (c->D - 2) : 1;
    auto there = [&]() {
        while (seen < words && __atomic_load_n(flags + seen, __ATOMIC_ACQUIRE) == seq) seen++;
        return seen == words;
    };
    for (int k = 0; k < 4096; k++) {
        if (there()) return EVT_OK;
        spin_pause();
    }
    auto asked = std::chrono::steady_clock::now();
    while (!there()) {
        std::this_thread::yield();
        const auto now = std::chrono::steady_clock::now();
        if (now - asked < std::chrono::milliseconds(200)) continue;
        asked = now;
        const hipError_t q = hipStreamQuery(c->stream);
        if (q == hipErrorNotReady) {
            (void)hipGetLastError();
        } else if (q != hipSuccess) {
            HIPCHK(q);
        } else if (!there()) {
            evt_set_error("internal: a tree's kernels have ended without it");
            return EVT_ERR_INTERNAL;
        }
    }
    return EVT_OK;
}

extern "C" int evt_grow_tree_end(evt_handle c, evt_tree_out *tree) {
    return guarded([&]() -> int {
    ARGCHK(c != nullptr, "handle is NULL");
    HIPCHK(hipSetDevice(c->device));
    if (!c->tree_in_flight) {
        evt_set_error("evt_grow_tree_end without evt_grow_tree_begin");
        return EVT_ERR_STATE;
    }
    // the older of the trees in flight
    const int slot = c->slot_r;
    c->tree_in_flight -= 1;
    c->slot_r ^= 1;
    const uint8_t *hs = c->h_stage_base + (size_t)slot * c->h_stage_bytes;
    const size_t o_stats = c->blob_stats;
    const int arrived = wait_for_tree(c, slot);
    if (arrived != EVT_OK) return arrived;
    const bool path = c->slot_path[slot];
    const PathNode *nodes = reinterpret_cast<const PathNode *>(hs + c->path_off);
    int64_t n_is = path ? nodes[0].rows : reinterpret_cast<const int64_t *>(hs + o_stats)[0];
    if (c->profiling || !c->recs.empty()) {
        if (c->profiling) c->prof_units[EVT_K_PARTITION] += n_is;
        int64_t rows[EVT_MAX_DEPTH + 2] = {n_is}; // of the levels
        for (int n = 1; path && n <= c->nnodes; n++) rows[32 - __builtin_clz((unsigned)n)] += nodes[n - 1].rows;
        prof_collect(c, path ? rows : reinterpret_cast<const int64_t *>(hs + o_stats), c->slot_seq[slot]);
    }
    if (n_is == 0) { // the tree grown on no rows is a single zero leaf; report it as the reference does
        evt_set_error("no subsample observation - choose larger rowsample");
        return EVT_ERR_EMPTY;
    }
    if (tree) return path ? fill_tree_out(c, nodes, tree) : fill_tree_out(c, hs, tree);
    return EVT_OK;
    });
}

// The tree arrays as they stand on the device, e.g. between the stages of a tree opened with evt_tree_open.
extern "C" int evt_peek_tree(evt_handle c, evt_tree_out *tree) {
    return guarded([&]() -> int {
    CTXCHK_STEP(c);
    ARGCHK(tree, "tree is NULL");
    int r = launch_copy_to_host(c, false);
    if (r != EVT_OK) return r;
    HIPCHK(hipStreamSynchronize(c->stream));
    return fill_tree_out(c, c->h_stage, tree);
    });
}

extern "C" int evt_grow_tree(evt_handle c, const uint8_t *mask, uint8_t cond, const uint32_t *js, int32_t n_js, const evt_params *p,
                             evt_tree_out *tree) {
    return guarded([&]() -> int {
    const int r = evt_grow_tree_begin(c, mask, cond, js, n_js, p);
    if (r != EVT_OK) return r;
    return evt_grow_tree_end(c, tree);
    });
}

// host tree -> packed device nodes; validates that every split node has both children in range
static int pack_tree(int32_t nn, const int64_t *feat, const uint8_t *cond_bin, const uint8_t *split, int F, const uint8_t *feattypes,
                     std::vector<uint32_t> &out) {
    out.assign(nn, 0u);
    for (int n = 1; n <= nn; n++) {
        if (split[n - 1]) {
            ARGCHK(2 * n + 1 <= nn, "split node without children inside the tree arrays");
            ARGCHK(feat[n - 1] >= 1 && feat[n - 1] <= F, "tree feature id outside 1..nfeats");
            out[n - 1] = evt_pack_node((int)feat[n - 1], cond_bin[n - 1], feattypes == nullptr || feattypes[feat[n - 1] - 1] != 0);
        }
    }
    return EVT_OK;
}

extern "C" int evt_predict_tree(evt_handle c, int32_t nnodes_tree, const int64_t *feat, const uint8_t *cond_bin, const float *pred,
                                const uint8_t *split) {
    return guarded([&]() -> int {
    CTXCHK(c);
    ARGCHK(feat && cond_bin && pred && split && nnodes_tree >= 1, "NULL tree arrays");
    if (!c->have_xbin || !c->have_target) {
        evt_set_error("x_bin and target must be set before evt_predict_tree");
        return EVT_ERR_STATE;
    }
    std::vector<uint32_t> nodes;
    int r = pack_tree(nnodes_tree, feat, cond_bin, split, c->F, c->h_feattypes.data(), nodes);
    if (r != EVT_OK) return r;
    r = launch_apply_pending(c);
    if (r != EVT_OK) return r;
    c->grads_ready = false; // the predictions change
    const size_t nn = (size_t)nnodes_tree;
    if (c->pt_busy) { // the last tree's upload must have been read before the pinned buffer is written again
        HIPCHK(hipStreamSynchronize(c->stream));
        c->pt_busy = false;
    }
    if (c->pt_cap < nn) { // device copies and upload buffer are kept between calls and grown on demand
        HIPCHK(hipStreamSynchronize(c->stream));
        dev_give(c->pt_nodes);
        pinned_give(c->pt_stage);
        c->pt_nodes = nullptr; c->pt_stage = nullptr; c->pt_stage_dev = nullptr; c->pt_cap = 0;
        const size_t cap = std::max(nn, (size_t)2047);
        c->pt_nodes = static_cast<uint32_t *>(dev_take(sizeof(uint32_t) * cap * (1 + c->K)));
        c->pt_stage = c->pt_stage_dev = static_cast<uint8_t *>(pinned_take(sizeof(uint32_t) * cap * (1 + c->K)));
        if (!c->pt_nodes || !c->pt_stage) return EVT_ERR_NOMEM;
        c->pt_cap = cap;
    }
    memcpy(c->pt_stage, nodes.data(), sizeof(uint32_t) * nn);
    memcpy(c->pt_stage + sizeof(uint32_t) * nn, pred, sizeof(float) * nn * c->K);
    r = launch_copy_words(c, c->pt_stage_dev, c->pt_nodes, sizeof(uint32_t) * nn * (1 + c->K)); // the leaf values behind the nodes
    if (r != EVT_OK) return r;
    c->pt_busy = true;
    prof_begin(c, EVT_K_PREDICT, 0);
    r = launch_predict_tree_nodes(c, c->pt_nodes, nnodes_tree, reinterpret_cast<const float *>(c->pt_nodes + nn));
    prof_end(c);
    if (r != EVT_OK) return r;
    if (c->profiling) {
        HIPCHK(hipStreamSynchronize(c->stream));
        c->pt_busy = false;
        c->prof_units[EVT_K_PREDICT] += c->N;
        prof_collect(c, nullptr);
    }
    return EVT_OK;
    });
}

extern "C" int evt_get_xbin(evt_handle c, uint8_t *out) {
    return guarded([&]() -> int {
    CTXCHK(c);
    ARGCHK(out, "out is NULL");
    if (!c->have_xbin) {
        evt_set_error("x_bin has not been set");
        return EVT_ERR_STATE;
    }
    HIPCHK(hipMemcpyAsync(out, c->xcm, (size_t)c->N * c->F, hipMemcpyDefault, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return EVT_OK;
    });
}
extern "C" int evt_get_pred(evt_handle c, float *out) {
    return guarded([&]() -> int {
    CTXCHK(c);
    ARGCHK(out, "out is NULL");
    {
        int r = launch_apply_pending(c);
        if (r != EVT_OK) return r;
    }
    HIPCHK(hipMemcpyAsync(out, c->pred, sizeof(float) * (size_t)c->N * c->K, hipMemcpyDefault, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return EVT_OK;
    });
}
extern "C" int evt_get_grads(evt_handle c, float *out) {
    return guarded([&]() -> int {
    CTXCHK(c);
    ARGCHK(out, "out is NULL");
    HIPCHK(hipMemcpyAsync(out, c->grad, sizeof(float) * (size_t)c->N * c->NK, hipMemcpyDefault, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return EVT_OK;
    });
}
extern "C" int evt_get_nidx(evt_handle c, uint32_t *out) {
    return guarded([&]() -> int {
    CTXCHK_STEP(c);
    ARGCHK(out, "out is NULL");
    if (c->n_js_last <= 0) {
        evt_set_error("no tree has been grown yet");
        return EVT_ERR_STATE;
    }
    if (c->step.phase >= 1 && c->step.phase <= 3) { // a tree in stages: rows still on their way down are in the level's row lists
        int r = launch_nidx_from_segments(c, c->step.level, c->step.is_cur);
        if (r != EVT_OK) return r;
    }
    if (!c->nidx_valid) { // not recorded while growing: walk the last tree (same decisions, row by row)
        {
            int r = launch_apply_pending(c); // the recorded leaves of all rows are about to be overwritten
            if (r != EVT_OK) return r;
        }
        int r = launch_nidx_from_tree(c, !c->last_all_rows, c->last_cond);
        if (r != EVT_OK) return r;
        c->nidx_valid = true;
    }
    HIPCHK(hipMemcpyAsync(out, c->nidx, sizeof(uint32_t) * (size_t)c->N, hipMemcpyDefault, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return EVT_OK;
    });
}
extern "C" int evt_get_hist(evt_handle c, double *out) {
    return guarded([&]() -> int {
    CTXCHK_STEP(c);
    ARGCHK(out, "out is NULL");
    if (c->n_js_last <= 0) {
        evt_set_error("no tree has been grown yet");
        return EVT_ERR_STATE;
    }
    const size_t n = (size_t)c->NK * c->B * c->F * c->nnodes;
    double *d = nullptr;
    HIPCHK(hipMalloc((void **)&d, sizeof(double) * n));
    hipError_t e = hipMemsetAsync(d, 0, sizeof(double) * n, c->stream);
    int r = EVT_OK;
    if (e == hipSuccess) r = launch_hist_export(c, d);
    if (e == hipSuccess) e = hipMemcpyAsync(out, d, sizeof(double) * n, hipMemcpyDefault, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    (void)hipFree(d);
    if (e != hipSuccess) {
        evt_set_error("hist export failed: %s", hipGetErrorString(e));
        return EVT_ERR_HIP;
    }
    return r;
    });
}
extern "C" int evt_get_quant(evt_handle c, int32_t *qbits, int32_t *qexp) {
    return guarded([&]() -> int {
    CTXCHK(c);
    ARGCHK(qbits && qexp, "NULL argument");
    int32_t e[EVT_MC_MAX_NK];
    const int r = finish_quantize(c);
    if (r != EVT_OK) return r;
    // the tables of the last tree's gradients, also when the next round's have been quantised behind it
    HIPCHK(hipMemcpyAsync(e, c->n_js_last > 0 ? c->qexp_buf[c->q_tree] : c->qexp, sizeof(int32_t) * EVT_MC_MAX_NK, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    for (int k = 0; k < c->NK; k++) {
        qbits[k] = c->h_qbits[k];
        qexp[k] = e[k];
    }
    return EVT_OK;
    });
}

// ---- evaluation metric ------------------------------------------------------------------------
extern "C" int evt_eval_metric_begin(evt_handle c, int32_t metric) {
    return guarded([&]() -> int {
    CTXCHK(c);
    ARGCHK(metric >= 0 && metric <= EVT_METRIC_MULTIQUANTILE, "unknown metric");
    ARGCHK(metric != EVT_METRIC_MULTIQUANTILE || c->loss == EVT_LOSS_MULTIQUANTILE,
           "multiquantile is the metric of the multiquantile loss (one target, a level per output) and of no other");
    ARGCHK((metric == EVT_METRIC_GAUSSIAN_MLE) == (c->loss == EVT_LOSS_GAUSSIAN_MLE),
           "gaussian_mle is the metric of the gaussian_mle loss and of no other");
    ARGCHK((metric == EVT_METRIC_LOGISTIC_MLE) == (c->loss == EVT_LOSS_LOGISTIC_MLE),
           "logistic_mle is the metric of the logistic_mle loss and of no other");
    ARGCHK((metric == EVT_METRIC_MLOGLOSS) == (c->loss == EVT_LOSS_MLOGLOSS), "mlogloss is the metric of the mlogloss loss and of no other");
    if (!c->have_target) {
        evt_set_error("evt_eval_metric: set the target first");
        return EVT_ERR_STATE;
    }
    c->metric_queued = false;
    prof_begin(c, EVT_K_OTHER, 0);
    int r = launch_apply_pending(c);
    if (r == EVT_OK) r = launch_eval_metric(c, metric, c->metric_host);
    prof_end(c);
    if (r != EVT_OK) return r;
    c->metric_queued = true;
    return EVT_OK;
    });
}

extern "C" int evt_eval_metric_end(evt_handle c, double *value_out) {
    return guarded([&]() -> int {
    ARGCHK(c != nullptr, "handle is NULL");
    ARGCHK(value_out, "value_out is NULL");
    HIPCHK(hipSetDevice(c->device));
    if (!c->metric_queued) {
        evt_set_error("evt_eval_metric_end without evt_eval_metric_begin");
        return EVT_ERR_STATE;
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    c->metric_queued = false;
    c->pt_busy = false;
    *value_out = *c->metric_host;
    return EVT_OK;
    });
}

extern "C" int evt_eval_metric(evt_handle c, int32_t metric, double *value_out) {
    return guarded([&]() -> int {
    ARGCHK(c != nullptr, "handle is NULL");
    ARGCHK(value_out, "value_out is NULL");
    const int r = evt_eval_metric_begin(c, metric);
    return r == EVT_OK ? evt_eval_metric_end(c, value_out) : r;
    });
}

// ---- inference ------------------------------------------------------------------------------
// Trees completed for the LDS kernel: every leaf above a tree's last level becomes a chain of always-left nodes that
// carries its value down to that level, so that all rows walk depth - 1 levels.  Returns false when a tree's arrays are
// not a full heap (2^depth - 1 entries) - the gather kernel takes such models.
struct ModelTreeHost {
    int32_t node_off, leaf_off, levels, n_int;
};
// EVT_PREDICT_SHAPE=1..4 in the environment picks the LDS kernel's launch shape when the model allows it (for sweeps)
static int predict_shape_hint() {
    const char *v = getenv("EVT_PREDICT_SHAPE");
    return v ? atoi(v) : 0;
}
// Largest number of internal nodes over the model's trees; false when a tree's arrays are not a full heap
// (2^depth - 1 entries): the gather kernel takes such models.
static bool model_max_internal(int ntrees, const int64_t *tree_off, int &max_int) {
    max_int = 0;
    for (int t = 0; t < ntrees; t++) {
        const int64_t nn = tree_off[t + 1] - tree_off[t];
        if (nn < 1 || (nn & (nn + 1)) != 0 || nn > (1 << 20)) return false;
        max_int = std::max(max_int, (int)((nn + 1) / 2 - 1));
    }
    return true;
}
// Every tree padded to `stride` node words and the list padded with trees of no levels to a multiple of `group`.
static void complete_trees(int ntrees, const int64_t *tree_off, const int64_t *feat, const uint8_t *cond_bin, const float *pred,
                           const uint8_t *split, const uint8_t *feattypes, int K, int stride, int group, std::vector<uint32_t> &cnodes,
                           std::vector<float> &cleaf, std::vector<ModelTreeHost> &meta, bool &all_numeric) {
    const int npad = ((ntrees + group - 1) / group) * group;
    cnodes.assign((size_t)npad * stride, 0u);
    cleaf.clear();
    meta.assign(npad, ModelTreeHost{0, 0, 0, 0});
    all_numeric = true;
    std::vector<int32_t> vsrc;
    const uint32_t always_left = 0u | (255u << 16) | EVT_NODE_NUMERIC; // feature 1, bin <= 255
    for (int t = 0; t < ntrees; t++) {
        const int64_t o = tree_off[t];
        const int64_t nn = tree_off[t + 1] - o;
        int depth = 0;
        while (((int64_t)1 << depth) - 1 < nn) depth++;
        const int n_int = (1 << (depth - 1)) - 1, n_leaf = 1 << (depth - 1);
        meta[t] = {(int32_t)((size_t)t * stride), (int32_t)(cleaf.size() / K), depth - 1, n_int};
        // vsrc[n]: 0 = a split node of the tree; otherwise the leaf whose value node n carries
        vsrc.assign(nn + 1, 0);
        for (int64_t n = 1; n <= nn; n++) {
            const int32_t up = (n == 1) ? 0 : vsrc[n >> 1];
            vsrc[n] = up ? up : (split[o + n - 1] ? 0 : (int32_t)n);
        }
        uint32_t *cn = cnodes.data() + (size_t)t * stride;
        for (int n = 1; n <= n_int; n++) {
            uint32_t w = always_left;
            if (vsrc[n] == 0) {
                const int f0 = (int)feat[o + n - 1] - 1;
                const bool numeric = feattypes == nullptr || feattypes[f0] != 0;
                all_numeric = all_numeric && numeric;
                w = (uint32_t)(((f0 >> 2) << 8) | (f0 & 3)) | ((uint32_t)cond_bin[o + n - 1] << 16) | (numeric ? EVT_NODE_NUMERIC : 0u);
            }
            cn[n - 1] = w;
        }
        for (int q = 0; q < n_leaf; q++) {
            const int32_t src = vsrc[n_int + 1 + q]; // never 0: a split node's children lie inside the arrays (checked when packing)
            for (int k = 0; k < K; k++) cleaf.push_back(pred[(size_t)K * (o + src - 1) + k]);
        }
    }
}

static int predict_common(int64_t nobs, int32_t nfeats, const uint8_t *x_bin, const uint8_t *feattypes, int32_t loss, int32_t K, int32_t ntrees,
                          const int64_t *tree_off, const int64_t *feat, const uint8_t *cond_bin, const float *pred, const uint8_t *split,
                          int32_t apply_link, float *out, uint32_t *leaf_out, const double *x_f64 = nullptr, const double *edges = nullptr,
                          const int32_t *edge_off = nullptr) {
    ARGCHK(nobs >= 1 && nfeats >= 1 && ntrees >= 1, "nobs, nfeats, ntrees must be >= 1");
    ARGCHK((x_bin || x_f64) && tree_off && feat && cond_bin && split, "NULL argument");
    ARGCHK(leaf_out || (pred && out && K >= 1 && K <= EVT_MAX_K && loss >= 0 && loss <= EVT_LOSS_LAST), "invalid prediction arguments");
    std::vector<int32_t> eoff;
    int max_edges = 0;
    if (x_f64) {
        ARGCHK(edges && edge_off, "NULL argument");
        eoff.assign(edge_off, edge_off + nfeats + 1);
        for (int j = 0; j < nfeats; j++) {
            ARGCHK(eoff[j] >= 0 && eoff[j + 1] - eoff[j] >= 1 && eoff[j + 1] - eoff[j] <= 254, "each feature needs 1..254 edges");
            max_edges = std::max(max_edges, eoff[j + 1] - eoff[j]);
        }
    }
    int ndev = 0;
    int r = evt_device_count(&ndev);
    if (r != EVT_OK) return r;
    // the offsets are checked before anything is sized by them
    ARGCHK(tree_off[0] == 0, "tree_off must start at 0");
    for (int t = 0; t < ntrees; t++)
        ARGCHK(tree_off[t + 1] > tree_off[t] && tree_off[t + 1] - tree_off[t] <= ((int64_t)1 << 24), "tree_off must be strictly ascending, at most 2^24 nodes per tree");
    const int64_t total = tree_off[ntrees];
    ARGCHK(total <= ((int64_t)1 << 31), "the model holds more than 2^31 nodes");
    std::vector<uint32_t> nodes((size_t)total, 0u), one;
    for (int t = 0; t < ntrees; t++) {
        const int64_t o = tree_off[t];
        const int64_t nn = tree_off[t + 1] - o;
        r = pack_tree((int32_t)nn, feat + o, cond_bin + o, split + o, nfeats, feattypes, one);
        if (r != EVT_OK) return r;
        memcpy(nodes.data() + o, one.data(), sizeof(uint32_t) * nn);
    }
    hipStream_t s = nullptr;
    uint8_t *d_x = nullptr;
    uint32_t *d_nodes = nullptr, *d_leaf = nullptr;
    float *d_lp = nullptr, *d_out = nullptr;
    int64_t *d_off = nullptr;
    // x_bin and the output are used in place when they already live on the device
    auto on_device = [](const void *p) {
        hipPointerAttribute_t attr;
        const bool dev = p && hipPointerGetAttributes(&attr, p) == hipSuccess && attr.type == hipMemoryTypeDevice;
        (void)hipGetLastError();
        return dev;
    };
    const bool x_in_place = !x_f64 && on_device(x_bin);
    const bool out_in_place = !leaf_out && on_device(out);
    // models whose trees are full heaps of moderate depth go through the LDS kernel, on trees completed here
    std::vector<uint32_t> cnodes;
    std::vector<float> cleaf;
    std::vector<ModelTreeHost> cmeta;
    int max_int = 0, shape = 0;
    bool all_numeric = true;
    bool use_lds = !leaf_out && ntrees >= 4 && !on_device(pred) && !on_device(feat) && model_max_internal(ntrees, tree_off, max_int);
    if (use_lds) {
        shape = predict_lds_shape(nfeats, max_int, K, predict_shape_hint());
        use_lds = shape > 0;
    }
    if (use_lds)
        complete_trees(ntrees, tree_off, feat, cond_bin, pred, split, feattypes, K, std::max(1, max_int), shape == 1 ? 4 : (shape == 2 ? 2 : 1), cnodes,
                       cleaf, cmeta, all_numeric);
    uint32_t *d_cn = nullptr;
    float *d_cl = nullptr;
    ModelTreeHost *d_cm = nullptr;
    hipError_t e = hipSuccess;
    if (x_in_place) d_x = const_cast<uint8_t *>(x_bin);
    else e = hipMalloc((void **)&d_x, (size_t)nobs * nfeats);
    if (use_lds) {
        if (e == hipSuccess) e = hipMalloc((void **)&d_cn, sizeof(uint32_t) * std::max<size_t>(1, cnodes.size()));
        if (e == hipSuccess) e = hipMalloc((void **)&d_cl, sizeof(float) * cleaf.size());
        if (e == hipSuccess) e = hipMalloc((void **)&d_cm, sizeof(ModelTreeHost) * cmeta.size());
    } else {
        if (e == hipSuccess) e = hipMalloc((void **)&d_nodes, sizeof(uint32_t) * total);
        if (e == hipSuccess) e = hipMalloc((void **)&d_off, sizeof(int64_t) * (ntrees + 1));
        if (e == hipSuccess && !leaf_out) e = hipMalloc((void **)&d_lp, sizeof(float) * (size_t)total * K);
    }
    if (out_in_place) d_out = out;
    else if (e == hipSuccess && !leaf_out) e = hipMalloc((void **)&d_out, sizeof(float) * (size_t)nobs * K);
    if (e == hipSuccess && leaf_out) e = hipMalloc((void **)&d_leaf, sizeof(uint32_t) * (size_t)nobs * ntrees);
    if (e == hipSuccess && !x_f64 && !x_in_place) r = upload_bytes(s, x_bin, d_x, (size_t)nobs * nfeats);
    if (e == hipSuccess && x_f64 && !on_device(x_f64)) {
        std::vector<double> ev(eoff[nfeats]);
        e = hipMemcpy(ev.data(), edges, sizeof(double) * eoff[nfeats], hipMemcpyDefault);
        if (e == hipSuccess) {
            HbPlan P;
            P.build(ev.data(), eoff.data(), nfeats, EVT_F64);
            r = upload_bins(s, P, HbSource{x_f64, EVT_F64, 1, nobs}, nobs, d_x, nobs);
        }
    } else if (e == hipSuccess && x_f64) {
        double *d_edges = nullptr;
        int32_t *d_eoff = nullptr;
        e = hipMalloc((void **)&d_edges, sizeof(double) * eoff[nfeats]);
        if (e == hipSuccess) e = hipMalloc((void **)&d_eoff, sizeof(int32_t) * (nfeats + 1));
        if (e == hipSuccess) e = hipMemcpy(d_edges, edges, sizeof(double) * eoff[nfeats], hipMemcpyDefault);
        if (e == hipSuccess) e = hipMemcpy(d_eoff, eoff.data(), sizeof(int32_t) * (nfeats + 1), hipMemcpyHostToDevice);
        if (e == hipSuccess) {
            r = launch_binarize(s, x_f64, EVT_F64, 1, nobs, d_edges, d_eoff, max_edges, d_x, nobs, nfeats, nobs);
            if (r == EVT_OK) e = hipStreamSynchronize(s);
        }
        void *tmp[] = {d_edges, d_eoff};
        for (void *p : tmp)
            if (p) (void)hipFree(p);
    }
    if (use_lds) {
        if (e == hipSuccess && !cnodes.empty()) e = hipMemcpy(d_cn, cnodes.data(), sizeof(uint32_t) * cnodes.size(), hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMemcpy(d_cl, cleaf.data(), sizeof(float) * cleaf.size(), hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMemcpy(d_cm, cmeta.data(), sizeof(ModelTreeHost) * cmeta.size(), hipMemcpyHostToDevice);
    } else {
        if (e == hipSuccess) e = hipMemcpy(d_nodes, nodes.data(), sizeof(uint32_t) * total, hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMemcpy(d_off, tree_off, sizeof(int64_t) * (ntrees + 1), hipMemcpyDefault);
        if (e == hipSuccess && !leaf_out) e = hipMemcpy(d_lp, pred, sizeof(float) * (size_t)total * K, hipMemcpyDefault);
    }
    if (e == hipSuccess && r == EVT_OK) {
        if (leaf_out) r = launch_leaf_idx_model(s, d_nodes, d_off, ntrees, d_x, nobs, d_leaf);
        else if (use_lds) r = launch_predict_model_lds(s, d_cn, d_cl, d_cm, ntrees, d_x, nobs, nfeats, max_int, K, K, loss, apply_link, all_numeric ? 1 : 0, shape, d_out);
        else r = launch_predict_model(s, d_nodes, d_lp, d_off, ntrees, d_x, nobs, K, loss, apply_link, d_out, nullptr);
        e = hipDeviceSynchronize();
    }
    if (e == hipSuccess && r == EVT_OK) {
        if (leaf_out) e = hipMemcpy(leaf_out, d_leaf, sizeof(uint32_t) * (size_t)nobs * ntrees, hipMemcpyDefault);
        else if (!out_in_place) e = hipMemcpy(out, d_out, sizeof(float) * (size_t)nobs * K, hipMemcpyDefault);
    }
    void *ptrs[] = {x_in_place ? nullptr : d_x, d_nodes, d_off, d_lp, out_in_place ? nullptr : d_out, d_leaf, d_cn, d_cl, d_cm};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    if (e != hipSuccess) {
        evt_set_error("predict failed: %s", hipGetErrorString(e));
        return EVT_ERR_HIP;
    }
    return r;
}

extern "C" int evt_predict(int64_t nobs, int32_t nfeats, const uint8_t *x_bin, const uint8_t *feattypes, int32_t loss, int32_t K, int32_t ntrees,
                           const int64_t *tree_off, const int64_t *feat, const uint8_t *cond_bin, const float *pred, const uint8_t *split,
                           int32_t apply_link, float *out) {
    return guarded([&]() -> int {
    return predict_common(nobs, nfeats, x_bin, feattypes, loss, K, ntrees, tree_off, feat, cond_bin, pred, split, apply_link, out, nullptr);
    });
}

extern "C" int evt_predict_f64(int64_t nobs, int32_t nfeats, const double *x_colmajor, const double *edges, const int32_t *edge_off,
                               const uint8_t *feattypes, int32_t loss, int32_t K, int32_t ntrees, const int64_t *tree_off, const int64_t *feat,
                               const uint8_t *cond_bin, const float *pred, const uint8_t *split, int32_t apply_link, float *out) {
    return guarded([&]() -> int {
    ARGCHK(x_colmajor, "x is NULL");
    return predict_common(nobs, nfeats, nullptr, feattypes, loss, K, ntrees, tree_off, feat, cond_bin, pred, split, apply_link, out, nullptr,
                          x_colmajor, edges, edge_off);
    });
}

extern "C" int evt_predict_leaf_idx(int64_t nobs, int32_t nfeats, const uint8_t *x_bin, const uint8_t *feattypes, int32_t ntrees,
                                    const int64_t *tree_off, const int64_t *feat, const uint8_t *cond_bin, const uint8_t *split, uint32_t *out) {
    return guarded([&]() -> int {
    ARGCHK(out, "out is NULL");
    return predict_common(nobs, nfeats, x_bin, feattypes, 0, 1, ntrees, tree_off, feat, cond_bin, nullptr, split, 0, nullptr, out);
    });
}

// ---- measurement ----------------------------------------------------------------------------
extern "C" int evt_set_profiling(evt_handle c, int32_t on) {
    return guarded([&]() -> int {
    CTXCHK_QUEUE(c); // applies to what is queued from here on; pairs already recorded are folded in when their work is done
    c->profiling = (on == 1) ? 0x7fffffff : on; // 1: every class; otherwise a bit mask of EVT_K_* classes
    return EVT_OK;
    });
}
extern "C" int evt_get_profile(evt_handle c, int64_t *launches, double *ms, int64_t *units) {
    return guarded([&]() -> int {
    CTXCHK(c);
    ARGCHK(launches && ms && units, "NULL argument");
    HIPCHK(hipStreamSynchronize(c->stream));
    prof_collect(c, nullptr);
    for (int k = 0; k < EVT_K_COUNT; k++) {
        launches[k] = c->prof_launches[k];
        ms[k] = c->prof_ms[k];
        units[k] = c->prof_units[k];
    }
    return EVT_OK;
    });
}
extern "C" int evt_reset_profile(evt_handle c) {
    return guarded([&]() -> int {
    CTXCHK(c);
    HIPCHK(hipStreamSynchronize(c->stream));
    prof_collect(c, nullptr);
    memset(c->prof_launches, 0, sizeof(c->prof_launches));
    memset(c->prof_ms, 0, sizeof(c->prof_ms));
    memset(c->prof_units, 0, sizeof(c->prof_units));
    return EVT_OK;
    });
}
extern "C" int evt_set_option(evt_handle c, const char *name, int64_t value) {
    return guarded([&]() -> int {
    CTXCHK(c);
    ARGCHK(name, "name is NULL");
    if (strcmp(name, "hist_blocks") == 0) {
        ARGCHK(value >= 1 && value <= 65535, "hist_blocks must be in [1, 65535]");
        c->hist_blocks = (int)value;
    } else if (strcmp(name, "hist_min_rows") == 0) {
        ARGCHK(value >= 1 && value <= EVT_HIST_MAX_ROWS_PER_BLOCK, "hist_min_rows must be in [1, 65535]");
        c->hist_min_rows = (int)value;
    } else if (strcmp(name, "hist_seg_cost") == 0) {
        ARGCHK(value >= 0 && value <= 65536, "hist_seg_cost must be in [0, 65536]");
        c->hist_seg_cost = (int)value;
    } else if (strcmp(name, "hist_variant") == 0) {
        ARGCHK(value >= 0 && value <= 2, "hist_variant must be 0 (auto), 1 (generic) or 2 (conflict-free where it applies)");
        ARGCHK(value != 1 || c->LPR <= 64, "hist_variant 1: the generic histogram kernel takes records of up to 1024 bytes");
        c->hist_variant = (int)value;
    } else if (strcmp(name, "hist_tile") == 0) {
        ARGCHK(value == 0 || (value >= 16 && value <= 512 && (value & (value - 1)) == 0), "hist_tile must be 0 (auto) or a power of two in [16, 512]");
        c->hist_tile = (int)value;
    } else if (strcmp(name, "bit_planes") == 0) {
        ARGCHK(value == 0 || value == 1, "bit_planes must be 0 or 1");
        c->use_planes = (int)value;
        if (value == 0) c->planes_ready = false;
    } else if (strcmp(name, "grads_ahead") == 0) {
        c->grads_ahead = value != 0;
        if (!c->grads_ahead) c->grads_ready = false;
    } else if (strcmp(name, "record_nidx") == 0) {
        c->record_nidx = value != 0;
    } else if (strcmp(name, "small_tree") == 0) {
        ARGCHK(value >= 0 && value <= 4, "small_tree must be 0 (never), 1 (inputs of few rows), 2 or 3 (a block, or several, per feature and level wherever it can) or 4 (one launch per tree wherever it can)");
        c->small_tree = (int)value;
    } else if (strcmp(name, "scan_fused") == 0) {
        c->scan_fused = value != 0;
    } else if (strcmp(name, "hist_in_scatter") == 0) {
        c->hist_in_scatter = value != 0;
    } else if (strcmp(name, "part_one_pass") == 0) {
        c->part_one_pass = value != 0;
    } else if (strcmp(name, "defer_pred") == 0) {
        c->defer_pred = value == 2 || value == 3 ? (int)value : value != 0; // 2, 3: always or never by walking the tree
    } else if (strcmp(name, "hist_threads") == 0) {
        ARGCHK(value == 256 || value == 512 || value == 1024, "hist_threads must be 256, 512 or 1024");
        c->hist_threads = (int)value;
    } else {
        evt_set_error("unknown option %s", name);
        return EVT_ERR_ARG;
    }
    return EVT_OK;
    });
}
extern "C" int evt_synchronize(evt_handle c) {
    return guarded([&]() -> int {
    ARGCHK(c != nullptr, "handle is NULL");
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipStreamSynchronize(c->stream));
    return EVT_OK;
    });
}

__global__ __launch_bounds__(256) void k_copy16(const uint4 *__restrict__ src, uint4 *__restrict__ dst, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) dst[i] = src[i];
}

__global__ __launch_bounds__(256) void k_read16(const uint4 *__restrict__ src, int64_t n, unsigned int *sink) {
    unsigned int acc = 0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const uint4 v = src[i];
        acc ^= v.x ^ v.y ^ v.z ^ v.w;
    }
    if (acc == 0x12345678u) sink[0] = acc; // keeps the loads alive without a write stream
}

extern "C" int evt_read_bandwidth(int64_t nbytes, int32_t iters, double *gbps_out) {
    return guarded([&]() -> int {
    ARGCHK(gbps_out && nbytes >= 4096 && iters >= 1, "invalid arguments");
    int ndev = 0;
    int r = evt_device_count(&ndev);
    if (r != EVT_OK) return r;
    const int64_t n = nbytes / 16;
    uint4 *a = nullptr;
    unsigned int *sink = nullptr;
    HIPCHK(hipMalloc((void **)&a, n * 16));
    hipError_t e = hipMalloc((void **)&sink, 64);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    float ms = 0.0f;
    if (e == hipSuccess) e = hipMemset(a, 1, n * 16);
    if (e == hipSuccess) e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_read16, dim3(8192), dim3(256), 0, 0, a, n, sink);
        e = hipEventRecord(e0, 0);
        for (int i = 0; i < iters; i++) hipLaunchKernelGGL(k_read16, dim3(8192), dim3(256), 0, 0, a, n, sink);
        if (e == hipSuccess) e = hipEventRecord(e1, 0);
        if (e == hipSuccess) e = hipEventSynchronize(e1);
        if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (a) (void)hipFree(a);
    if (sink) (void)hipFree(sink);
    if (e != hipSuccess) {
        evt_set_error("read bandwidth probe failed: %s", hipGetErrorString(e));
        return EVT_ERR_HIP;
    }
    *gbps_out = (double)(n * 16) * iters / ((double)ms * 1e-3) / 1e9;
    return EVT_OK;
    });
}

extern "C" int evt_copy_bandwidth(int64_t nbytes, int32_t iters, double *gbps_out) {
    return guarded([&]() -> int {
    ARGCHK(gbps_out && nbytes >= 4096 && iters >= 1, "invalid arguments");
    int ndev = 0;
    int r = evt_device_count(&ndev);
    if (r != EVT_OK) return r;
    const int64_t n = nbytes / 16;
    uint4 *a = nullptr, *b = nullptr;
    HIPCHK(hipMalloc((void **)&a, n * 16));
    hipError_t e = hipMalloc((void **)&b, n * 16);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    float ms = 0.0f;
    if (e == hipSuccess) e = hipMemset(a, 1, n * 16);
    if (e == hipSuccess) e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_copy16, dim3(8192), dim3(256), 0, 0, a, b, n); // warm-up
        e = hipEventRecord(e0, 0);
        for (int i = 0; i < iters; i++) hipLaunchKernelGGL(k_copy16, dim3(8192), dim3(256), 0, 0, a, b, n);
        if (e == hipSuccess) e = hipEventRecord(e1, 0);
        if (e == hipSuccess) e = hipEventSynchronize(e1);
        if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (a) (void)hipFree(a);
    if (b) (void)hipFree(b);
    if (e != hipSuccess) {
        evt_set_error("copy bandwidth probe failed: %s", hipGetErrorString(e));
        return EVT_ERR_HIP;
    }
    *gbps_out = 2.0 * (double)(n * 16) * iters / ((double)ms * 1e-3) / 1e9;
    return EVT_OK;
    });
}
