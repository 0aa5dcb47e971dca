// Pinned buffers, and the pipeline that bins a host matrix on its way to the device.
#include "upload.h"

#include <algorithm>
#include <mutex>

namespace {
std::mutex g_pin_m;
std::vector<void *> g_pin_idle;
} // namespace

void *pinned_take() {
    {
        std::lock_guard<std::mutex> lk(g_pin_m);
        if (!g_pin_idle.empty()) {
            void *p = g_pin_idle.back();
            g_pin_idle.pop_back();
            return p;
        }
    }
    void *p = nullptr;
    const hipError_t e = hipHostMalloc(&p, PINNED_BYTES, hipHostMallocPortable);
    if (e == hipSuccess) return p;
    evt_set_error("hipHostMalloc failed: %s", hipGetErrorString(e));
    return nullptr;
}
void pinned_give(void *p) {
    {
        std::lock_guard<std::mutex> lk(g_pin_m);
        if ((int)g_pin_idle.size() < PINNED_KEPT) {
            g_pin_idle.push_back(p);
            return;
        }
    }
    (void)hipHostFree(p);
}
extern "C" int evt_trim(void) {
    return guarded([&]() -> int {
    std::vector<void *> idle;
    {
        std::lock_guard<std::mutex> lk(g_pin_m);
        idle.swap(g_pin_idle);
    }
    for (void *p : idle) (void)hipHostFree(p);
    return EVT_OK;
    });
}

BinPieces::BinPieces(int64_t N_, int F_, bool rows_contiguous, size_t bytes) : N(N_), F(F_) {
    const int64_t cells = (int64_t)bytes;
    if (rows_contiguous) {
        cols = F;
        rows = std::min(N, std::max<int64_t>(64, cells / F / 64 * 64));
    } else if (N <= cells) {
        rows = N;
        cols = (int)std::max<int64_t>(1, std::min<int64_t>(F, cells / N));
    } else {
        rows = cells;
        cols = 1;
    }
    row_pieces = (N + rows - 1) / rows;
    np = row_pieces * ((F + cols - 1) / cols);
}
void BinPieces::at(int64_t p, int64_t *r0, int64_t *n, int *f0, int *f1) const {
    *r0 = (p % row_pieces) * rows;
    *n = std::min(rows, N - *r0);
    *f0 = (int)(p / row_pieces) * cols;
    *f1 = std::min(F, *f0 + cols);
}

// the bins of task t of a piece: a block of rows of all its features, or a block of rows of one
struct PieceTasks {
    int64_t block;
    int per_piece, row_blocks;
    bool rowwise;
    PieceTasks(const BinPieces &B, bool rows_contiguous) : rowwise(rows_contiguous) {
        // about 64k cells: 25 us of work, against 0.1 us to hand it out
        block = rowwise ? std::max<int64_t>(64, 65536 / B.F / 64 * 64) : 65536;
        row_blocks = (int)((B.rows + block - 1) / block);
        per_piece = rowwise ? row_blocks : row_blocks * B.cols;
    }
    void run(const HbPlan &P, const HbSource &S, int64_t r0, int64_t n, int f0, int f1, uint8_t *out, int t) const {
        const int64_t b0 = (int64_t)(t % row_blocks) * block;
        if (b0 >= n) return;
        const int64_t m = std::min(block, n - b0);
        if (rowwise) {
            hb_bin(P, S, r0 + b0, m, f0, f1, out + b0, n);
        } else {
            const int f = f0 + t / row_blocks;
            if (f < f1) hb_bin(P, S, r0 + b0, m, f, f + 1, out + (size_t)(f - f0) * n + b0, n);
        }
    }
};

int upload_bins(hipStream_t s, const HbPlan &P, const HbSource &S, int64_t N, uint8_t *xcm, int64_t ldo) {
    const bool rowwise = S.rows_contiguous();
    const BinPieces B(N, P.F, rowwise, PINNED_BYTES);
    const PieceTasks T(B, rowwise);
    const int NS = (int)std::min<int64_t>(PinnedSlots::NS, B.np);
    PinnedSlots U(s);
    int r = U.init(NS);
    if (r != EVT_OK) return r;
    auto send = [&](int64_t p) -> hipError_t {
        int64_t r0, n;
        int f0, f1;
        B.at(p, &r0, &n, &f0, &f1);
        uint8_t *dst = xcm + (size_t)f0 * ldo + r0;
        const void *src = U.host[p % NS];
        hipError_t e = (n == ldo || f1 - f0 == 1) ? hipMemcpyAsync(dst, src, (size_t)n * (f1 - f0), hipMemcpyHostToDevice, s)
                                                  : hipMemcpy2DAsync(dst, (size_t)ldo, src, (size_t)n, (size_t)n, (size_t)(f1 - f0), hipMemcpyHostToDevice, s);
        return e == hipSuccess ? hipEventRecord(U.ev[p % NS], s) : e;
    };
    auto bin = [&](int64_t p, int t) {
        int64_t r0, n;
        int f0, f1;
        B.at(p, &r0, &n, &f0, &f1);
        T.run(P, S, r0, n, f0, f1, static_cast<uint8_t *>(U.host[p % NS]), t);
    };
    const int workers = hb_workers(N * P.F);
    if (B.np <= 2 || workers == 0) { // the calling thread works too
        for (int64_t p = 0; p < B.np; p++) {
            if (p >= NS) HIPCHK(hipEventSynchronize(U.ev[p % NS]));
            hb_parallel(T.per_piece, workers, [&](int t) { bin(p, t); });
            HIPCHK(send(p));
        }
        HIPCHK(hipStreamSynchronize(s));
        U.idle = true;
        return EVT_OK;
    }
    // Many pieces: the workers run through the tasks of all of them, as far as buffers are free; the calling thread sends a piece when
    // its last task is done and frees a buffer when its copy has arrived.
    const int64_t total = B.np * T.per_piece;
    std::atomic<int64_t> next{0}, released{NS};
    std::vector<std::atomic<int>> done((size_t)B.np);
    for (auto &d : done) d.store(0, std::memory_order_relaxed);
    std::atomic<bool> stop{false};
    auto work = [&] {
        for (int64_t t; (t = next.fetch_add(1, std::memory_order_relaxed)) < total;) {
            const int64_t p = t / T.per_piece;
            while (p >= released.load(std::memory_order_acquire)) {
                if (stop.load(std::memory_order_relaxed)) return;
                std::this_thread::yield();
            }
            bin(p, (int)(t % T.per_piece));
            done[(size_t)p].fetch_add(1, std::memory_order_release);
        }
    };
    struct Joined {
        std::atomic<bool> &stop;
        std::vector<std::thread> th;
        ~Joined() {
            stop.store(true);
            for (auto &t : th) t.join();
        }
    } ws{stop, {}};
    for (int w = 0; w < workers; w++) ws.th.emplace_back(work);
    int64_t freed = NS; // pieces whose buffer is free for binning, as far as released
    for (int64_t p = 0; p < B.np; p++) {
        while (done[(size_t)p].load(std::memory_order_acquire) < T.per_piece) {
            if (freed < B.np && freed - NS < p) { // the oldest piece sent whose buffer has not been handed on
                const hipError_t q = hipEventQuery(U.ev[freed % NS]);
                if (q == hipSuccess) released.store(++freed, std::memory_order_release);
                else if (q == hipErrorNotReady) (void)hipGetLastError();
                else HIPCHK(q);
            }
            std::this_thread::yield();
        }
        HIPCHK(send(p));
    }
    HIPCHK(hipStreamSynchronize(s));
    U.idle = true;
    return EVT_OK;
}

// ---- host-only entry points ---------------------------------------------------------------------
static int take_columns(const void *v, int32_t ncols, std::vector<HbColumn> &out) {
    const evt_column *cols = static_cast<const evt_column *>(v);
    ARGCHK(cols && ncols >= 1, "columns missing");
    out.resize(ncols);
    for (int j = 0; j < ncols; j++) {
        ARGCHK(cols[j].data && cols[j].dtype >= EVT_F32 && cols[j].dtype <= EVT_U64, "a column without data or of an unknown type");
        out[j] = {static_cast<const char *>(cols[j].data), cols[j].stride, (int32_t)cols[j].dtype};
    }
    return EVT_OK;
}
extern "C" int evt_bin_columns(const void *cols, int32_t ncols, int64_t nobs, const double *edges, const int32_t *edge_off, uint8_t *out) {
    return guarded([&]() -> int {
    std::vector<HbColumn> c;
    int r = take_columns(cols, ncols, c);
    if (r != EVT_OK) return r;
    ARGCHK(nobs >= 1 && edge_off && out, "NULL argument");
    for (int j = 0; j < ncols; j++)
        ARGCHK(edge_off[j] >= 0 && edge_off[j + 1] >= edge_off[j] && edge_off[j + 1] - edge_off[j] <= 254, "each feature has at most 254 edges");
    ARGCHK(edges || edge_off[ncols] == 0, "NULL argument");
    hb_bin_columns(c.data(), ncols, nobs, edges, edge_off, out);
    return EVT_OK;
    });
}
extern "C" int evt_order_stats(const void *cols, int32_t ncols, const int64_t *idx, int64_t n, const int64_t *ranks, int32_t n_ranks, double *out) {
    return guarded([&]() -> int {
    std::vector<HbColumn> c;
    int r = take_columns(cols, ncols, c);
    if (r != EVT_OK) return r;
    ARGCHK(n >= 1 && n <= 0x7fffffff && ranks && n_ranks >= 1 && out, "invalid arguments");
    for (int i = 0; i < n_ranks; i++) ARGCHK(ranks[i] >= 0 && ranks[i] < n && (i == 0 || ranks[i] >= ranks[i - 1]), "ranks must ascend within the sample");
    hb_order_stats(c.data(), ncols, idx, n, ranks, n_ranks, out);
    return EVT_OK;
    });
}
