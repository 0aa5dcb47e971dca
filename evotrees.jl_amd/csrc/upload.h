// Feature matrices on their way from host memory to the device.
#pragma once
#include "evt_internal.h"
#include "host_bin.h"
#include "pool.h"

#include <thread>

static const size_t PINNED_BYTES = (size_t)8 << 20; // a piece on its way up

struct PinnedSlots { // NS of them, with an event each for the work that reads or writes them
    static const int NS = 4;
    void *host[NS] = {};
    hipEvent_t ev[NS] = {};
    hipStream_t s;
    bool idle = false; // the stream has been waited for since the buffers were last used
    explicit PinnedSlots(hipStream_t s_) : s(s_) {}
    int init(int n) {
        for (int k = 0; k < n; k++) {
            host[k] = pinned_take(PINNED_BYTES);
            if (!host[k]) return EVT_ERR_NOMEM;
            HIPCHK(hipEventCreateWithFlags(&ev[k], hipEventDisableTiming));
        }
        return EVT_OK;
    }
    ~PinnedSlots() {
        if (!idle) (void)hipStreamSynchronize(s);
        for (int k = 0; k < NS; k++) {
            if (ev[k]) (void)hipEventDestroy(ev[k]);
            if (host[k]) pinned_give(host[k]);
        }
    }
};

// How a matrix of N rows and F features is cut into pieces: row ranges of all features, or whole columns (or row ranges of one).
struct BinPieces {
    int64_t N, rows; // rows of a piece
    int F, cols;     // features of a piece
    int64_t np;      // pieces
    int64_t row_pieces;
    bool rowwise;    // the source's rows are contiguous
    // tasks of a piece: blocks of rows, of all its features or of one
    int64_t block;
    int per_piece, row_blocks;
    BinPieces(int64_t N_, int F_, bool src_rows_contiguous, bool by_rows, int64_t rows_most, int64_t cells_most);
    void at(int64_t p, int64_t *r0, int64_t *n, int *f0, int *f1) const;
    void bin(const HbPlan &P, const HbSource &S, int64_t p, int t, uint8_t *out) const; // the bin of (r, f) to out[(f - f0) * n + r - r0]
    void copy(const HbSource &S, int64_t p, int t, void *out) const; // its value there, or to out[(r - r0) * cols + f] when rowwise
};

// Pieces that go up as they lie and are binned by a kernel: for hosts whose cores are slower at it than the bus.
bool bins_by_device(int dtype, int64_t cells);
class DeviceBins {
    uint8_t *edges = nullptr, *stage = nullptr;
    size_t off_at = 0, slot = 0;
    int max_edges = 0;

  public: // declared before the pinned buffers: they wait for the stream
    int init(hipStream_t s, const HbPlan &P, size_t slot_bytes, int slots);
    // queues piece data of n rows and features [f0, f1) from h, by way of buffer k; its bins go to out + (f - f0) * ldo
    int send(hipStream_t s, int k, const void *h, const HbSource &S, int64_t n, int f0, int f1, uint8_t *out, int64_t ldo);
    ~DeviceBins() {
        dev_give(edges);
        dev_give(stage);
    }
};

// The pieces 0 .. np - 1 through NS buffers: piece p is filled by its `tasks` calls of fill(p, t), on worker threads or this one; then send(p) queues
// what the device does with it and records U.ev[p % NS]; when that event has come, retire(p), on the calling thread, and the buffer
// is free for piece p + NS.  Everything has been retired when the call returns EVT_OK.
template <typename Fill, typename Send, typename Retire>
static int run_pieces(PinnedSlots &U, int NS, int64_t np, int tasks, int workers, Fill fill, Send send, Retire retire) {
    if (np <= 2 || workers == 0) { // the calling thread fills too
        int64_t back = 0;
        for (int64_t p = 0; p < np; p++) {
            if (p >= NS) {
                HIPCHK(hipEventSynchronize(U.ev[back % NS]));
                retire(back++);
            }
            hb_parallel(tasks, workers, [&](int t) { fill(p, t); });
            const int r = send(p);
            if (r != EVT_OK) return r;
        }
        for (; back < np; back++) {
            HIPCHK(hipEventSynchronize(U.ev[back % NS]));
            retire(back);
        }
        U.idle = true;
        return EVT_OK;
    }
    // Many pieces: the workers run through the tasks of all of them, as far as buffers are free
    const int64_t total = np * tasks;
    std::atomic<int64_t> next{0}, released{NS};
    std::vector<std::atomic<int>> done((size_t)np);
    for (auto &d : done) d.store(0, std::memory_order_relaxed);
    std::atomic<bool> stop{false};
    auto step = [&]() -> bool {
        int64_t t = next.load(std::memory_order_relaxed);
        if (t >= total || stop.load(std::memory_order_relaxed)) return false;
        if (t / tasks >= released.load(std::memory_order_acquire)) std::this_thread::yield();
        else if (next.compare_exchange_weak(t, t + 1, std::memory_order_relaxed)) {
            fill(t / tasks, (int)(t % tasks));
            done[(size_t)(t / tasks)].fetch_add(1, std::memory_order_release);
        }
        return true;
    };
    struct Stop { // whatever ends the call, workers that wait for a buffer stop waiting
        std::atomic<bool> &flag;
        ~Stop() { flag.store(true); }
    };
    HbWorkers ws(workers, step);
    Stop on_return{stop};
    int64_t back = 0;
    for (int64_t p = 0; p < np; p++) {
        while (done[(size_t)p].load(std::memory_order_acquire) < tasks) {
            if (back < p && back + NS < np) { // the oldest piece sent that has not been retired, while a piece needs its buffer
                const hipError_t q = hipEventQuery(U.ev[back % NS]);
                if (q == hipSuccess) {
                    retire(back++);
                    released.store(back + NS, std::memory_order_release);
                } else if (q == hipErrorNotReady) {
                    (void)hipGetLastError();
                } else {
                    HIPCHK(q);
                }
            }
            if (ws.failed()) ws.join(); // throws
            if (ws.none()) step();
            else std::this_thread::yield();
        }
        const int r = send(p);
        if (r != EVT_OK) return r;
    }
    ws.join(); // the workers are free for what retire() shares out
    for (; back < np; back++) {
        HIPCHK(hipEventSynchronize(U.ev[back % NS]));
        retire(back);
    }
    U.idle = true;
    return EVT_OK;
}

// nbytes from the caller's memory, on the host or the device, to the device.  The data has arrived when the call returns.
int upload_bytes(hipStream_t s, const void *src, void *dst, size_t nbytes);
// Binned matrix -> device, column j to xcm + j * ldo.  The data has arrived when the call returns.
int upload_bins(hipStream_t s, const HbPlan &P, const HbSource &S, int64_t N, uint8_t *xcm, int64_t ldo);
