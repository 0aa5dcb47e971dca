// Feature matrices on their way from host memory to the device.
#pragma once
#include "evt_internal.h"
#include "host_bin.h"

// Pinned buffers of PINNED_BYTES each, kept between calls: pinning 8 MB costs the host more than filling them.  At most
// PINNED_KEPT stay behind when nobody uses them (32 MB); evt_trim gives those back.  Any thread, any device (portable).
static const size_t PINNED_BYTES = (size_t)8 << 20;
static const int PINNED_KEPT = 4;
void *pinned_take();          // nullptr: out of memory (the error is set)
void pinned_give(void *p);    // nothing on the device may still use it

struct PinnedSlots { // NS of them, with an event each for the work that reads or writes them
    static const int NS = PINNED_KEPT;
    void *host[NS] = {};
    hipEvent_t ev[NS] = {};
    hipStream_t s;
    bool idle = false; // the stream has been waited for since the buffers were last used
    explicit PinnedSlots(hipStream_t s_) : s(s_) {}
    int init(int n) {
        for (int k = 0; k < n; k++) {
            host[k] = pinned_take();
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

// How a matrix of N rows and F features is cut into pieces of at most `bytes` bins: row ranges of all features where its rows are
// contiguous, whole columns (or row ranges of one) where its columns are.
struct BinPieces {
    int64_t N, rows; // rows of a piece
    int F, cols;     // features of a piece
    int64_t np;      // pieces
    int64_t row_pieces;
    BinPieces(int64_t N_, int F_, bool rows_contiguous, size_t bytes);
    void at(int64_t p, int64_t *r0, int64_t *n, int *f0, int *f1) const;
};
// Binned matrix -> device, column j to xcm + j * ldo.  Workers bin pieces into pinned buffers while earlier ones are copied; the
// data has arrived when the call returns.
int upload_bins(hipStream_t s, const HbPlan &P, const HbSource &S, int64_t N, uint8_t *xcm, int64_t ldo);
