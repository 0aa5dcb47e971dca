// The pipeline that bins a host matrix on its way to the device.
#include "upload.h"

#include <string.h>

#include <algorithm>

BinPieces::BinPieces(int64_t N_, int F_, bool src_rows_contiguous, bool by_rows, int64_t rows_most, int64_t cells_most)
    : N(N_), F(F_), rowwise(src_rows_contiguous) {
    if (by_rows) {
        cols = F;
        rows = std::min(N, rows_most);
    } else if (N <= cells_most) {
        rows = N;
        cols = (int)std::max<int64_t>(1, std::min<int64_t>(F, cells_most / N));
    } else {
        rows = cells_most;
        cols = 1;
    }
    row_pieces = (N + rows - 1) / rows;
    np = row_pieces * ((F + cols - 1) / cols);
    // a task is 64k cells at most (25 us of work, against 0.1 us to hand it out), less when they would be few
    const int64_t cells = std::max<int64_t>(4096, std::min<int64_t>(65536, rows * cols / 64));
    block = std::max<int64_t>(64, (rowwise ? cells / F : std::min(cells, rows)) / 64 * 64);
    row_blocks = (int)((rows + block - 1) / block);
    per_piece = rowwise ? row_blocks : row_blocks * cols;
}
void BinPieces::at(int64_t p, int64_t *r0, int64_t *n, int *f0, int *f1) const {
    *r0 = (p % row_pieces) * rows;
    *n = std::min(rows, N - *r0);
    *f0 = (int)(p / row_pieces) * cols;
    *f1 = std::min(F, *f0 + cols);
}
void BinPieces::bin(const HbPlan &P, const HbSource &S, int64_t p, int t, uint8_t *out) const {
    int64_t r0, n;
    int f0, f1;
    at(p, &r0, &n, &f0, &f1);
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

void BinPieces::copy(const HbSource &S, int64_t p, int t, void *out) const {
    int64_t r0, n;
    int f0, f1;
    at(p, &r0, &n, &f0, &f1);
    const int64_t b0 = (int64_t)(t % row_blocks) * block;
    if (b0 >= n) return;
    const int64_t m = std::min(block, n - b0);
    const size_t es = S.esize();
    char *o = static_cast<char *>(out);
    if (rowwise) {
        const char *x = static_cast<const char *>(S.base) + es * ((size_t)(r0 + b0) * S.rs + f0);
        const size_t row = es * (f1 - f0);
        o += row * b0;
        if (S.rs == f1 - f0) memcpy(o, x, row * m);
        else
            for (int64_t i = 0; i < m; i++) memcpy(o + row * i, x + es * i * S.rs, row);
    } else {
        const int f = f0 + t / row_blocks;
        if (f < f1) memcpy(o + es * ((size_t)(f - f0) * n + b0), static_cast<const char *>(S.base) + es * ((size_t)f * S.cs + r0 + b0), es * m);
    }
}

// Nanoseconds by c cores (measured on a 16-core EPYC at 64 bins): the AVX-512 search takes 0.5 for a Float32 value and 0.65 for a Float64
// one, / c; the plain search 20 / c.  The device's form is a copy into pinned memory at 30 GB/s a core and the bus at 43 GB/s: ahead for
// Float64 below 4 cores, for Float32 below 6, and always without AVX-512, once the matrix repays its 100 us.
bool bins_by_device(int dtype, int64_t cells) {
    if (cells < 4096) return false;
    const double c = hb_cores(), es = dtype == EVT_F32 ? 4 : 8;
    const double host = (!hb_has_avx512() ? 20.0 : dtype == EVT_F32 ? 0.5 : 0.65) / c, device = std::max(es / 43, es / 30 / c);
    return 100e3 + device * cells < host * cells;
}
int DeviceBins::init(hipStream_t s, const HbPlan &P, size_t slot_bytes, int slots) {
    std::vector<int32_t> off(P.F + 1);
    for (int j = 0; j < P.F; j++) off[j] = (int32_t)(P.feat[j].e - P.edges.data());
    off[P.F] = (int32_t)P.edges.size();
    for (const HbFeature &f : P.feat) max_edges = std::max(max_edges, f.ne);
    slot = (slot_bytes + 255) / 256 * 256;
    off_at = (8 * P.edges.size() + 255) / 256 * 256;
    edges = static_cast<uint8_t *>(dev_take(off_at + 4 * off.size()));
    stage = static_cast<uint8_t *>(dev_take(slot * slots));
    if (!edges || !stage) return EVT_ERR_NOMEM;
    const hipError_t e = hipMemcpyAsync(edges, P.edges.data(), 8 * P.edges.size(), hipMemcpyHostToDevice, s);
    const hipError_t e2 = hipMemcpyAsync(edges + off_at, off.data(), 4 * off.size(), hipMemcpyHostToDevice, s);
    HIPCHK(hipStreamSynchronize(s)); // the copies read `off`
    HIPCHK(e);
    HIPCHK(e2);
    return EVT_OK;
}
int DeviceBins::send(hipStream_t s, int k, const void *h, const HbSource &S, int64_t n, int f0, int f1, uint8_t *out, int64_t ldo) {
    uint8_t *x = stage + k * slot;
    const bool rowwise = S.rows_contiguous();
    HIPCHK(hipMemcpyAsync(x, h, S.esize() * n * (f1 - f0), hipMemcpyHostToDevice, s));
    return launch_binarize(s, x, S.dtype, rowwise ? f1 - f0 : 1, rowwise ? 1 : n, reinterpret_cast<const double *>(edges),
                           reinterpret_cast<const int32_t *>(edges + off_at) + f0, max_edges, out, n, f1 - f0, ldo);
}

int upload_bins(hipStream_t s, const HbPlan &P, const HbSource &S, int64_t N, uint8_t *xcm, int64_t ldo) {
    const bool rowwise = S.rows_contiguous(), raw = bins_by_device(S.dtype, N * P.F);
    const int64_t cell = raw ? (int64_t)S.esize() : 1; // bytes of one in a pinned buffer
    const int64_t rows = (int64_t)PINNED_BYTES / (P.F * cell);
    const BinPieces B(N, P.F, rowwise, rowwise, rows >= 64 ? rows / 64 * 64 : std::max<int64_t>(1, rows), (int64_t)PINNED_BYTES / cell);
    const int NS = (int)std::min<int64_t>(PinnedSlots::NS, B.np);
    DeviceBins D;
    PinnedSlots U(s);
    int r = U.init(NS);
    if (r == EVT_OK && raw) r = D.init(s, P, PINNED_BYTES, NS);
    if (r != EVT_OK) return r;
    auto send = [&](int64_t p) -> int {
        int64_t r0, n;
        int f0, f1;
        B.at(p, &r0, &n, &f0, &f1);
        uint8_t *dst = xcm + (size_t)f0 * ldo + r0;
        const void *src = U.host[p % NS];
        if (raw) {
            const int rs = D.send(s, (int)(p % NS), src, S, n, f0, f1, dst, ldo);
            if (rs != EVT_OK) return rs;
        } else if (n == ldo || f1 - f0 == 1) {
            HIPCHK(hipMemcpyAsync(dst, src, (size_t)n * (f1 - f0), hipMemcpyHostToDevice, s));
        } else {
            HIPCHK(hipMemcpy2DAsync(dst, (size_t)ldo, src, (size_t)n, (size_t)n, (size_t)(f1 - f0), hipMemcpyHostToDevice, s));
        }
        HIPCHK(hipEventRecord(U.ev[p % NS], s));
        return EVT_OK;
    };
    auto fill = [&](int64_t p, int t) {
        if (raw) B.copy(S, p, t, U.host[p % NS]);
        else B.bin(P, S, p, t, static_cast<uint8_t *>(U.host[p % NS]));
    };
    return run_pieces(U, NS, B.np, B.per_piece, hb_workers(N * P.F), fill, send, [](int64_t) {});
}

// From 64 MB on by way of pinned buffers that the workers fill while the bus empties others: a copy straight from pageable memory is
// staged by the runtime at 31 GB/s on this bus.  set_xbin of 100 MB 2.4 ms, of 1 GB 23.4 ms (43 GB/s); 32 MB pieces and threads started for each
// call took 5.4 and 25 to 27.
int upload_bytes(hipStream_t s, const void *src, void *dst, size_t nbytes) {
    hipPointerAttribute_t attr;
    const bool on_dev = (hipPointerGetAttributes(&attr, src) == hipSuccess) && attr.type == hipMemoryTypeDevice;
    (void)hipGetLastError();
    if (on_dev || nbytes < (size_t)64 << 20) {
        HIPCHK(hipMemcpyAsync(dst, src, nbytes, hipMemcpyDefault, s));
        HIPCHK(hipStreamSynchronize(s));
        return EVT_OK;
    }
    const size_t task = (size_t)512 << 10;
    PinnedSlots U(s);
    const int r = U.init(PinnedSlots::NS);
    if (r != EVT_OK) return r;
    auto size = [&](int64_t p) { return std::min(PINNED_BYTES, nbytes - (size_t)p * PINNED_BYTES); };
    auto fill = [&](int64_t p, int t) {
        const size_t at = t * task, n = size(p);
        if (at < n) memcpy(static_cast<char *>(U.host[p % PinnedSlots::NS]) + at, static_cast<const char *>(src) + (size_t)p * PINNED_BYTES + at, std::min(task, n - at));
    };
    auto send = [&](int64_t p) -> int {
        HIPCHK(hipMemcpyAsync(static_cast<char *>(dst) + (size_t)p * PINNED_BYTES, U.host[p % PinnedSlots::NS], size(p), hipMemcpyHostToDevice, s));
        HIPCHK(hipEventRecord(U.ev[p % PinnedSlots::NS], s));
        return EVT_OK;
    };
    return run_pieces(U, PinnedSlots::NS, (int64_t)((nbytes + PINNED_BYTES - 1) / PINNED_BYTES), (int)(PINNED_BYTES / task), hb_workers(nbytes / 8), fill, send,
                      [](int64_t) {});
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
        ARGCHK(edge_off[j] >= 0 && edge_off[j + 1] >= edge_off[j], "edge offsets must ascend");
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
