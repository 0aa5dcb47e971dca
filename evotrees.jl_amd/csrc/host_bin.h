// Binarize on the host's cores (src/fit-utils.jl:66-72): bins leave the host as bytes, an eighth of a Float64 matrix's way over
// the bus.
#pragma once
#include <stdint.h>

#include <atomic>
#include <functional>
#include <memory>
#include <vector>

#include "../../include/evotrees_hip.h"

// A matrix in host memory: element (i, j) at base + i * rs + j * cs elements; one of the two strides is 1.
struct HbSource {
    const void *base;
    int32_t dtype; // EVT_F32 / EVT_F64
    int64_t rs, cs;
    bool rows_contiguous() const { return cs == 1 && rs != 1; }
    size_t esize() const { return dtype == EVT_F32 ? 4 : 8; }
};

#define HB_SLOW 1  // an edge is NaN or -0.0, or there are more than 254: compared by isless, value by value
#define HB_EXACT 2 // the Float32 search decides alone; otherwise a value that meets an edge there is compared in Float64

// One feature's edges for a source type, laid out for the search.
struct HbFeature {
    int32_t levels; // steps of the search: 4 .. 8, 2^levels - 1 >= ne unless the feature is HB_SLOW
    int32_t flags;
    int32_t ne;
    int32_t heap;      // first word of the feature's search heap in HbPlan::heap
    const double *e;   // its edges
};
struct HbPlan {
    int32_t dtype = 0, F = 0;
    std::vector<HbFeature> feat;
    std::vector<double> edges;
    std::vector<float> heap_store; // over-allocated: heap() is 64-byte aligned
    float *heap = nullptr;
    void build(const double *edges_flat, const int32_t *off, int F, int dtype);
};
// rows [r0, r0 + n) of features [f0, f1): the bin of (r, f) goes to out + (f - f0) * ldo + (r - r0)
void hb_bin(const HbPlan &P, const HbSource &S, int64_t r0, int64_t n, int f0, int f1, uint8_t *out, int64_t ldo);
bool hb_has_avx512();
int hb_cores(); // that the calling thread may use: its affinity, within the container's CPU quota
// worker threads worth starting for this much work, the calling thread not counted (0: none)
int hb_workers(int64_t cells);

// the AVX-512 forms (host_bin_avx512.cpp), chosen at run time
void hb512_col(const void *x, int dtype, int64_t n, const HbFeature &f, const float *heap, uint8_t *out);
void hb512_rows(const void *x, int dtype, int64_t rs, int64_t n, const HbFeature *feat, int nf, const float *heap, uint8_t *out, int64_t ldo);

// A column of a table in host memory.
struct HbColumn {
    const char *data;
    int64_t stride; // bytes
    int32_t dtype;
};
// n values of a column, from row r0, as Float64
void hb_column_f64(const HbColumn &c, int64_t r0, int64_t n, double *out);
// bins of every row of `nc` columns (column j to out + j * n): the search of off[j + 1] - off[j] edges, or value + 1 where there are none
void hb_bin_columns(const HbColumn *cols, int nc, int64_t n, const double *edges, const int32_t *off, uint8_t *out);
// out[j * nr + i] = the ranks[i]-th smallest (from 0, ascending ranks) of column j's values at the rows idx[0 .. n) (all rows when idx is NULL);
// a column with a NaN among them gets NaN throughout
void hb_order_stats(const HbColumn *cols, int nc, const int64_t *idx, int64_t n, const int64_t *ranks, int nr, double *out);

// step() again and again on up to n worker threads (fewer, or none, when others use them) until it returns false: no task is left.  A
// task is short (tens of us): between two of them a worker may move to another caller's region, and come back.  join() waits for
// the workers that are in a task, and throws what a task threw first (failed(): no further one is begun); what no worker has taken
// by then is the caller's to do.
class HbWorkers {
    struct State;
    std::unique_ptr<State> state;

  public:
    HbWorkers(int n, std::function<bool()> step);
    ~HbWorkers();
    HbWorkers(const HbWorkers &) = delete;
    bool failed() const;
    bool none() const; // no worker is at it now: the caller does its tasks itself
    void join();
};
// fn(0) .. fn(ntasks - 1) on the calling thread and up to nworkers more; all are done when it returns
void hb_parallel(int ntasks, int nworkers, const std::function<void(int)> &fn);
