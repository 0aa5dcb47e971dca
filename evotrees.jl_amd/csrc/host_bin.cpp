#include "host_bin.h"

#include <math.h>
#include <sched.h>
#include <stdio.h>
#include <string.h>
#include <unistd.h>

#include <algorithm>
#include <condition_variable>
#include <exception>
#include <mutex>
#include <thread>

bool hb_has_avx512() {
#if defined(__x86_64__)
    static const bool has = __builtin_cpu_supports("avx512f") && __builtin_cpu_supports("avx512bw") && __builtin_cpu_supports("avx512vl") &&
                            __builtin_cpu_supports("avx512dq");
    return has;
#else
    return false;
#endif
}

// Cores that the container's CPU quota pays for (a process that runs on more is stopped for the rest of each period), or no limit.
static int quota_cores(const char *cpu_max, const char *cfs_quota, const char *cfs_period) {
    auto words = [](const char *path, long long *v, int most) { // the numbers a file starts with
        int n = 0;
        if (FILE *f = fopen(path, "r")) {
            while (n < most && fscanf(f, "%lld", &v[n]) == 1) n++;
            fclose(f);
        }
        return n;
    };
    long long v[2];
    const bool have = words(cpu_max, v, 2) == 2 || (words(cfs_quota, v, 1) == 1 && words(cfs_period, v + 1, 1) == 1);
    return have && v[0] > 0 && v[1] > 0 ? (int)std::max(1ll, std::min(1ll << 20, (v[0] + v[1] - 1) / v[1])) : 1 << 20;
}
int hb_cores() {
    static const int quota = quota_cores("/sys/fs/cgroup/cpu.max", "/sys/fs/cgroup/cpu/cpu.cfs_quota_us", "/sys/fs/cgroup/cpu/cpu.cfs_period_us");
    cpu_set_t set;
    const int mine = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : (int)std::thread::hardware_concurrency();
    return std::max(1, std::min(mine, quota));
}
int hb_workers(int64_t cells) {
    // a worker takes about 5 us to wake, in which the calling thread bins 8k cells
    const int64_t worth = cells / 16384 - 1;
    return worth <= 0 ? 0 : (int)std::min<int64_t>(hb_cores() - 1, worth);
}

// The worker threads: started when first needed, kept asleep between calls (waking one costs about 5 us, starting one 15 and more), at
// most one per core less the caller's in the whole process.  Any number of regions use them at a time, each caller beside its own:
// a worker that comes free joins the region with the fewest, and between two tasks leaves one that has more than its share while
// another waits.
namespace {
struct Region {
    const std::function<bool()> *step;
    int wanted;                // workers that may still join; changed under Pool::m, as `active` is
    std::atomic<int> active{0};
    bool closed = false;
    std::atomic<bool> failed{false};
    std::exception_ptr error; // the first exception of a task; the caller's to throw
    cpu_set_t cpus;           // the caller's: its workers run there too
};
struct Pool {
    const pid_t pid = getpid();
    int most = 0; // threads: the most that a region has asked for, each caller's cores less one
    std::mutex m;
    std::condition_variable cv, cv_done;
    int threads = 0;
    std::vector<Region *> regions;
    std::atomic<int> open{0}; // regions, for a look without the lock
    Region *hungriest() {
        Region *best = nullptr;
        for (Region *r : regions)
            if (r->wanted > 0 && (!best || r->active.load() < best->active.load())) best = r;
        return best;
    }
    bool should_leave(const Region *r) { // one worker more there than here would still be no more than here now
        if (open.load(std::memory_order_relaxed) < 2) return false;
        std::lock_guard<std::mutex> lk(m);
        for (const Region *o : regions)
            if (o != r && o->wanted > 0 && o->active + 1 < r->active) return true;
        return false;
    }
    void loop() {
        cpu_set_t cpus;
        CPU_ZERO(&cpus);
        std::unique_lock<std::mutex> lk(m);
        for (;;) {
            Region *r;
            cv.wait(lk, [&] { return (r = hungriest()) != nullptr; });
            r->wanted--;
            r->active++;
            lk.unlock();
            if (!CPU_EQUAL(&cpus, &r->cpus)) {
                cpus = r->cpus;
                (void)sched_setaffinity(0, sizeof(cpus), &cpus); // of this thread
            }
            bool more = true, leave = false;
            std::exception_ptr error;
            try {
                while (!leave && (more = !r->failed.load(std::memory_order_relaxed) && (*r->step)())) leave = should_leave(r);
            } catch (...) {
                error = std::current_exception();
                more = false;
            }
            lk.lock();
            if (error && !r->failed.exchange(true)) r->error = error;
            if (!more) r->wanted = 0; // nothing left to hand out
            else if (!r->closed) r->wanted++;
            if (--r->active == 0) cv_done.notify_all();
        }
    }
    void enter(Region *r) {
        const int n = r->wanted;
        {
            std::lock_guard<std::mutex> lk(m);
            regions.push_back(r);
            open.store((int)regions.size(), std::memory_order_relaxed);
            most = std::max(most, n);
            int need = 0;
            for (const Region *o : regions) need += o->wanted + o->active;
            try {
                for (; threads < std::min(need, most); threads++) std::thread([this] { loop(); }).detach();
            } catch (const std::exception &) { // no more threads to be had: the callers do their work themselves
            }
        }
        for (int i = 0; i < n; i++) cv.notify_one(); // the lock is free: a worker that wakes does not wait for it
    }
    void leave(Region *r) { // workers that have not joined by now do not; those that have are waited for
        std::unique_lock<std::mutex> lk(m);
        r->closed = true;
        r->wanted = 0;
        cv_done.wait(lk, [&] { return r->active == 0; });
        regions.erase(std::find(regions.begin(), regions.end(), r));
        open.store((int)regions.size(), std::memory_order_relaxed);
    }
    static Pool &get() { // never destroyed: its threads outlive main.  After a fork the child has none of them and starts afresh
        static std::mutex gm;
        static Pool *p = nullptr;
        std::lock_guard<std::mutex> lk(gm);
        if (!p || p->pid != getpid()) p = new Pool();
        return *p;
    }
};
} // namespace

struct HbWorkers::State {
    std::function<bool()> step;
    Pool &pool;
    Region region;
    State(int n, std::function<bool()> &&f) : step(std::move(f)), pool(Pool::get()) {
        region.step = &step;
        region.wanted = n;
        CPU_ZERO(&region.cpus);
        (void)sched_getaffinity(0, sizeof(region.cpus), &region.cpus);
    }
};
HbWorkers::HbWorkers(int n, std::function<bool()> step) {
    if (n <= 0) return;
    std::unique_ptr<State> s(new State(n, std::move(step)));
    s->pool.enter(&s->region);
    state = std::move(s);
}
bool HbWorkers::none() const { return !state || state->region.active.load(std::memory_order_relaxed) == 0; }
bool HbWorkers::failed() const { return state && state->region.failed.load(std::memory_order_relaxed); }
void HbWorkers::join() {
    if (!state) return;
    const std::unique_ptr<State> s = std::move(state);
    s->pool.leave(&s->region);
    if (s->region.error) std::rethrow_exception(s->region.error);
}
HbWorkers::~HbWorkers() {
    if (!state) return;
    state->region.failed.store(true); // left by an exception or an error: no further task
    state->pool.leave(&state->region);
}

void hb_parallel(int ntasks, int nworkers, const std::function<void(int)> &fn) {
    const int n = std::min(nworkers, ntasks - 1);
    if (n <= 0) { // the leaf ids of one row, 62 trees: 0.8 us of 23 less than by way of a region
        for (int t = 0; t < ntasks; t++) fn(t);
        return;
    }
    std::atomic<int> next{0};
    auto step = [&]() -> bool {
        const int t = next.fetch_add(1, std::memory_order_relaxed);
        if (t >= ntasks) return false;
        fn(t);
        return true;
    };
    HbWorkers ws(n, step);
    while (!ws.failed() && step()) {
    }
    ws.join();
}

// Float32 neighbours of a Float64 value: the largest not above it, the smallest not below it
static float round_down(double v) {
    const float f = (float)v;
    return (double)f > v ? nextafterf(f, -INFINITY) : f;
}
static float round_up(double v) {
    const float f = (float)v;
    return (double)f < v ? nextafterf(f, INFINITY) : f;
}

static void fill_heap(const float *sorted, int n, int levels, float *heap) {
    // node h of level l (from the top, 0) is element (2 (h - 2^l) + 1) 2^(levels - 1 - l) - 1 of the sorted list
    const int cap = (1 << levels) - 1;
    heap[0] = 0.0f;
    for (int l = 0; l < levels; l++)
        for (int k = 0; k < (1 << l); k++) {
            const int at = (2 * k + 1) * (1 << (levels - 1 - l)) - 1;
            heap[(1 << l) + k] = at < n && at < cap ? sorted[at] : INFINITY;
        }
}

// The search runs on Float32 keys and is exact all the same.  A Float32 value x passes the Float64 edge e iff it passes
// the largest Float32 not above e.  A Float64 value is rounded up to a Float32 key, as the edges are: rounding up keeps
// the order, so different keys order as the values do; equal keys leave it open (unless every edge IS a Float32: then a
// value rounded up passes an edge iff it did before), and the value is compared with the edges of that key in Float64.
void HbPlan::build(const double *edges_flat, const int32_t *off, int F_, int dtype_) {
    F = F_;
    dtype = dtype_;
    edges.assign(edges_flat, edges_flat + off[F]);
    feat.resize(F);
    int64_t words = 0;
    for (int j = 0; j < F; j++) {
        HbFeature &f = feat[j];
        f.ne = off[j + 1] - off[j];
        f.e = edges.data() + off[j];
        f.levels = 4;
        while ((1 << f.levels) - 1 < f.ne && f.levels < 8) f.levels++;
        f.heap = (int32_t)words;
        words += std::max(16, 1 << f.levels);
    }
    heap_store.resize((size_t)words + 16);
    heap = reinterpret_cast<float *>((reinterpret_cast<uintptr_t>(heap_store.data()) + 63) & ~(uintptr_t)63);
    std::vector<float> key;
    for (int j = 0; j < F; j++) {
        HbFeature &f = feat[j];
        key.resize(std::max(1, f.ne));
        bool slow = f.ne > 254, all32 = true;
        for (int i = 0; i < f.ne; i++) {
            const double e = f.e[i];
            slow |= e != e || (e == 0.0 && signbit(e)) || (i > 0 && !(f.e[i - 1] <= e));
            key[i] = dtype == EVT_F32 ? round_down(e) : round_up(e);
            all32 &= (double)key[i] == e;
        }
        f.flags = (slow ? HB_SLOW : 0) | (dtype == EVT_F32 || all32 ? HB_EXACT : 0);
        fill_heap(key.data(), f.ne, f.levels, heap + f.heap);
    }
}

// Julia's isless on Float64: NaN after everything, -0.0 before 0.0
static inline bool isless_f64(double a, double b) {
    if (a != a) return false;
    if (b != b) return true;
    if (a == 0.0 && b == 0.0) return signbit(a) && !signbit(b);
    return a < b;
}
static inline uint8_t bin_one(const HbFeature &f, double v) {
    if (f.flags & HB_SLOW) {
        int lo = 0, hi = f.ne;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (isless_f64(f.e[mid], v)) lo = mid + 1;
            else hi = mid;
        }
        return (uint8_t)(lo + 1);
    }
    const double *b = f.e; // !(e >= v): passes the edges below v, and all of them when v is NaN
    int n = f.ne;
    while (n > 0) {
        const int half = n >> 1;
        const bool right = !(b[half] >= v);
        b = right ? b + half + 1 : b;
        n = right ? n - half - 1 : half;
    }
    return (uint8_t)(b - f.e + 1);
}
template <typename T>
static void bin_strided(const HbFeature &f, const T *x, int64_t stride, int64_t n, uint8_t *out) {
    for (int64_t i = 0; i < n; i++) out[i] = bin_one(f, (double)x[i * stride]);
}
static void bin_plain(const HbFeature &f, const HbSource &S, const char *x, int64_t n, uint8_t *out) {
    if (S.dtype == EVT_F32) bin_strided(f, reinterpret_cast<const float *>(x), S.rs, n, out);
    else bin_strided(f, reinterpret_cast<const double *>(x), S.rs, n, out);
}

void hb_bin(const HbPlan &P, const HbSource &S, int64_t r0, int64_t n, int f0, int f1, uint8_t *out, int64_t ldo) {
    const size_t es = S.esize();
    const char *base = static_cast<const char *>(S.base) + es * (size_t)r0 * S.rs;
    const bool wide = hb_has_avx512() && n >= 16; // a few rows: a scalar search each costs less than filling vectors
    if (wide && S.rows_contiguous()) hb512_rows(base + es * f0, S.dtype, S.rs, n, P.feat.data() + f0, f1 - f0, P.heap, out, ldo);
    for (int f = f0; f < f1; f++) {
        const char *x = base + es * (size_t)f * S.cs;
        uint8_t *o = out + (size_t)(f - f0) * ldo;
        if (!wide || (P.feat[f].flags & HB_SLOW)) bin_plain(P.feat[f], S, x, n, o);
        else if (!S.rows_contiguous()) hb512_col(x, S.dtype, n, P.feat[f], P.heap, o);
    }
}

// ---- tables -----------------------------------------------------------------------------------
template <typename T>
static void gather_f64(const HbColumn &c, int64_t r0, int64_t n, double *out) {
    const char *p = c.data + r0 * c.stride;
    for (int64_t i = 0; i < n; i++, p += c.stride) {
        T v;
        memcpy(&v, p, sizeof(T));
        out[i] = (double)v;
    }
}
void hb_column_f64(const HbColumn &c, int64_t r0, int64_t n, double *out) {
    switch (c.dtype) {
        case EVT_F32: return gather_f64<float>(c, r0, n, out);
        case EVT_F64: return gather_f64<double>(c, r0, n, out);
        case EVT_I8: return gather_f64<int8_t>(c, r0, n, out);
        case EVT_I16: return gather_f64<int16_t>(c, r0, n, out);
        case EVT_I32: return gather_f64<int32_t>(c, r0, n, out);
        case EVT_I64: return gather_f64<int64_t>(c, r0, n, out);
        case EVT_U8: return gather_f64<uint8_t>(c, r0, n, out);
        case EVT_U16: return gather_f64<uint16_t>(c, r0, n, out);
        case EVT_U32: return gather_f64<uint32_t>(c, r0, n, out);
        default: return gather_f64<uint64_t>(c, r0, n, out);
    }
}
void hb_bin_columns(const HbColumn *cols, int nc, int64_t n, const double *edges, const int32_t *off, uint8_t *out) {
    HbPlan P;
    P.build(edges, off, nc, EVT_F64);
    const int64_t block = 4096; // 32 KB of Float64: stays in the core's own cache
    const int64_t nb = (n + block - 1) / block;
    hb_parallel((int)(nb * nc), hb_workers(n * nc), [&](int t) {
        const int j = (int)(t / nb);
        const int64_t r0 = (t % nb) * block, m = std::min(block, n - r0);
        double buf[4096];
        hb_column_f64(cols[j], r0, m, buf);
        uint8_t *o = out + (size_t)j * n + r0;
        if (P.feat[j].ne == 0) {
            for (int64_t i = 0; i < m; i++) o[i] = (uint8_t)(buf[i] + 1.0);
        } else {
            hb_bin(P, HbSource{buf, EVT_F64, 1, 0}, 0, m, j, j + 1, o, m); // column stride 0: `buf` is column j
        }
    });
}

// ---- order statistics -------------------------------------------------------------------------
// The ranks asked for (63 of 64000 values, say) touch few values once these are dealt into buckets: one pass finds the range, one
// counts equal slices of it, one collects the slices that hold a rank; those are sorted, or dealt again while they are large
// (skewed values).  O(n): 0.25 ms for 64000 values where selecting them one after the other takes 1.2 ms.
template <typename T>
static void select_ranks(T *v, int64_t n, const int64_t *ranks, int nr, double *out, int depth, std::vector<uint16_t> &scratch) {
    if (nr == 0) return;
    T lo = v[0], hi = v[0];
    for (int64_t i = 1; i < n; i++) {
        lo = v[i] < lo ? v[i] : lo;
        hi = v[i] > hi ? v[i] : hi;
    }
    const double width = (double)hi - (double)lo;
    // sorted where the slices have no width that Float64 holds: all values equal (0), an infinity among them (inf), or so close that
    // nb / width would overflow (denormals, also those that a skewed column leaves in one slice)
    if (n <= 64 || depth >= 8 || !(width > 1e-300 && width < 1e300)) {
        if (hi > lo) std::sort(v, v + n);
        for (int i = 0; i < nr; i++) out[i] = (double)v[ranks[i]];
        return;
    }
    int nb = 64; // counts and places of 4096 slices stay in the core's first cache; a slice's sixteen or so values are sorted in no time
    while (nb < n / 2 && nb < 4096) nb <<= 1;
    const double l = (double)lo, scale = (double)nb / width;
    // (v - lo) * scale lies in [0, nb] up to rounding and is monotone in v, in rounded arithmetic too: a bucket's values all lie
    // between its neighbours'
    std::vector<uint32_t> first((size_t)nb + 1, 0);
    scratch.resize((size_t)n);
    uint16_t *bucket = scratch.data();
    for (int64_t i = 0; i < n; i++) {
        int b = (int)(((double)v[i] - l) * scale);
        b = b < nb ? b : nb - 1;
        bucket[i] = (uint16_t)b;
        first[b + 1]++;
    }
    for (int b = 0; b < nb; b++) first[b + 1] += first[b];
    // the buckets that hold a rank, in order; kept[b] = where its values are collected (from 1; 0: not asked for)
    std::vector<uint32_t> kept((size_t)nb, 0);
    std::vector<int> held;
    int64_t total = 0;
    for (int i = 0, b = 0; i < nr; i++) {
        while ((int64_t)first[b + 1] <= ranks[i]) b++;
        if (held.empty() || held.back() != b) {
            held.push_back(b);
            kept[b] = (uint32_t)total + 1;
            total += first[b + 1] - first[b];
        }
    }
    std::vector<T> part((size_t)total);
    for (int64_t i = 0; i < n; i++)
        if (uint32_t &k = kept[bucket[i]]) part[(size_t)(k++ - 1)] = v[i];
    std::vector<int64_t> sub;
    int i = 0;
    int64_t at = 0;
    for (int b : held) {
        const int64_t m = first[b + 1] - first[b];
        sub.clear();
        int i1 = i;
        for (; i1 < nr && ranks[i1] < (int64_t)first[b + 1]; i1++) sub.push_back(ranks[i1] - first[b]);
        select_ranks(part.data() + at, m, sub.data(), i1 - i, out + i, depth + 1, scratch);
        i = i1;
        at += m;
    }
}
template <typename T>
static void order_stats_of(T *v, int64_t n, const int64_t *ranks, int nr, double *out, std::vector<uint16_t> &scratch) {
    bool nan = false;
    for (int64_t i = 0; i < n; i++) nan |= v[i] != v[i];
    if (nan) std::fill(out, out + nr, (double)NAN);
    else select_ranks(v, n, ranks, nr, out, 0, scratch);
}

// neighbouring columns of a matrix whose rows are contiguous are gathered together: a sampled row's cache line is read once
template <typename T>
static void order_stats_group(const HbColumn *cols, int g, const int64_t *idx, int64_t n, const int64_t *ranks, int nr, double *out) {
    std::vector<T> v((size_t)g * n);
    std::vector<uint16_t> scratch;
    for (int64_t i = 0; i < n; i++) {
        if (idx && i + 32 < n) { // sampled rows lie apart: their lines are asked for ahead (64000 of 500k rows x 50 columns 2.3 -> 0.9 ms, of 1M x 100 3.3 -> 1.2)
            const char *q = cols[0].data + idx[i + 32] * cols[0].stride;
            __builtin_prefetch(q);
            __builtin_prefetch(q + g * sizeof(T) - 1);
        }
        const char *p = cols[0].data + (idx ? idx[i] : i) * cols[0].stride;
        for (int j = 0; j < g; j++) {
            T t;
            memcpy(&t, p + j * sizeof(T), sizeof(T));
            v[(size_t)j * n + i] = t;
        }
    }
    for (int j = 0; j < g; j++) order_stats_of(v.data() + (size_t)j * n, n, ranks, nr, out + (size_t)j * nr, scratch);
}

void hb_order_stats(const HbColumn *cols, int nc, const int64_t *idx, int64_t n, const int64_t *ranks, int nr, double *out) {
    auto size = [](int32_t d) { return d == EVT_F32 ? (int64_t)4 : (int64_t)8; };
    // the groups: up to 8 columns side by side in memory, fewer where cores would be left without one; or one.  (16 cores, 64000 rows: 10 columns in
    // groups of 8 2.2 ms, of one 0.46; 50 columns in groups of 8 3.9, of 4 2.3.)
    const int workers = hb_workers(n * nc), most = std::max(1, std::min(8, (nc + workers) / (workers + 1)));
    std::vector<int> start;
    for (int j = 0; j < nc; j++) {
        const int f = start.empty() ? -1 : start.back();
        const bool join = f >= 0 && j - f < most && cols[j].dtype == cols[f].dtype && cols[f].dtype <= EVT_F64 && cols[j].stride == cols[f].stride &&
                          cols[f].stride > size(cols[f].dtype) && cols[j].data - cols[f].data == (j - f) * size(cols[f].dtype);
        if (!join) start.push_back(j);
    }
    start.push_back(nc);
    hb_parallel((int)start.size() - 1, workers, [&](int t) {
        const HbColumn *c = cols + start[t];
        const int g = start[t + 1] - start[t];
        double *o = out + (size_t)start[t] * nr;
        if (c->dtype == EVT_F32) {
            order_stats_group<float>(c, g, idx, n, ranks, nr, o);
        } else if (c->dtype == EVT_F64) {
            order_stats_group<double>(c, g, idx, n, ranks, nr, o);
        } else {
            std::vector<double> v((size_t)n);
            std::vector<uint16_t> scratch;
            if (!idx) hb_column_f64(*c, 0, n, v.data());
            else
                for (int64_t i = 0; i < n; i++) hb_column_f64(*c, idx[i], 1, &v[(size_t)i]);
            order_stats_of(v.data(), n, ranks, nr, o, scratch);
        }
    });
}
