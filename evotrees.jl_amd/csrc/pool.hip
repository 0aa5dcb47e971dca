#include "pool.h"

#include <map>
#include <mutex>
#include <unordered_map>

namespace {

std::mutex g_mu;
struct Block {
    size_t size;
    int device;
};
enum { DEVICE, PINNED, COHERENT, KINDS };
std::unordered_map<void *, Block> g_out[KINDS];                        // blocks in use
std::multimap<std::pair<int, size_t>, void *> g_idle[KINDS];           // by (device, size); pinned blocks under device 0
std::map<int, size_t> g_kept[KINDS];                                   // idle bytes by device
std::map<int, std::vector<hipStream_t>> g_streams[2];                  // idle ones by device, the last used at the end: blocking, non-blocking
const size_t STREAMS_KEPT = 16; // per device and kind

// sizes are rounded up by an eighth at most, so that inputs of about the same size find each other's blocks; those of blocks that are
// never kept only to whole pages
size_t size_class(size_t n) {
    if (n > POOL_BLOCK_KEPT) return (n + 4095) / 4096 * 4096;
    size_t step = 4096;
    while (step * 16 <= n) step <<= 1;
    return (n + step - 1) / step * step;
}
int current_device() {
    int d = 0;
    return hipGetDevice(&d) == hipSuccess ? d : 0;
}
void release(int kind, void *p) {
    if (kind == DEVICE) (void)hipFree(p);
    else (void)hipHostFree(p);
}
void trim(int kind) {
    std::vector<void *> idle;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        for (auto &e : g_idle[kind]) idle.push_back(e.second);
        g_idle[kind].clear();
        g_kept[kind].clear();
    }
    for (void *p : idle) release(kind, p);
}
void *take(int kind, size_t bytes) {
    const int dev = kind == DEVICE ? current_device() : 0;
    const size_t n = size_class(bytes ? bytes : 1);
    {
        std::lock_guard<std::mutex> lk(g_mu);
        auto it = g_idle[kind].find({dev, n});
        if (it != g_idle[kind].end()) {
            void *p = it->second;
            g_idle[kind].erase(it);
            g_kept[kind][dev] -= n;
            g_out[kind][p] = {n, dev};
            return p;
        }
    }
    void *p = nullptr;
    hipError_t e = hipSuccess;
    for (int attempt = 0; attempt < 2; attempt++) {
        e = kind == DEVICE ? hipMalloc(&p, n) : hipHostMalloc(&p, n, hipHostMallocPortable | (kind == COHERENT ? hipHostMallocCoherent : 0u));
        if (e == hipSuccess) break;
        (void)hipGetLastError();
        // idle blocks of other sizes make room
        if (kind == DEVICE) trim(DEVICE);
        else trim(PINNED), trim(COHERENT);
    }
    if (e != hipSuccess) {
        evt_set_error("%s of %zu bytes failed: %s", kind == DEVICE ? "hipMalloc" : "hipHostMalloc", n, hipGetErrorString(e));
        return nullptr;
    }
    if (kind != DEVICE) {
        void *d = nullptr;
        if (hipHostGetDevicePointer(&d, p, 0) != hipSuccess || d != p) {
            evt_set_error("pinned memory is not addressable from the device");
            release(kind, p);
            return nullptr;
        }
    }
    std::lock_guard<std::mutex> lk(g_mu);
    g_out[kind][p] = {n, dev};
    return p;
}
void give(int kind, void *p) {
    if (!p) return;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        auto it = g_out[kind].find(p);
        if (it != g_out[kind].end()) {
            const Block b = it->second;
            g_out[kind].erase(it);
            if (b.size <= POOL_BLOCK_KEPT && g_kept[kind][b.device] + b.size <= (kind == DEVICE ? POOL_DEVICE_KEPT : POOL_PINNED_KEPT)) {
                g_idle[kind].insert({{b.device, b.size}, p});
                g_kept[kind][b.device] += b.size;
                return;
            }
        }
    }
    release(kind, p);
}

} // namespace

void *dev_take(size_t bytes) { return take(DEVICE, bytes); }
void dev_give(void *p) { give(DEVICE, p); }
void *pinned_take(size_t bytes) { return take(PINNED, bytes); }
void pinned_give(void *p) { give(PINNED, p); }
void *coherent_take(size_t bytes) { return take(COHERENT, bytes); }
void coherent_give(void *p) { give(COHERENT, p); }

hipError_t stream_take(hipStream_t *s, bool non_blocking) {
    const int dev = current_device();
    {
        std::lock_guard<std::mutex> lk(g_mu);
        std::vector<hipStream_t> &idle = g_streams[non_blocking][dev];
        if (!idle.empty()) {
            *s = idle.back();
            idle.pop_back();
            return hipSuccess;
        }
    }
    return hipStreamCreateWithFlags(s, non_blocking ? hipStreamNonBlocking : hipStreamDefault);
}
void stream_give(hipStream_t s, bool non_blocking, int dev) {
    {
        std::lock_guard<std::mutex> lk(g_mu);
        std::vector<hipStream_t> &idle = g_streams[non_blocking][dev];
        if (idle.size() < STREAMS_KEPT) {
            idle.push_back(s);
            return;
        }
    }
    (void)hipStreamDestroy(s);
}

extern "C" int evt_trim(void) {
    return guarded([&]() -> int {
    models_trim();
    for (int k = 0; k < KINDS; k++) trim(k);
    std::vector<hipStream_t> idle;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        for (auto &q : g_streams) {
            for (auto &e : q) idle.insert(idle.end(), e.second.begin(), e.second.end());
            q.clear();
        }
    }
    for (hipStream_t s : idle) (void)hipStreamDestroy(s);
    return EVT_OK;
    });
}
