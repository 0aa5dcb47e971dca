// Data-layout kernels: observation-major copy of x_bin, device binarize, small fills.
#include "evt_internal.h"

// 4 and 16 bytes from any address
__device__ __forceinline__ uint32_t load4(const uint8_t *p) {
    uint32_t v;
    __builtin_memcpy(&v, p, 4);
    return v;
}
__device__ __forceinline__ uint4 load16(const uint8_t *p) {
    uint4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}
// 4 x 4 bytes: byte j of v[i] becomes byte i of v[j]
__device__ __forceinline__ void transpose4(uint32_t (&v)[4]) {
    const uint32_t a = __builtin_amdgcn_perm(v[1], v[0], 0x05010400u), b = __builtin_amdgcn_perm(v[3], v[2], 0x05010400u); // 0.0 1.0 0.1 1.1 | 2.0 3.0 2.1 3.1
    const uint32_t c = __builtin_amdgcn_perm(v[1], v[0], 0x07030602u), d = __builtin_amdgcn_perm(v[3], v[2], 0x07030602u);
    v[0] = __builtin_amdgcn_perm(b, a, 0x05040100u);
    v[1] = __builtin_amdgcn_perm(b, a, 0x07060302u);
    v[2] = __builtin_amdgcn_perm(d, c, 0x05040100u);
    v[3] = __builtin_amdgcn_perm(d, c, 0x07060302u);
}

// x_bin column by column -> the observation-major records.  Bins outside 1..B raise the device error flag (the histogram kernels index LDS with them).
// Padding bytes of a record are set to 1, so that a kernel may index with them unchecked.
// Byte p of a record holds feature (p / PBL) * PU + p % PBL when p % PBL < PU, padding otherwise (evt_ctx::PBL).
// A block takes 256 rows of up to 128 bytes of their records: a lane loads four rows of four columns, a word each, and what it has is transposed in registers and
// put together in LDS, so that whole lines are read and written.  Bound by the bytes.  10M rows x 100 (1.0 GB read, 1.28 written) 3.6 ms -> 0.57 ms, 1M x 100 0.25 -> 0.064, with 16-byte pieces of
// records written by a thread that loaded single bytes before.
#define TR_ROWS 256
#define TR_BYTES 128
__global__ __launch_bounds__(256) void k_transpose_validate(const uint8_t *__restrict__ xcm, uint8_t *__restrict__ xrm,
                                                           int64_t N, int F, int B, int RS, int PBL, int PU, int32_t *errflag) {
    constexpr int LD = TR_BYTES / 4 + 1; // words from row to row: lanes four rows apart write to 16 banks
    __shared__ uint32_t s_rec[TR_ROWS * LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t row0 = (int64_t)blockIdx.x * TR_ROWS, row = row0 + 4 * lane;
    const int p0 = blockIdx.y * TR_BYTES, nw = min(TR_BYTES, RS - p0) >> 2; // words of a record here
    const bool whole = row + 4 <= N;
    bool bad = false;
    for (int w = wave; w < nw; w += 4) {
        uint32_t v[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int p = p0 + 4 * w + t, f = (p / PBL) * PU + p % PBL;
            v[t] = 0x01010101u; // padding reads as bin 1: always a valid histogram index
            if (p % PBL < PU && f < F) {
                const uint8_t *col = xcm + (size_t)f * N;
                if (whole) {
                    v[t] = load4(col + row);
                } else {
                    for (int i = 0; i < 4; i++)
                        if (row + i < N) v[t] = (v[t] & ~(0xFFu << (8 * i))) | ((uint32_t)col[row + i] << (8 * i));
                }
            }
        }
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) bad |= ((v[t] >> (8 * i)) & 0xFFu) - 1u >= (uint32_t)B;
        transpose4(v);
#pragma unroll
        for (int i = 0; i < 4; i++) s_rec[(4 * lane + i) * LD + w] = v[i];
    }
    if (bad) atomicOr(errflag, 1);
    __syncthreads();
    const int n16 = nw >> 2; // 16 bytes of a record at a time: a record is a multiple of them
    const int64_t rows = N - row0 < TR_ROWS ? N - row0 : TR_ROWS;
    for (int k = tid; k < TR_ROWS * n16; k += 256) {
        const int r = k / n16, q = k - r * n16;
        if (r >= rows) break;
        const uint32_t *s = s_rec + r * LD + 4 * q;
        *reinterpret_cast<uint4 *>(xrm + (size_t)(row0 + r) * RS + p0 + 16 * q) = make_uint4(s[0], s[1], s[2], s[3]);
    }
}

int launch_transpose_validate(evt_ctx *c) {
    dim3 grid((unsigned)((c->N + TR_ROWS - 1) / TR_ROWS), (unsigned)((c->RS + TR_BYTES - 1) / TR_BYTES));
    hipLaunchKernelGGL(k_transpose_validate, grid, dim3(256), 0, c->stream, c->xcm, c->xrm, c->N, c->F, c->B, c->RS, c->PBL, c->PU, c->errflag);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

// Threshold bit planes of x_bin: word w of plane (f, b) holds, for rows 32 w .. 32 w + 31, the bit x_bin[row, f] <= b.
// One thread reads its 32 bins once and writes one word of each of the feature's B - 1 planes (consecutive threads,
// consecutive words).  Rows past the end read as bin 255: their bits are 0 in every plane.
// The 32 bins are turned into eight words of one bit each, on which a comparison of all 32 with b is a few instructions: with b = 16 H + L, below H in the high
// four bits, or equal there and at most L in the low ones - one instruction and a store for a plane.  Bound by the planes' bytes.  10M rows x 100 of 64 bins
// (7.9 GB) 4.15 ms -> 1.80 with 32 comparisons a word before, 1M x 28 of 128 bins 0.26 -> 0.071.
__global__ __launch_bounds__(256) void k_build_planes(const uint8_t *__restrict__ xcm, uint32_t *__restrict__ planes, int64_t N, int B,
                                                     int64_t W) {
    const int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int f = blockIdx.y;
    if (w >= W) return;
    const uint8_t *col = xcm + (size_t)f * N;
    uint32_t v[8]; // bytes: rows 4 i .. 4 i + 3
    if (32 * w + 32 <= N) {
        const uint4 a = load16(col + 32 * w), b = load16(col + 32 * w + 16);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            v[i] = 0xFFFFFFFFu;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int64_t row = 32 * w + 4 * i + k;
                if (row < N) v[i] = (v[i] & ~(0xFFu << (8 * k))) | ((uint32_t)col[row] << (8 * k));
            }
        }
    }
    // bits[j]: bit j of the 32 bins.  Bit j of a word's four bytes (places 0, 8, 16, 24) is gathered to its low four by one multiplication.
    uint32_t bits[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        bits[j] = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) bits[j] |= ((((v[i] >> j) & 0x01010101u) * 0x01020408u) >> 24 & 0xFu) << (4 * i);
    }
    uint32_t le[16]; // low four bits at most L
    {
        uint32_t eq, lt = 0;
#pragma unroll
        for (int L = 0; L < 16; L++) {
            eq = (L & 1 ? bits[0] : ~bits[0]) & (L & 2 ? bits[1] : ~bits[1]) & (L & 4 ? bits[2] : ~bits[2]) & (L & 8 ? bits[3] : ~bits[3]);
            lt |= eq;
            le[L] = lt;
        }
    }
    uint32_t *out = planes + ((size_t)f * (B - 1)) * W + w - W; // plane b at out + b * W
    uint32_t below = 0;                                         // high four bits below H
    for (int H = 0; 16 * H < B; H++) {
        uint32_t eq = ~0u;
#pragma unroll
        for (int j = 0; j < 4; j++) eq &= (H >> j) & 1 ? bits[4 + j] : ~bits[4 + j];
#pragma unroll
        for (int L = 0; L < 16; L++) {
            const int b = 16 * H + L;
            if (b >= 1 && b < B) out[(size_t)b * W] = below | (eq & le[L]);
        }
        below |= eq;
    }
}

int launch_build_planes(evt_ctx *c) {
    dim3 grid((unsigned)((c->plane_words + 255) / 256), (unsigned)c->F);
    hipLaunchKernelGGL(k_build_planes, grid, dim3(256), 0, c->stream, c->xcm, c->planes, c->N, c->B, c->plane_words);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

// Julia's isless on Float64 (the default order of searchsortedfirst): IEEE `<`, except that NaN sorts after everything and
// -0.0 before 0.0.
__device__ __forceinline__ bool jl_isless(double a, double b) {
    if (a != a) return false;
    if (b != b) return true;
    if (a == 0.0 && b == 0.0) return (__double_as_longlong(a) < 0) && (__double_as_longlong(b) >= 0);
    return a < b;
}

// searchsortedfirst(edges_j, x) = 1 + number of edges that are isless than x (src/fit-utils.jl:69); a NaN lands in the last bin.
// Element (i, j) of x at i * rs + j * cs.  A block takes 16 features, whose edges it holds in LDS (32 KB: four blocks a compute unit), so
// that a thread's 16 loads of a row are two or one 64-byte lines where rows are contiguous, and a wavefront's are where columns
// are; its stores are the consecutive rows of a column either way.  evt_binarize_f64 of 2M x 50 values on the device, records and all:
// 0.63 ms (a block per feature with that one's edges: 0.66); behind the bus (19 ms for these) its time does not show.
template <typename T>
__global__ __launch_bounds__(256) void k_binarize(const T *__restrict__ x, int64_t rs, int64_t cs, const double *__restrict__ edges,
                                                 const int32_t *__restrict__ edge_off, uint8_t *__restrict__ xcm, int64_t n, int F, int64_t ldo) {
    extern __shared__ double s_edges[]; // of 16 features
    __shared__ int s_off[17];
    const int f0 = blockIdx.y * 16, nf = min(16, F - f0), e0 = edge_off[f0], total = edge_off[f0 + nf] - e0;
    for (int t = threadIdx.x; t < total; t += 256) s_edges[t] = edges[e0 + t];
    if (threadIdx.x <= nf) s_off[threadIdx.x] = edge_off[f0 + threadIdx.x] - e0;
    __syncthreads();
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        T v[16];
#pragma unroll
        for (int k = 0; k < 16; k++) v[k] = k < nf ? x[i * rs + (f0 + k) * cs] : (T)0;
#pragma unroll
        for (int k = 0; k < 16; k++) {
            if (k < nf) {
                const double d = (double)v[k];
                const int first = s_off[k];
                int lo = first, hi = s_off[k + 1];
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (jl_isless(s_edges[mid], d)) lo = mid + 1; else hi = mid;
                }
                xcm[(size_t)(f0 + k) * ldo + i] = (uint8_t)(lo - first + 1);
            }
        }
    }
}

// n rows of F columns of at most max_edges (<= 254) edges each: column j's bins to xcm + j * ldo
int launch_binarize(hipStream_t s, const void *x_dev, int dtype, int64_t rs, int64_t cs, const double *edges_dev, const int32_t *edge_off_dev, int max_edges,
                    uint8_t *xcm, int64_t n, int F, int64_t ldo) {
    ARGCHK(max_edges >= 0 && max_edges <= 254, "at most 254 edges per feature");
    const size_t lds = sizeof(double) * 16 * (max_edges > 0 ? max_edges : 1);
    int64_t nb = (n + 255) / 256;
    if (nb > 4096) nb = 4096;
    const dim3 grid((unsigned)nb, (unsigned)((F + 15) / 16));
    if (dtype == EVT_F32)
        hipLaunchKernelGGL(k_binarize<float>, grid, dim3(256), lds, s, static_cast<const float *>(x_dev), rs, cs, edges_dev, edge_off_dev, xcm, n, F, ldo);
    else
        hipLaunchKernelGGL(k_binarize<double>, grid, dim3(256), lds, s, static_cast<const double *>(x_dev), rs, cs, edges_dev, edge_off_dev, xcm, n, F, ldo);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

__global__ __launch_bounds__(256) void k_iota(uint32_t *dst, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) dst[i] = (uint32_t)i;
}
int launch_iota(evt_ctx *c, uint32_t *dst, int64_t n) {
    int64_t nb = (n + 255) / 256;
    if (nb > 8192) nb = 8192;
    if (nb < 1) nb = 1;
    hipLaunchKernelGGL(k_iota, dim3((unsigned)nb), dim3(256), 0, c->stream, dst, n);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

// A tree's arrays to its pinned slot by a kernel (blob_send: system-scope stores of 8 bytes).  A stream-ordered
// hipMemcpyAsync goes through the copy engine, and handing the stream over to it and back stalls the kernels queued
// behind it for tens of microseconds; a kernel's stores over the bus do not.
__global__ __launch_bounds__(256) void k_copy_to_host(BlobOut O) { blob_send(O, (int)blockIdx.x); }

// the arrays of the tree queued last, to its staging slot
void blob_out(evt_ctx *c, BlobOut &O) {
    O.src = reinterpret_cast<const uint4 *>(c->tree_blob);
    O.dst = reinterpret_cast<uint4 *>(c->h_stage_dev);
    O.n = (int64_t)(c->blob_bytes / 16);
    O.blocks = (int)std::min<int64_t>(64, (O.n + 255) / 256);
    O.arrived = c->blob_arrived;
    O.flag = c->slot_flag[c->slot_w];
    O.seq = (unsigned long long)c->tree_seq;
}
// flag: the tree is finished
int launch_copy_to_host(evt_ctx *c, bool flag) {
    BlobOut O;
    blob_out(c, O);
    if (!flag) O.flag = nullptr;
    hipLaunchKernelGGL(k_copy_to_host, dim3((unsigned)O.blocks), dim3(256), 0, c->stream, O);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

// the same for small pinned host -> device uploads, in 4-byte words
__global__ __launch_bounds__(256) void k_copy_words(const uint32_t *__restrict__ src, uint32_t *__restrict__ dst, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) dst[i] = src[i];
}
int launch_copy_words(evt_ctx *c, const void *src, void *dst, size_t nbytes) {
    const int64_t n = (int64_t)(nbytes / 4);
    if (n <= 0) return EVT_OK;
    int64_t nb = (n + 255) / 256;
    if (nb > 64) nb = 64;
    hipLaunchKernelGGL(k_copy_words, dim3((unsigned)nb), dim3(256), 0, c->stream, static_cast<const uint32_t *>(src), static_cast<uint32_t *>(dst), n);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

__global__ __launch_bounds__(256) void k_fill_u32(uint32_t *dst, uint32_t v, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) dst[i] = v;
}
int launch_fill_u32(evt_ctx *c, uint32_t *dst, uint32_t v, int64_t n) {
    if (n <= 0) return EVT_OK;
    int64_t nb = (n + 255) / 256;
    if (nb > 8192) nb = 8192;
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)nb), dim3(256), 0, c->stream, dst, v, n);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}
// zero-fill of a byte range whose size is a multiple of 4
int launch_fill_bytes(evt_ctx *c, void *dst, int64_t nbytes) { return launch_fill_u32(c, (uint32_t *)dst, 0u, nbytes / 4); }

// grad[NK-1, i] = w[i] (or 1): the weight row is written once (src/init.jl:173-174).
__global__ __launch_bounds__(256) void k_set_weight_row(float *grad, const float *w, int64_t N, int NK) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= N) return;
    float *g = grad + (size_t)NK * i;
    for (int k = 0; k < NK - 1; k++) g[k] = 0.0f;
    g[NK - 1] = w ? w[i] : 1.0f;
}
int launch_set_weight_row(evt_ctx *c, const float *w_dev) {
    hipLaunchKernelGGL(k_set_weight_row, dim3((unsigned)((c->N + 255) / 256)), dim3(256), 0, c->stream, c->grad, w_dev, c->N, c->NK);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

// pred[:, i] = mu (+ offset[:, i])  (src/init.jl:168-170)
__global__ __launch_bounds__(256) void k_init_pred(float *pred, const float *mu, const float *offset, int64_t N, int K) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= N) return;
    for (int k = 0; k < K; k++) {
        float v = mu[k];
        if (offset) v += offset[(size_t)K * i + k];
        pred[(size_t)K * i + k] = v;
    }
}
int launch_init_pred(evt_ctx *c, const float *mu_dev, const float *offset_dev) {
    hipLaunchKernelGGL(k_init_pred, dim3((unsigned)((c->N + 255) / 256)), dim3(256), 0, c->stream, c->pred, mu_dev, offset_dev, c->N, c->K);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}

// Multi-class targets are level codes 1..K stored as Float32; the gradient and metric kernels index with them.
__global__ __launch_bounds__(256) void k_validate_classes(const float *__restrict__ y, int64_t N, int K, int32_t *errflag) {
    bool bad = false;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < N; i += (int64_t)gridDim.x * 256) {
        const float v = y[i];
        bad |= !(v >= 1.0f && v <= (float)K && v == floorf(v));
    }
    if (bad) atomicOr(errflag, 1);
}
int launch_validate_classes(evt_ctx *c) {
    int64_t nb = (c->N + 255) / 256;
    if (nb > 2048) nb = 2048;
    hipLaunchKernelGGL(k_validate_classes, dim3((unsigned)nb), dim3(256), 0, c->stream, c->y, c->N, c->K, c->errflag);
    HIPCHK(hipGetLastError());
    return EVT_OK;
}
