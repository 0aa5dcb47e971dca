// The searches of host_bin.cpp, sixteen values at a time.  Compiled for AVX-512 and called only where the processor has it:
// plain functions, no inline library code that another file could be linked to.
//
// A feature's edges sit in vector registers as a search heap (node h at lane h & 15 of register h >> 4): a step of the search is
// a register permute that fetches every lane's own node, a compare, and h = 2 h + passed.  63 edges take six steps, 22
// instructions for 16 values: 0.59 ns per Float64 value read from memory on one core of the host this was measured on (a plain search: 21), and
// 170 to 180 GB/s of Float64 read and binned on 16 (the same matrix moved to the device as it lies: 43 GB/s).
#include "host_bin.h"

#if defined(__AVX512F__)
#include <immintrin.h>

namespace {

struct Tables {
    __m512 t[16];
};

template <int L>
inline __attribute__((always_inline)) void load_tables(Tables &T, const float *heap) {
#pragma unroll
    for (int k = 0; k < (1 << L) / 16; k++) T.t[k] = _mm512_load_ps(heap + 16 * k);
}

// rank of each value among the heap's keys, padding included; *last: the first key not passed (a value that equals it is open)
template <int L, bool CHECK>
inline __attribute__((always_inline)) __m512i search16(const Tables &T, __m512 v, __m512 *last) {
    const __m512i one = _mm512_set1_epi32(1);
    __m512i h = one;
    __m512 lb = _mm512_set1_ps(__builtin_inff());
#pragma unroll
    for (int l = 0; l < L; l++) {
        __m512 node;
        if (l < 4) {
            node = _mm512_permutexvar_ps(h, T.t[0]);
        } else if (l == 4) {
            node = _mm512_permutexvar_ps(h, T.t[1]);
        } else if (l == 5) {
            node = _mm512_permutex2var_ps(T.t[2], h, T.t[3]);
        } else if (l == 6) {
            const __mmask16 hi = _mm512_test_epi32_mask(h, _mm512_set1_epi32(32));
            node = _mm512_mask_blend_ps(hi, _mm512_permutex2var_ps(T.t[4], h, T.t[5]), _mm512_permutex2var_ps(T.t[6], h, T.t[7]));
        } else {
            const __mmask16 b5 = _mm512_test_epi32_mask(h, _mm512_set1_epi32(32)), b6 = _mm512_test_epi32_mask(h, _mm512_set1_epi32(64));
            const __m512 lo = _mm512_mask_blend_ps(b5, _mm512_permutex2var_ps(T.t[8], h, T.t[9]), _mm512_permutex2var_ps(T.t[10], h, T.t[11]));
            const __m512 hi = _mm512_mask_blend_ps(b5, _mm512_permutex2var_ps(T.t[12], h, T.t[13]), _mm512_permutex2var_ps(T.t[14], h, T.t[15]));
            node = _mm512_mask_blend_ps(b6, lo, hi);
        }
        const __mmask16 pass = _mm512_cmp_ps_mask(node, v, _CMP_NGE_UQ); // node < v, or v is NaN: it passes every edge
        h = _mm512_add_epi32(h, h);
        h = _mm512_mask_add_epi32(h, pass, h, one);
        if (CHECK) lb = _mm512_mask_mov_ps(node, pass, lb);
    }
    if (CHECK) *last = lb;
    return _mm512_sub_epi32(h, _mm512_set1_epi32(1 << L));
}

inline __attribute__((always_inline)) __m512 load16_f64(const double *x) { // rounded up, as the keys are
    const __m256 a = _mm512_cvt_roundpd_ps(_mm512_loadu_pd(x), _MM_FROUND_TO_POS_INF | _MM_FROUND_NO_EXC);
    const __m256 b = _mm512_cvt_roundpd_ps(_mm512_loadu_pd(x + 8), _MM_FROUND_TO_POS_INF | _MM_FROUND_NO_EXC);
    return _mm512_insertf32x8(_mm512_castps256_ps512(a), b, 1);
}
inline __attribute__((always_inline)) __m512 mask_load16_f64(const double *x, __mmask16 m) {
    const __m256 a = _mm512_cvt_roundpd_ps(_mm512_maskz_loadu_pd((__mmask8)m, x), _MM_FROUND_TO_POS_INF | _MM_FROUND_NO_EXC);
    const __m256 b = _mm512_cvt_roundpd_ps(_mm512_maskz_loadu_pd((__mmask8)(m >> 8), x + 8), _MM_FROUND_TO_POS_INF | _MM_FROUND_NO_EXC);
    return _mm512_insertf32x8(_mm512_castps256_ps512(a), b, 1);
}

// the values of `open` met a key: their rank goes on past the edges of that key that they pass in Float64
inline void settle(__mmask16 open, uint8_t *bins, const double *x, int64_t stride, const HbFeature &f) {
    for (unsigned m = open; m; m &= m - 1) {
        const int i = __builtin_ctz(m);
        int c = bins[i] - 1;
        const double v = x[i * stride];
        while (c < f.ne && f.e[c] < v) c++;
        bins[i] = (uint8_t)(c + 1);
    }
}

// bins of 16 keys; x, stride: the Float64 values behind them (CHECK only)
template <int L, bool CHECK>
inline __attribute__((always_inline)) void bin16(const Tables &T, __m512 v, __m512i ne, uint8_t *out, const double *x, int64_t stride, const HbFeature &f) {
    __m512 last;
    __m512i r = search16<L, CHECK>(T, v, &last);
    r = _mm512_add_epi32(_mm512_min_epi32(r, ne), _mm512_set1_epi32(1));
    _mm_storeu_si128(reinterpret_cast<__m128i *>(out), _mm512_cvtepi32_epi8(r));
    if (CHECK) {
        const __mmask16 open = _mm512_cmp_ps_mask(last, v, _CMP_EQ_OQ);
        if (__builtin_expect(open, 0)) settle(open, out, x, stride, f);
    }
}

template <int L, bool CHECK>
void col_f64(const double *x, int64_t n, const HbFeature &f, const float *heap, uint8_t *out) {
    Tables T;
    load_tables<L>(T, heap);
    const __m512i ne = _mm512_set1_epi32(f.ne);
    int64_t i = 0;
    for (; i + 16 <= n; i += 16) bin16<L, CHECK>(T, load16_f64(x + i), ne, out + i, x + i, 1, f);
    if (i < n) { // the last values again with some before them: n >= 16
        i = n - 16;
        bin16<L, CHECK>(T, load16_f64(x + i), ne, out + i, x + i, 1, f);
    }
}
template <int L>
void col_f32(const float *x, int64_t n, const HbFeature &f, const float *heap, uint8_t *out) {
    Tables T;
    load_tables<L>(T, heap);
    const __m512i ne = _mm512_set1_epi32(f.ne);
    int64_t i = 0;
    for (; i + 16 <= n; i += 16) bin16<L, false>(T, _mm512_loadu_ps(x + i), ne, out + i, nullptr, 0, f);
    if (i < n) {
        i = n - 16;
        bin16<L, false>(T, _mm512_loadu_ps(x + i), ne, out + i, nullptr, 0, f);
    }
}

// 16 rows of 16 keys -> 16 columns of 16 keys
inline __attribute__((always_inline)) void transpose16(__m512 *r) {
    __m512 a[16];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        a[2 * i] = _mm512_unpacklo_ps(r[2 * i], r[2 * i + 1]);
        a[2 * i + 1] = _mm512_unpackhi_ps(r[2 * i], r[2 * i + 1]);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) { // r[4 i + q]: column q of each 128-bit lane, rows 4 i .. 4 i + 3
        r[4 * i + 0] = _mm512_castpd_ps(_mm512_unpacklo_pd(_mm512_castps_pd(a[4 * i]), _mm512_castps_pd(a[4 * i + 2])));
        r[4 * i + 1] = _mm512_castpd_ps(_mm512_unpackhi_pd(_mm512_castps_pd(a[4 * i]), _mm512_castps_pd(a[4 * i + 2])));
        r[4 * i + 2] = _mm512_castpd_ps(_mm512_unpacklo_pd(_mm512_castps_pd(a[4 * i + 1]), _mm512_castps_pd(a[4 * i + 3])));
        r[4 * i + 3] = _mm512_castpd_ps(_mm512_unpackhi_pd(_mm512_castps_pd(a[4 * i + 1]), _mm512_castps_pd(a[4 * i + 3])));
    }
#pragma unroll
    for (int q = 0; q < 4; q++) { // columns q, 4 + q, 8 + q, 12 + q from the four row groups' lanes
        const __m512 p0 = _mm512_shuffle_f32x4(r[q], r[4 + q], 0x88), p1 = _mm512_shuffle_f32x4(r[q], r[4 + q], 0xdd);
        const __m512 p2 = _mm512_shuffle_f32x4(r[8 + q], r[12 + q], 0x88), p3 = _mm512_shuffle_f32x4(r[8 + q], r[12 + q], 0xdd);
        a[q] = _mm512_shuffle_f32x4(p0, p2, 0x88);
        a[8 + q] = _mm512_shuffle_f32x4(p0, p2, 0xdd);
        a[4 + q] = _mm512_shuffle_f32x4(p1, p3, 0x88);
        a[12 + q] = _mm512_shuffle_f32x4(p1, p3, 0xdd);
    }
#pragma unroll
    for (int i = 0; i < 16; i++) r[i] = a[i];
}

// 64 keys of one feature (contiguous in `key`) -> 64 bins; x: the Float64 values behind them
template <int L, bool CHECK>
void tile_col(const float *key, const HbFeature &f, const float *heap, uint8_t *bins, const double *x, int64_t stride) {
    Tables T;
    load_tables<L>(T, heap);
    const __m512i ne = _mm512_set1_epi32(f.ne);
#pragma unroll
    for (int g = 0; g < 4; g++) bin16<L, CHECK>(T, _mm512_load_ps(key + 16 * g), ne, bins + 16 * g, x + 16 * g * stride, stride, f);
}

#define HB_LEVELS(call)                 \
    switch (f.levels) {                 \
        case 4: { call(4); } break;     \
        case 5: { call(5); } break;     \
        case 6: { call(6); } break;     \
        case 7: { call(7); } break;     \
        default: { call(8); } break;    \
    }

} // namespace

void hb512_col(const void *x, int dtype, int64_t n, const HbFeature &f, const float *heap, uint8_t *out) {
    const float *h = heap + f.heap;
    if (dtype == EVT_F32) {
#define HB_CALL(L) col_f32<L>(static_cast<const float *>(x), n, f, h, out)
        HB_LEVELS(HB_CALL)
#undef HB_CALL
    } else if (f.flags & HB_EXACT) {
#define HB_CALL(L) col_f64<L, false>(static_cast<const double *>(x), n, f, h, out)
        HB_LEVELS(HB_CALL)
#undef HB_CALL
    } else {
#define HB_CALL(L) col_f64<L, true>(static_cast<const double *>(x), n, f, h, out)
        HB_LEVELS(HB_CALL)
#undef HB_CALL
    }
}

// Rows one after the other in memory: tiles of 64 rows x 16 features are turned over in registers (16 x 16 keys at a time)
// into a 4 KB buffer of columns, then binned a feature at a time and written as whole 64-byte lines.  The next tile's rows are one
// run of memory, read here in strides no hardware prefetcher follows: it is requested a share with every group of features.
void hb512_rows(const void *x, int dtype, int64_t rs, int64_t n, const HbFeature *feat, int nf, const float *heap, uint8_t *out, int64_t ldo) {
    alignas(64) float key[16][64] = {};
    alignas(64) uint8_t bins[64];
    const int64_t row_bytes = rs * (dtype == EVT_F32 ? 4 : 8), used = nf * (dtype == EVT_F32 ? 4 : 8);
    const int groups = (nf + 15) / 16;
    for (int64_t r0 = 0; r0 < n; r0 += 64) {
        const int64_t nr = n - r0 < 64 ? n - r0 : 64;
        const char *ahead = static_cast<const char *>(x) + (r0 + 64) * row_bytes;
        const int64_t na = n - r0 - 64 < 64 ? n - r0 - 64 : 64;                                   // rows of the next tile
        const int64_t dense = na <= 0 ? 0 : (row_bytes <= used + 64 ? (na - 1) * row_bytes + used : 0); // bytes, when nearly all are used
        for (int f0 = 0; f0 < nf; f0 += 16) {
            const int fc = nf - f0 < 16 ? nf - f0 : 16;
            for (int64_t b = dense * (f0 / 16) / groups, e = dense * (f0 / 16 + 1) / groups; b < e; b += 64) _mm_prefetch(ahead + b, _MM_HINT_T0);
            const __mmask16 m = (__mmask16)((1u << fc) - 1);
            for (int g = 0; 16 * g < nr; g++) {
                __m512 r[16];
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int64_t row = r0 + (16 * g + i < nr ? 16 * g + i : nr - 1);
                    if (dtype == EVT_F32) r[i] = _mm512_maskz_loadu_ps(m, static_cast<const float *>(x) + row * rs + f0);
                    else r[i] = mask_load16_f64(static_cast<const double *>(x) + row * rs + f0, m);
                }
                transpose16(r);
#pragma unroll
                for (int i = 0; i < 16; i++) _mm512_store_ps(&key[i][16 * g], r[i]);
            }
            for (int j = 0; j < fc; j++) {
                const HbFeature &f = feat[f0 + j];
                if (f.flags & HB_SLOW) continue; // the caller compares these value by value
                const float *h = heap + f.heap;
                const bool full = nr == 64;
                uint8_t *o = out + (int64_t)(f0 + j) * ldo + r0;
                uint8_t *b = full ? o : bins;
                const double *xd = dtype == EVT_F32 ? nullptr : static_cast<const double *>(x) + r0 * rs + f0 + j;
                if (full && (dtype == EVT_F32 || (f.flags & HB_EXACT))) {
#define HB_CALL(L) tile_col<L, false>(key[j], f, h, b, nullptr, 0)
                    HB_LEVELS(HB_CALL)
#undef HB_CALL
                } else if (full) {
#define HB_CALL(L) tile_col<L, true>(key[j], f, h, b, xd, rs)
                    HB_LEVELS(HB_CALL)
#undef HB_CALL
                } else { // the last rows: the keys past them are stale, and no value stands behind them to compare
#define HB_CALL(L) tile_col<L, false>(key[j], f, h, b, nullptr, 0)
                    HB_LEVELS(HB_CALL)
#undef HB_CALL
                    for (int64_t i = 0; i < nr; i++) {
                        int c = b[i] - 1;
                        if (dtype != EVT_F32 && !(f.flags & HB_EXACT))
                            while (c < f.ne && f.e[c] < xd[i * rs]) c++;
                        o[i] = (uint8_t)(c + 1);
                    }
                }
            }
        }
    }
}

#else // a compiler without AVX-512: never called (hb_has_avx512)
void hb512_col(const void *, int, int64_t, const HbFeature &, const float *, uint8_t *) {}
void hb512_rows(const void *, int, int64_t, int64_t, const HbFeature *, int, const float *, uint8_t *, int64_t) {}
#endif
