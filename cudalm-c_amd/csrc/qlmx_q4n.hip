/* qlmx_q4n.hip -- the reference's "q4n" wire format (qtype 3): how a model quantised on the 4-bit
 * grid travels in a checkpoint. Host code only; no device is needed.
 *
 * Writer quantize_params(..., qtype 3, ...) cudalm.cu:638-656, reader dequantize_params
 * cudalm.cu:688-696. Layout per group of `group` values (the last group may be shorter):
 *   fp32 scale, then ceil(g/2) bytes of two's-complement nibbles, even element in the low nibble
 *   (the nibble rule of the packed digits, qlm.cuh:96-101); value = scale * nibble.
 *   A NaN scale marks a group stored as g raw fp32 values instead.
 * The writer accepts a group only if some candidate scale reproduces every value exactly:
 * candidates are amax/k for k = 7..1, each with its two neighbours below and above; the first hit
 * wins. A rendered QLM view (P = s * digit) always passes, possibly with a scale one or two ulps
 * away from s; anything else is kept bit-exact as raw fp32.
 */
#include "qlmx_dev.h"
#include <immintrin.h>
#include <math.h>
#include <string.h>
#include <algorithm>
#include <atomic>
#include <new>
#include <stdexcept>
#include <thread>
#include <vector>

/* What bounds it: one division per value when a group is tried against a scale, then the copy of the bytes. Eight
 * values at a time where the CPU has AVX2 (division, rounding and product are the IEEE ones of the scalar form, so the
 * bytes are the same), and by several threads where each has a share worth the 10 us or so that it takes to start: 128 K
 * values when writing, 256 K when reading, eight threads at most (sixteen were slower). The writer finds the groups'
 * scales first, which says where each part's bytes start, and the digits again behind that; the reader walks the group
 * headers first. 4 M values, a tenth of the groups raw, on the 16 CPUs of a GPU's share: write 7.9 ms -> 0.65,
 * read 0.99 -> 0.22. */
#define Q4N_WRITE_SHARE (128 * 1024)
#define Q4N_READ_SHARE (256 * 1024)
#define Q4N_MAX_THREADS 8
static int q4n_parts(size_t n, size_t ngroups, size_t share){
    const unsigned hw = std::thread::hardware_concurrency();
    return (int)std::max<size_t>(1, std::min({n / share, ngroups, (size_t)std::min<unsigned>(Q4N_MAX_THREADS, hw)}));
}
static size_t q4n_groups(size_t n, int group){ return n / (size_t)group + (n % (size_t)group != 0); }
/* first(part) for every part, and once all are done, second(part) */
template<class F, class S> static void q4n_run(int parts, const F &first, const S &second){
    std::atomic<int> done(0);
    auto finish = [&](int p0, int p1){
        done.fetch_add(p1 - p0, std::memory_order_acq_rel);
        while(done.load(std::memory_order_acquire) < parts) std::this_thread::yield();
        for(int p = p0; p < p1; p++) second(p);
    };
    std::thread th[Q4N_MAX_THREADS];
    int own = 0;                                           /* parts from here on are this thread's */
    for(; own + 1 < parts; own++){
        const int p = own;
        try { th[p] = std::thread([&, p]{ first(p); finish(p, p + 1); }); }
        catch(const std::exception &){ break; }            /* no more threads, or no memory for one, to be had */
    }
    for(int p = own; p < parts; p++) first(p);
    finish(own, parts);
    for(int p = 0; p < own; p++) th[p].join();
}
static bool q4n_avx2(){ static const bool yes = __builtin_cpu_supports("avx2"); return yes; }

/* ---- the pieces of a group, from element j0 on ---- */
static float amax_from(const float *v, int j0, int g, float amax){
    for(int j = j0; j < g; j++) amax = fmaxf(amax, fabsf(v[j]));
    return amax;
}
/* whether every value is scale * (-7..7) exactly; the digits on the way */
static bool try_from(const float *v, int j0, int g, float scale, signed char *digit){
    for(int j = j0; j < g; j++){
        const float dgt = rintf(v[j] / scale);
        if(fabsf(dgt) > 7.0f || dgt * scale != v[j]) return false;
        digit[j] = (signed char)(int)dgt;
    }
    return true;
}
static void pack_from(const signed char *digit, int j0, int g, unsigned char *b){       /* digit[g] is read where g is odd */
    for(int j = j0; j < g; j += 2) b[j >> 1] = (unsigned char)((digit[j] & 15) | ((digit[j + 1] & 15) << 4));
}
static void unpack_from(const unsigned char *b, int j0, int g, float scale, float *P){
    for(int j = j0; j < g; j += 2){
        const unsigned char x = b[j >> 1];
        P[j] = (float)((int)((x & 15) ^ 8) - 8) * scale;
        if(j + 1 < g) P[j + 1] = (float)((int)((x >> 4) ^ 8) - 8) * scale;
    }
}
__attribute__((target("avx2"))) static float amax_avx2(const float *v, int g){
    const __m256 mag = _mm256_castsi256_ps(_mm256_set1_epi32(0x7FFFFFFF));
    __m256 m = _mm256_setzero_ps();
    int j = 0;
    for(; j + 8 <= g; j += 8) m = _mm256_max_ps(_mm256_and_ps(_mm256_loadu_ps(v + j), mag), m);     /* a NaN leaves m, as fmaxf does */
    float e[8]; _mm256_storeu_ps(e, m);
    float amax = 0.0f;
    for(int k = 0; k < 8; k++) amax = fmaxf(amax, e[k]);
    return amax_from(v, j, g, amax);
}
__attribute__((target("avx2"))) static bool try_avx2(const float *v, int g, float scale, signed char *digit){
    const __m256 s = _mm256_set1_ps(scale), seven = _mm256_set1_ps(7.0f), mag = _mm256_castsi256_ps(_mm256_set1_epi32(0x7FFFFFFF));
    int j = 0;
    for(; j + 8 <= g; j += 8){
        const __m256 x = _mm256_loadu_ps(v + j), d = _mm256_round_ps(_mm256_div_ps(x, s), _MM_FROUND_CUR_DIRECTION);
        const __m256 off = _mm256_or_ps(_mm256_cmp_ps(_mm256_and_ps(d, mag), seven, _CMP_GT_OQ), _mm256_cmp_ps(_mm256_mul_ps(d, s), x, _CMP_NEQ_UQ));
        if(_mm256_movemask_ps(off)) return false;
        const __m256i i = _mm256_cvttps_epi32(d);
        const __m128i w = _mm_packs_epi32(_mm256_castsi256_si128(i), _mm256_extracti128_si256(i, 1));
        _mm_storel_epi64((__m128i *)(digit + j), _mm_packs_epi16(w, w));
    }
    return try_from(v, j, g, scale, digit);
}
__attribute__((target("avx2"))) static void pack_avx2(const signed char *digit, int g, unsigned char *b){
    const __m128i low = _mm_set1_epi8(15), place = _mm_set1_epi16(0x1001);                /* low digit * 1 + high digit * 16 */
    int j = 0;
    for(; j + 16 <= g; j += 16){
        const __m128i w = _mm_maddubs_epi16(_mm_and_si128(_mm_loadu_si128((const __m128i *)(digit + j)), low), place);
        _mm_storel_epi64((__m128i *)(b + (j >> 1)), _mm_packus_epi16(w, w));
    }
    pack_from(digit, j, g, b);
}
__attribute__((target("avx2"))) static void unpack_avx2(const unsigned char *b, int g, float scale, float *P){
    const __m256 s = _mm256_set1_ps(scale);
    const __m128i low = _mm_set1_epi8(15), eight = _mm_set1_epi8(8);
    int j = 0;
    for(; j + 16 <= g; j += 16){
        const __m128i x = _mm_loadl_epi64((const __m128i *)(b + (j >> 1)));
        const __m128i lo = _mm_and_si128(x, low), hi = _mm_and_si128(_mm_srli_epi16(x, 4), low);
        const __m128i d = _mm_sub_epi8(_mm_xor_si128(_mm_unpacklo_epi8(lo, hi), eight), eight);
        _mm256_storeu_ps(P + j, _mm256_mul_ps(_mm256_cvtepi32_ps(_mm256_cvtepi8_epi32(d)), s));
        _mm256_storeu_ps(P + j + 8, _mm256_mul_ps(_mm256_cvtepi32_ps(_mm256_cvtepi8_epi32(_mm_srli_si128(d, 8))), s));
    }
    unpack_from(b, j, g, scale, P);
}
static float group_amax(const float *v, int g){ return q4n_avx2() ? amax_avx2(v, g) : amax_from(v, 0, g, 0.0f); }
static bool group_try(const float *v, int g, float scale, signed char *digit){ return q4n_avx2() ? try_avx2(v, g, scale, digit) : try_from(v, 0, g, scale, digit); }
static void group_pack(const signed char *digit, int g, unsigned char *b){ if(q4n_avx2()) pack_avx2(digit, g, b); else pack_from(digit, 0, g, b); }
static void group_unpack(const unsigned char *b, int g, float scale, float *P){ if(q4n_avx2()) unpack_avx2(b, g, scale, P); else unpack_from(b, 0, g, scale, P); }

/* the neighbours of a value >= 0: nextafterf towards 0 and towards infinity, without the calls (35 candidates in a raw group) */
static inline float toward_zero(float x){ unsigned u; memcpy(&u, &x, 4); if(u) u--; memcpy(&x, &u, 4); return x; }
static inline float toward_inf(float x){ unsigned u; memcpy(&u, &x, 4); if(u != 0x7F800000u) u++; memcpy(&x, &u, 4); return x; }
/* the group's scale, the first candidate that fits (0 for a group of zeros), or NaN for a group that is kept raw */
static float group_scale(const float *v, int g, signed char *digit){
    const float amax = group_amax(v, g);
    if(amax == 0.0f) return 0.0f;
    for(int k = 7; k >= 1; k--){
        const float s0 = amax / (float)k;
        const float below = toward_zero(s0), above = toward_inf(s0);
        const float cand[5] = {s0, below, above, toward_zero(below), toward_inf(above)};
        for(int t = 0; t < 5; t++) if(group_try(v, g, cand[t], digit)) return cand[t];
    }
    return NAN;
}

extern "C" size_t qlmx_q4n_bound(size_t n, int group){
    if(group <= 0) return 0;
    return 4 * ((n + (size_t)group - 1) / (size_t)group) + 4 * n;
}

static int q4n_write(const float *P, size_t n, int group, unsigned char *out, size_t *out_len, size_t *nraw){
    const size_t ngroups = q4n_groups(n, group);
    const int parts = q4n_parts(n, ngroups, Q4N_WRITE_SHARE);
    std::vector<float> scales(ngroups);
    const size_t stride = std::min((size_t)group, n) + 256;     /* a part's digits share no cache line with another's */
    std::vector<signed char> digits((size_t)parts * stride);
    size_t len[Q4N_MAX_THREADS] = {}, raw[Q4N_MAX_THREADS] = {};
    auto begin = [&](int p){ return ngroups * (size_t)p / (size_t)parts; };
    auto size_of = [&](size_t q){ return (int)std::min((size_t)group, n - q * (size_t)group); };
    q4n_run(parts, [&](int p){
        signed char *digit = digits.data() + (size_t)p * stride;
        size_t l = 0, r = 0;
        for(size_t q = begin(p); q < begin(p + 1); q++){
            const int g = size_of(q);
            const float s = group_scale(P + q * (size_t)group, g, digit);
            scales[q] = s;
            if(s != s){ l += 4 + 4 * (size_t)g; r++; } else l += 4 + (size_t)(g + 1) / 2;
        }
        len[p] = l; raw[p] = r;
    }, [&](int p){
        signed char *digit = digits.data() + (size_t)p * stride;
        unsigned char *o = out;
        for(int i = 0; i < p; i++) o += len[i];
        for(size_t q = begin(p); q < begin(p + 1); q++){
            const float *v = P + q * (size_t)group;
            const int g = size_of(q);
            const float s = scales[q];
            memcpy(o, &s, 4); o += 4;
            if(s != s){ memcpy(o, v, 4 * (size_t)g); o += 4 * (size_t)g; continue; }
            if(s == 0.0f) memset(digit, 0, (size_t)g); else group_try(v, g, s, digit);
            digit[g] = 0;                                  /* the partner of an odd group's last digit */
            group_pack(digit, g, o); o += (g + 1) / 2;
        }
    });
    size_t o = 0, nr = 0;
    for(int p = 0; p < parts; p++){ o += len[p]; nr += raw[p]; }
    *out_len = o;
    if(nraw) *nraw = nr;
    return QLMX_OK;
}

static int q4n_read(const unsigned char *buf, size_t len, float *P, size_t n, int group, size_t *used){
    const size_t ngroups = q4n_groups(n, group);
    /* where a group starts: for as many as the buffer can hold at most (all but the last are whole), not as n names */
    std::vector<size_t> at(std::min(ngroups, len / (4 + ((size_t)group + 1) / 2) + 1));
    size_t o = 0;
    for(size_t q = 0; q < ngroups; q++){
        const size_t g = std::min((size_t)group, n - q * (size_t)group);
        float scale;
        QLMX_REQUIRE(len - o >= 4, "qlmx_q4n_dequantize: buffer ends inside group %zu", q);
        memcpy(&scale, buf + o, 4);
        at[q] = o; o += 4;
        if(scale != scale){
            QLMX_REQUIRE((len - o) / 4 >= g, "qlmx_q4n_dequantize: buffer ends inside raw group %zu", q);
            o += 4 * g;
        } else {
            QLMX_REQUIRE(len - o >= (g + 1) / 2, "qlmx_q4n_dequantize: buffer ends inside group %zu", q);
            o += (g + 1) / 2;
        }
    }
    const int parts = q4n_parts(n, ngroups, Q4N_READ_SHARE);
    q4n_run(parts, [&](int p){
        for(size_t q = ngroups * (size_t)p / (size_t)parts; q < ngroups * (size_t)(p + 1) / (size_t)parts; q++){
            const size_t i = q * (size_t)group;
            const int g = (int)std::min((size_t)group, n - i);
            const unsigned char *b = buf + at[q];
            float scale; memcpy(&scale, b, 4);
            if(scale != scale) memcpy(P + i, b + 4, 4 * (size_t)g);
            else group_unpack(b + 4, g, scale, P + i);
        }
    }, [](int){});
    if(used) *used = o;
    return QLMX_OK;
}

/* What a call does, with an allocation that fails as an error of the call: no exception passes a C entry point. */
template<class F> static int q4n_guarded(const char *who, const F &body){
    try { return body(); }
    catch(const std::bad_alloc &){}
    catch(const std::length_error &){}                     /* more than a vector can name */
    qlmx_set_error("%s: out of memory for the scratch", who);
    return QLMX_E_LIMIT;
}
extern "C" int qlmx_q4n_quantize(const float *P, size_t n, int group, unsigned char *out, size_t cap,
                                 size_t *out_len, size_t *nraw){
    QLMX_REQUIRE(P && out && out_len, "qlmx_q4n_quantize: NULL buffer");
    QLMX_REQUIRE(group > 0 && group % 2 == 0, "qlmx_q4n_quantize: group %d must be positive and even", group);
    QLMX_REQUIRE(cap >= qlmx_q4n_bound(n, group), "qlmx_q4n_quantize: output buffer smaller than qlmx_q4n_bound()");
    return q4n_guarded("qlmx_q4n_quantize", [&]{ return q4n_write(P, n, group, out, out_len, nraw); });
}

extern "C" int qlmx_q4n_dequantize(const unsigned char *buf, size_t len, float *P, size_t n, int group, size_t *used){
    QLMX_REQUIRE(buf && P, "qlmx_q4n_dequantize: NULL buffer");
    QLMX_REQUIRE(group > 0, "qlmx_q4n_dequantize: group %d", group);
    return q4n_guarded("qlmx_q4n_dequantize", [&]{ return q4n_read(buf, len, P, n, group, used); });
}
