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
#include <sched.h>
#include <signal.h>
#include <sys/resource.h>
#include <unistd.h>
#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <functional>
#include <mutex>
#include <new>
#include <stdexcept>
#include <thread>
#include <vector>

/* What bounds it: reading the values, twice when writing -- the writer finds the groups' scales first, which says where each part's bytes
 * start, and the digits again behind that -- the first touch of the output's pages, and the reader's walk over the group headers. Whether a group fits a scale is
 * tried eight values at a time where the CPU has AVX2, with one reciprocal for the group instead of a division per value (fits_avx2), also behind the last whole 32 of a
 * group: with scalar divisions there, as the remainders of 32 had, 40 K values in groups of 24 took 350 us to write, of 16 384, of 56 175; now 66, 91, 42 (with divisions eight at a time
 * 87, 116, 67). All of it in parts by up to eight threads (sixteen were slower). Seven threads take 80 us to start and 15 to wake, so they are kept (Q4nCrew below).
 * 4 M values, a tenth of the groups raw, on the 16 CPUs of a GPU's share, us: write and read by one thread with scalar arithmetic 7900 + 990, divisions and threads started in
 * each call 350-410 + 230-260, as here 180-190 + 160-170, into memory that has been written before. A caller that takes new memory for each call, as the Python calls do, pays for the first touch
 * of its pages: 510-540 + 160-170 (large pages, in part used ones; all new, of 4 KB, 850-930 + 3200-3500). */
#define Q4N_WRITE_PART (48 * 1024)              /* values to a part: several parts a thread, since threads wake one after the other */
#define Q4N_READ_PART (128 * 1024)
#define Q4N_MAX_THREADS 8
static size_t q4n_groups(size_t n, int group){ return n / (size_t)group + (n % (size_t)group != 0); }
/* groups longer than 4096: no more parts than threads, as each part has scratch for the digits of a group */
static int q4n_parts(size_t n, size_t ngroups, int group, size_t part){ return (int)std::max<size_t>(1, std::min<size_t>({n / part, ngroups, (size_t)(group > 4096 ? Q4N_MAX_THREADS : 4096)})); }

/* Threads for the calls' parts: started as calls ask for them, at most seven whatever the number of callers, and gone after a second without work. A call
 * takes part in its own job and needs none of them; several calls at once share them. A job is on its caller's stack: the caller leaves when its
 * parts are done and no thread has hold of it any more. A thread works on a job in its caller's floating-point mode (rounding, small values flushed to
 * zero or not) and on the CPUs that the caller may run on: a new thread has those of whoever started it, which here is some earlier caller (4 M values written behind a
 * call bound to one CPU, 8 CPUs, us: on the CPU of that call 1600-2000, with this 580-630, as behind any other). A priority cannot be
 * given back once lowered, so the threads serve callers of the one that they were started with; a caller of another starts its own for the call. The crew itself is never destroyed, so threads asleep at exit touch nothing that is; a
 * child of fork() has none of the threads and starts with a crew of its own. */
struct Q4nJob {
    const std::function<void(int)> *phase[2]; int parts;
    const unsigned mode = _mm_getcsr() & ~(unsigned)_MM_EXCEPT_MASK;
    cpu_set_t cpus; bool placed;                           /* not placed: more CPUs than the set has room for */
    std::atomic<int> next[2], done[2];
    int holders; Q4nJob *link;                             /* both under the crew's lock */
    Q4nJob() : parts(0), holders(0), link(nullptr) { for(int i = 0; i < 2; i++){ phase[i] = nullptr; next[i] = 0; done[i] = 0; } }
    bool open() const { return next[0].load(std::memory_order_relaxed) < parts || (phase[1] && next[1].load(std::memory_order_relaxed) < parts); }
    /* parts that nobody has begun; the second phase only when all of the first are done */
    void work(){
        for(int ph = 0; ph < 2 && phase[ph]; ph++){
            for(int p; (p = next[ph].fetch_add(1, std::memory_order_relaxed)) < parts; ){
                (*phase[ph])(p);
                done[ph].fetch_add(1, std::memory_order_acq_rel);
            }
            while(done[ph].load(std::memory_order_acquire) < parts) std::this_thread::yield();
        }
    }
};
struct Q4nPriority {                                      /* of the calling thread */
    int policy = sched_getscheduler(0), level = 0, nice = getpriority(PRIO_PROCESS, 0);
    Q4nPriority(){ sched_param p; if(sched_getparam(0, &p) == 0) level = p.sched_priority; }
    bool operator==(const Q4nPriority &o) const { return policy == o.policy && level == o.level && nice == o.nice; }
};
struct Q4nCrew {
    std::mutex lock; std::condition_variable wake, left;
    Q4nJob *jobs = nullptr; int threads = 0, idle = 0;
    Q4nPriority theirs;                                    /* while there are threads */
    const pid_t owner = getpid();

    void member(){
        sigset_t sent;                                     /* signals are for the program's own threads, but a fault is the faulting thread's: blocked, it ends the process past any handler */
        sigfillset(&sent);
        for(int fault : {SIGSEGV, SIGBUS, SIGFPE, SIGILL, SIGTRAP, SIGSYS}) sigdelset(&sent, fault);
        pthread_sigmask(SIG_BLOCK, &sent, nullptr);
        cpu_set_t cpus; CPU_ZERO(&cpus);
        std::unique_lock<std::mutex> l(lock);
        for(;;){
            Q4nJob *j = jobs;
            while(j && !j->open()) j = j->link;
            if(!j){
                idle++;
                const bool late = wake.wait_for(l, std::chrono::seconds(1)) == std::cv_status::timeout;
                idle--;
                if(late){
                    for(j = jobs; j && !j->open(); j = j->link) ;
                    if(!j) break;
                }
                continue;
            }
            j->holders++;
            l.unlock();
            if(j->placed && !CPU_EQUAL(&cpus, &j->cpus) && sched_setaffinity(0, sizeof cpus, &j->cpus) == 0) cpus = j->cpus;
            const unsigned own = _mm_getcsr();
            _mm_setcsr(j->mode);
            j->work();
            _mm_setcsr(own);
            l.lock();
            if(--j->holders == 0) left.notify_all();
        }
        threads--;
    }
    bool run(Q4nJob &j, int wanted){                       /* false: not for this caller */
        const Q4nPriority mine;
        j.placed = sched_getaffinity(0, sizeof j.cpus, &j.cpus) == 0;
        {
            std::lock_guard<std::mutex> l(lock);
            if(threads == 0) theirs = mine;
            else if(!(theirs == mine)) return false;
            j.link = jobs; jobs = &j;
            for(int more = wanted - idle; more > 0 && threads < Q4N_MAX_THREADS - 1; more--){
                try { std::thread([this]{ member(); }).detach(); threads++; }
                catch(const std::exception &){ break; }    /* no more threads, or no memory for one, to be had */
            }
        }
        wake.notify_all();
        j.work();
        std::unique_lock<std::mutex> l(lock);
        Q4nJob **at = &jobs;
        while(*at != &j) at = &(*at)->link;
        *at = j.link;
        while(j.holders) left.wait(l);
        return true;
    }
};
static Q4nCrew *q4n_crew(){
    static std::atomic<Q4nCrew *> crew(nullptr);
    Q4nCrew *c = crew.load(std::memory_order_acquire);
    while(!c || c->owner != getpid()){
        Q4nCrew *n = new Q4nCrew;
        if(crew.compare_exchange_strong(c, n, std::memory_order_acq_rel)) return n;
        delete n;
    }
    return c;
}
/* first(part) for every part, and once all are done, second(part) for every part */
static void q4n_run(int parts, const std::function<void(int)> &first, const std::function<void(int)> *second){
    Q4nJob j;
    j.parts = parts; j.phase[0] = &first; j.phase[1] = second;
    const int wanted = std::min({parts, Q4N_MAX_THREADS, (int)std::thread::hardware_concurrency()}) - 1;
    if(wanted > 0 && q4n_crew()->run(j, wanted)) return;
    std::thread own[Q4N_MAX_THREADS];
    for(int i = 0; i < wanted; i++){
        try { own[i] = std::thread([&j]{ j.work(); }); }
        catch(const std::exception &){ break; }
    }
    j.work();
    for(std::thread &t : own) if(t.joinable()) t.join();
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
    __m256 m = _mm256_setzero_ps(), m1 = m, m2 = m, m3 = m;       /* four chains: a maximum takes four cycles */
    int j = 0;
    for(; j + 32 <= g; j += 32){
        m  = _mm256_max_ps(_mm256_and_ps(_mm256_loadu_ps(v + j), mag), m);                             /* a NaN leaves m, as fmaxf does */
        m1 = _mm256_max_ps(_mm256_and_ps(_mm256_loadu_ps(v + j + 8), mag), m1);
        m2 = _mm256_max_ps(_mm256_and_ps(_mm256_loadu_ps(v + j + 16), mag), m2);
        m3 = _mm256_max_ps(_mm256_and_ps(_mm256_loadu_ps(v + j + 24), mag), m3);
    }
    for(; j + 8 <= g; j += 8) m1 = _mm256_max_ps(_mm256_and_ps(_mm256_loadu_ps(v + j), mag), m1);
    m = _mm256_max_ps(_mm256_max_ps(m, m1), _mm256_max_ps(m2, m3));
    __m128 t = _mm_max_ps(_mm256_castps256_ps128(m), _mm256_extractf128_ps(m, 1));
    t = _mm_max_ps(t, _mm_movehl_ps(t, t));
    const float amax = _mm_cvtss_f32(_mm_max_ss(t, _mm_shuffle_ps(t, t, 1)));
    return amax_from(v, j, g, amax);
}
/* A group against one of its candidates amax / k, in the range and the direction of rounding that q4n_mid names: whether every value is a digit times the scale, with a reciprocal for the division. The
 * answer is that of try_from. A digit d passes there when |d| <= 7 and the rounded product d * scale is v. Then v is d * scale within 2^-24 of itself, and v * (1/scale), two
 * roundings further, d within 2^-22 of itself: it rounds to the same d. The other way round, a digit that passes here has v = rounded d * scale, so that
 * v / scale rounds to it too; and it is at most 7, as no value is more than amax and no candidate less than amax / 7 by more than two units in its last place. */
__attribute__((target("avx2"))) static bool fits_avx2(const float *v, int g, float scale){
    const __m256 s = _mm256_set1_ps(scale), inv = _mm256_set1_ps(1.0f / scale);
    int j = 0;
    auto off8 = [&](int at) __attribute__((target("avx2"))) {
        const __m256 x = _mm256_loadu_ps(v + at), d = _mm256_round_ps(_mm256_mul_ps(x, inv), _MM_FROUND_CUR_DIRECTION);
        return _mm256_cmp_ps(_mm256_mul_ps(d, s), x, _CMP_NEQ_UQ);
    };
    for(; j + 32 <= g; j += 32)
        if(_mm256_movemask_ps(_mm256_or_ps(_mm256_or_ps(off8(j), off8(j + 8)), _mm256_or_ps(off8(j + 16), off8(j + 24))))) return false;
    for(; j + 8 <= g; j += 8) if(_mm256_movemask_ps(off8(j))) return false;
    if(j < g && g >= 8) return !_mm256_movemask_ps(off8(g - 8));          /* the last eight, some of them once more */
    for(; j < g; j++){
        const float d = rintf(v[j] / scale);
        if(fabsf(d) > 7.0f || d * scale != v[j]) return false;
    }
    return true;
}
/* the nibbles of a group that fits, one of the range */
__attribute__((target("avx2"))) static void put_avx2(const float *v, int g, float scale, unsigned char *b){
    const __m256 inv = _mm256_set1_ps(1.0f / scale);
    const __m256i low = _mm256_set1_epi32(0x000F000F), byte = _mm256_set1_epi32(0xFF);
    int j = 0;
    for(; j + 32 <= g; j += 32){
        __m256i h[2];
        for(int i = 0; i < 2; i++){
            const __m256i u = _mm256_cvtps_epi32(_mm256_mul_ps(_mm256_loadu_ps(v + j + 16 * i), inv)), w = _mm256_cvtps_epi32(_mm256_mul_ps(_mm256_loadu_ps(v + j + 16 * i + 8), inv));
            const __m256i x = _mm256_and_si256(_mm256_permute4x64_epi64(_mm256_packs_epi32(u, w), 0xD8), low);      /* 16 digits in order, a 16-bit word each */
            h[i] = _mm256_and_si256(_mm256_or_si256(x, _mm256_srli_epi32(x, 12)), byte);
        }
        const __m256i t = _mm256_permute4x64_epi64(_mm256_packus_epi32(h[0], h[1]), 0xD8);
        _mm_storeu_si128((__m128i *)(b + (j >> 1)), _mm_packus_epi16(_mm256_castsi256_si128(t), _mm256_extracti128_si256(t, 1)));
    }
    auto put8 = [&](int at) __attribute__((target("avx2"))) {
        const __m256i u = _mm256_cvtps_epi32(_mm256_mul_ps(_mm256_loadu_ps(v + at), inv));
        const __m128i x = _mm_and_si128(_mm_packs_epi32(_mm256_castsi256_si128(u), _mm256_extracti128_si256(u, 1)), _mm256_castsi256_si128(low));
        const __m128i h = _mm_and_si128(_mm_or_si128(x, _mm_srli_epi32(x, 12)), _mm256_castsi256_si128(byte)), t = _mm_packus_epi32(h, h);
        const int four = _mm_cvtsi128_si32(_mm_packus_epi16(t, t));
        memcpy(b + (at >> 1), &four, 4);
    };
    for(; j + 8 <= g; j += 8) put8(j);
    if(j < g && g >= 8 && !(g & 1)){ put8(g - 8); return; }                /* the last eight, some of them once more */
    for(; j < g; j += 2){
        const int d0 = (int)rintf(v[j] / scale), d1 = j + 1 < g ? (int)rintf(v[j + 1] / scale) : 0;
        b[j >> 1] = (unsigned char)((d0 & 15) | ((d1 & 15) << 4));
    }
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
/* Whether the first eight values may be amax / k times whole numbers, for the candidates of this k: a value that is a digit times one of them, rounded, is
 * amax / k times that digit within 2^-21 of itself, so that v * (1 / amax) * k is within 2^-17 of a whole number. What fails here fails with all five; a raw group, which has no
 * scale, is seen off with 7 of these instead of 35 tries (4 M values, half the groups raw: 580 -> 376 us). */
__attribute__((target("avx2"))) static bool maybe_avx2(const float *v, float inv, int k){       /* inv = 1 / amax */
    const __m256 t = _mm256_mul_ps(_mm256_mul_ps(_mm256_loadu_ps(v), _mm256_set1_ps(inv)), _mm256_set1_ps((float)k)), off = _mm256_sub_ps(t, _mm256_round_ps(t, _MM_FROUND_CUR_DIRECTION));
    const __m256 mag = _mm256_castsi256_ps(_mm256_set1_epi32(0x7FFFFFFF));
    return _mm256_movemask_ps(_mm256_cmp_ps(_mm256_and_ps(off, mag), _mm256_set1_ps(0x1p-17f), _CMP_NLE_UQ)) == 0;
}
/* the callers that round to nearest, as the bounds of fits_avx2 and maybe_avx2 have it; asked once per part */
static bool q4n_nearest(){ return q4n_avx2() && _MM_GET_ROUNDING_MODE() == _MM_ROUND_NEAREST; }
/* and largest magnitudes, and scales, whose quotients and products neither overflow nor lose bits */
static bool q4n_mid(float x, bool nearest){ return nearest && x >= 0x1p-90f && x <= 0x1p90f; }
static float group_amax(const float *v, int g){ return q4n_avx2() ? amax_avx2(v, g) : amax_from(v, 0, g, 0.0f); }
static bool group_try(const float *v, int g, float scale, signed char *digit){ return q4n_avx2() ? try_avx2(v, g, scale, digit) : try_from(v, 0, g, scale, digit); }
static void group_pack(const signed char *digit, int g, unsigned char *b){ if(q4n_avx2()) pack_avx2(digit, g, b); else pack_from(digit, 0, g, b); }
static void group_unpack(const unsigned char *b, int g, float scale, float *P){ if(q4n_avx2()) unpack_avx2(b, g, scale, P); else unpack_from(b, 0, g, scale, P); }

/* the neighbours of a value >= 0: nextafterf towards 0 and towards infinity, without the calls (35 candidates in a raw group) */
static inline float toward_zero(float x){ unsigned u; memcpy(&u, &x, 4); if(u) u--; memcpy(&x, &u, 4); return x; }
static inline float toward_inf(float x){ unsigned u; memcpy(&u, &x, 4); if(u != 0x7F800000u) u++; memcpy(&x, &u, 4); return x; }
/* the first candidate that fits, or NaN for a group that is kept raw */
template<class Worth, class Fits> static inline float first_scale(float amax, const Worth &worth, const Fits &fits){
    for(int k = 7; k >= 1; k--){
        if(!worth(k)) continue;
        const float s0 = amax / (float)k;
        const float below = toward_zero(s0), above = toward_inf(s0);
        const float cand[5] = {s0, below, above, toward_zero(below), toward_inf(above)};
        for(int t = 0; t < 5; t++) if(fits(cand[t])) return cand[t];
    }
    return NAN;
}
/* the group's scale: 0 for a group of zeros, NaN for one that is kept raw */
static float group_scale(const float *v, int g, bool nearest, signed char *digit){
    const float amax = group_amax(v, g);
    if(amax == 0.0f) return 0.0f;
    if(q4n_mid(amax, nearest)){
        const float inv = 1.0f / amax;
        return first_scale(amax, [&](int k){ return g < 8 || maybe_avx2(v, inv, k); }, [&](float s){ return fits_avx2(v, g, s); });
    }
    return first_scale(amax, [](int){ return true; }, [&](float s){ return group_try(v, g, s, digit); });
}

extern "C" size_t qlmx_q4n_bound(size_t n, int group){
    if(group <= 0) return 0;
    return 4 * ((n + (size_t)group - 1) / (size_t)group) + 4 * n;
}

static int q4n_write(const float *P, size_t n, int group, unsigned char *out, size_t *out_len, size_t *nraw){
    const size_t ngroups = q4n_groups(n, group);
    const int parts = q4n_parts(n, ngroups, group, Q4N_WRITE_PART);
    std::vector<float> scales(ngroups);
    const size_t stride = std::min((size_t)group, n) + 256;     /* a part's digits share no cache line with another's */
    std::vector<signed char> digits((size_t)parts * stride);
    std::vector<size_t> len(parts), raw(parts);
    auto begin = [&](int p){ return ngroups * (size_t)p / (size_t)parts; };
    auto size_of = [&](size_t q){ return (int)std::min((size_t)group, n - q * (size_t)group); };
    const std::function<void(int)> find = [&](int p){
        signed char *digit = digits.data() + (size_t)p * stride;
        const bool nearest = q4n_nearest();
        size_t l = 0, r = 0;
        for(size_t q = begin(p); q < begin(p + 1); q++){
            const int g = size_of(q);
            const float s = group_scale(P + q * (size_t)group, g, nearest, digit);
            scales[q] = s;
            if(s != s){ l += 4 + 4 * (size_t)g; r++; } else l += 4 + (size_t)(g + 1) / 2;
        }
        len[p] = l; raw[p] = r;
    }, put = [&](int p){
        signed char *digit = digits.data() + (size_t)p * stride;
        const bool nearest = q4n_nearest();
        unsigned char *o = out;
        for(int i = 0; i < p; i++) o += len[i];
        for(size_t q = begin(p); q < begin(p + 1); q++){
            const float *v = P + q * (size_t)group;
            const int g = size_of(q);
            const float s = scales[q];
            memcpy(o, &s, 4); o += 4;
            if(s != s){ memcpy(o, v, 4 * (size_t)g); o += 4 * (size_t)g; continue; }
            if(q4n_mid(s, nearest)) put_avx2(v, g, s, o);
            else {
                if(s == 0.0f) memset(digit, 0, (size_t)g); else group_try(v, g, s, digit);
                digit[g] = 0;                              /* the partner of an odd group's last digit */
                group_pack(digit, g, o);
            }
            o += (g + 1) / 2;
        }
    };
    q4n_run(parts, find, &put);
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
    const int parts = q4n_parts(n, ngroups, group, Q4N_READ_PART);
    q4n_run(parts, [&](int p){
        for(size_t q = ngroups * (size_t)p / (size_t)parts; q < ngroups * (size_t)(p + 1) / (size_t)parts; q++){
            const size_t i = q * (size_t)group;
            const int g = (int)std::min((size_t)group, n - i);
            const unsigned char *b = buf + at[q];
            float scale; memcpy(&scale, b, 4);
            if(scale != scale) memcpy(P + i, b + 4, 4 * (size_t)g);
            else group_unpack(b + 4, g, scale, P + i);
        }
    }, nullptr);
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
