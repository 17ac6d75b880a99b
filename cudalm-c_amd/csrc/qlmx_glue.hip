/* qlmx_glue.hip -- the pieces of a top-K MoE layer that sit between the expert GEMMs: router,
 * grouping permutation, row gather / gated scatter, gate gradient, SwiGLU forward and backward.
 *
 * Reference: k_router_topk (cudalm.cu:2515-2534, CPU cpu_kern.h:413-425), k_gp_hist / k_gp_scan /
 * k_gp_scatter (cudalm.cu:3504-3530; the host form of the same permutation is 3586-3599),
 * k_gather / k_scatter_gate / k_gather4 / k_scatter_add4 (cudalm.cu:2536-2567, cpu_kern.h:426-450),
 * k_moe_dgate (cudalm.cu:2591, cpu_kern.h:454-468), k_swiglu / k_swiglu_bwd (cudalm.cu:2430-2453,
 * cpu_kern.h:376-394).
 *
 * Indices (assign, perm, off) and gate probabilities are part of the bit-exact contract: the
 * router restates the CPU build's polynomial exponential operation for operation (this file is
 * compiled without FMA contraction), sums the softmax in expert order, and breaks ties towards
 * the lower expert index; the permutation is the stable counting sort. Everything here is bound by
 * HBM: one read and one write per element, rows moved with 16-byte accesses.
 */
#include "qlmx_dev.h"
#include "qlmx_gemm.h"

/* ---- router, more than 64 experts: one thread per token, experts visited in order so the softmax sum rounds
 * exactly as the reference's loop does. `logit` points at the token's E logits and `pr` at E floats for its
 * probabilities (the two may be the same place). ---- */
__device__ __forceinline__ void route_token(const float *logit, float *pr, int n, int *assign, float *gate,
                                            int N, int E, int K, const float *bias, int bs){
    float mx = -1e30f;
    for(int e = 0; e < E; e++) if(logit[e] > mx) mx = logit[e];
    float sum = 0.0f;
    for(int e = 0; e < E; e++){ const float p = qx_fexp(logit[e] - mx); pr[e] = p; sum += p; }
    const float inv = 1.0f / sum;
    for(int e = 0; e < E; e++) pr[e] *= inv;
    int chosen[8];
    for(int k = 0; k < K; k++){
        int best = -1; float bestp = -1e30f;
        for(int e = 0; e < E; e++){
            bool taken = false;
#pragma unroll
            for(int j = 0; j < 8; j++) taken = taken || (j < k && chosen[j] == e);
            if(taken) continue;
            const float sc = pr[e] + (bias ? bias[k * bs + e] : 0.0f);
            if(sc > bestp){ bestp = sc; best = e; }
        }
        if(best < 0) best = k;
#pragma unroll
        for(int j = 0; j < 8; j++) if(j == k) chosen[j] = best;
        assign[(size_t)k * N + n] = best;
        gate[(size_t)k * N + n] = pr[best];
    }
}

/* rows straight from memory: consecutive threads are E floats apart, for any E */
__global__ void __launch_bounds__(256) k_router_topk(const float *rt, float *rprobs, int *assign, float *gate,
                                                     int N, int E, int K, const float *bias, int bs){
    const int n = blockIdx.x * 256 + threadIdx.x;
    if(n >= N) return;
    route_token(rt + (size_t)n * E, rprobs + (size_t)n * E, n, assign, gate, N, E, K, bias, bs);
}

/* The rows of RT_TOK consecutive tokens are one contiguous piece of `rt`: it is copied to LDS with
 * consecutive threads on consecutive floats, each thread then routes its token out of LDS (rows an odd
 * number of floats apart, so the lanes of a wavefront hit different banks), and the probabilities go
 * back the way the logits came. Same arithmetic in the same order as the kernel above. */
#define RT_TOK 64
#define RT_MAXE 96
__global__ void __launch_bounds__(RT_TOK) k_router_topk_lds(const float *rt, float *rprobs, int *assign, float *gate,
                                                            int N, int E, int K, const float *bias, int bs){
    extern __shared__ float rows[];
    const int n0 = blockIdx.x * RT_TOK, tid = threadIdx.x;
    const int ld = E | 1;
    const int cnt = min(RT_TOK, N - n0) * E;
    const float *src = rt + (size_t)n0 * E;
    int t = tid / E, e = tid - t * E;
    const int dt = RT_TOK / E, de = RT_TOK - dt * E;
    for(int i = tid; i < cnt; i += RT_TOK){
        rows[t * ld + e] = src[i];
        t += dt; e += de; if(e >= E){ e -= E; t++; }
    }
    __syncthreads();
    if(n0 + tid < N) route_token(rows + tid * ld, rows + tid * ld, n0 + tid, assign, gate, N, E, K, bias, bs);
    __syncthreads();
    float *dst = rprobs + (size_t)n0 * E;
    t = tid / E; e = tid - t * E;
    for(int i = tid; i < cnt; i += RT_TOK){
        dst[i] = rows[t * ld + e];
        t += dt; e += de; if(e >= E){ e -= E; t++; }
    }
}

/* At most 64 experts: a token on G lanes, one expert each (G = 8, 16, 32 or 64, 64/G tokens per wavefront). A thread
 * per token walked its experts one after the other, K + 3 times, each time a chain of dependent instructions: 6-10 us
 * for one to sixteen tokens, 20 for a few hundred, 48 for 32768 x 64, against 2.4-4.6 and 22 with a lane per expert. What
 * the contract fixes is the softmax sum: in expert order from 0. Every lane adds the G terms in that order, read
 * from LDS four at a time (the lanes past E hold zeros, which change no sum). A pick is the largest score, ties to the
 * lowest expert: the group's maximum, then the lowest lane that holds it; a score not above -1e30 (or NaN) is no
 * candidate, and without a candidate the pick is expert k, as in the loop above. */
template<int G> __device__ __forceinline__ float rt_group_max(float v){
    v = fmaxf(v, qx_dpp<0xB1>(v));
    v = fmaxf(v, qx_dpp<0x4E>(v));
    v = fmaxf(v, qx_dpp<0x141>(v));
    if(G >= 16) v = fmaxf(v, qx_dpp<0x140>(v));
    if(G >= 32) v = fmaxf(v, __shfl_xor(v, 16, 64));
    if(G >= 64) v = fmaxf(v, __shfl_xor(v, 32, 64));
    return v;
}
#define RT_WG 256
template<int G>
__global__ void __launch_bounds__(RT_WG) k_router_topk_lanes(const float *rt, float *rprobs, int *assign, float *gate,
                                                            int N, int E, int K, const float *bias, int bs){
    __shared__ __attribute__((aligned(16))) float terms[RT_WG];
    const int tid = threadIdx.x, lane = tid & 63, e = tid & (G - 1), g0 = lane & ~(G - 1);
    const int n = blockIdx.x * (RT_WG / G) + tid / G;
    const bool on = n < N && e < E;
    const size_t at = (size_t)n * E + e;
    const float l = on ? rt[at] : -INFINITY;
    const float mx = fmaxf(rt_group_max<G>(l), -1e30f);
    float p = on ? qx_fexp(l - mx) : 0.0f;
    terms[tid] = p;
    __syncthreads();
    float sum = 0.0f;
    const float4 *row = (const float4 *)(terms + (tid & ~(G - 1)));
#pragma unroll
    for(int i = 0; i < G / 4; i++){ const float4 v = row[i]; sum += v.x; sum += v.y; sum += v.z; sum += v.w; }
    p *= 1.0f / sum;
    if(on) rprobs[at] = p;
    bool open = on;                                       /* an expert of this token that is not picked yet */
    for(int k = 0; k < K; k++){
        const float sc = p + (bias && on ? bias[k * bs + e] : 0.0f);
        const float v = (open && sc > -1e30f) ? sc : -INFINITY;
        const float m = rt_group_max<G>(v);
        unsigned long long hit = __ballot(v == m && v > -INFINITY) >> g0;
        if(G < 64) hit &= (1ull << G) - 1;
        const int best = hit ? __ffsll((long long)hit) - 1 : k;
        const float gv = __shfl(p, g0 + best, 64);
        if(e == 0 && n < N){ assign[(size_t)k * N + n] = best; gate[(size_t)k * N + n] = gv; }
        open = open && e != best;
    }
}

/* ---- grouping permutation of one pass: perm lists the tokens expert by expert, tokens of one
 * expert in ascending order; off[e] is the first row of expert e, off[E] = N.
 * A workgroup places the tokens of one chunk, its wavefronts one contiguous segment each, 64 tokens at a time: the
 * lanes that share an expert are found with one ballot per bit of the expert's number, a token's row is the next free
 * row of (wavefront, expert) plus the number of earlier lanes with its expert. Up to GP_ONE tokens are one chunk and
 * one launch; more are cut into at most 64 chunks, whose histograms a first launch leaves in the workspace and every
 * workgroup of the second adds up for itself. Kernel times for 386 tokens: 3.9 us (clear, histograms, scan and placement
 * as four launches: 17); 16384: 11 us (20); 131072: 13 us (33). ---- */
#define GP_ONE 4096
static inline int gp_chunk(int N){ return N <= GP_ONE ? N : 2048 * ((N + 2048 * 64 - 1) / (2048 * 64)); }
static inline int gp_threads(int E){ return E <= 896 ? 1024 : E <= 2600 ? 256 : 64; }   /* [wavefronts + 2][E] counters in 64 KB of LDS */
/* workspace: hist[K][NC][E], then seen[K][NC] (0, or -1-e for an expert number e out of range) and, at the offset that
 * qlmx_moe_perm_status reads, bad[K], the same for each whole pass: every pass has a workgroup of its own that writes its
 * word, so no word has to be cleared first and none is written by two */
__global__ void __launch_bounds__(1024) k_gp_hist(const int *asn, int N, int E, int chunk, int *hist, int *seen){
    extern __shared__ int cnt[];                          /* [E], then the flag */
    const int c = blockIdx.x, k = blockIdx.y, end = min(N, (c + 1) * chunk);
    for(int e = threadIdx.x; e <= E; e += blockDim.x) cnt[e] = 0;
    __syncthreads();
    for(int n = c * chunk + threadIdx.x; n < end; n += blockDim.x){
        const int e = asn[(size_t)k * N + n];
        if((unsigned)e < (unsigned)E) atomicAdd(&cnt[e], 1); else cnt[E] = -1 - e;
    }
    __syncthreads();
    const size_t at = (size_t)k * gridDim.x + c;
    for(int e = threadIdx.x; e < E; e += blockDim.x) hist[at * E + e] = cnt[e];
    if(threadIdx.x == 0) seen[at] = cnt[E];
}
__device__ __forceinline__ int wave_incl_scan(int v, int lane){
#pragma unroll
    for(int d = 1; d < 64; d <<= 1){ const int u = __shfl_up(v, d, 64); if(lane >= d) v += u; }
    return v;
}
__global__ void __launch_bounds__(1024) k_gp_place(const int *asn, int N, int E, int chunk, const int *hist, const int *seen,
                                                   int *perm, int *off, int *bad){
    extern __shared__ int lds[];                          /* next[waves][E], first[E + 1] (totals, then first rows), earlier[E], flag */
    const int c = blockIdx.x, k = blockIdx.y, NC = gridDim.x, NT = blockDim.x, NW = NT >> 6;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int *next = lds, *mine = lds + wave * E, *first = lds + NW * E, *earlier = first + E + 1, *flag = earlier + E;
    const int *a = asn + (size_t)k * N;
    const int n0 = c * chunk, n1 = min(N, n0 + chunk);
    const int seg = ((n1 - n0 + NW - 1) / NW + 63) & ~63, s0 = n0 + wave * seg, s1 = min(n1, s0 + seg);
    for(int i = tid; i < (NW + 2) * E + 2; i += NT) lds[i] = 0;
    __syncthreads();
    for(int n = s0 + lane; n < s1; n += 64){
        const int e = a[n];
        if((unsigned)e < (unsigned)E) atomicAdd(&mine[e], 1); else *flag = -1 - e;
    }
    __syncthreads();
    /* an expert's tokens in the chunks before this one, and in all of them */
    if(NC > 1){
        for(int x = tid; x < NC * E; x += NT){
            const int h = hist[(size_t)k * NC * E + x], i = x / E, e = x - i * E;
            if(h){ atomicAdd(&first[e], h); if(i < c) atomicAdd(&earlier[e], h); }
        }
        __syncthreads();
    }
    for(int e = tid; e < E; e += NT){
        int row = earlier[e];
        for(int w = 0; w < NW; w++){ const int h = next[w * E + e]; next[w * E + e] = row; row += h; }
        if(NC == 1) first[e] = row;
    }
    __syncthreads();
    if(wave == 0){
        int run = 0;
        for(int e0 = 0; e0 < E; e0 += 64){
            const int e = e0 + lane, t = e < E ? first[e] : 0, incl = wave_incl_scan(t, lane);
            if(e < E) first[e] = run + incl - t;
            run += __shfl(incl, 63, 64);
        }
        if(lane == 0) first[E] = run;
    }
    __syncthreads();
    if(c == 0){
        for(int e = tid; e <= E; e += NT) off[(size_t)k * (E + 1) + e] = first[e];
        if(wave == 0){
            int f = *flag;
            if(seen) for(int i = lane; i < NC; i += 64) if(seen[(size_t)k * NC + i]) f = seen[(size_t)k * NC + i];
            const unsigned long long any = __ballot(f != 0);
            f = any ? __shfl(f, __ffsll((long long)any) - 1, 64) : 0;
            if(lane == 0) bad[k] = f;
        }
    }
    const int bits = 32 - __clz(E);
    for(int n = s0 + lane; n - lane < s1; n += 64){
        const int e = n < s1 ? a[n] : -1;
        const bool ok = (unsigned)e < (unsigned)E;
        unsigned long long same = __ballot(ok);
        for(int b = 0; b < bits; b++){ const unsigned long long m = __ballot((e >> b) & 1); same &= ((e >> b) & 1) ? m : ~m; }
        if(ok){
            const int row = mine[e], rank = __popcll(same & ((1ull << lane) - 1));
            perm[(size_t)k * N + first[e] + row + rank] = n;
            if(rank == 0) mine[e] = row + __popcll(same);
        }
        qx_wave_sync();
    }
}

__global__ void __launch_bounds__(256) k_fill_i32(int *p, int v, int n){
    const int i = blockIdx.x * 256 + threadIdx.x;
    if(i < n) p[i] = v;
}

/* ---- row movers. One workgroup per row; D % 4 == 0. Bound by HBM. What a launch touches once goes past the caches (NT)
 * where it is more than the last-level cache holds: it would only push out the rows that the K experts of a token read
 * again, and plain loads of such a stream reach 5.1 TB/s, these 6.1. 131072 rows of 2048: combine 316 -> 263 us, gate
 * gradient 437 -> 355, gather 222 -> 219. Smaller buffers are partly in the cache, left there by the GEMM before or kept for
 * the one after (16384 rows of 768 again and again: gate gradient 19.1 us, 20.3 with NT). ---- */
#define PAST_CACHE (256ull << 20)                      /* bytes of the launch's rows in fp32 */
typedef float gl_f4 __attribute__((ext_vector_type(4)));
typedef uint32_t gl_u2 __attribute__((ext_vector_type(2)));
template<bool NT> __device__ __forceinline__ float4 row_load(const float4 *p){
    if(!NT) return *p;
    const gl_f4 v = __builtin_nontemporal_load((const gl_f4 *)p);
    return make_float4(v.x, v.y, v.z, v.w);
}
/* v as unit i of four values of a row buffer of either type */
template<bool OUT_BF16, bool NT> __device__ __forceinline__ void row_store(void *rows, size_t i, float4 v){
    if(OUT_BF16){
        const gl_u2 o = {(uint32_t)qx_f32_to_bf16(v.x) | ((uint32_t)qx_f32_to_bf16(v.y) << 16),
                         (uint32_t)qx_f32_to_bf16(v.z) | ((uint32_t)qx_f32_to_bf16(v.w) << 16)};
        if(NT) __builtin_nontemporal_store(o, (gl_u2 *)rows + i); else ((gl_u2 *)rows)[i] = o;
    } else {
        const gl_f4 o = {v.x, v.y, v.z, v.w};
        if(NT) __builtin_nontemporal_store(o, (gl_f4 *)rows + i); else ((gl_f4 *)rows)[i] = o;
    }
}
template<bool OUT_BF16, bool NT>
__global__ void __launch_bounds__(256) k_gather_rows(const float4 *src, const int *perm, void *Xp, int D4){
    const int j = blockIdx.x, n = perm[j];
    const float4 *s = src + (size_t)(n < 0 ? 0 : n) * D4;
    for(int d = threadIdx.x; d < D4; d += 256){
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if(n >= 0) v = s[d];
        row_store<OUT_BF16, NT>(Xp, (size_t)j * D4 + d, v);
    }
}
/* out[perm[j],:] = out[perm[j],:] + gate[perm[j]] * yp[j,:] (multiply, then add); a pass names every
 * token at most once, so rows do not collide */
__global__ void __launch_bounds__(256) k_scatter_gate(const float4 *yp, const int *perm, const float *gate, float4 *out, int D4){
    const int j = blockIdx.x, n = perm[j];
    if(n < 0) return;
    const float g = gate[n];
    float4 *o = out + (size_t)n * D4; const float4 *y = yp + (size_t)j * D4;
    for(int d = threadIdx.x; d < D4; d += 256){
        float4 a = o[d]; const float4 b = y[d];
        a.x = a.x + g * b.x; a.y = a.y + g * b.y; a.z = a.z + g * b.z; a.w = a.w + g * b.w;
        o[d] = a;
    }
}
__global__ void __launch_bounds__(256) k_scatter_add(const float4 *dXp, const int *perm, float4 *dst, int D4){
    const int j = blockIdx.x, n = perm[j];
    if(n < 0) return;
    float4 *o = dst + (size_t)n * D4; const float4 *s = dXp + (size_t)j * D4;
    for(int d = threadIdx.x; d < D4; d += 256){
        float4 a = o[d]; const float4 b = s[d];
        a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
        o[d] = a;
    }
}
/* d_gate[n] = dout[n,:] . yp[j,:];  dyp[j,:] = gate[n] * dout[n,:] */
template<bool OUT_BF16, bool NT>
__global__ void __launch_bounds__(256) k_moe_dgate(const float4 *dout, const float4 *yp, const int *perm, const float *gate,
                                                   float *d_gate, void *dyp, int D4, int tokens){
    __shared__ float red[4];
    /* one pass (tokens = 0): perm names the token, which also indexes gate and d_gate; all passes as one grouped
     * list: perm names pass * tokens + token, which indexes gate and d_gate, and the token is the remainder */
    const int j = blockIdx.x, m = perm[j], n = (tokens && m >= 0) ? m % tokens : m;
    if(n < 0){
        for(int d = threadIdx.x; d < D4; d += 256) row_store<OUT_BF16, NT>(dyp, (size_t)j * D4 + d, make_float4(0.0f, 0.0f, 0.0f, 0.0f));
        return;
    }
    const float4 *dr = dout + (size_t)n * D4, *y = yp + (size_t)j * D4;
    const float g = gate[m];
    float acc = 0.0f;
    for(int d = threadIdx.x; d < D4; d += 256){
        const float4 a = dr[d], b = row_load<NT>(&y[d]);
        acc += a.x * b.x; acc += a.y * b.y; acc += a.z * b.z; acc += a.w * b.w;
        row_store<OUT_BF16, NT>(dyp, (size_t)j * D4 + d, make_float4(g * a.x, g * a.y, g * a.z, g * a.w));
    }
    acc = qx_wave_sum(acc);
    if((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if(threadIdx.x == 0) d_gate[m] = (red[0] + red[1]) + (red[2] + red[3]);
}

/* ---- all K passes as ONE expert-grouped list of K*N rows (the reference's merged top-K, cudalm.cu:3532-3561,
 * 4022-4034): the grouping permutation of the K*N assignments names entries m = pass * N + token; row p of the
 * grouped buffers holds token perm[p] % N, and inv[m] is the row that holds entry m. ---- */
/* A workgroup reads the whole permutation and keeps the inverse of its own MR_WINDOW entries in LDS: one launch, where a fill
 * and the kernel that overwrites it are two. The reading grows with the square of the rows; beyond MR_WHOLE of them two
 * launches are the faster (12004 rows 5.7 -> 3.4 us, 32768 5.8 -> 5.5, 131072 5.4 and 16.5). */
#define MR_WINDOW 1024
#define MR_WHOLE 32768
__global__ void __launch_bounds__(MR_WINDOW) k_merge_rows_windows(const int *perm, int KN, int N, int *tok, int *inv){
    __shared__ int at[MR_WINDOW];
    const int first = (int)blockIdx.x * MR_WINDOW, own = first + (int)threadIdx.x;
    at[threadIdx.x] = -1;
    __syncthreads();
    for(int p0 = 0; p0 < KN; p0 += 8 * MR_WINDOW){
        int m[8];
#pragma unroll
        for(int k = 0; k < 8; k++) m[k] = perm[min(p0 + k * MR_WINDOW + (int)threadIdx.x, KN - 1)];
#pragma unroll
        for(int k = 0; k < 8; k++){
            const int p = p0 + k * MR_WINDOW + (int)threadIdx.x;
            if(p >= KN) continue;
            if(m[k] >= first && m[k] - first < MR_WINDOW) at[m[k] - first] = p;
            if(p == own) tok[p] = m[k] < 0 ? -1 : m[k] % N;
        }
    }
    __syncthreads();
    if(own < KN) inv[own] = at[threadIdx.x];
}
__global__ void __launch_bounds__(256) k_merge_rows(const int *perm, int KN, int N, int *tok, int *inv){
    const int p = blockIdx.x * 256 + threadIdx.x;
    if(p >= KN) return;
    const int m = perm[p];
    tok[p] = m < 0 ? -1 : m % N;
    if(m >= 0) inv[m] = p;
}
/* out[n,:] = (..(out[n,:] + g[0*N+n] * y[inv[0*N+n],:]) + ..) + g[(K-1)*N+n] * y[inv[(K-1)*N+n],:], pass after pass:
 * the sums the per-pass scatters build, in their order (g NULL: plain additions; inv < 0: the pass dropped the token).
 * The rows of KU passes are requested together: one after the other, a trip to memory each, they were the kernel where it is short (193 rows of 768,
 * two passes: 4.8 -> 4.2 us; 3001 of 2048, four passes: 29.4 -> 26.0). A dropped pass reads the output row once more. */
template<bool NT, int KU>
__global__ void __launch_bounds__(256) k_combine(const float4 *y, const int *inv, const float *g, float4 *out, int N, int K, int D4){
    const int n = blockIdx.x;
    float4 *o = out + (size_t)n * D4;
    for(int d = threadIdx.x; d < D4; d += 256){
        float4 a = o[d];
        for(int k0 = 0; k0 < K; k0 += KU){
            int p[KU]; float4 b[KU]; float w[KU];
#pragma unroll
            for(int j = 0; j < KU; j++){
                const size_t i = (size_t)min(k0 + j, K - 1) * N + n;
                p[j] = k0 + j < K ? inv[i] : -1;
                w[j] = g ? g[i] : 0.0f;
            }
#pragma unroll
            for(int j = 0; j < KU; j++) b[j] = row_load<NT>(p[j] >= 0 ? &y[(size_t)p[j] * D4 + d] : &o[d]);
#pragma unroll
            for(int j = 0; j < KU; j++){
                if(p[j] < 0) continue;
                if(g){ a.x = a.x + w[j] * b[j].x; a.y = a.y + w[j] * b[j].y; a.z = a.z + w[j] * b[j].z; a.w = a.w + w[j] * b[j].w; }
                else { a.x += b[j].x; a.y += b[j].y; a.z += b[j].z; a.w += b[j].w; }
            }
        }
        o[d] = a;
    }
}

/* ---- SwiGLU between the GEMMs: O = g * sigmoid(g) * u with the polynomial sigmoid ---- */
template<bool OUT_BF16>
__global__ void __launch_bounds__(256) k_swiglu(const float4 *G, const float4 *U, void *O, size_t n4){
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if(i >= n4) return;
    const float4 g = G[i], u = U[i];
    float4 o;
    o.x = g.x * qx_fsig(g.x) * u.x; o.y = g.y * qx_fsig(g.y) * u.y;
    o.z = g.z * qx_fsig(g.z) * u.z; o.w = g.w * qx_fsig(g.w) * u.w;
    if(OUT_BF16){
        uint2 p;
        p.x = (uint32_t)qx_f32_to_bf16(o.x) | ((uint32_t)qx_f32_to_bf16(o.y) << 16);
        p.y = (uint32_t)qx_f32_to_bf16(o.z) | ((uint32_t)qx_f32_to_bf16(o.w) << 16);
        ((uint2 *)O)[i] = p;
    } else ((float4 *)O)[i] = o;
}
template<bool OUT_BF16>
__global__ void __launch_bounds__(256) k_swiglu_bwd(const float4 *Gg, const float4 *U, const float4 *dact, void *dg, void *du, size_t n4){
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if(i >= n4) return;
    const float4 g = Gg[i], u = U[i], a = dact[i];
    float4 x, y;
    qx_swiglu_bwd1(g.x, u.x, a.x, x.x, y.x); qx_swiglu_bwd1(g.y, u.y, a.y, x.y, y.y);
    qx_swiglu_bwd1(g.z, u.z, a.z, x.z, y.z); qx_swiglu_bwd1(g.w, u.w, a.w, x.w, y.w);
    if(OUT_BF16){
        uint2 p, q;
        p.x = (uint32_t)qx_f32_to_bf16(x.x) | ((uint32_t)qx_f32_to_bf16(x.y) << 16);
        p.y = (uint32_t)qx_f32_to_bf16(x.z) | ((uint32_t)qx_f32_to_bf16(x.w) << 16);
        q.x = (uint32_t)qx_f32_to_bf16(y.x) | ((uint32_t)qx_f32_to_bf16(y.y) << 16);
        q.y = (uint32_t)qx_f32_to_bf16(y.z) | ((uint32_t)qx_f32_to_bf16(y.w) << 16);
        ((uint2 *)dg)[i] = p; ((uint2 *)du)[i] = q;
    } else { ((float4 *)dg)[i] = x; ((float4 *)du)[i] = y; }
}

/* ------------------------------------------------------------------------------------------
 * C ABI
 * ---------------------------------------------------------------------------------------- */
#define GLUE_ALIGN16(p) ((((uintptr_t)(p)) & 15) == 0)

extern "C" int qlmx_router_topk(const float *rt, float *rprobs, int *assign, float *gate, int N, int E, int K,
                                const float *bias, int bs, void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(rt && rprobs && assign && gate, "qlmx_router_topk: NULL buffer");
    QLMX_REQUIRE(N >= 0 && E > 0 && K > 0 && K <= 8 && K <= E, "qlmx_router_topk: N=%d E=%d K=%d (K at most 8 and at most E)", N, E, K);
    if(N == 0) return QLMX_OK;
#define ROUTE_LANES(G) hipLaunchKernelGGL(k_router_topk_lanes<G>, dim3((N + RT_WG / G - 1) / (RT_WG / G)), dim3(RT_WG), 0, (hipStream_t)stream, \
                                          rt, rprobs, assign, gate, N, E, K, bias, bs)
    if(E <= 8) ROUTE_LANES(8);
    else if(E <= 16) ROUTE_LANES(16);
    else if(E <= 32) ROUTE_LANES(32);
    else if(E <= 64) ROUTE_LANES(64);
#undef ROUTE_LANES
    else if(E <= RT_MAXE)
        hipLaunchKernelGGL(k_router_topk_lds, dim3((N + RT_TOK - 1) / RT_TOK), dim3(RT_TOK), (size_t)RT_TOK * (E | 1) * sizeof(float),
                           (hipStream_t)stream, rt, rprobs, assign, gate, N, E, K, bias, bs);
    else
        hipLaunchKernelGGL(k_router_topk, dim3((N + 255) / 256), dim3(256), 0, (hipStream_t)stream, rt, rprobs, assign, gate, N, E, K, bias, bs);
    QLMX_LAUNCH_CHECK("router launch");
    return QLMX_OK;
}

#define GP_CHUNK 256          /* the workspace has room for a histogram per 256 tokens, more than gp_chunk cuts */
static size_t gp_flag_at(int N, int E, int K){ return (size_t)K * ((size_t)(N + GP_CHUNK - 1) / GP_CHUNK) * E; }
extern "C" size_t qlmx_moe_perm_workspace(int N, int E, int K){
    return (gp_flag_at(N, E, K) + 4 + (size_t)K * E) * sizeof(int);       /* the flags are the first K of the words behind the histograms */
}

extern "C" int qlmx_moe_perm(const int *assign, int N, int E, int K, int *perm, int *off, void *workspace, void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    QLMX_REQUIRE(assign && perm && off && workspace, "qlmx_moe_perm: NULL buffer");
    QLMX_REQUIRE(N > 0 && E > 0 && E <= 4096 && K > 0, "qlmx_moe_perm: N=%d E=%d K=%d", N, E, K);
    const int chunk = gp_chunk(N), NC = (N + chunk - 1) / chunk, NT = gp_threads(E);
    int *hist = (int *)workspace, *seen = hist + (size_t)K * NC * E, *bad = hist + gp_flag_at(N, E, K);
    if(NC > 1){
        hipLaunchKernelGGL(k_gp_hist, dim3(NC, K), dim3(NT), (E + 1) * sizeof(int), st, assign, N, E, chunk, hist, seen);
        QLMX_LAUNCH_CHECK("perm histogram launch");
    }
    hipLaunchKernelGGL(k_gp_place, dim3(NC, K), dim3(NT), ((size_t)(NT / 64 + 2) * E + 2) * sizeof(int), st, assign, N, E, chunk,
                       (const int *)hist, (const int *)(NC > 1 ? seen : nullptr), perm, off, bad);
    QLMX_LAUNCH_CHECK("perm placement launch");
    return QLMX_OK;
}

/* 0 when every assignment of the last qlmx_moe_perm on this workspace was in range, else -1-e for
 * one offending expert index e (the reference aborts the run, cudalm.cu:3476-3478). Synchronises. */
extern "C" int qlmx_moe_perm_status(const void *workspace, int N, int E, int K, void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(workspace, "qlmx_moe_perm_status: NULL workspace");
    enum { AT_ONCE = 64 };                                 /* more passes than any caller has */
    int bad[AT_ONCE];
    for(int k0 = 0; k0 < K; k0 += AT_ONCE){
        const int n = K - k0 < AT_ONCE ? K - k0 : AT_ONCE;
        QLMX_HIP(hipMemcpyAsync(bad, (const int *)workspace + gp_flag_at(N, E, K) + k0, (size_t)n * sizeof(int), hipMemcpyDeviceToHost, (hipStream_t)stream), "perm flag read");
        QLMX_HIP(hipStreamSynchronize((hipStream_t)stream), "perm flag sync");
        for(int k = 0; k < n; k++)
            if(bad[k]){ qlmx_set_error("qlmx_moe_perm: expert index %d out of range [0, %d)", -1 - bad[k], E); return QLMX_E_ARG; }
    }
    return QLMX_OK;
}

#define GLUE_ROWS_CHECK(name, D)                                                                   \
    QLMX_REQUIRE((D) > 0 && (D) % 4 == 0, name ": D=%d must be a positive multiple of 4", (D))

extern "C" int qlmx_moe_gather(const float *src, const int *perm, void *Xp, int N, int D, int out_dtype, void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(src && perm && Xp, "qlmx_moe_gather: NULL buffer");
    GLUE_ROWS_CHECK("qlmx_moe_gather", D);
    QLMX_REQUIRE(GLUE_ALIGN16(src) && GLUE_ALIGN16(Xp), "qlmx_moe_gather: buffers must be 16-byte aligned");
    QLMX_REQUIRE(out_dtype == QLMX_ACT_F32 || out_dtype == QLMX_ACT_BF16, "qlmx_moe_gather: unknown output type %d", out_dtype);
    if(N <= 0) return QLMX_OK;
    const bool bf = out_dtype == QLMX_ACT_BF16, nt = (unsigned long long)N * D * 4 >= PAST_CACHE;
    hipLaunchKernelGGL((bf ? nt ? k_gather_rows<true, true> : k_gather_rows<true, false> : nt ? k_gather_rows<false, true> : k_gather_rows<false, false>),
                       dim3(N), dim3(256), 0, (hipStream_t)stream, (const float4 *)src, perm, Xp, D / 4);
    QLMX_LAUNCH_CHECK("gather launch");
    return QLMX_OK;
}

extern "C" int qlmx_moe_scatter_gate(const float *yp, const int *perm, const float *gate, float *out, int N, int D, void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(yp && perm && gate && out, "qlmx_moe_scatter_gate: NULL buffer");
    GLUE_ROWS_CHECK("qlmx_moe_scatter_gate", D);
    QLMX_REQUIRE(GLUE_ALIGN16(yp) && GLUE_ALIGN16(out), "qlmx_moe_scatter_gate: buffers must be 16-byte aligned");
    if(N <= 0) return QLMX_OK;
    hipLaunchKernelGGL(k_scatter_gate, dim3(N), dim3(256), 0, (hipStream_t)stream, (const float4 *)yp, perm, gate, (float4 *)out, D / 4);
    QLMX_LAUNCH_CHECK("scatter launch");
    return QLMX_OK;
}

extern "C" int qlmx_moe_scatter_add(const float *dXp, const int *perm, float *dst, int N, int D, void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(dXp && perm && dst, "qlmx_moe_scatter_add: NULL buffer");
    GLUE_ROWS_CHECK("qlmx_moe_scatter_add", D);
    QLMX_REQUIRE(GLUE_ALIGN16(dXp) && GLUE_ALIGN16(dst), "qlmx_moe_scatter_add: buffers must be 16-byte aligned");
    if(N <= 0) return QLMX_OK;
    hipLaunchKernelGGL(k_scatter_add, dim3(N), dim3(256), 0, (hipStream_t)stream, (const float4 *)dXp, perm, (float4 *)dst, D / 4);
    QLMX_LAUNCH_CHECK("scatter-add launch");
    return QLMX_OK;
}

static void dgate_launch(const float *dout, const float *yp, const int *perm, const float *gate, float *d_gate, void *dyp, int rows, int D, int out_dtype,
                         int tokens, hipStream_t stream){
    const bool bf = out_dtype == QLMX_ACT_BF16, nt = (unsigned long long)rows * D * 4 >= PAST_CACHE;
    hipLaunchKernelGGL((bf ? nt ? k_moe_dgate<true, true> : k_moe_dgate<true, false> : nt ? k_moe_dgate<false, true> : k_moe_dgate<false, false>),
                       dim3(rows), dim3(256), 0, stream, (const float4 *)dout, (const float4 *)yp, perm, gate, d_gate, dyp, D / 4, tokens);
}

extern "C" int qlmx_moe_dgate(const float *dout, const float *yp, const int *perm, const float *gate,
                              float *d_gate, void *dyp, int N, int D, int out_dtype, void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(dout && yp && perm && gate && d_gate && dyp, "qlmx_moe_dgate: NULL buffer");
    GLUE_ROWS_CHECK("qlmx_moe_dgate", D);
    QLMX_REQUIRE(GLUE_ALIGN16(dout) && GLUE_ALIGN16(yp) && GLUE_ALIGN16(dyp), "qlmx_moe_dgate: buffers must be 16-byte aligned");
    QLMX_REQUIRE(out_dtype == QLMX_ACT_F32 || out_dtype == QLMX_ACT_BF16, "qlmx_moe_dgate: unknown output type %d", out_dtype);
    if(N <= 0) return QLMX_OK;
    dgate_launch(dout, yp, perm, gate, d_gate, dyp, N, D, out_dtype, 0, (hipStream_t)stream);
    QLMX_LAUNCH_CHECK("dgate launch");
    return QLMX_OK;
}

/* ---- merged passes ---- */
extern "C" int qlmx_moe_merge_rows(const int *perm, int N, int K, int *tok, int *inv, void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(perm && tok && inv, "qlmx_moe_merge_rows: NULL buffer");
    QLMX_REQUIRE(N > 0 && K > 0 && (long long)N * K < (1LL << 31), "qlmx_moe_merge_rows: N=%d K=%d", N, K);
    const int KN = N * K;
    if(KN <= MR_WHOLE && tok != perm){                     /* over the permutation: a workgroup there reads what another may have overwritten */
        hipLaunchKernelGGL(k_merge_rows_windows, dim3((KN + MR_WINDOW - 1) / MR_WINDOW), dim3(MR_WINDOW), 0, (hipStream_t)stream, perm, KN, N, tok, inv);
        QLMX_LAUNCH_CHECK("merge rows launch");
        return QLMX_OK;
    }
    /* rows a caller dropped (perm < 0) leave no inverse: -1 everywhere first, by a kernel so that a capture holds no memset node */
    hipLaunchKernelGGL(k_fill_i32, dim3((KN + 255) / 256), dim3(256), 0, (hipStream_t)stream, inv, -1, KN);
    QLMX_LAUNCH_CHECK("merge rows: inverse fill");
    hipLaunchKernelGGL(k_merge_rows, dim3((KN + 255) / 256), dim3(256), 0, (hipStream_t)stream, perm, KN, N, tok, inv);
    QLMX_LAUNCH_CHECK("merge rows launch");
    return QLMX_OK;
}

extern "C" int qlmx_moe_combine(const float *y, const int *inv, const float *gate, float *out, int N, int K, int D, void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(y && inv && out, "qlmx_moe_combine: NULL buffer");
    GLUE_ROWS_CHECK("qlmx_moe_combine", D);
    QLMX_REQUIRE(K > 0 && GLUE_ALIGN16(y) && GLUE_ALIGN16(out), "qlmx_moe_combine: K=%d, buffers must be 16-byte aligned", K);
    if(N <= 0) return QLMX_OK;
    const bool nt = (unsigned long long)N * K * D * 4 >= PAST_CACHE;
    hipLaunchKernelGGL((K == 1 ? nt ? k_combine<true, 1> : k_combine<false, 1> : K == 2 ? nt ? k_combine<true, 2> : k_combine<false, 2>
                                                                               : nt ? k_combine<true, 4> : k_combine<false, 4>), dim3(N), dim3(256), 0, (hipStream_t)stream, (const float4 *)y, inv, gate, (float4 *)out, N, K, D / 4);
    QLMX_LAUNCH_CHECK("combine launch");
    return QLMX_OK;
}

extern "C" int qlmx_moe_dgate_merged(const float *dout, const float *yp, const int *perm, const float *gate,
                                     float *d_gate, void *dyp, int N, int K, int D, int out_dtype, void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(dout && yp && perm && gate && d_gate && dyp, "qlmx_moe_dgate_merged: NULL buffer");
    GLUE_ROWS_CHECK("qlmx_moe_dgate_merged", D);
    QLMX_REQUIRE(GLUE_ALIGN16(dout) && GLUE_ALIGN16(yp) && GLUE_ALIGN16(dyp), "qlmx_moe_dgate_merged: buffers must be 16-byte aligned");
    QLMX_REQUIRE(out_dtype == QLMX_ACT_F32 || out_dtype == QLMX_ACT_BF16, "qlmx_moe_dgate_merged: unknown output type %d", out_dtype);
    QLMX_REQUIRE(K > 0 && (long long)N * K < (1LL << 31), "qlmx_moe_dgate_merged: N=%d K=%d", N, K);
    if(N <= 0) return QLMX_OK;
    const int KN = N * K;
    dgate_launch(dout, yp, perm, gate, d_gate, dyp, KN, D, out_dtype, N, (hipStream_t)stream);
    QLMX_LAUNCH_CHECK("merged dgate launch");
    return QLMX_OK;
}

extern "C" int qlmx_swiglu(const float *G, const float *U, void *O, size_t n, int out_dtype, void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(G && U && O, "qlmx_swiglu: NULL buffer");
    QLMX_REQUIRE(n % 4 == 0 && GLUE_ALIGN16(G) && GLUE_ALIGN16(U) && GLUE_ALIGN16(O), "qlmx_swiglu: n must be a multiple of 4 and the buffers 16-byte aligned");
    QLMX_REQUIRE(out_dtype == QLMX_ACT_F32 || out_dtype == QLMX_ACT_BF16, "qlmx_swiglu: unknown output type %d", out_dtype);
    if(n == 0) return QLMX_OK;
    const size_t n4 = n / 4; const unsigned grid = (unsigned)((n4 + 255) / 256);
    if(out_dtype == QLMX_ACT_BF16) hipLaunchKernelGGL(k_swiglu<true>, dim3(grid), dim3(256), 0, (hipStream_t)stream, (const float4 *)G, (const float4 *)U, O, n4);
    else                           hipLaunchKernelGGL(k_swiglu<false>, dim3(grid), dim3(256), 0, (hipStream_t)stream, (const float4 *)G, (const float4 *)U, O, n4);
    QLMX_LAUNCH_CHECK("swiglu launch");
    return QLMX_OK;
}

extern "C" int qlmx_swiglu_bwd(const float *Gg, const float *U, const float *dact, void *dg, void *du, size_t n, int out_dtype, void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(Gg && U && dact && dg && du, "qlmx_swiglu_bwd: NULL buffer");
    QLMX_REQUIRE(n % 4 == 0 && GLUE_ALIGN16(Gg) && GLUE_ALIGN16(U) && GLUE_ALIGN16(dact) && GLUE_ALIGN16(dg) && GLUE_ALIGN16(du),
                 "qlmx_swiglu_bwd: n must be a multiple of 4 and the buffers 16-byte aligned");
    QLMX_REQUIRE(out_dtype == QLMX_ACT_F32 || out_dtype == QLMX_ACT_BF16, "qlmx_swiglu_bwd: unknown output type %d", out_dtype);
    if(n == 0) return QLMX_OK;
    const size_t n4 = n / 4; const unsigned grid = (unsigned)((n4 + 255) / 256);
    if(out_dtype == QLMX_ACT_BF16) hipLaunchKernelGGL(k_swiglu_bwd<true>, dim3(grid), dim3(256), 0, (hipStream_t)stream, (const float4 *)Gg, (const float4 *)U, (const float4 *)dact, dg, du, n4);
    else                           hipLaunchKernelGGL(k_swiglu_bwd<false>, dim3(grid), dim3(256), 0, (hipStream_t)stream, (const float4 *)Gg, (const float4 *)U, (const float4 *)dact, dg, du, n4);
    QLMX_LAUNCH_CHECK("swiglu backward launch");
    return QLMX_OK;
}
