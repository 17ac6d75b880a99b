/* qlmx_gemm_small.hip -- forward (nn, fp16 matrix core) and input-gradient (tn, bf16 matrix core) grouped GEMMs of
 * experts with few rows: a short prompt, a small training batch.
 *
 * The tiled kernels (qlmx_gemm_nn_h.hip, qlmx_gemm_tn_body.h) give a workgroup a column strip of an expert and the
 * whole contraction, one LDS tile and one barrier per 32 of it. With a dozen rows a step is some 1000 cycles of
 * LDS, barrier and issue latency around four matrix products, and a call has too few strips to hide it: 36 us for the
 * down projection of 32 experts (2048 x 768, 12 rows each), whose 25 MB of weights take 5. Here nothing passes
 * through LDS on the way in, four (input gradient: eight) wavefronts split the contraction and add up at the end:
 *
 * A wavefront owns 128 (64) columns and its share of the contraction. v_mfma_f32_16x16x32 wants eight consecutive k of one
 * column per lane (lane = column lane%16, k group lane/16). Weights of the forward lie along the columns: the lane
 * loads, for its eight k, the 4-byte word of eight neighbouring columns, and product j takes digit j of the eight words
 * -- the columns of a product are then eight apart, which only the store has to know. Weights of the input
 * gradient lie along k as they should; a lane loads 16 or 32 k of four columns sixteen apart. Activations come from
 * L2 straight as operands (16 bytes of a row per lane). All loads of a step are plain register loads, one to four steps
 * ahead, without a barrier in the loop.
 *
 * Arithmetic as in the tiled kernels: forward weights fp16(s * digit * 2^8), activations converted exactly; the input
 * gradient multiplies exact digits and applies the scale to the fp32 sums of each group of k.
 *
 * Which calls come here (qlmx_small_rows): all problems of at most 32 rows, or of at most 64 when the call has few column
 * strips. The rule looks at what the forms of a call that are documented to agree bit for bit have in common -- with and
 * without gather, SwiGLU, scatter, inside a pair or not -- so that they run the same arithmetic in the same order.
 * 32 experts, 768 x 2048, us per call at 4 / 30 rows each, tiled kernels -> these: gate|up + SwiGLU 37 / 33 -> 20 / 22, down
 * 27 / 26 -> 12 / 16, its input gradient + SwiGLU 20 / 22 -> 11 / 20, paired input gradient 56 / 58 -> 27 / 33. At 60 rows
 * (two row tiles of 32, the weights converted twice): 192 strips 27 -> 23 and 58 -> 49, 512 strips 35 -> 39 and 25 -> 36.
 * What bounds them now: the conversion of the weights (some 220 vector instructions for 32 x 128 of them) on as many
 * wavefronts as there are, and the round trips in front of and behind it.
 */
#include "qlmx_gemm.h"
#include <type_traits>

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float  f32x2 __attribute__((ext_vector_type(2)));
typedef float  f32x4 __attribute__((ext_vector_type(4)));
typedef int    i32x2 __attribute__((ext_vector_type(2)));
typedef int    i32x4 __attribute__((ext_vector_type(4)));

#define SM_COLS 128
#define SM_WAVES 4                              /* along the forward's contraction (eight: the same for 2048, 20 % slower for 768) */
#define SM_TWAVES 8                             /* along the input gradient's */
#define SM_WSCALE 4096.0f                       /* 16 (digits come as digit/16) * 2^8, as NH_WSCALE */
#define SM_UNSCALE (1.0f / 256.0f)
#define SM_ROWS 32
#define SM_STRIPS 256

enum { SM_PLAIN = 0, SM_GATHER = 1, SM_SCATTER = 2, SM_SWIGLU_BWD = 3 };
struct SmArgs { const DevProb *pr; int nprob, ntiles; const signed char *d; const float *s; int gshift; int K, N;
                const char *xsrc; float *out; const float *gate;
                const float *gp, *up; unsigned short *dg, *du; };

static __device__ __align__(16) unsigned char sm_zero_row[32768];       /* what a dropped row of a gather reads */

bool qlmx_small_rows(const qlmx_gemm_prob *probs, int nprob, int N, int group){
    if(group < 64) return false;
    int most = 0;
    for(int i = 0; i < nprob; i++) if(probs[i].M > most) most = probs[i].M;
    return most <= SM_ROWS || (most <= 2 * SM_ROWS && (long long)nprob * (N / SM_COLS) <= SM_STRIPS);
}

__device__ __forceinline__ int sm_pk_f16(float lo, float hi){ f32x2 v = {lo, hi}; return __builtin_bit_cast(int, __builtin_convertvector(v, f16x2)); }
__device__ __forceinline__ int sm_pk_bf16(float lo, float hi){ f32x2 v = {lo, hi}; return __builtin_bit_cast(int, __builtin_convertvector(v, bf16x2)); }
__device__ __forceinline__ int sm_bf16x2_to_f16x2(int w){
    return __builtin_bit_cast(int, __builtin_amdgcn_cvt_pkrtz(__uint_as_float((uint32_t)w << 16), __uint_as_float((uint32_t)w & 0xFFFF0000u)));
}
/* value of lane I of every row of 16 lanes (row_newbcast) */
template<int I> __device__ __forceinline__ float sm_bcast(float v){
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + I, 0xF, 0xF, true));
}
/* and of lane 8 + I for the upper half of the row */
template<int I> __device__ __forceinline__ float sm_bcast_hi(float low, float v){
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(low), __float_as_int(v), 0x158 + I, 0xF, 0xC, false));
}
template<int I, int N, class F> __device__ __forceinline__ void sm_each(const F &f){ if constexpr(I < N){ f(std::integral_constant<int, I>()); sm_each<I + 1, N>(f); } }

/* The sums of the SM_WAVES wavefronts from `first` on, of one 16-row tile, through LDS: `mine(e, j)` is a lane's sum of
 * row (lane/16)*4 + e, column j of its eight. total[u] belongs to place u * threads + thread of the tile's 16 x 32
 * places of four columns. */
template<int NT, class F> __device__ __forceinline__ void sm_reduce(float *red, int first, const F &mine, f32x4 (&total)[512 / NT]){
    const int tid = threadIdx.x, lane = tid & 63, wave = (tid >> 6) - first, c = lane & 15, g = lane >> 4;
    __syncthreads();                                      /* the tile before has been read */
    if(wave >= 0 && wave < SM_WAVES){
        float *w = red + wave * (16 * SM_COLS);
#pragma unroll
        for(int e = 0; e < 4; e++){
            *(f32x4 *)&w[(g * 4 + e) * SM_COLS + c * 8]     = (f32x4){mine(e, 0), mine(e, 1), mine(e, 2), mine(e, 3)};
            *(f32x4 *)&w[(g * 4 + e) * SM_COLS + c * 8 + 4] = (f32x4){mine(e, 4), mine(e, 5), mine(e, 6), mine(e, 7)};
        }
    }
    __syncthreads();
    constexpr int U = 512 / NT;
#pragma unroll
    for(int u = 0; u < U; u++){
        const int x = u * NT + tid;                       /* four columns of one row */
        f32x4 v = *(const f32x4 *)&red[x * 4];
#pragma unroll
        for(int k = 1; k < SM_WAVES; k++) v += *(const f32x4 *)&red[k * (16 * SM_COLS) + x * 4];
        total[u] = v * SM_UNSCALE;
    }
}

/* ---- forward. DUAL: gate | up, as many wavefronts again on the second matrix (wq, wg of Q) ---- */
template<int RT, int IO, bool DUAL, bool G64>
__device__ __forceinline__ void sm_nn_tile(const SmArgs &a, const DevProb &P, const DevProb &Q, int i0, int j0, float *red){
    constexpr int PF = RT == 1 ? (DUAL ? 3 : 4) : (DUAL ? 1 : 2);        /* steps on their way */
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
    const int steps = a.K / 32, ks = wave & (SM_WAVES - 1), st0 = steps * ks / SM_WAVES, st1 = steps * (ks + 1) / SM_WAVES;
    const bool second = DUAL && wave >= SM_WAVES;
    const char *pa[RT];
#pragma unroll
    for(int r = 0; r < RT; r++){
        const int row = min(i0 + r * 16 + c, P.M - 1);
        if(IO == SM_GATHER){
            const int tok = ((const int *)P.A)[row];
            pa[r] = tok >= 0 ? a.xsrc + (size_t)tok * a.K * 2 : (const char *)sm_zero_row;
        } else pa[r] = (const char *)P.A + (size_t)row * a.K * 2;
        pa[r] += g * 16;
    }
    const size_t gpr = (size_t)a.N >> a.gshift, rowb = (size_t)a.N >> 1;       /* scale groups and bytes per row of weights */
    const signed char *pw = a.d + (((second ? Q.wq : P.wq) + (size_t)(g * 8) * a.N + j0 + c * 8) >> 1);
    const float *ps = a.s + (second ? Q.wg : P.wg) + (size_t)(g * 8 + (c & 7)) * gpr + (j0 >> a.gshift) + (G64 ? c >> 3 : 0);
    f32x4 acc[RT][8];
#pragma unroll
    for(int r = 0; r < RT; r++)
#pragma unroll
        for(int j = 0; j < 8; j++) acc[r][j] = (f32x4)(0.0f);
    uint32_t w[PF][8]; float s[PF]; i32x4 x[PF][RT];
    auto load = [&](int set, int st){
        const int t = min(st, st1 - 1);                   /* past the end: the last step again, never used */
        s[set] = ps[(size_t)t * 32 * gpr];
#pragma unroll
        for(int i = 0; i < 8; i++) w[set][i] = *(const uint32_t *)(pw + ((size_t)t * 32 + i) * rowb);
#pragma unroll
        for(int r = 0; r < RT; r++) x[set][r] = *(const i32x4 *)(pa[r] + (size_t)t * 64);
    };
    auto step = [&](auto IC, int st){
        constexpr int I = decltype(IC)::value;
        f16x8 xa[RT];
#pragma unroll
        for(int r = 0; r < RT; r++){
            i32x4 v;
#pragma unroll
            for(int q = 0; q < 4; q++) v[q] = sm_bf16x2_to_f16x2(x[I][r][q]);
            xa[r] = __builtin_bit_cast(f16x8, v);
        }
        const float sv = s[I] * SM_WSCALE;
        float sk[8]; QxNibs nb[8];
        sm_each<0, 8>([&](auto KC){
            constexpr int k = decltype(KC)::value;
            sk[k] = sm_bcast<k>(sv);
            if(G64) sk[k] = sm_bcast_hi<k>(sk[k], sv);
            nb[k] = qx_nibs(w[I][k]);
        });
        load(I, st + PF);
        /* two operands at a time: left alone, the compiler builds all eight first and runs out of registers */
#pragma unroll
        for(int j = 0; j < 8; j++){
            i32x4 b;
#pragma unroll
            for(int q = 0; q < 4; q++) b[q] = sm_pk_f16(sk[2 * q] * qx_nib16(nb[2 * q], j), sk[2 * q + 1] * qx_nib16(nb[2 * q + 1], j));
#pragma unroll
            for(int r = 0; r < RT; r++)
                acc[r][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[r], __builtin_bit_cast(f16x8, b), acc[r][j], 0, 0, 0);
            if(j & 1) __builtin_amdgcn_sched_barrier(0);
        }
    };
    if(st0 < st1){
        sm_each<0, PF>([&](auto IC){ load(decltype(IC)::value, st0 + decltype(IC)::value); });
        int st = st0;
        for(; st + PF <= st1; st += PF) sm_each<0, PF>([&](auto IC){ step(IC, st + decltype(IC)::value); });
        sm_each<0, PF - 1>([&](auto IC){ if(st + decltype(IC)::value < st1) step(IC, st + decltype(IC)::value); });
    }
    /* ---- totals ---- */
    constexpr int NT = 64 * SM_WAVES * (DUAL ? 2 : 1), U = 512 / NT;
#pragma unroll
    for(int r = 0; r < RT; r++){
        auto mine = [&](int e, int j){ return acc[r][j][e]; };
        f32x4 ty[U], tu[U];
        sm_reduce<NT>(red, 0, mine, ty);
        if constexpr(DUAL) sm_reduce<NT>(red, SM_WAVES, mine, tu);
#pragma unroll
        for(int v = 0; v < U; v++){
            const int x = v * NT + tid, lr = i0 + r * 16 + (x >> 5);
            if(lr >= P.M) continue;
            const f32x4 y = ty[v];
            const size_t o = (size_t)lr * a.N + j0 + (x & 31) * 4;
            if constexpr(DUAL){
                const f32x4 u = tu[v];
                if(P.C){ *(f32x4 *)(P.C + o) = y; *(f32x4 *)(Q.C + o) = u; }
                ushort4 h;
                h.x = qx_f32_to_bf16(y[0] * qx_fsig_hw(y[0]) * u[0]); h.y = qx_f32_to_bf16(y[1] * qx_fsig_hw(y[1]) * u[1]);
                h.z = qx_f32_to_bf16(y[2] * qx_fsig_hw(y[2]) * u[2]); h.w = qx_f32_to_bf16(y[3] * qx_fsig_hw(y[3]) * u[3]);
                *(ushort4 *)((unsigned short *)Q.B + o) = h;
            } else if constexpr(IO == SM_SCATTER){
                const int tok = ((const int *)P.C)[lr];
                if(tok >= 0){
                    qx_gfloat *t = (qx_gfloat *)(a.out + (size_t)tok * a.N + j0 + (x & 31) * 4);
                    const float gt = a.gate ? a.gate[tok] : 1.0f;
#pragma unroll
                    for(int q = 0; q < 4; q++) (void)__builtin_amdgcn_global_atomic_fadd_f32(t + q, a.gate ? gt * y[q] : y[q]);
                }
            } else *(f32x4 *)(P.C + o) = y;
        }
    }
}

template<int RT, int IO, bool DUAL>
__global__ void __launch_bounds__(64 * SM_WAVES * (DUAL ? 2 : 1), RT == 1 || DUAL ? 4 : 2) k_gemm_nn_small(SmArgs a){
    __shared__ __attribute__((aligned(16))) float red[SM_WAVES * 16 * SM_COLS];
    const int t = qx_xcd_tile(blockIdx.x, gridDim.x);
    if(t >= a.ntiles) return;
    const int pi = qx_find_problem(a.pr, a.nprob, t);
    const DevProb P = a.pr[pi], Q = a.pr[DUAL ? pi + 1 : pi];
    const int lt = t - P.tile0, ti = lt / P.tiles_n, tj = lt - ti * P.tiles_n;
    const int i0 = ti * (RT * 16), j0 = tj * SM_COLS, left = P.M - i0;
    if(a.gshift == 6){
        if(RT == 2 && left > 16) sm_nn_tile<RT, IO, DUAL, true>(a, P, Q, i0, j0, red);
        else                     sm_nn_tile<1, IO, DUAL, true>(a, P, Q, i0, j0, red);
    } else {
        if(RT == 2 && left > 16) sm_nn_tile<RT, IO, DUAL, false>(a, P, Q, i0, j0, red);
        else                     sm_nn_tile<1, IO, DUAL, false>(a, P, Q, i0, j0, red);
    }
}

/* ---- input gradient: 64 columns per wavefront; nseg operand pairs (a continued problem's second pair comes from the
 * table entry behind it). A lane loads ND words of eight k from each of four rows of weights (16 bytes each where the scale
 * group is 128 or more: the 16 lanes of a k group must share a scale group, and the four k groups of a product too). ---- */
#define SM_TCOLS 64
template<int RT, int IO, int ND>
__device__ __forceinline__ void sm_tn_tile(const SmArgs &a, const DevProb &P, const DevProb &Q, int nseg, int i0, int j0, float *red){
    constexpr int PF = RT == 1 ? 2 : 1, KS = ND * 32;     /* steps on their way; contraction values of a step */
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
    /* the wavefronts take the steps in turn: a step reads 16 ND bytes of a weight row, the eight of them 128 ND side by side */
    const int steps1 = a.K / KS, steps = steps1 * nseg, mine = (steps - wave + SM_TWAVES - 1) / SM_TWAVES;
    const int ngroups = a.K >> a.gshift;
    f32x4 acc[RT][4];
#pragma unroll
    for(int r = 0; r < RT; r++)
#pragma unroll
        for(int j = 0; j < 4; j++) acc[r][j] = (f32x4)(0.0f);
    size_t ra[RT];                                        /* the lane's rows of A, in bytes */
#pragma unroll
    for(int r = 0; r < RT; r++) ra[r] = (size_t)min(i0 + r * 16 + c, P.M - 1) * a.K * 2 + g * (ND * 16);
    int w[PF][4][ND]; float s[PF][4]; i32x4 x[PF][RT][ND];
    auto load = [&](int set, int st){
        const int t = wave + SM_TWAVES * min(st, mine - 1);
        const bool two = t >= steps1;
        const int u = two ? t - steps1 : t;
        const char *A = (const char *)(two ? Q.A : P.A) + (size_t)u * (KS * 2);
        const signed char *W = a.d + (((two ? Q.wq : P.wq) + (size_t)(j0 + c) * a.K + (size_t)u * KS) >> 1) + g * (ND * 4);
        const float *S = a.s + (two ? Q.wg : P.wg) + (size_t)(j0 + c) * ngroups + ((u * KS) >> a.gshift);
#pragma unroll
        for(int j = 0; j < 4; j++){
            if constexpr(ND == 4){ const i32x4 v = *(const i32x4 *)(W + (size_t)(j * 16) * a.K / 2); w[set][j][0] = v[0]; w[set][j][1] = v[1]; w[set][j][2] = v[2]; w[set][j][3] = v[3]; }
            else                 { const i32x2 v = *(const i32x2 *)(W + (size_t)(j * 16) * a.K / 2); w[set][j][0] = v[0]; w[set][j][1] = v[1]; }
            s[set][j] = S[(size_t)(j * 16) * ngroups];
        }
#pragma unroll
        for(int r = 0; r < RT; r++)
#pragma unroll
            for(int i = 0; i < ND; i++) x[set][r][i] = *(const i32x4 *)(A + ra[r] + i * 16);
    };
    auto step = [&](auto IC, int st){
        constexpr int I = decltype(IC)::value;
#pragma unroll
        for(int j = 0; j < 4; j++){
            f32x4 p[RT];
#pragma unroll
            for(int r = 0; r < RT; r++) p[r] = (f32x4)(0.0f);
#pragma unroll
            for(int i = 0; i < ND; i++){
                const QxNibs nb = qx_nibs((uint32_t)w[I][j][i]);
                i32x4 b;
#pragma unroll
                for(int q = 0; q < 4; q++) b[q] = sm_pk_bf16(qx_nib16(nb, 2 * q), qx_nib16(nb, 2 * q + 1));
#pragma unroll
                for(int r = 0; r < RT; r++)
                    p[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x[I][r][i]), __builtin_bit_cast(bf16x8, b), p[r], 0, 0, 0);
            }
            const float sc = s[I][j] * 16.0f;
#pragma unroll
            for(int r = 0; r < RT; r++)
#pragma unroll
                for(int e = 0; e < 4; e++) acc[r][j][e] = fmaf(sc, p[r][e], acc[r][j][e]);
        }
        load(I, st + PF);
    };
    if(mine > 0){
        sm_each<0, PF>([&](auto IC){ load(decltype(IC)::value, decltype(IC)::value); });
        int st = 0;
        for(; st + PF <= mine; st += PF) sm_each<0, PF>([&](auto IC){ step(IC, st + decltype(IC)::value); });
        sm_each<0, PF - 1>([&](auto IC){ if(st + decltype(IC)::value < mine) step(IC, st + decltype(IC)::value); });
    }
    /* ---- totals: the thread holds row tid/32, two columns ---- */
    const int row = tid >> 5, col = (tid & 31) * 2;
#pragma unroll
    for(int r = 0; r < RT; r++){
        __syncthreads();                                  /* the tile before has been read */
#pragma unroll
        for(int e = 0; e < 4; e++)
#pragma unroll
            for(int j = 0; j < 4; j++) red[(wave * 16 + g * 4 + e) * SM_TCOLS + j * 16 + c] = acc[r][j][e];
        __syncthreads();
        f32x2 y = *(const f32x2 *)&red[tid * 2];
#pragma unroll
        for(int k = 1; k < SM_TWAVES; k++) y += *(const f32x2 *)&red[k * (16 * SM_TCOLS) + tid * 2];
        const int lr = i0 + r * 16 + row;
        if(lr >= P.M) continue;
        if constexpr(IO == SM_SCATTER){
            const int tok = ((const int *)P.C)[lr];
            if(tok >= 0){
                qx_gfloat *t = (qx_gfloat *)(a.out + (size_t)tok * a.N + j0 + col);
                (void)__builtin_amdgcn_global_atomic_fadd_f32(t, y[0]);
                (void)__builtin_amdgcn_global_atomic_fadd_f32(t + 1, y[1]);
            }
        } else if constexpr(IO == SM_SWIGLU_BWD){
            const size_t o = (size_t)(P.C - a.gp) + (size_t)lr * a.N + j0 + col;      /* even: pairs of bf16 are 4-byte aligned */
            float dg[2], du[2];
#pragma unroll
            for(int q = 0; q < 2; q++) qx_swiglu_bwd1<true>(a.gp[o + q], a.up[o + q], y[q], dg[q], du[q]);
            *(uint32_t *)(a.dg + o) = (uint32_t)qx_f32_to_bf16(dg[0]) | ((uint32_t)qx_f32_to_bf16(dg[1]) << 16);
            *(uint32_t *)(a.du + o) = (uint32_t)qx_f32_to_bf16(du[0]) | ((uint32_t)qx_f32_to_bf16(du[1]) << 16);
        } else {
            f32x2 *o = (f32x2 *)(P.C + (size_t)lr * a.N + j0 + col);
            if(P.beta != 0.0f) y = *o + y;
            *o = y;
        }
    }
}

template<int RT, int IO>
__global__ void __launch_bounds__(64 * SM_TWAVES, 4) k_gemm_tn_small(SmArgs a){
    __shared__ __attribute__((aligned(16))) float red[SM_TWAVES * 16 * SM_TCOLS];
    const int t = qx_xcd_tile(blockIdx.x, gridDim.x);
    if(t >= a.ntiles) return;
    const int pi = qx_find_problem(a.pr, a.nprob, t);
    const DevProb P = a.pr[pi];
    const DevProb Q = a.pr[P.chunk ? pi + 1 : pi];
    const int lt = t - P.tile0, ti = lt / P.tiles_n, tj = lt - ti * P.tiles_n;
    const int i0 = ti * (RT * 16), j0 = tj * SM_TCOLS, left = P.M - i0, nseg = P.chunk ? 2 : 1;
    if(a.gshift >= 7 && a.K % 128 == 0){
        if(RT == 2 && left > 16) sm_tn_tile<RT, IO, 4>(a, P, Q, nseg, i0, j0, red);
        else                     sm_tn_tile<1, IO, 4>(a, P, Q, nseg, i0, j0, red);
    } else {
        if(RT == 2 && left > 16) sm_tn_tile<RT, IO, 2>(a, P, Q, nseg, i0, j0, red);
        else                     sm_tn_tile<1, IO, 2>(a, P, Q, nseg, i0, j0, red);
    }
}

/* ---- launches ---- */
static int sm_row_tiles(const qlmx_gemm_prob *probs, int nprob){
    for(int i = 0; i < nprob; i++) if(probs[i].M > 16) return 2;
    return 1;
}
static SmArgs sm_args(const signed char *d, const float *s, int group, int K, int N, const ProbUpload &up){
    SmArgs a = {};
    a.pr = up.dev; a.nprob = up.nprob; a.ntiles = up.ntiles; a.d = d; a.s = s; a.K = K; a.N = N;
    while((1 << a.gshift) < group) a.gshift++;
    return a;
}
#define SM_LAUNCH(KERNEL, WAVES) hipLaunchKernelGGL(KERNEL, dim3((a.ntiles + 7) & ~7), dim3(64 * (WAVES)), 0, st, a)

/* N % 128 == 0, K % 32 == 0, group a power of two >= 64; io, xsrc, out, gate as in qlmx_gemm_nn_h_launch */
int qlmx_gemm_nn_small_launch(const signed char *d, const float *s, int group, const qlmx_gemm_prob *probs, int nprob, int K, int N,
                              int io, const void *xsrc, float *out, const float *gate, hipStream_t st){
    const int rt = sm_row_tiles(probs, nprob);
    ProbUpload up; int slot;
    int rc = qlmx_upload_problems(probs, nprob, GEMM_NN, K, N, rt * 16, SM_COLS, st, &up, &slot); if(rc) return rc;
    if(up.ntiles == 0) return QLMX_OK;
    SmArgs a = sm_args(d, s, group, K, N, up);
    a.xsrc = (const char *)xsrc; a.out = out; a.gate = gate;
#define SM_NN(IO) do{ if(rt == 1) SM_LAUNCH((k_gemm_nn_small<1, IO, false>), SM_WAVES); else SM_LAUNCH((k_gemm_nn_small<2, IO, false>), SM_WAVES); }while(0)
    if(io == SM_GATHER) SM_NN(SM_GATHER); else if(io == SM_SCATTER) SM_NN(SM_SCATTER); else SM_NN(SM_PLAIN);
#undef SM_NN
    QLMX_LAUNCH_CHECK("grouped gemm nn (few rows) launch");
    return qlmx_upload_done(slot, st);
}
/* gate|up with the SwiGLU behind; N % 128 == 0 */
int qlmx_gemm_nn_small_swiglu_launch(const signed char *d, const float *s, int group, const qlmx_gemm_prob *gate, const qlmx_gemm_prob *up_, int nprob,
                                     int K, int N, const void *xsrc, hipStream_t st){
    const int rt = sm_row_tiles(gate, nprob);
    ProbUpload up; int slot;
    int rc = qlmx_upload_problem_pairs(gate, up_, nprob, GEMM_NN, K, N, rt * 16, SM_COLS, st, &up, &slot); if(rc) return rc;
    if(up.ntiles == 0) return QLMX_OK;
    SmArgs a = sm_args(d, s, group, K, N, up);
    a.xsrc = (const char *)xsrc;
#define SM_DUAL(IO) do{ if(rt == 1) SM_LAUNCH((k_gemm_nn_small<1, IO, true>), 2 * SM_WAVES); else SM_LAUNCH((k_gemm_nn_small<2, IO, true>), 2 * SM_WAVES); }while(0)
    if(xsrc) SM_DUAL(SM_GATHER); else SM_DUAL(SM_PLAIN);
#undef SM_DUAL
    QLMX_LAUNCH_CHECK("grouped gemm nn + swiglu (few rows) launch");
    return qlmx_upload_done(slot, st);
}
/* N % 128 == 0, K % 64 == 0, group a power of two >= 64; the rest as in qlmx_gemm_tn_lds_launch */
int qlmx_gemm_tn_small_launch(const signed char *d, const float *s, int group, const qlmx_gemm_prob *probs, const qlmx_gemm_prob *second, int nprob,
                              int K, int N, float *out, const float *gp, const float *up_, void *dg, void *du, hipStream_t st){
    const int rt = sm_row_tiles(probs, nprob);
    ProbUpload up; int slot;
    int rc = second ? qlmx_upload_problem_pairs(probs, second, nprob, GEMM_TN, K, N, rt * 16, SM_TCOLS, st, &up, &slot)
                    : qlmx_upload_problems(probs, nprob, GEMM_TN, K, N, rt * 16, SM_TCOLS, st, &up, &slot);
    if(rc) return rc;
    if(up.ntiles == 0) return QLMX_OK;
    SmArgs a = sm_args(d, s, group, K, N, up);
    a.out = out; a.gp = gp; a.up = up_; a.dg = (unsigned short *)dg; a.du = (unsigned short *)du;
#define SM_TN(IO) do{ if(rt == 1) SM_LAUNCH((k_gemm_tn_small<1, IO>), SM_TWAVES); else SM_LAUNCH((k_gemm_tn_small<2, IO>), SM_TWAVES); }while(0)
    if(out) SM_TN(SM_SCATTER); else if(gp) SM_TN(SM_SWIGLU_BWD); else SM_TN(SM_PLAIN);
#undef SM_TN
    QLMX_LAUNCH_CHECK("grouped gemm tn (few rows) launch");
    return qlmx_upload_done(slot, st);
}
