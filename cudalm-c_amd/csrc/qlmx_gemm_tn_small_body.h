/* qlmx_gemm_tn_small_body.h -- the input gradient (tn) of experts with few rows, shared by its own kernel (qlmx_gemm_small.hip, whose head says
 * which calls come here) and by the grid that holds a weight gradient too (qlmx_gemm_bwd.hip). */
#ifndef QLMX_GEMM_TN_SMALL_BODY_H
#define QLMX_GEMM_TN_SMALL_BODY_H
#include "qlmx_gemm.h"
#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float  f32x2 __attribute__((ext_vector_type(2)));
typedef float  f32x4 __attribute__((ext_vector_type(4)));
typedef int    i32x2 __attribute__((ext_vector_type(2)));
typedef int    i32x4 __attribute__((ext_vector_type(4)));

#define SM_TCOLS 64                             /* of an input-gradient strip */
#define SM_WAVES 4                              /* along the contraction (the forward of few rows: eight where sm_few_shape says so) */

enum { SM_PLAIN = 0, SM_GATHER = 1, SM_SCATTER = 2, SM_SWIGLU_BWD = 3 };
struct SmArgs { const DevProb *pr; int nprob, ntiles; const signed char *d; const float *s; int gshift; int K, N;
                const char *xsrc; float *out; const float *gate;
                const float *gp, *up; unsigned short *dg, *du; };

__device__ __forceinline__ int sm_pk_bf16(float lo, float hi){ f32x2 v = {lo, hi}; return __builtin_bit_cast(int, __builtin_convertvector(v, bf16x2)); }
template<int I, int N, class F> __device__ __forceinline__ void sm_each(const F &f){ if constexpr(I < N){ f(std::integral_constant<int, I>()); sm_each<I + 1, N>(f); } }

/* ---- input gradient: 64 columns per workgroup; nseg operand pairs (a continued problem's second pair comes from the
 * table entry behind it). A wavefront's step is 64 of the contraction: 16 RT rows of activations (128 bytes each) and 64
 * rows of weights (32 bytes each) go straight into stages of LDS of its own, so there is no barrier in the loop, only the
 * wavefront's own wait counts. Loaded as operands (lane = row lane%16) instead, sixteen bytes each with neighbouring lanes in
 * different rows, a load takes 66 cycles of a CU where four lanes per row of 64 bytes take 17.5, and that set the pace. Piece q of row r of a stage
 * lies at q ^ ((r >> 1) & 7): the sixteen rows of an operand read hit sixteen different units.
 * LDS accesses are inline assembly: the compiler would wait for every load to LDS in front of them. ---- */
#define SM_TSTAGE(RT) (2048 * ((RT) + 1) + 256)      /* activations, weights, scales */
#define SM_TSTAGES(RT) ((RT) == 1 ? 4 : 3)            /* 70, 77, 126 KB: two workgroups per CU, for 64 rows one */
#define SM_TLDS(RT) (SM_WAVES * SM_TSTAGES(RT) * SM_TSTAGE(RT))
typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void glb_void;
template<int OFF> __device__ __forceinline__ i32x4 sm_rd128(uint32_t addr){
    i32x4 v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
    return v;
}
template<int OFF> __device__ __forceinline__ i32x2 sm_rd64(uint32_t addr){
    i32x2 v;
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
    return v;
}
template<int OFF> __device__ __forceinline__ int sm_rd32(uint32_t addr){
    int v;
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
    return v;
}
template<int RT, int IO>
__device__ __forceinline__ void sm_tn_tile(const SmArgs &a, const DevProb &P, const DevProb &Q, int nseg, int i0, int j0, unsigned char *lds){
    constexpr int ST = SM_TSTAGES(RT), STAGE = SM_TSTAGE(RT), LOADS = 2 * RT + 3;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
    /* the wavefronts take pairs of steps in turn: 128 of the contraction, which share a scale group where it is that long */
    const int steps1 = a.K / 64, steps = steps1 * nseg, pairs = (steps + 1) / 2, mypairs = (pairs - wave + SM_WAVES - 1) / SM_WAVES;
    const int mine = 2 * mypairs - ((steps & 1) && mypairs > 0 && (mypairs - 1) * SM_WAVES + wave == pairs - 1 ? 1 : 0);
    const int ngroups = a.K >> a.gshift;
    f32x4 acc[RT][4];
#pragma unroll
    for(int r = 0; r < RT; r++)
#pragma unroll
        for(int j = 0; j < 4; j++) acc[r][j] = (f32x4)(0.0f);
    /* what this lane loads: piece lane%8 of rows n*8 + lane/8 of the activations, half lane%2 of rows n*32 + lane/2 of the
     * weights, the scale of column `lane` */
    size_t ra[2 * RT];
#pragma unroll
    for(int n = 0; n < 2 * RT; n++){
        const int r = n * 8 + (lane >> 3);
        ra[n] = (size_t)min(i0 + r, P.M - 1) * a.K * 2 + ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    }
    const size_t rw = (((size_t)(j0 + (lane >> 1)) * a.K) >> 1) + (lane & 1) * 16, rs = (size_t)(j0 + lane) * ngroups;
    unsigned char *base = lds + wave * (ST * STAGE);
    auto load = [&](auto SC, int n){
        constexpr int S = decltype(SC)::value;
        const int m = min(n, mine - 1), t = ((m >> 1) * SM_WAVES + wave) * 2 + (m & 1);   /* past the end: the last step again, never used */
        const bool two = t >= steps1;
        const int u = two ? t - steps1 : t;
        const char *A = (const char *)(two ? Q.A : P.A) + (size_t)u * 128;
        const signed char *W = a.d + ((two ? Q.wq : P.wq) >> 1) + (size_t)u * 32 + rw;
#pragma unroll
        for(int k = 0; k < 2 * RT; k++) __builtin_amdgcn_global_load_lds((glb_void *)(A + ra[k]), (lds_void *)(base + S * STAGE + k * 1024), 16, 0, 0);
#pragma unroll
        for(int k = 0; k < 2; k++) __builtin_amdgcn_global_load_lds((glb_void *)(W + (size_t)(k * 16) * a.K), (lds_void *)(base + S * STAGE + RT * 2048 + k * 1024), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((glb_void *)(a.s + (two ? Q.wg : P.wg) + rs + ((u * 64) >> a.gshift)), (lds_void *)(base + S * STAGE + RT * 2048 + 2048), 4, 0, 0);
        asm volatile("" ::: "memory");                    /* the stages' loads stay in order: the waits count them */
    };
    const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_void *)base;
    uint32_t rdx[2];                                      /* activations of product i, row lane%16 of the first 16 */
#pragma unroll
    for(int i = 0; i < 2; i++) rdx[i] = lds_base + c * 128 + (((2 * g + i) ^ (c >> 1)) << 4);
    const uint32_t rdw = lds_base + c * 32 + g * 8, rds = lds_base + c * 4;
    auto step = [&](auto SC, int n){
        constexpr int S = decltype(SC)::value;
        asm volatile("s_waitcnt vmcnt(%0)" :: "n"((ST - 1) * LOADS) : "memory");
        i32x4 x[RT][2]; i32x2 w[4]; int sc[4];
        sm_each<0, 4>([&](auto JC){ constexpr int j = decltype(JC)::value; w[j] = sm_rd64<S * STAGE + RT * 2048 + j * 512>(rdw); });
        sm_each<0, RT>([&](auto RC){
            constexpr int r = decltype(RC)::value;
            x[r][0] = sm_rd128<S * STAGE + r * 2048>(rdx[0]); x[r][1] = sm_rd128<S * STAGE + r * 2048>(rdx[1]);
        });
        sm_each<0, 4>([&](auto JC){ constexpr int j = decltype(JC)::value; sc[j] = sm_rd32<S * STAGE + RT * 2048 + 2048 + j * 64>(rds); });
        /* everything is in registers before the stage is loaded again */
#pragma unroll
        for(int r = 0; r < RT; r++) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(x[r][0]), "+v"(x[r][1]) :: "memory");
        asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]), "+v"(sc[0]), "+v"(sc[1]), "+v"(sc[2]), "+v"(sc[3]));
        load(SC, n + ST);
#pragma unroll
        for(int j = 0; j < 4; j++){
            f32x4 p[RT];
#pragma unroll
            for(int r = 0; r < RT; r++) p[r] = (f32x4)(0.0f);
#pragma unroll
            for(int i = 0; i < 2; i++){
                const QxNibs nb = qx_nibs((uint32_t)w[j][i]);
                i32x4 b;
#pragma unroll
                for(int q = 0; q < 4; q++) b[q] = sm_pk_bf16(qx_nib16(nb, 2 * q), qx_nib16(nb, 2 * q + 1));
#pragma unroll
                for(int r = 0; r < RT; r++)
                    p[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x[r][i]), __builtin_bit_cast(bf16x8, b), p[r], 0, 0, 0);
            }
            const float f = __int_as_float(sc[j]) * 16.0f;
#pragma unroll
            for(int r = 0; r < RT; r++)
#pragma unroll
                for(int e = 0; e < 4; e++) acc[r][j][e] = fmaf(f, p[r][e], acc[r][j][e]);
        }
    };
    if(mine > 0){
        sm_each<0, ST>([&](auto IC){ load(IC, decltype(IC)::value); });
        int n = 0;
        for(; n + ST <= mine; n += ST) sm_each<0, ST>([&](auto IC){ step(IC, n + decltype(IC)::value); });
        sm_each<0, ST - 1>([&](auto IC){ if(n + decltype(IC)::value < mine) step(IC, n + decltype(IC)::value); });
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);                   /* vmcnt(0): no load may land in a stage any more */
    /* ---- totals: [row tile][wavefront][16 rows][64 columns]; the thread holds row tid/16, four columns ---- */
    float *red = (float *)lds;
    __syncthreads();
#pragma unroll
    for(int r = 0; r < RT; r++)
#pragma unroll
        for(int e = 0; e < 4; e++)
#pragma unroll
            for(int j = 0; j < 4; j++) red[((r * SM_WAVES + wave) * 16 + g * 4 + e) * SM_TCOLS + j * 16 + c] = acc[r][j][e];
    __syncthreads();
    const int row = tid >> 4, col = (tid & 15) * 4;
#pragma unroll
    for(int r = 0; r < RT; r++){
        const int lr = i0 + r * 16 + row;
        if(lr >= P.M) continue;
        f32x4 y = *(const f32x4 *)&red[(r * SM_WAVES * 16 + row) * SM_TCOLS + col];
#pragma unroll
        for(int k = 1; k < SM_WAVES; k++) y += *(const f32x4 *)&red[((r * SM_WAVES + k) * 16 + row) * SM_TCOLS + col];
        if constexpr(IO == SM_SCATTER){
            const int tok = ((const int *)P.C)[lr];
            if(tok >= 0){
                qx_gfloat *t = (qx_gfloat *)(a.out + (size_t)tok * a.N + j0 + col);
#pragma unroll
                for(int q = 0; q < 4; q++) (void)__builtin_amdgcn_global_atomic_fadd_f32(t + q, y[q]);
            }
        } else if constexpr(IO == SM_SWIGLU_BWD){
            const size_t o = (size_t)(P.C - a.gp) + (size_t)lr * a.N + j0 + col;      /* even: pairs of bf16 are 4-byte aligned */
            float dg[4], du[4];
#pragma unroll
            for(int q = 0; q < 4; q++) qx_swiglu_bwd1<true>(a.gp[o + q], a.up[o + q], y[q], dg[q], du[q]);
#pragma unroll
            for(int q = 0; q < 4; q += 2){
                *(uint32_t *)(a.dg + o + q) = (uint32_t)qx_f32_to_bf16(dg[q]) | ((uint32_t)qx_f32_to_bf16(dg[q + 1]) << 16);
                *(uint32_t *)(a.du + o + q) = (uint32_t)qx_f32_to_bf16(du[q]) | ((uint32_t)qx_f32_to_bf16(du[q + 1]) << 16);
            }
        } else {
            f32x4 *o = (f32x4 *)(P.C + (size_t)lr * a.N + j0 + col);
            if(P.beta != 0.0f) y = *o + y;
            *o = y;
        }
    }
}

/* the tile of workgroup b of `grid`, a multiple of 8 */
template<int RT, int IO> __device__ __forceinline__ void sm_tn_block(const SmArgs &a, int b, int grid, unsigned char *lds){
    const int t = qx_xcd_tile(b, grid);
    if(t >= a.ntiles) return;
    const int pi = qx_find_problem(a.pr, a.nprob, t);
    const DevProb P = a.pr[pi];
    const DevProb Q = a.pr[P.chunk ? pi + 1 : pi];
    const int lt = t - P.tile0, ti = lt / P.tiles_n, tj = lt - ti * P.tiles_n;
    const int i0 = ti * (RT * 16), j0 = tj * SM_TCOLS, left = P.M - i0, nseg = P.chunk ? 2 : 1;
    if(RT == 4 && left > 32)      sm_tn_tile<RT, IO>(a, P, Q, nseg, i0, j0, lds);
    else if(RT >= 2 && left > 16) sm_tn_tile<RT >= 2 ? 2 : 1, IO>(a, P, Q, nseg, i0, j0, lds);
    else                          sm_tn_tile<1, IO>(a, P, Q, nseg, i0, j0, lds);
}

#endif
