/* qlmx_gemm_small.hip -- forward (nn, fp16 matrix core) and input-gradient (tn, bf16 matrix core) grouped GEMMs of
 * experts with few rows: a short prompt, a small training batch.
 *
 * The tiled kernels (qlmx_gemm_nn_h.hip, qlmx_gemm_tn_body.h) give a workgroup a column strip of an expert and the
 * whole contraction, one LDS tile and one barrier per 32 or 64 of it. With a dozen rows a step is some 1000 cycles of
 * LDS, barrier and issue latency around four matrix products, and a call has too few strips to hide it: 36 us for the
 * down projection of 32 experts (2048 x 768, 12 rows each), whose 25 MB of weights take 5. Here nothing meets
 * a barrier on the way in, four wavefronts split the contraction and add up at the end:
 *
 * A wavefront owns 128 (64) columns and its share of the contraction. v_mfma_f32_16x16x32 wants eight consecutive k of one
 * column per lane (lane = column lane%16, k group lane/16). Weights of the forward lie along the columns: the lane
 * loads, for its eight k, the 4-byte word of eight neighbouring columns, and product j takes digit j of the eight words
 * -- the columns of a product are then eight apart, which only the store has to know. Activations come from
 * L2 straight as operands (16 bytes of a row per lane), all loads are plain register loads, one to four steps ahead. Weights
 * of the input gradient lie along k as they should; they and the activations go through LDS, each wavefront its own stages.
 *
 * Arithmetic as in the tiled kernels: forward weights fp16(s * digit * 2^8), activations converted exactly; the input
 * gradient multiplies exact digits and applies the scale to the fp32 sums of each group of k.
 *
 * Which calls come here (qlmx_small_rows): all whose problems have at most 32 rows, and those that would leave the tiled
 * kernels with few workgroups, each walking the whole contraction, or with tiles that are mostly padding: a prompt or a small batch whose router prefers
 * some experts has a few problems of a hundred rows beside many of five, each a tile of 128 there and of 32 here. The forward's rule looks at what the
 * forms of a call that are documented to agree bit for bit have in common -- with and without gather, SwiGLU, scatter -- so that they run the same
 * arithmetic in the same order. The lines count in CUs of the device; the numbers here are a device's with 256. us for the plain and the SwiGLU call, these : tiled --
 *   contractions over 512, tiles of 32 rows x 128 columns up to 256, one to a CU. 16 problems, largest 43 rows, 896 x 1152 8.3:13.6, 1152 x 896 14.6:19.0; 8 of 49,
 *     768 x 896 8.3:11.9, 896 x 768 12.2:13.8. Shorter ones stay with the tiled kernel (plain and SwiGLU call, 8 of 104,
 *     384 x 384 6.0:7.7 and 8.3:8.6; 8 of 21, 384 x 1152 6.0:8.3 and 8.6:9.0): the SwiGLU call gains little, and the plain call's gain is given up for layers of such widths, whose passes one by one
 *     and merged into one list then run the same kernel in more cases;
 *   tiles of 32 rows at most 1.5 times the 128-row tiles; from 257 to 352 of them 1.125 times (a second round that is nearly empty). Zipf shares: 1096 rows of 64, 896 x 512
 *     12.5:18.0, 512 x 896 22:24; 617 of 64, 1664 x 1920 41:60, 1920 x 1664 62:109; 362 of 32, 2304 x 896 18:31, 896 x 2304 32:50. On the other side 4832 of 64,
 *     1536 x 768 41:33, 768 x 1536 77:70; and with 330 tiles, 16 of 31 rows, 1024 x 1920 14:16 and 26:20;
 *   strips of 64 x 128 up to 256, where the contraction is not shorter than the width, or over 1024 with no problem of more than 64 rows: the plain
 *     call gains what the SwiGLU call (two rounds) loses. 1536 x 512, 64 of 40 18:22 and 29:28; 1408 x 2048, 16 of 40 17:20 and 32:28.
 *   up to 512, where the contraction is four times the width: the down projection of a wide layer, whose SwiGLU call has other
 *     sizes. 2304 x 512, 64 of 77 39:43 (a SwiGLU call 79:59, as at twice the width: 2048 x 768, 32 of 100 30:26 and 56:38).
 *   beyond, contractions over 1024 and not shorter than the width, of at most 64 rows to a problem and 48 on average, which the tiled kernel pads to 128: 2048 x 1664,
 *     64 of 41 59:63 and 102:116, 2048 x 768, 64 of 40 31:33 and 57:68; on the other side 64 of 64 56:63 and 121:103.
 * Over 160 calls of 1 to 64 problems of 5 to 400 rows on average, in even and in Zipf shares, 256 to 2048 in and out, a plain call takes 0.88 and a SwiGLU call 0.96 of what they took
 * when the rule counted strips of 64 rows only and problems of over 32 rows had tiles of 64 (mean of the ratios; 68 of the calls are as they were).
 * The lines look at a call's own sizes, so a layer whose passes run one by one may take the one path and its merged list the other: where both take the same, bits agree, and that is
 * promised for no size.
 * Input gradient, strips of 64 x 64: up to 512, 1024 where the contraction is twice the width.
 * us per call, tiled kernels of 256 x 128 (128 x 128) as these were written -> these: 32 experts, 768 x 2048, 12 rows each: gate|up + SwiGLU 34 -> 21, down 26 -> 12, its
 * input gradient + SwiGLU 21 -> 13, paired input gradient 56 -> 19; 8 experts of 125 (250) rows, 512 x 1536: down 24 -> 16
 * (35 -> 17), its input gradient 18 -> 13 (28 -> 22), paired input gradient 50 -> 14 (72 -> 16).
 * Shapes of the forward of at most 32 rows per problem, groups of 128 or 256 (sm_few_shape). What takes the time there is the CU's address unit
 * as much as vector issue: an instruction that loads a word per lane from four rows of weights takes it as long as one that loads two.
 *   wide: 256 columns to a strip, a lane's words of a row of weights in one load (RT * 64 registers of sums), two workgroups of four wavefronts to a CU; gate|up is eight wavefronts and one
 *     workgroup to a CU. Lines (sm_wide) from 2700 pairs of calls, K 256-2048, N 512-4096, 136-512 strips, and 3000 drawn ones; time of wide over narrow, with rows, K x N:
 *     one round of CUs, from 11/16 of it on (gate|up 10/16; with half of the CUs 1.3-1.7). Up to 16 rows K from 512: 0.66-0.97, at 384 and 256 0.97-1.13; gate|up from 384: 0.67-0.94, at 256 1.02-1.16.
 *       More rows, plain: K from 768 0.72-1.04, at 512 1.0-1.1 and at 256 1.07-1.18. More rows, gate|up: twice the registers against half the loads, and it takes a large matrix: from
 *       3 M weights 0.78-1.02 (20 rows, 1408 x 2304 0.98, 2048 x 1536 0.96, 1280 x 2560 0.94; below it 768 x 1536 1.08, 1408 x 768 1.04, 2048 x 768 1.02). Rows of weights a
 *       multiple of 1 KB apart, where narrow strips meet in the same memory channels, gain earlier: 768 x 2048 0.93-0.99, 896 x 4096 0.90, beside 768 x 2304 1.08, 768 x 2816 1.06, 896 x 3072
 *       0.99; 512 x 2048 1.05. They take the plain call from K = 512: 0.93, others 1.0-1.05. More rows and two strips for three narrow ones (N = 384): 1.07;
 *     beyond: plain, not where narrow strips, 2 to a CU, still come in one round (43 of 1408 1.40-1.44), K from 512: up to 16 rows 0.60-1.03, more rows from three narrow strips to a CU 0.64-0.97, with
 *       fewer a large matrix or rows 1 KB apart 0.85-1.04, others, and half strips, up to 1.14. Shorter ones with six rounds and more 0.85-0.98, fewer 0.9-1.3. Gate|up of up to 16 rows, K from 768,
 *       where the rounds are 25/32 full (a large matrix 22/32 or 23/32): 0.70-1.09; K from 384 two that are 27/32 full, or five: 0.84-1.0; others up to 1.25, at 256 1.1-1.5. Gate|up of more rows in
 *       one round only (1.0-1.5, with a round and a half and more 0.8-1.2).
 *   eight wavefronts along the contraction, where few strips walk a long one: K from 2048, up to 7/8 of a strip of 128 to a CU, above 16 rows K from 2 N. All forms of a call split alike. Eight over four,
 *     K 1024-4096, N 128-3840: plain 0.81-0.95. Gate|up, up to half a strip to a CU, on strips of 64 columns of each matrix, one to a CU: 0.59-0.88; on strips of 128, as with more of them, 0.97-1.03
 *     up to 16 rows and 1.04-1.10 above, where the rule takes that for the plain call's 0.75-0.90 (2048 x 768, 20 rows of 32: 14.3:16.7). Shorter contractions: plain 0.86-0.95 and 0.90-0.99 from K = 1024 on,
 *     gate|up on strips of 128 0.96-1.07 and 1.05-1.2. All eight put their sums into LDS at once; four after four took gate|up 2-4 % longer. One step of a wavefront is on its way in both: two are slower (18.3 -> 19.6
 *     for gate|up of 32, 768 x 2048).
 * What bounds them now: a wavefront's chain -- the round trip in front of its loop, the steps one behind the other, the sum over
 * the wavefronts behind it: 7 us of a gate|up call of 18, whose 50 MB stream at 4 TB/s beside it. Without the conversions it took 10. Other ways to them: scales on the
 * activations, as two bf16 parts, and digits as denormal bf16 took half the vector instructions and no less time, the address unit being as busy; and they round otherwise than
 * the tiled kernel. Vector issue is at 15-29 % in the input gradient, the address units at 24-51 %, the matrix cores at 4-14 %.
 */
#include "qlmx_gemm_tn_small_body.h"
#include <algorithm>

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

#define SM_COLS 128                             /* of a forward strip */
#define SM_WSCALE 4096.0f                       /* 16 (digits come as digit/16) * 2^8, as NH_WSCALE */
#define SM_UNSCALE (1.0f / 256.0f)


static __device__ __align__(16) unsigned char sm_zero_row[32768];       /* what a dropped row of a gather reads */

/* a call's row tiles of 32, 64 and 128 */
struct SmRows { long long t32, t64, t128, rows, busy; int most; };
static SmRows sm_rows(const qlmx_gemm_prob *probs, int nprob){
    SmRows r = {0, 0, 0, 0, 0, 0};
    for(int i = 0; i < nprob; i++){
        const int m = probs[i].M;
        r.t32 += (m + 31) / 32; r.t64 += (m + 63) / 64; r.t128 += (m + 127) / 128;
        r.rows += m; r.busy += m > 0;
        if(m > r.most) r.most = m;
    }
    return r;
}
/* tiles of 32 rows on so many strips, against `high` taller ones: not many more of them, by a line that depends on whether they come in two rounds; see the head of this file */
static bool sm_low(long long t32, long long high, int strips){
    const long long tiles = t32 * strips, cu = qlmx_cu_count();
    return tiles > cu && 8 * tiles <= 11 * cu ? 8 * t32 <= 9 * high : 2 * t32 <= 3 * high;
}
/* see the head of this file */
bool qlmx_small_rows(const qlmx_gemm_prob *probs, int nprob, int mode, int K, int N, int nseg, int group){
    if(group < 64) return false;
    const SmRows r = sm_rows(probs, nprob);
    const int cu = qlmx_cu_count();
    if(r.most <= 32) return true;
    if(mode == GEMM_NN){
        const long long tiles = r.t64 * (N / SM_COLS);
        if((K > 512 && r.t32 * (N / SM_COLS) <= cu) || sm_low(r.t32, r.t128, N / SM_COLS)) return true;
        if(tiles <= cu) return K >= N || (r.most <= 64 && K > 1024);
        if(tiles <= 2 * cu && K >= 4 * N) return true;
        return K > 1024 && K >= N && r.most <= 64 && r.rows <= 48 * r.busy;
    }
    const long long tiles = r.t64 * (N / SM_TCOLS);
    return tiles <= 2 * cu || (tiles <= 4 * cu && (long long)K * nseg >= 2 * N);
}

__device__ __forceinline__ int sm_pk_f16(float lo, float hi){ f32x2 v = {lo, hi}; return __builtin_bit_cast(int, __builtin_convertvector(v, f16x2)); }
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

/* The sums of KW wavefronts from `first` on, of one 16-row tile, through LDS: acc holds a lane's sums of rows
 * (lane/16)*4 + e, columns (lane%16)*CL + j. */
template<int CL, int KW> __device__ __forceinline__ void sm_put(float *red, int first, const f32x4 (&acc)[CL]){
    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) - first, c = lane & 15, g = lane >> 4;
    __syncthreads();                                      /* the tile before has been read */
    if(wave >= 0 && wave < KW){
        float *w = red + wave * (16 * 16 * CL);
#pragma unroll
        for(int e = 0; e < 4; e++)
#pragma unroll
            for(int j = 0; j < CL; j += 4)
                *(f32x4 *)&w[(g * 4 + e) * (16 * CL) + c * CL + j] = (f32x4){acc[j][e], acc[j + 1][e], acc[j + 2][e], acc[j + 3][e]};
    }
    __syncthreads();
}
/* four columns of a row; of eight wavefronts, first k and k + 4 */
template<int CL, int KW> __device__ __forceinline__ f32x4 sm_get(const float *red, int row, int col){
    f32x4 sum;
#pragma unroll
    for(int k = 0; k < 4; k++){
        f32x4 v = *(const f32x4 *)&red[k * (16 * 16 * CL) + row * (16 * CL) + col];
        if(KW == 8) v += *(const f32x4 *)&red[(k + 4) * (16 * 16 * CL) + row * (16 * CL) + col];
        sum = k ? sum + v : v;
    }
    return sum * SM_UNSCALE;
}

/* ---- forward, and gate | up in one (the second matrix at wq, wg of Q): SM_BY_WAVE, four more wavefronts work on 128 columns
 * of up; SM_BY_LANE, the strip is 64 columns of gate (lanes 0-7 of each 16) and 64 of up (lanes 8-15). By wave a row of
 * weights is read in 64-byte pieces, which is what counts while the weights set the pace (32 experts of 12 rows, 768 x 2048:
 * 20.6 against 26.3 us); by lane a workgroup is half as large and twice as many fit where 64 rows need 216 registers (8
 * experts of 250 rows, 512 x 1536: 24.5 against 30.2). TWO: the halves of the strip have scales of their own. ---- */
enum { SM_ONE = 0, SM_BY_WAVE = 1, SM_BY_LANE = 2 };
template<int RT, int IO, int DUAL, bool TWO, int CL, int KW>
__device__ __forceinline__ void sm_nn_tile(const SmArgs &a, const DevProb &P, const DevProb &Q, int i0, int j0, float *red){
    /* gate|up on narrow strips of 16 rows, several steps ahead, has registers for the addresses and is 3 % faster with them */
    constexpr bool SCALAR = DUAL == SM_ONE || (DUAL == SM_BY_WAVE && !(CL == 8 && KW == 4 && RT == 1));
    constexpr int COLS = 16 * CL, PF = CL == 16 || KW == 8 ? 1 : RT == 1 ? (DUAL == SM_BY_WAVE ? 3 : 4) : RT == 2 ? (DUAL == SM_BY_WAVE ? 1 : 2) : 1;        /* steps on their way */
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
    const int steps = a.K / 32, ks = wave & (KW - 1), st0 = steps * ks / KW, st1 = steps * (ks + 1) / KW;
    const size_t gpr = (size_t)a.N >> a.gshift, rowb = (size_t)a.N >> 1;       /* scale groups and bytes per row of weights */
    const bool second = DUAL == SM_BY_WAVE ? wave >= KW : DUAL == SM_BY_LANE && c >= 8;
    /* where the strip's weights and scales start, the same in all lanes (by lane: in those of a half), and the lane's way from there */
    const signed char *pw = a.d + (((second ? Q.wq : P.wq) + j0) >> 1);
    const float *ps = a.s + (second ? Q.wg : P.wg) + (j0 >> a.gshift);
    const int cw = DUAL == SM_BY_LANE || (CL == 16 && j0 + 128 >= a.N) ? c & 7 : c;      /* past the last column: the strip's first half once more, not stored */
    const uint32_t vw = (uint32_t)((g * 8) * rowb) + cw * (CL / 2);
    const uint32_t vs = (uint32_t)((g * 8 + (c & 7)) * gpr) + (CL == 16 ? ((j0 + (cw & 8) * 16) >> a.gshift) - (j0 >> a.gshift) : TWO && DUAL != SM_BY_LANE ? c >> 3 : 0);
    const char *pa[RT];
    f32x4 acc[RT][CL];
#pragma unroll
    for(int r = 0; r < RT; r++)
#pragma unroll
        for(int j = 0; j < CL; j++) acc[r][j] = (f32x4)(0.0f);
    typedef uint32_t Word __attribute__((ext_vector_type(CL / 8)));
    Word w[PF][8]; float s[PF]; i32x4 x[PF][RT];
    auto load_w = [&](int set, int st){
        const int t = min(st, st1 - 1);                   /* past the end: the last step again, never used */
        const float *sc = ps + (size_t)t * 32 * gpr;
        const signed char *row = pw + (size_t)t * 32 * rowb;
        s[set] = sc[vs];
#pragma unroll
        for(int i = 0; i < 8; i++){
            if(SCALAR) asm("" : "+s"(row));               /* stays in scalar registers: seen through, every load adds 64 bits per lane */
            w[set][i] = *(const Word *)(row + vw);
            row += rowb;
        }
    };
    auto load_x = [&](int set, int st){
        const int t = min(st, st1 - 1);
#pragma unroll
        for(int r = 0; r < RT; r++) x[set][r] = *(const i32x4 *)(pa[r] + (size_t)t * 64);
    };
    auto load = [&](int set, int st){ load_w(set, st); load_x(set, st); };
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
        float sk[8]; QxNibs nb[8][CL / 8];
        sm_each<0, 8>([&](auto KC){
            constexpr int k = decltype(KC)::value;
            sk[k] = sm_bcast<k>(sv);
            if(TWO) sk[k] = sm_bcast_hi<k>(sk[k], sv);
#pragma unroll
            for(int h = 0; h < CL / 8; h++) nb[k][h] = qx_nibs(w[I][k][h]);
        });
        load(I, st + PF);
        /* two operands at a time: left alone, the compiler builds all eight first and runs out of registers */
#pragma unroll
        for(int j = 0; j < CL; j++){
            i32x4 b;
#pragma unroll
            for(int q = 0; q < 4; q++) b[q] = sm_pk_f16(sk[2 * q] * qx_nib16(nb[2 * q][j / 8], j & 7), sk[2 * q + 1] * qx_nib16(nb[2 * q + 1][j / 8], j & 7));
#pragma unroll
            for(int r = 0; r < RT; r++)
                acc[r][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[r], __builtin_bit_cast(f16x8, b), acc[r][j], 0, 0, 0);
            if(j & 1) __builtin_amdgcn_sched_barrier(0);
        }
    };
    if(st0 < st1){
        /* a gather's row indices are a round trip of their own: behind the first weights */
        if(SCALAR) sm_each<0, PF>([&](auto IC){ load_w(decltype(IC)::value, st0 + decltype(IC)::value); });
#pragma unroll
        for(int r = 0; r < RT; r++){
            const int row = min(i0 + r * 16 + c, P.M - 1);
            if(IO == SM_GATHER){
                const int tok = ((const int *)P.A)[row];
                pa[r] = tok >= 0 ? a.xsrc + (size_t)tok * a.K * 2 : (const char *)sm_zero_row;
            } else pa[r] = (const char *)P.A + (size_t)row * a.K * 2;
            pa[r] += g * 16;
        }
        sm_each<0, PF>([&](auto IC){ if(!SCALAR) load_w(decltype(IC)::value, st0 + decltype(IC)::value); load_x(decltype(IC)::value, st0 + decltype(IC)::value); });
        int st = st0;
        for(; st + PF <= st1; st += PF) sm_each<0, PF>([&](auto IC){ step(IC, st + decltype(IC)::value); });
        sm_each<0, PF - 1>([&](auto IC){ if(st + decltype(IC)::value < st1) step(IC, st + decltype(IC)::value); });
    }
    /* ---- totals ---- */
    auto swiglu = [&](int lr, int col, const f32x4 &y, const f32x4 &u){
        if(lr >= P.M || (CL == 16 && j0 + col >= a.N)) return;
        const size_t o = (size_t)lr * a.N + j0 + col;
        if(P.C){ *(f32x4 *)(P.C + o) = y; *(f32x4 *)(Q.C + o) = u; }
        ushort4 h;
        h.x = qx_f32_to_bf16(y[0] * qx_fsig_hw(y[0]) * u[0]); h.y = qx_f32_to_bf16(y[1] * qx_fsig_hw(y[1]) * u[1]);
        h.z = qx_f32_to_bf16(y[2] * qx_fsig_hw(y[2]) * u[2]); h.w = qx_f32_to_bf16(y[3] * qx_fsig_hw(y[3]) * u[3]);
        *(ushort4 *)((unsigned short *)Q.B + o) = h;
    };
    constexpr int THREADS = 64 * KW * (DUAL == SM_BY_WAVE ? 2 : 1), PER_ROW = COLS / 4, V = (16 * PER_ROW + THREADS - 1) / THREADS;
#pragma unroll
    for(int r = 0; r < RT; r++){
        const int i = i0 + r * 16;
        sm_put<CL, KW>(red, 0, acc[r]);
        if constexpr(DUAL == SM_BY_LANE){
            const int row = tid >> 4, col = (tid & 15) * 4;
            if(THREADS <= 256 || row < 16) swiglu(i + row, col, sm_get<CL, KW>(red, row, col), sm_get<CL, KW>(red, row, 64 + col));
        } else if constexpr(DUAL == SM_BY_WAVE){
            f32x4 y[V];
#pragma unroll
            for(int v = 0; v < V; v++){ const int at = (v * THREADS + tid) % (16 * PER_ROW); y[v] = sm_get<CL, KW>(red, at / PER_ROW, at % PER_ROW * 4); }
            sm_put<CL, KW>(red, KW, acc[r]);
#pragma unroll
            for(int v = 0; v < V; v++){
                const int at = v * THREADS + tid, row = at / PER_ROW, col = at % PER_ROW * 4;
                if(at < 16 * PER_ROW) swiglu(i + row, col, y[v], sm_get<CL, KW>(red, row, col));
            }
        } else {
#pragma unroll
            for(int v = 0; v < V; v++){
                const int at = v * THREADS + tid, row = at / PER_ROW, col = at % PER_ROW * 4, lr = i + row;
                const f32x4 y = sm_get<CL, KW>(red, row, col);
                if(lr >= P.M || (CL == 16 && j0 + col >= a.N)) continue;
                if constexpr(IO == SM_SCATTER){
                    const int tok = ((const int *)P.C)[lr];
                    if(tok >= 0){
                        qx_gfloat *t = (qx_gfloat *)(a.out + (size_t)tok * a.N + j0 + col);
                        const float gt = a.gate ? a.gate[tok] : 1.0f;
#pragma unroll
                        for(int q = 0; q < 4; q++) (void)__builtin_amdgcn_global_atomic_fadd_f32(t + q, a.gate ? gt * y[q] : y[q]);
                    }
                } else *(f32x4 *)(P.C + (size_t)lr * a.N + j0 + col) = y;
            }
        }
    }
}

template<int RT, int IO, int DUAL, int CL, int KW>
__global__ void __launch_bounds__(64 * KW * (DUAL == SM_BY_WAVE ? 2 : 1), CL == 16 ? 2 : RT == 1 || DUAL == SM_BY_WAVE ? 4 : 2) k_gemm_nn_small(SmArgs a){
    __shared__ __attribute__((aligned(16))) float red[KW * 16 * 16 * CL];
    const int t = qx_xcd_tile(blockIdx.x, gridDim.x);
    if(t >= a.ntiles) return;
    const int pi = qx_find_problem(a.pr, a.nprob, t);
    const DevProb P = a.pr[pi], Q = a.pr[DUAL ? pi + 1 : pi];
    const int lt = t - P.tile0, ti = lt / P.tiles_n, tj = lt - ti * P.tiles_n;
    const int i0 = ti * (RT * 16), j0 = tj * (DUAL == SM_BY_LANE ? 8 * CL : 16 * CL), left = P.M - i0;
    auto tile = [&](auto TW){
        constexpr bool TWO = decltype(TW)::value;
        if(RT == 4 && left > 32)      sm_nn_tile<RT, IO, DUAL, TWO, CL, KW>(a, P, Q, i0, j0, red);
        else if(RT >= 2 && left > 16) sm_nn_tile<RT >= 2 ? 2 : 1, IO, DUAL, TWO, CL, KW>(a, P, Q, i0, j0, red);
        else                          sm_nn_tile<1, IO, DUAL, TWO, CL, KW>(a, P, Q, i0, j0, red);
    };
    if constexpr(DUAL == SM_BY_LANE || CL == 16) tile(std::true_type());
    else if(a.gshift == 6) tile(std::true_type());
    else tile(std::false_type());
}

template<int RT, int IO>
__global__ void __launch_bounds__(64 * SM_WAVES, 2) k_gemm_tn_small(SmArgs a){
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    sm_tn_block<RT, IO>(a, blockIdx.x, gridDim.x, lds);
}

/* ---- launches ---- */
/* Shape of the forward of at most 32 rows per problem. Eight wavefronts along the contraction change the order of the sums, so that line looks at what the
 * forms of a call have in common; the width of a strip does not, and looks at the form too. See the head of this file. */
enum { SM_NARROW = 0, SM_WIDE = 1, SM_EIGHT = 2, SM_EIGHT_HALF = 3 };
static bool sm_wide(long long narrow, long long wide, int K, int N, bool dual, int rt){
    const int cu = qlmx_cu_count();
    const bool apart = N % 2048 == 0, large = (long long)K * N >= 3000000;
    if(16 * wide < (dual ? 10 : 11) * cu || (rt == 2 && 8 * wide > 5 * narrow)) return false;
    if(wide <= cu) return rt == 1 ? K >= (dual ? 384 : 512) : dual ? K >= 768 && (apart || large) : K >= (apart ? 512 : 768);
    if(dual){
        const long long rounds = (wide + cu - 1) / cu, full = 32 * wide / (rounds * cu);          /* in 32nds */
        if(rt == 2) return false;
        if(K < 768) return K >= 384 && (rounds == 2 ? full >= 27 : rounds >= 5);
        return full >= (!large ? 25 : rounds == 2 ? 22 : 23);
    }
    if(narrow <= 2 * cu) return false;
    if(rt == 2 && narrow < 3 * cu && (N % 256 != 0 || !(large || apart))) return false;
    return K >= 512 || wide >= 6 * cu;
}
static int sm_few_shape(const qlmx_gemm_prob *probs, int nprob, int K, int N, int group, bool dual, int rt){
    if(group < 128) return SM_NARROW;                     /* a wide strip has room for two scales in a row of weights */
    long long narrow = 0, wide = 0;
    for(int i = 0; i < nprob; i++) if(probs[i].M > 0){ narrow += N / SM_COLS; wide += (N + 2 * SM_COLS - 1) / (2 * SM_COLS); }
    if(8 * narrow <= 7 * qlmx_cu_count() && K >= 2048 && (rt == 1 || K >= 2 * N)) return dual && 2 * narrow <= qlmx_cu_count() ? SM_EIGHT_HALF : SM_EIGHT;
    return sm_wide(narrow, wide, K, N, dual, rt) ? SM_WIDE : SM_NARROW;
}
/* Height, in sixteens, of the row tiles of a call with more than 32 rows to a problem: 64 rows share the weights' conversion or loads, 32 are less padding and more
 * workgroups. The order of a sum is the same in both, so the forms of a call need not agree on it. us, 32 : 64 rows:
 *   forward: 32 where these are at most one to a CU, or beyond that not many more than the tiles of 64 (sm_low): 8 problems of 125, 1536 x 512, 11.9:15.1, 16 of 64, 2048 x 768
 *     16.5:20.8, 107 rows of 16, largest 41, 896 x 1920 8.4:10.9, 1040 of 64, largest 245, 1920 x 1152 33.5:46.3; on the other side 16, largest 555, 1920 x 896, 20.5:18.4, 64 of 31, 1024 x 384, 13.0:11.6;
 *   gate|up: also 64 where there are at most 128 of 32, whose strips would leave half the CUs idle (those of 64 rows are half as wide): 8 of 11, 896 x 256, 11.8:10.7, 32 of 9,
 *     1152 x 384, 13.8:12.8; but 16 of 23, 1792 x 1024, 22.7:28.9, and 1040 of 64, 1920 x 1152, 56:78;
 *   input gradient: 32 where at most one to a CU and the contraction is long enough for a workgroup's loop to be what takes the time: paired, 8 of 125, 1536 x 512, 11.6:14.5, of 64, 2048 x 768
 *     14:18.1; more than one to a CU 16 of 64, 1536 x 768 19.5:16.2, 32 of 64, 2048 x 1024 47:40; short, 8 of 64, 512 x 512, 7.5:6.5. */
static int sm_few_height(const SmRows &r){ return r.most > 16 ? 2 : 1; }
static int sm_nn_height(const SmRows &r, int strips, bool dual){
    if(r.most <= 32) return sm_few_height(r);
    const long long tiles = r.t32 * strips, cu = qlmx_cu_count();
    return tiles <= cu ? (dual && 2 * tiles <= cu ? 4 : 2) : sm_low(r.t32, r.t64, strips) ? 2 : 4;
}
static int sm_tn_height(const SmRows &r, long long contraction, int strips){
    if(r.most <= 32) return sm_few_height(r);
    return r.t32 * strips <= qlmx_cu_count() && contraction >= 1024 ? 2 : 4;
}
bool qlmx_pair_open(hipStream_t st);
bool qlmx_pair_waits(hipStream_t st);
int qlmx_pair_hold_tn_few(const SmArgs &a, int rt, int io, int slot, hipStream_t st, bool *held);
static SmArgs sm_args(const signed char *d, const float *s, int group, int K, int N, const ProbUpload &up){
    SmArgs a = {};
    a.pr = up.dev; a.nprob = up.nprob; a.ntiles = up.ntiles; a.d = d; a.s = s; a.K = K; a.N = N;
    while((1 << a.gshift) < group) a.gshift++;
    return a;
}
#define SM_LAUNCH(KERNEL, WAVES, LDS) hipLaunchKernelGGL(KERNEL, dim3((a.ntiles + 7) & ~7), dim3(64 * (WAVES)), LDS, st, a)

/* N % 128 == 0, K % 32 == 0, group a power of two >= 64; io, xsrc, out, gate as in qlmx_gemm_nn_h_launch */
int qlmx_gemm_nn_small_launch(const signed char *d, const float *s, int group, const qlmx_gemm_prob *probs, int nprob, int K, int N,
                              int io, const void *xsrc, float *out, const float *gate, hipStream_t st){
    const SmRows rows = sm_rows(probs, nprob);
    const int rt = sm_nn_height(rows, N / SM_COLS, false);
    ProbUpload up; int slot;
    const int shape = rows.most <= 32 ? sm_few_shape(probs, nprob, K, N, group, false, rt) : SM_NARROW;
    int rc = qlmx_upload_problems(probs, nprob, GEMM_NN, K, N, rt * 16, shape == SM_WIDE ? 2 * SM_COLS : SM_COLS, st, &up, &slot); if(rc) return rc;
    if(up.ntiles == 0) return QLMX_OK;
    SmArgs a = sm_args(d, s, group, K, N, up);
    a.xsrc = (const char *)xsrc; a.out = out; a.gate = gate;
#define SM_FEW(RT, IO) do{ if(shape == SM_WIDE) SM_LAUNCH((k_gemm_nn_small<RT, IO, SM_ONE, 16, 4>), 4, 0); \
                           else if(shape == SM_EIGHT) SM_LAUNCH((k_gemm_nn_small<RT, IO, SM_ONE, 8, 8>), 8, 0); else SM_LAUNCH((k_gemm_nn_small<RT, IO, SM_ONE, 8, 4>), 4, 0); }while(0)
#define SM_NN(IO) do{ if(rt == 1) SM_FEW(1, IO); else if(rt == 2) SM_FEW(2, IO); else SM_LAUNCH((k_gemm_nn_small<4, IO, SM_ONE, 8, 4>), 4, 0); }while(0)
    if(io == SM_GATHER) SM_NN(SM_GATHER); else if(io == SM_SCATTER) SM_NN(SM_SCATTER); else SM_NN(SM_PLAIN);
#undef SM_NN
#undef SM_FEW
    QLMX_LAUNCH_CHECK("grouped gemm nn (few rows) launch");
    return qlmx_upload_done(slot, st);
}
/* gate|up with the SwiGLU behind; N % 128 == 0 */
int qlmx_gemm_nn_small_swiglu_launch(const signed char *d, const float *s, int group, const qlmx_gemm_prob *gate, const qlmx_gemm_prob *up_, int nprob,
                                     int K, int N, const void *xsrc, hipStream_t st){
    const SmRows rows = sm_rows(gate, nprob);
    const int rt = sm_nn_height(rows, N / SM_COLS, true);
    ProbUpload up; int slot;
    const int shape = rows.most <= 32 ? sm_few_shape(gate, nprob, K, N, group, true, rt) : SM_NARROW;
    int rc = qlmx_upload_problem_pairs(gate, up_, nprob, GEMM_NN, K, N, rt * 16, rt == 4 || shape == SM_EIGHT_HALF ? SM_COLS / 2 : shape == SM_WIDE ? 2 * SM_COLS : SM_COLS, st, &up, &slot); if(rc) return rc;
    if(up.ntiles == 0) return QLMX_OK;
    SmArgs a = sm_args(d, s, group, K, N, up);
    a.xsrc = (const char *)xsrc;
#define SM_FEW(RT, IO) do{ if(shape == SM_WIDE) SM_LAUNCH((k_gemm_nn_small<RT, IO, SM_BY_WAVE, 16, 4>), 8, 0); \
                           else if(shape == SM_EIGHT_HALF) SM_LAUNCH((k_gemm_nn_small<RT, IO, SM_BY_LANE, 8, 8>), 8, 0); \
                           else if(shape == SM_EIGHT) SM_LAUNCH((k_gemm_nn_small<RT, IO, SM_BY_WAVE, 8, 8>), 16, 0); else SM_LAUNCH((k_gemm_nn_small<RT, IO, SM_BY_WAVE, 8, 4>), 8, 0); }while(0)
#define SM_DUAL(IO) do{ if(rt == 1) SM_FEW(1, IO); else if(rt == 2) SM_FEW(2, IO); else SM_LAUNCH((k_gemm_nn_small<4, IO, SM_BY_LANE, 8, 4>), 4, 0); }while(0)
    if(xsrc) SM_DUAL(SM_GATHER); else SM_DUAL(SM_PLAIN);
#undef SM_DUAL
#undef SM_FEW
    QLMX_LAUNCH_CHECK("grouped gemm nn + swiglu (few rows) launch");
    return qlmx_upload_done(slot, st);
}
/* the launch itself (also what issues a launch that was held for a pair and found no partner) */
int qlmx_gemm_tn_small_issue(const SmArgs &a, int rt, int io, int slot, hipStream_t st){
#define SM_TN1(RT, IO) do{ \
        static bool attr_set = false; \
        if(!attr_set){ QLMX_HIP(hipFuncSetAttribute((const void *)k_gemm_tn_small<RT, IO>, hipFuncAttributeMaxDynamicSharedMemorySize, SM_TLDS(RT)), "tn (few rows) LDS size"); attr_set = true; } \
        SM_LAUNCH((k_gemm_tn_small<RT, IO>), SM_WAVES, SM_TLDS(RT)); }while(0)
#define SM_TN(IO) do{ if(rt == 1) SM_TN1(1, IO); else if(rt == 2) SM_TN1(2, IO); else SM_TN1(4, IO); }while(0)
    if(io == SM_SCATTER) SM_TN(SM_SCATTER); else if(io == SM_SWIGLU_BWD) SM_TN(SM_SWIGLU_BWD); else SM_TN(SM_PLAIN);
#undef SM_TN
#undef SM_TN1
    QLMX_LAUNCH_CHECK("grouped gemm tn (few rows) launch");
    return qlmx_upload_done(slot, st);
}
/* N % 128 == 0, K % 64 == 0, group a power of two >= 64; the rest as in qlmx_gemm_tn_lds_launch */
int qlmx_gemm_tn_small_launch(const signed char *d, const float *s, int group, const qlmx_gemm_prob *probs, const qlmx_gemm_prob *second, int nprob,
                              int K, int N, float *out, const float *gp, const float *up_, void *dg, void *du, hipStream_t st){
    /* In one grid with a weight gradient the tiles are of 32 rows, two workgroups to a CU as that kernel's: 0.58-0.99 of the two launches, this one on its own height (60 drawn pairs).
     * On its own where it would be 64 rows, that takes 0.63-1.25, so it is held only for a weight gradient that is there already: one that comes later finds it launched. */
    const int alone = sm_tn_height(sm_rows(probs, nprob), (long long)K * (second ? 2 : 1), N / SM_TCOLS);
    bool pair = alone <= 2 ? qlmx_pair_open(st) : qlmx_pair_waits(st);
    if(!pair){ const int rc = qlmx_pair_flush(); if(rc) return rc; }
    int rt = pair ? std::min(alone, 2) : alone;
    ProbUpload up; int slot;
    auto upload = [&]{
        return second ? qlmx_upload_problem_pairs(probs, second, nprob, GEMM_TN, K, N, rt * 16, SM_TCOLS, st, &up, &slot)
                      : qlmx_upload_problems(probs, nprob, GEMM_TN, K, N, rt * 16, SM_TCOLS, st, &up, &slot);
    };
    int rc = upload(); if(rc) return rc;
    if(rt != alone && !qlmx_pair_waits(st)){               /* the slot opened a segment of the ring, which issues what is held */
        pair = false; rt = alone;
        rc = upload(); if(rc) return rc;
    }
    if(up.ntiles == 0) return QLMX_OK;
    SmArgs a = sm_args(d, s, group, K, N, up);
    a.out = out; a.gp = gp; a.up = up_; a.dg = (unsigned short *)dg; a.du = (unsigned short *)du;
    const int io = out ? SM_SCATTER : gp ? SM_SWIGLU_BWD : SM_PLAIN;
    if(pair){
        bool held;
        rc = qlmx_pair_hold_tn_few(a, rt, io, slot, st, &held); if(rc) return rc;
        if(held) return QLMX_OK;
    }
    return qlmx_gemm_tn_small_issue(a, rt, io, slot, st);
}
