/* qlmx_gemm_f32s.hip -- grouped expert GEMMs on fp32 activations with fp32 results, on the bf16 matrix core.
 *
 * The fp32 matrix core multiplies at a sixteenth of the bf16 rate. An fp32 value is exactly the sum of three bf16 values
 * (hi = bf16(x), mid = bf16(x - hi), lo = x - hi - mid: 8 significant bits each, every difference exact), a digit is one,
 * and products of bf16 values are exact in fp32. So:
 *
 *   nn: out[m,n] = sum_k fl(A[m,k] * s[k, group of n]) * digit[k,n]: a tile's columns lie in one scale group, so the scale is
 *       a factor of the activation; one rounding of the product as in fl(s * digit) before, then three exact products.
 *   tn: out[m,n] = sum over groups of s[n, group] * sum_{k in group} A[m,k] * digit[n,k]: three exact products.
 *   nt: out[k,n] (+)= sum_m A[m,k] * B[m,n]: of the nine products of the parts six; mid*lo, lo*mid and lo*lo, together below
 *       2^-24 of a product (2^-27.5 root mean square), are left out of sums of 32 rows, where 1 % of the error comes from that.
 *       In the last rows of a problem, which may be one or two and all it has, only lo*lo is, below 2^-32.
 *
 * Every matrix product rounds what it adds to, so the parts of a step (64 of the contraction, 32 rows in nt) are added up by themselves, smallest
 * first, and the total takes one rounding a step. With the total in the matrix core it took six per 32 rows (nt) or three per 16 (nn), and long
 * sums of few outputs, which the fp32 core spreads over sixteen wavefronts, came out further off than there. Error against 64 bits, so / with
 * the total in the matrix core / fp32 core: nt 32 rows 3.8e-8 / 3.9e-8 / 7.9e-8, 1024 rows 512 x 512 8.6e-8 / 2.3e-7 / 2.9e-7, 4096 rows 256 x 512 1.2e-7 /
 * 4.9e-7 / 3.0e-7, 16384 rows 256 x 256 2.2e-7 / 1.1e-6 / 5.8e-7; nn one row, 8192 x 512, 1.6e-7 / 4.4e-7 / 3.4e-7; 1024 x 1024 1.0e-7 /
 * 1.6e-7 / 1.7e-7; tn, which always did, 1.4e-7 / 4.0e-7 (core) and 9.6e-8 / 1.8e-7.
 *
 * What bounds it: with three (six) bf16 products for an fp32 one the matrix core needs a fifth (two fifths) of the time, and vector issue sets the
 * pace: splitting (4 instructions a value, 5 in tn and nt), converting digits (1.6), addresses; one wavefront's splitting and products hardly overlap.
 * 1024 rows, 512 x 1536: 10-12 us a forward or input gradient, 16-17 a weight gradient (22-29 all six before; 20 with four wavefronts to a
 * tile), of which about 4 are the launch and the ends of a workgroup.
 *
 * Small values: the last bit of lo is the value's own, 23 places below its first, and bf16 ends where fp32 ends, at 2^-133. So what is
 * split has been multiplied by a power of two, F3_UP, that makes the parts of every fp32 value normal numbers; the sums are divided by it at the
 * end. In nn that rides in the scale, in tn and nt it is an instruction per value.
 * Large ones: infinities have no parts, and what has been multiplied can overflow where fp32 sums do not. Either leaves sums that are not
 * finite: a workgroup that has one, or a NaN, drops its sums and runs the plain fp32 matrix core loop (f3_plain). Looking at the sums
 * and not for the largest of what is split pays for most of the multiplication: six launches of 1024 rows, 512 x 1536 and back, 83.5 us
 * when small values beside large ones kept as little as eight bits, 85 so, 88.5 with both (all three with the total in the matrix core).
 */
#include "qlmx_gemm.h"
#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float  f32x4  __attribute__((ext_vector_type(4)));
/* operands named in the problem table: known to be global memory (a load from an address of unknown kind counts as an LDS access too,
 * and every wait for LDS then waits for it) */
typedef const __attribute__((address_space(1))) f32x4 gf32x4;
typedef int    i32x2  __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(1))) float gfloat;
typedef const __attribute__((address_space(1))) char gchar;
typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void glb_void;

/* Powers of two on what is split and back: the smallest fp32 value, 2^-149, has its parts at 2^-121 (2^-125 in nt, where both operands are
 * multiplied), and a sixteenth of that (digits come as digit / 16) is still a normal number. */
#define F3_UP(MODE)   ((MODE) == GEMM_NT ? 0x1p24f : 0x1p28f)
#define F3_DOWN(MODE) ((MODE) == GEMM_NT ? 0x1p-48f : (MODE) == GEMM_NN ? 0x1p-24f : 0x1p-28f)     /* nn: with digit / 16 */

struct F3Args { const DevProb *pr; int nprob, ntiles; const signed char *d; const float *s; int group, gshift; int K, N; };

/* eight values into their three parts */
__device__ __forceinline__ void f3_split(const QxMinus &k, const float (&f)[8], uint4 (&p)[3]){
    uint32_t w[3][4];
#pragma unroll
    for(int i = 0; i < 4; i++){
        const float a = f[2 * i], b = f[2 * i + 1];
        w[0][i] = qx_pk_bf16(a, b);
        const float a1 = qx_dot2(a, w[0][i], k.lo), b1 = qx_dot2(b, w[0][i], k.hi);
        w[1][i] = qx_pk_bf16(a1, b1);
        w[2][i] = qx_pk_bf16(qx_dot2(a1, w[1][i], k.lo), qx_dot2(b1, w[1][i], k.hi));
    }
#pragma unroll
    for(int q = 0; q < 3; q++) p[q] = make_uint4(w[q][0], w[q][1], w[q][2], w[q][3]);
}
/* eight digits as bf16(digit / 16) */
__device__ __forceinline__ uint4 f3_digits(uint32_t w){
    const QxNibs n = qx_nibs(w);
    uint32_t r[4];
#pragma unroll
    for(int i = 0; i < 4; i++)                            /* the upper halves of both: exact */
        r[i] = __builtin_amdgcn_perm(__float_as_uint(qx_nib16(n, 2 * i + 1)), __float_as_uint(qx_nib16(n, 2 * i)), 0x07060302u);
    return make_uint4(r[0], r[1], r[2], r[3]);
}
/* The tile once more on the fp32 matrix core, operands straight from memory, s * digit as one product: what the parts do not hold. */
template<int MODE, int BM, int BN, int NWAVE>
__device__ __forceinline__ void f3_plain(const F3Args &a, const DevProb &P, int i0, int j0){
    const int lane = threadIdx.x & 63, fr = lane & 31, hf = lane >> 5;
    const int rows = MODE == GEMM_NT ? a.K : P.M, depth = MODE == GEMM_NT ? P.M : a.K;
    gfloat *A = (gfloat *)P.A, *B = (gfloat *)P.B;
    for(int t = threadIdx.x >> 6; t < (BM / 32) * (BN / 32); t += NWAVE){
        const int i = i0 + t / (BN / 32) * 32, j = j0 + t % (BN / 32) * 32;
        const int r = min(i + fr, rows - 1), c = min(j + fr, a.N - 1);
        qx_f32x16 acc = (qx_f32x16)(0.0f);
        for(int p = 0; p < depth; p += 2){
            const int k = min(p + hf, depth - 1);
            float x = MODE == GEMM_NT ? A[(size_t)k * a.K + r] : A[(size_t)r * a.K + k], y;
            if constexpr(MODE == GEMM_NT) y = B[(size_t)k * a.N + c];
            else {
                const size_t e = MODE == GEMM_NN ? (size_t)k * a.N + c : (size_t)c * a.K + k;
                const uint32_t b = (unsigned char)a.d[(P.wq + e) >> 1];
                y = a.s[P.wg + (e >> a.gshift)] * (float)qx_nib(b, (int)(e & 1));
            }
            if(p + hf >= depth) x = y = 0.0f;
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x, y, acc, 0, 0, 0);
        }
#pragma unroll
        for(int e = 0; e < 16; e++){
            const int ro = i + (e >> 2) * 8 + (e & 3) + hf * 4;
            if(ro < rows && j + fr < a.N){ qx_gfloat *o = (qx_gfloat *)P.C + (size_t)ro * a.N + j + fr; *o = P.beta != 0.0f ? *o + acc[e] : acc[e]; }
        }
    }
}

/* zero if the four sums are finite, else NaN */
__device__ __forceinline__ float f3_odd(f32x4 v){ return fmaf(v[0], 0.0f, v[1] * 0.0f) + fmaf(v[2], 0.0f, v[3] * 0.0f); }
/* whether a thread of the workgroup's NWAVE wavefronts has an odd sum; `flag`: LDS words that nothing else is in */
template<int NWAVE> __device__ __forceinline__ bool f3_any(float odd, int *flag){
    const bool mine = __ballot(odd != 0.0f) != 0;         /* NaN is not equal to zero */
    if(NWAVE == 1) return mine;
    if((threadIdx.x & 63) == 0) flag[threadIdx.x >> 6] = mine;
    __syncthreads();
    int any = 0;
#pragma unroll
    for(int w = 0; w < NWAVE; w++) any |= flag[w];
    return any != 0;
}

/* ---- wavefronts on their own: each computes a tile of outputs over its share of the contraction from operands that it brings in itself,
 * without a barrier before the sums are added up in LDS, in the order of the wavefronts ---- */
template<int I, int N, class F> __device__ __forceinline__ void f3_each(const F &f){ if constexpr(I < N){ f(std::integral_constant<int, I>()); f3_each<I + 1, N>(f); } }
/* nt: 64 x 64 outputs per wavefront, KS of them along the contraction. Lane l loads sixteen bytes, columns 4 (l % 16) .. + 3, of rows 8 (l / 16)
 * .. + 7 of both operands: the operand of v_mfma_f32_16x16x32 for column q of each four is then in the lane that needs it, the columns of a
 * product are four apart, which only the store has to know, and a request moves four rows of 256 bytes (with four bytes per lane a step of the
 * loop waited for the issue of its requests). FEW: every problem has fewer than 32 rows. The loads of the next step go out as this step's values have been split. */
template<int KS, bool FEW>
__global__ void __launch_bounds__(64 * KS, KS == 8 ? 1 : 2) k_gemm_f32s_nt(F3Args a){
    constexpr int B = 64, LD = B + 4;
    constexpr float up = F3_UP(GEMM_NT), down = F3_DOWN(GEMM_NT);
    extern __shared__ __attribute__((aligned(16))) unsigned char f3_lds[];
    const int tile = qx_xcd_tile(blockIdx.x, gridDim.x);
    if(tile >= a.ntiles) return;
    const DevProb P = a.pr[qx_find_problem(a.pr, a.nprob, tile)];
    const int lt = tile - P.tile0, ti = lt / P.tiles_n, tj = lt - ti * P.tiles_n;
    const int i0 = ti * B, j0 = tj * B, M = P.M;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, g = lane >> 4;
    const QxMinus minus = qx_minus();
    /* the lane's byte offset in a step's rows, and with its columns alone */
    const uint32_t ca = (uint32_t)min(i0 + c * 4, a.K - 4) * 4u, cb = (uint32_t)min(j0 + c * 4, a.N - 4) * 4u;
    const uint32_t oa = (uint32_t)(g * 8 * a.K) * 4u + ca, ob = (uint32_t)(g * 8 * a.N) * 4u + cb;
    const int whole = M / 32, mine = (whole - wave + KS - 1) / KS;               /* steps of 32 rows; of this wavefront */
    f32x4 va[8], vb[8];
    auto load = [&](f32x4 (&v)[8], gchar *base, int ld, uint32_t off, int n){
        base += (size_t)(min(n, mine - 1) * KS + wave) * 128 * ld;                /* past the end: the last step again, never used */
#pragma unroll
        for(int r = 0; r < 8; r++) v[r] = *(gf32x4 *)(base + (size_t)r * 4 * ld + off);
        asm volatile("" ::: "memory");                    /* they are requested here, not where they are needed */
    };
    f32x4 acc[4][4];
#pragma unroll
    for(int i = 0; i < 4; i++)
#pragma unroll
        for(int j = 0; j < 4; j++) acc[i][j] = (f32x4)(0.0f);
    auto multiply = [&](auto NEXT, int n){
        constexpr bool next = decltype(NEXT)::value;
        uint4 x[4][3];
#pragma unroll
        for(int i = 0; i < 4; i++){
            const float f[8] = {up * va[0][i], up * va[1][i], up * va[2][i], up * va[3][i], up * va[4][i], up * va[5][i], up * va[6][i], up * va[7][i]};
            f3_split(minus, f, x[i]);
        }
        if(next) load(va, (gchar *)P.A, a.K, oa, n + 1);
#pragma unroll
        for(int j = 0; j < 4; j++){
            const float f[8] = {up * vb[0][j], up * vb[1][j], up * vb[2][j], up * vb[3][j], up * vb[4][j], up * vb[5][j], up * vb[6][j], up * vb[7][j]};
            uint4 y[3];
            f3_split(minus, f, y);
            if(next && j == 3) load(vb, (gchar *)P.B, a.N, ob, n + 1);
            auto product = [&](int i, int p, int q, f32x4 v){
                return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x[i][p]), __builtin_bit_cast(bf16x8, y[q]), v, 0, 0, 0);
            };
            constexpr int order[8][2] = {{2, 1}, {1, 2}, {2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
            if constexpr(next){                           /* a whole step: one rounding of the total */
                f32x4 t[4] = {(f32x4)(0.0f), (f32x4)(0.0f), (f32x4)(0.0f), (f32x4)(0.0f)};
#pragma unroll
                for(int o = 2; o < 8; o++)
#pragma unroll
                    for(int i = 0; i < 4; i++) t[i] = product(i, order[o][0], order[o][1], t[i]);
#pragma unroll
                for(int i = 0; i < 4; i++) acc[i][j] += t[i];
            } else {
                /* The last rows, perhaps one or two and no others: eight of the products, the large ones and the small ones apart, added to
                 * the total by rounded additions, which is what a single product needs to be as close as fp32's. */
#pragma unroll
                for(int h = 0; h < 4; h += 2){
                    f32x4 small[2] = {(f32x4)(0.0f), (f32x4)(0.0f)}, large[2];
#pragma unroll
                    for(int i = 0; i < 2; i++) large[i] = product(h + i, 0, 0, small[i]);
#pragma unroll
                    for(int o = 0; o < 7; o++)
#pragma unroll
                        for(int i = 0; i < 2; i++) small[i] = product(h + i, order[o][0], order[o][1], small[i]);
#pragma unroll
                    for(int i = 0; i < 2; i++) acc[h + i][j] += large[i] + small[i];
                }
            }
        }
    };
    if(!FEW && mine > 0){
        load(va, (gchar *)P.A, a.K, oa, 0); load(vb, (gchar *)P.B, a.N, ob, 0);
        for(int n = 0; n < mine; n++) multiply(std::true_type(), n);
    }
    if(M % 32 != 0 && whole % KS == wave){                /* the last rows: past the end zeros */
#pragma unroll
        for(int r = 0; r < 8; r++){
            const int m = whole * 32 + g * 8 + r;
            const size_t at = (size_t)min(m, M - 1) * 4;
            const f32x4 p = *(gf32x4 *)((gchar *)P.A + at * a.K + ca), q = *(gf32x4 *)((gchar *)P.B + at * a.N + cb);
            va[r] = m < M ? p : (f32x4)(0.0f); vb[r] = m < M ? q : (f32x4)(0.0f);
        }
        multiply(std::false_type(), 0);
    }
    /* element e of acc[i][j]: row 4 (4 g + e) + i, column 4 c + j; four columns at a time */
    auto out = [&](int r, int col, f32x4 v){
        if(i0 + r >= a.K || j0 + col >= a.N) return;
        v *= down;
        qx_gf4 *o = (qx_gf4 *)((qx_gfloat *)P.C + (size_t)(i0 + r) * a.N + j0 + col);      /* at any float */
        if(P.beta != 0.0f){ const qx_f4 old = *o; v += (f32x4){old[0], old[1], old[2], old[3]}; }
        *o = (qx_f4){v[0], v[1], v[2], v[3]};
    };
    float odd = 0.0f;
    if constexpr(KS == 1){
#pragma unroll
        for(int i = 0; i < 4; i++)
#pragma unroll
            for(int j = 0; j < 4; j++) odd += f3_odd(acc[i][j]);
        if(f3_any<KS>(odd, nullptr)){ f3_plain<GEMM_NT, B, B, KS>(a, P, i0, j0); return; }
#pragma unroll
        for(int i = 0; i < 4; i++)
#pragma unroll
            for(int e = 0; e < 4; e++) out((g * 4 + e) * 4 + i, c * 4, (f32x4){acc[i][0][e], acc[i][1][e], acc[i][2][e], acc[i][3][e]});
    } else {
        constexpr int U = B * B / 4 / (64 * KS);
        float *red = (float *)f3_lds;
#pragma unroll
        for(int i = 0; i < 4; i++)
#pragma unroll
            for(int e = 0; e < 4; e++)
                *(f32x4 *)(red + (wave * B + (g * 4 + e) * 4 + i) * LD + c * 4) = (f32x4){acc[i][0][e], acc[i][1][e], acc[i][2][e], acc[i][3][e]};
        __syncthreads();
        f32x4 v[U];
#pragma unroll
        for(int u = 0; u < U; u++){
            const int x = u * 64 * KS + threadIdx.x, r = x / (B / 4), col = x % (B / 4) * 4;
            v[u] = *(const f32x4 *)(red + r * LD + col);
#pragma unroll
            for(int q = 1; q < KS; q++) v[u] += *(const f32x4 *)(red + (q * B + r) * LD + col);
            odd += f3_odd(v[u]);
        }
        if(f3_any<KS>(odd, (int *)(red + KS * B * LD))){ f3_plain<GEMM_NT, B, B, KS>(a, P, i0, j0); return; }
#pragma unroll
        for(int u = 0; u < U; u++){
            const int x = u * 64 * KS + threadIdx.x;
            out(x / (B / 4), x % (B / 4) * 4, v[u]);
        }
    }
}

/* nn, tn: 32 x 64 outputs per workgroup; its four wavefronts take 64 of the contraction in turn, in two steps of 32. All operands of a step go
 * straight into a stage of LDS of the wavefront's own. Activations: 128 bytes of 32 rows, piece q of row r at q ^ (r / 2 % 8), so that the
 * sixteen rows of an operand read hit sixteen different units; lane = row lane % 32, lanes 0-31 take the first 16 of the 32 k, eight for each
 * of two products. Digits of nn: 32 rows of 32 bytes, and the transposing read of four-bit elements, in which lane i of 16 receives element i
 * of the sixteen lanes' eight bytes, hands a lane the sixteen k of its column. Digits of tn lie along k: 16 bytes of 64 columns. LDS reads are
 * inline assembly: the compiler would wait for every load to LDS in front of them.
 * Two stages let three workgroups onto a CU (43 KB each), which is worth more than a third stage (1024 rows, 512 x 1536, us: 11.8 against 13.2;
 * 4096, 1024 x 2048: 78 against 93) or 64 rows per wavefront with half the digit conversions and two thirds of the wavefronts (13.4, 74). Eight
 * wavefronts: 17 and 119. */
#define F3_WAVES 4
#define F3_ST 2
#define F3_A_BYTES 4096
#define F3_STAGE (F3_A_BYTES + 1024 + 256)       /* activations, digits, scales */
#define F3_LOADS 6
template<int OFF> __device__ __forceinline__ f32x4 f3_rd128(uint32_t addr){
    f32x4 v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
    return v;
}
template<int OFF> __device__ __forceinline__ i32x2 f3_rd64(uint32_t addr){
    i32x2 v;
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
    return v;
}
template<int OFF> __device__ __forceinline__ float f3_rd32(uint32_t addr){
    float v;
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
    return v;
}
template<int OFF> __device__ __forceinline__ i32x2 f3_tr4(uint32_t addr){
    i32x2 v;
    asm volatile("ds_read_b64_tr_b4 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
    return v;
}
/* lane I's value of every row of 16 lanes */
template<int I> __device__ __forceinline__ float f3_bcast(float v){
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + I, 0xF, 0xF, true));
}
template<int MODE>
__global__ void __launch_bounds__(64 * F3_WAVES, 2) k_gemm_f32s(F3Args a){
    constexpr int BM = 32, BN = 64, LD = BM + 4, KS = F3_WAVES, ST = F3_ST, AB = F3_A_BYTES;
    constexpr float up = F3_UP(MODE), down = F3_DOWN(MODE);
    extern __shared__ __attribute__((aligned(16))) unsigned char f3_lds[];
    const int tile = qx_xcd_tile(blockIdx.x, gridDim.x);
    if(tile >= a.ntiles) return;
    const DevProb P = a.pr[qx_find_problem(a.pr, a.nprob, tile)];
    const int lt = tile - P.tile0, ti = lt / P.tiles_n, tj = lt - ti * P.tiles_n;
    const int i0 = ti * BM, j0 = tj * BN;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 31, hf = lane >> 5;
    const QxMinus minus = qx_minus();
    const int chunks = a.K / 64, mine = 2 * ((chunks - wave + KS - 1) / KS);        /* steps of this wavefront */
    unsigned char *base = f3_lds + wave * (ST * F3_STAGE);
    uint32_t ra[4];
#pragma unroll
    for(int n = 0; n < 4; n++){
        const int r = n * 8 + (lane >> 3);
        ra[n] = (uint32_t)min(r, P.M - 1 - i0) * (uint32_t)a.K * 4u + ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    }
    gchar *A = (gchar *)P.A + (size_t)i0 * a.K * 4;
    const signed char *W = MODE == GEMM_NN ? a.d + ((P.wq + (size_t)(lane >> 1) * a.N + j0) >> 1) + (lane & 1) * 16
                                           : a.d + ((P.wq + (size_t)min(j0 + lane, a.N - 1) * a.K) >> 1);
    const float *S = a.s + P.wg + (MODE == GEMM_NN ? ((size_t)c * a.N + j0) >> a.gshift : ((size_t)min(j0 + lane, a.N - 1) * a.K) >> a.gshift);
    auto load = [&](int stage, int n){
        const int k0 = ((n >> 1) * KS + wave) * 64 + (n & 1) * 32;
        unsigned char *st = base + stage * F3_STAGE;
#pragma unroll
        for(int q = 0; q < 4; q++) __builtin_amdgcn_global_load_lds((glb_void *)(A + (size_t)k0 * 4 + ra[q]), (lds_void *)(st + q * 1024), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((glb_void *)(W + ((MODE == GEMM_NN ? (size_t)k0 * a.N : (size_t)k0) >> 1)), (lds_void *)(st + AB), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((glb_void *)(S + ((MODE == GEMM_NN ? (size_t)k0 * a.N : (size_t)k0) >> a.gshift)), (lds_void *)(st + AB + 1024), 4, 0, 0);
        asm volatile("" ::: "memory");                    /* the loads of a step stay together: the waits count them */
    };
    qx_f32x16 acc[2] = {(qx_f32x16)(0.0f), (qx_f32x16)(0.0f)}, part[2];
    const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_void *)base;
    uint32_t rdx[4];
#pragma unroll
    for(int p = 0; p < 4; p++) rdx[p] = lds_base + c * 128 + (((hf * 4 + p) ^ ((c >> 1) & 7)) << 4);
    const uint32_t rdw = lds_base + (MODE == GEMM_NN ? (hf * 16 + (lane & 15)) * 32 + (lane >> 4 & 1) * 8 : c * 16 + hf * 8);
    const uint32_t rds = lds_base + (MODE == GEMM_NN ? hf * 16 + (lane & 15) : c) * 4;
    auto step = [&](auto HALF, int stage, int n){
        /* the step behind this one, except at the end, may still be on its way */
        if(n + ST <= mine) asm volatile("s_waitcnt vmcnt(%0)" :: "n"((ST - 1) * F3_LOADS) : "memory");
        else               asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const uint32_t so = stage * F3_STAGE;
        f32x4 x[4]; i32x2 w[2]; float sv[2];
        if constexpr(MODE == GEMM_NN){ w[0] = f3_tr4<AB>(rdw + so); w[1] = f3_tr4<AB + 16>(rdw + so); sv[0] = f3_rd32<AB + 1024>(rds + so); sv[1] = 0.0f; }
        else {
            w[0] = f3_rd64<AB>(rdw + so); w[1] = f3_rd64<AB + 512>(rdw + so);
            sv[0] = f3_rd32<AB + 1024>(rds + so); sv[1] = f3_rd32<AB + 1024 + 128>(rds + so);
        }
#pragma unroll
        for(int p = 0; p < 4; p++) x[p] = f3_rd128<0>(rdx[p] + so);
        /* everything is in registers before the stage is loaded again */
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(w[0]), "+v"(w[1]), "+v"(sv[0]), "+v"(sv[1]) :: "memory");
        if(n + ST < mine) load(stage, n + ST);
        if(MODE == GEMM_NN) sv[0] *= up;
        else { sv[0] *= 16.0f; sv[1] *= 16.0f; }          /* digits come as digit / 16 */
        constexpr bool first = decltype(HALF)::value == 0;
        if(first) part[0] = part[1] = (qx_f32x16)(0.0f);
        f3_each<0, 2>([&](auto UC){
            constexpr int u = decltype(UC)::value;
            uint4 y[2], xp[3];
#pragma unroll
            for(int j = 0; j < 2; j++) y[j] = f3_digits((uint32_t)w[j][u]);
            float f[8];
#pragma unroll
            for(int q = 0; q < 8; q++) f[q] = MODE == GEMM_TN ? up * x[u * 2 + (q >> 2)][q & 3] : x[u * 2 + (q >> 2)][q & 3];
            if constexpr(MODE == GEMM_NN) f3_each<0, 8>([&](auto QC){ constexpr int q = decltype(QC)::value; f[q] *= f3_bcast<u * 8 + q>(sv[0]); });
            f3_split(minus, f, xp);
#pragma unroll
            for(int q = 2; q >= 0; q--)
#pragma unroll
                for(int j = 0; j < 2; j++)
                    part[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, xp[q]), __builtin_bit_cast(bf16x8, y[j]), part[j], 0, 0, 0);
        });
        if(!first)
#pragma unroll
            for(int j = 0; j < 2; j++)
#pragma unroll
                for(int e = 0; e < 16; e++) acc[j][e] = MODE == GEMM_TN ? fmaf(sv[j], part[j][e], acc[j][e]) : acc[j][e] + part[j][e];
    };
#pragma unroll
    for(int n = 0; n < ST; n++) if(n < mine) load(n, n);
    for(int n = 0; n < mine; n += 2){
        step(std::integral_constant<int, 0>(), 0, n);
        step(std::integral_constant<int, 1>(), 1, n + 1);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);                   /* vmcnt(0): no load may land in a stage any more */
    /* Sums of a wavefront, in its own stages, as columns of 32 rows (a lane holds four consecutive rows of a column), columns 36 words
     * apart: the 16-byte writes and reads of eight lanes hit all banks once. */
    constexpr int U = BM * BN / 4 / (64 * KS), STRIDE = ST * F3_STAGE / 4;
    static_assert(BN * LD + KS <= STRIDE, "a wavefront's sums and a flag fit its stages");
    float *red = (float *)f3_lds;
#pragma unroll
    for(int j = 0; j < 2; j++)
#pragma unroll
        for(int q = 0; q < 4; q++)
            *(f32x4 *)(red + wave * STRIDE + (j * 32 + c) * LD + q * 8 + hf * 4) = (f32x4){acc[j][q * 4], acc[j][q * 4 + 1], acc[j][q * 4 + 2], acc[j][q * 4 + 3]};
    __syncthreads();
    f32x4 v[U];
    float odd = 0.0f;
#pragma unroll
    for(int u = 0; u < U; u++){
        const int x = u * 64 * KS + threadIdx.x, col = x % BN, row = x / BN * 4;
        v[u] = *(const f32x4 *)(red + col * LD + row);
#pragma unroll
        for(int q = 1; q < KS; q++) v[u] += *(const f32x4 *)(red + q * STRIDE + col * LD + row);
        odd += f3_odd(v[u]);
    }
    if(f3_any<KS>(odd, (int *)(red + (KS - 1) * STRIDE + BN * LD))){ f3_plain<MODE, BM, BN, KS>(a, P, i0, j0); return; }
#pragma unroll
    for(int u = 0; u < U; u++){
        const int x = u * 64 * KS + threadIdx.x, col = x % BN, row = x / BN * 4, left = P.M - (i0 + row);
        if(j0 + col >= a.N) continue;
        v[u] *= down;
        qx_gfloat *o = (qx_gfloat *)P.C + (size_t)(i0 + row) * a.N + j0 + col;
        if(P.beta != 0.0f)
#pragma unroll
            for(int e = 0; e < 4; e++) if(e < left) v[u][e] += o[(size_t)e * a.N];
#pragma unroll
        for(int e = 0; e < 4; e++) if(e < left) o[(size_t)e * a.N] = v[u][e];
    }
}

template<int MODE, int BM, int BN, int NT, int LDS, void (*KERNEL)(F3Args)>
static int launch_tiles(const F3Args &args, const qlmx_gemm_prob *probs, int nprob, hipStream_t st){
    F3Args a = args;
    ProbUpload up; int slot;
    int rc = qlmx_upload_problems(probs, nprob, MODE, a.K, a.N, BM, BN, st, &up, &slot); if(rc) return rc;
    if(up.ntiles == 0) return QLMX_OK;
    a.pr = up.dev; a.nprob = up.nprob; a.ntiles = up.ntiles;
    static bool attr_set = false;
    if(!attr_set){
        QLMX_HIP(hipFuncSetAttribute((const void *)KERNEL, hipFuncAttributeMaxDynamicSharedMemorySize, LDS), "fp32 gemm LDS size");
        attr_set = true;
    }
    hipLaunchKernelGGL(KERNEL, dim3((up.ntiles + 7) & ~7), dim3(NT), LDS, st, a);
    QLMX_LAUNCH_CHECK("grouped gemm (fp32 in parts) launch");
    return qlmx_upload_done(slot, st);
}

static long long f3_nt_tiles(const qlmx_gemm_prob *probs, int nprob, int K, int N){
    long long n = 0;
    for(int i = 0; i < nprob; i++) if(probs[i].M > 0) n += (long long)((K + 63) / 64) * ((N + 63) / 64);
    return n;
}
/* Weight gradients: eight wavefronts along the rows where every compute unit has at most one tile, two wavefronts to a matrix core, one splitting
 * while the other multiplies; four up to three tiles per unit; each where there are rows enough for all of them; else one, without LDS. us with one /
 * four / eight: 192 tiles of 512 x 1536, 128 rows 9 / 6.0 / 6.1, 192 rows 12 / 7.5 / 7.2, 1024 rows 55 / 20 / 17; 256 tiles, 1024 rows 55 / 20 / 18; 320 tiles
 * 55 / 28 / 29; 512 tiles, 4096 rows 213 / 111 / 111; 4 x 75 rows, 640 x 1408, 880 tiles 11 / 14; 4 x 1024, 2048 x 1024, 2048 tiles 99 / 111. */
int qlmx_gemm_f32s_launch(int mode, const signed char *d, const float *s, int group, const qlmx_gemm_prob *probs, int nprob, int K, int N, hipStream_t st){
    F3Args a; a.pr = nullptr; a.nprob = a.ntiles = 0; a.d = d; a.s = s; a.gshift = 0; a.K = K; a.N = N;
    while(mode != GEMM_NT && (1 << a.gshift) < group) a.gshift++;
    constexpr int lds = F3_WAVES * F3_ST * F3_STAGE;
    if(mode == GEMM_NN) return launch_tiles<GEMM_NN, 32, 64, 64 * F3_WAVES, lds, k_gemm_f32s<GEMM_NN>>(a, probs, nprob, st);
    if(mode == GEMM_TN) return launch_tiles<GEMM_TN, 32, 64, 64 * F3_WAVES, lds, k_gemm_f32s<GEMM_TN>>(a, probs, nprob, st);
    int most = 0;
    for(int i = 0; i < nprob; i++) if(probs[i].M > most) most = probs[i].M;
    const long long tiles = f3_nt_tiles(probs, nprob, K, N);
    if(tiles <= qlmx_cu_count() && most >= 192) return launch_tiles<GEMM_NT, 64, 64, 512, (8 * 64 * 68 + 8) * 4, k_gemm_f32s_nt<8, false>>(a, probs, nprob, st);
    if(tiles < 3LL * qlmx_cu_count() && most >= 128) return launch_tiles<GEMM_NT, 64, 64, 256, (4 * 64 * 68 + 4) * 4, k_gemm_f32s_nt<4, false>>(a, probs, nprob, st);
    return most < 32 ? launch_tiles<GEMM_NT, 64, 64, 64, 64, k_gemm_f32s_nt<1, true>>(a, probs, nprob, st)
                     : launch_tiles<GEMM_NT, 64, 64, 64, 64, k_gemm_f32s_nt<1, false>>(a, probs, nprob, st);
}

/* Whether these kernels take a call: 64 columns (nn) or 64 of the contraction (tn) inside one scale group, whole units of 16 bytes. Everything else
 * goes to qlmx_gemm_f32.hip, as do weight gradients of few rows and few tiles, whose rows it spreads over more wavefronts (2 to 16 rows of 256 x
 * 512: 4.5 us against 5.0). Elsewhere these are the faster ones, few-row forwards but those of qlmx_gemv_nn_gains included (us, before / here: two rows of eight experts, 512 x
 * 1024, 24.8 / 5.4 with the GEMV; 1024 rows, 512 x 1536, and back, forward 28.2, 27.6 / 11.6, 10.3, input gradient 28.7, 25.3 / 11.2, 10.5,
 * weight gradient 23.7, 22.4 / 17.0, 15.8; 4096 rows, 1024 x 2048: 175, 168, 197 / 77, 69, 106). The error against 64 bits is no larger at any size
 * tried, one to 32768 rows and contractions of up to 16384 (head of the file). */
bool qlmx_gemm_f32s_takes(int mode, const signed char *d, int group, const qlmx_gemm_prob *probs, int nprob, int K, int N){
    if(mode == GEMM_NT){
        int most = 0;
        for(int i = 0; i < nprob; i++) if(probs[i].M > most) most = probs[i].M;
        if(most <= 32 && f3_nt_tiles(probs, nprob, K, N) < qlmx_cu_count()) return false;
    }
    if(mode == GEMM_NT ? K % 4 || N % 4 : K % 64 || (group != 64 && group != 128 && group != 256) || ((uintptr_t)d & 15)) return false;
    for(int i = 0; i < nprob; i++)
        if((((uintptr_t)probs[i].A | (mode == GEMM_NT ? (uintptr_t)probs[i].B : 0)) & 15) != 0) return false;
    return true;
}
