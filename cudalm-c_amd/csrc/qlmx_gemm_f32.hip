/* qlmx_gemm_f32.hip -- grouped expert GEMMs in fp32 on the fp32 matrix core, dequantisation fused into the
 * weight-tile load.
 *
 * This is the path whose results track the reference's CPU SGEMM to rounding error: the weight is
 * formed as the single fp32 product s*digit (exactly the value the reference renders into P,
 * qlm.cuh:177) and every multiply-accumulate is an fp32 FMA (v_mfma_f32_32x32x2_f32 multiplies and adds
 * fp32 values), as in the reference's 6x16 micro-kernel (cpu_rt.h:196-208); only the summation order
 * differs. Under QLMX_MATH_F32 (the default of the host mirror's mg_bind) it serves what the kernels of
 * qlmx_gemm_f32s.hip, twice as fast, do not take: bf16 activations, groups below 64, odd sizes and addresses, and
 * weight gradients of a few rows and tiles.
 *
 *   nn: out[m,n] = sum_k A[m,k] * W[k,n]      W row-major [K,N], groups along n
 *   tn: out[m,n] = sum_k A[m,k] * W[n,k]      W row-major [N,K], groups along k   (+ beta*out)
 *   nt: out[k,n] += sum_m A[m,k] * B[m,n]     no weight operand
 * A flattened tile list covers every problem of the call, so one launch serves all experts.
 *
 * What bounds it: the fp32 matrix core (256 operations per cycle and CU, a sixteenth of the bf16 rate: one
 * 32x32x2 product holds it for 64 cycles), so that a wavefront needs one 4-byte read of each operand per 64 cycles
 * and neither LDS, L2 nor the dequantisation comes near a limit, even on 32x32 tiles. The split of the work therefore
 * serves one thing, matrix cores that are all busy: a workgroup is WM x WN wavefronts of 32x32 outputs times KS
 * wavefronts that share the contraction and add up through LDS in a fixed order (see f32_shape for the choice).
 * One expert of 1024 rows, 512 x 1536, six GEMMs of 1.6 GFLOP each: 970 us with 4x4 outputs per thread on the vector
 * ALU (80-263 us a launch); 22-28 us a launch here. A step is 64 deep where four wavefronts share the contraction (32
 * and 128 deep: 167 and 162 us for the six launches against 154), since what is left is the start and end of a
 * workgroup and the wait for its operands, which more resident workgroups cover.
 *
 * Operand layouts in LDS. An operand whose contraction index is contiguous in memory keeps rows of consecutive k
 * ("KMAJ", 128-bit reads of four k), the other kind keeps rows of consecutive outputs ("IMAJ", 32-bit reads).
 * Both use the same order of the contraction inside eight k: product i takes k = i from lanes 0-31 and k = 4 + i from
 * lanes 32-63. The row padding (4 and 8 words) makes both kinds of reads conflict-free. Two LDS buffers: the next
 * step's operands are loaded into registers before this step's products and written behind them.
 */
#include "qlmx_gemm.h"

struct F32Args { const DevProb *pr; int nprob, ntiles; const signed char *d; const float *s; int group; int K, N; };

template<bool BF16> __device__ __forceinline__ float ld_act(const void *p, size_t i){
    if constexpr(BF16) return qx_bf16_to_f32(((const unsigned short *)p)[i]);
    return ((const float *)p)[i];
}
/* four consecutive activations, 16-byte (fp32) or 8-byte (bf16) aligned */
template<bool BF16> __device__ __forceinline__ float4 ld_act4(const void *p, size_t i){
    if constexpr(BF16){
        const ushort4 h = *(const ushort4 *)((const unsigned short *)p + i);
        return make_float4(qx_bf16_to_f32(h.x), qx_bf16_to_f32(h.y), qx_bf16_to_f32(h.z), qx_bf16_to_f32(h.w));
    }
    return *(const float4 *)((const float *)p + i);
}
/* s*digit for element e of the packed digit array; group index relative to the matrix start */
__device__ __forceinline__ float ld_weight(const signed char *d, const float *s, unsigned long long wq,
                                           unsigned long long wg, size_t e, int group){
    const unsigned long long q = wq + e;
    const unsigned b = (unsigned char)d[q >> 1];
    const int v = (q & 1ULL) ? (int)(b >> 4) : (int)(b & 15u);
    return s[wg + e / (size_t)group] * (float)(v >= 8 ? v - 16 : v);
}

template<int WM, int WN, int KS> struct F32Shape {
    static constexpr int NT = 64 * WM * WN * KS, BM = 32 * WM, BN = 32 * WN, BK = KS == 1 ? 32 : KS == 4 ? 64 : 128;
    static constexpr int KW = BK / KS;                       /* contraction values of a wavefront per step */
};

/* FAST: K, N and the group are multiples of 8, every problem's pointers are 16-byte and weight offsets 8-element
 * aligned, so that operands move in units of four activations or eight digits (which share one scale);
 * otherwise units are put together element by element. */
template<int MODE, bool BF16, bool FAST, int WM, int WN, int KS>
__global__ void __launch_bounds__(64 * WM * WN * KS) k_gemm_f32(F32Args a){
    typedef F32Shape<WM, WN, KS> SH;
    constexpr int NT = SH::NT, BM = SH::BM, BN = SH::BN, BK = SH::BK, KW = SH::KW;
    constexpr bool KMAJ_A = MODE != GEMM_NT, KMAJ_B = MODE == GEMM_TN, WEIGHT = MODE != GEMM_NT;
    constexpr int LDA = KMAJ_A ? BK + 4 : BM + 8, LDB = KMAJ_B ? BK + 4 : BN + 8;
    constexpr int A_WORDS = (KMAJ_A ? BM : BK) * LDA, B_WORDS = (KMAJ_B ? BN : BK) * LDB;
    constexpr int UA = BM * BK / 4 / NT;                                     /* units of four per thread */
    constexpr int EB = WEIGHT ? 8 : 4, NB = BN * BK / EB, UB = (NB + NT - 1) / NT;
    constexpr int RED_WORDS = KS > 1 ? KS * BM * BN : 0;
    constexpr int WORDS = 2 * (A_WORDS + B_WORDS) > RED_WORDS ? 2 * (A_WORDS + B_WORDS) : RED_WORDS;
    extern __shared__ __attribute__((aligned(16))) float f32_lds[];
    static_assert(WORDS * 4 <= 160 * 1024, "LDS");

    const int t = qx_xcd_tile(blockIdx.x, gridDim.x);
    if(t >= a.ntiles) return;
    const DevProb P = a.pr[qx_find_problem(a.pr, a.nprob, t)];
    const int lt = t - P.tile0;
    const int ti = lt / P.tiles_n, tj = lt - ti * P.tiles_n;
    const int i0 = ti * BM, j0 = tj * BN;
    const int rows = MODE == GEMM_NT ? a.K : P.M;      /* output rows   */
    const int cols = a.N;                              /* output cols   */
    const int depth = MODE == GEMM_NT ? P.M : a.K;     /* contraction   */
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ks = wave / (WM * WN), wi = (wave % (WM * WN)) / WN * 32, wj = wave % WN * 32;

    /* ---- operands of the step from contraction index p0 on, in registers ---- */
    float4 va[UA]; uint32_t wb[UB]; float sb[UB]; float4 vb[WEIGHT ? 1 : UB]; float eb[WEIGHT && !FAST ? UB * 8 : 1];
    auto load = [&](int p0){
#pragma unroll
        for(int u = 0; u < UA; u++){
            const int x = u * NT + tid;
            const int i = KMAJ_A ? x / (BK / 4) : x % (BM / 4) * 4, k = KMAJ_A ? x % (BK / 4) * 4 : x / (BM / 4), p = p0 + k;
            float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if constexpr(FAST){
                if constexpr(KMAJ_A){ const int r = min(i0 + i, rows - 1); if(p < depth) v = ld_act4<BF16>(P.A, (size_t)r * a.K + p); }
                else { const int r = min(i0 + i, rows - 4); if(p < depth) v = ld_act4<BF16>(P.A, (size_t)p * a.K + r); }
            } else {
                float e[4];
#pragma unroll
                for(int q = 0; q < 4; q++){
                    const int r = i0 + i + (KMAJ_A ? 0 : q), c = p + (KMAJ_A ? q : 0);
                    e[q] = (r < rows && c < depth) ? ld_act<BF16>(P.A, KMAJ_A ? (size_t)r * a.K + c : (size_t)c * a.K + r) : 0.0f;
                }
                v = make_float4(e[0], e[1], e[2], e[3]);
            }
            va[u] = v;
        }
#pragma unroll
        for(int u = 0; u < UB; u++){
            const int x = u * NT + tid;
            if(NB % NT != 0 && x >= NB) break;
            const int j = KMAJ_B ? x / (BK / EB) : x % (BN / EB) * EB, k = KMAJ_B ? x % (BK / EB) * EB : x / (BN / EB), p = p0 + k;
            if constexpr(WEIGHT && FAST){
                const int c = KMAJ_B ? min(j0 + j, cols - 1) : min(j0 + j, cols - 8);
                wb[u] = 0; sb[u] = 0.0f;
                if(p < depth){
                    const size_t e = KMAJ_B ? (size_t)c * a.K + p : (size_t)p * a.N + c;
                    wb[u] = *(const uint32_t *)(a.d + ((P.wq + e) >> 1));
                    sb[u] = a.s[P.wg + e / (size_t)a.group];
                }
            } else if constexpr(WEIGHT){
#pragma unroll
                for(int q = 0; q < 8; q++){
                    const int c = j0 + j + (KMAJ_B ? 0 : q), pp = p + (KMAJ_B ? q : 0);
                    eb[u * 8 + q] = (c < cols && pp < depth) ? ld_weight(a.d, a.s, P.wq, P.wg, KMAJ_B ? (size_t)c * a.K + pp : (size_t)pp * a.N + c, a.group) : 0.0f;
                }
            } else if constexpr(FAST){
                const int c = min(j0 + j, cols - 4);
                vb[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if(p < depth) vb[u] = ld_act4<BF16>(P.B, (size_t)p * a.N + c);
            } else {
                float e[4];
#pragma unroll
                for(int q = 0; q < 4; q++) e[q] = (j0 + j + q < cols && p < depth) ? ld_act<BF16>(P.B, (size_t)p * a.N + j0 + j + q) : 0.0f;
                vb[u] = make_float4(e[0], e[1], e[2], e[3]);
            }
        }
    };
    /* ---- and from the registers into an LDS buffer ---- */
    auto store = [&](float *As, float *Bs){
#pragma unroll
        for(int u = 0; u < UA; u++){
            const int x = u * NT + tid;
            const int i = KMAJ_A ? x / (BK / 4) : x % (BM / 4) * 4, k = KMAJ_A ? x % (BK / 4) * 4 : x / (BM / 4);
            *(float4 *)&As[KMAJ_A ? i * LDA + k : k * LDA + i] = va[u];
        }
#pragma unroll
        for(int u = 0; u < UB; u++){
            const int x = u * NT + tid;
            if(NB % NT != 0 && x >= NB) break;
            const int j = KMAJ_B ? x / (BK / EB) : x % (BN / EB) * EB, k = KMAJ_B ? x % (BK / EB) * EB : x / (BN / EB);
            float *dst = &Bs[KMAJ_B ? j * LDB + k : k * LDB + j];
            if constexpr(WEIGHT){
                float e[8];
                if constexpr(FAST){
                    /* fl(s * digit); with the 16 on s it would be infinite from s = 2^124 on */
                    const QxNibs nb = qx_nibs(wb[u]);
#pragma unroll
                    for(int q = 0; q < 8; q++) e[q] = sb[u] * (16.0f * qx_nib16(nb, q));
                } else {
#pragma unroll
                    for(int q = 0; q < 8; q++) e[q] = eb[u * 8 + q];
                }
                *(float4 *)dst = make_float4(e[0], e[1], e[2], e[3]);
                *(float4 *)(dst + 4) = make_float4(e[4], e[5], e[6], e[7]);
            } else *(float4 *)dst = vb[u];
        }
    };

    qx_f32x16 acc = (qx_f32x16)(0.0f);
    const int fr = lane & 31, hf = lane >> 5;
    constexpr int BUF = A_WORDS + B_WORDS;
    load(0);
    store(f32_lds, f32_lds + A_WORDS);
    __syncthreads();
    for(int p0 = 0, b = 0; p0 < depth; p0 += BK, b ^= 1){
        const bool more = p0 + BK < depth;
        if(more) load(p0 + BK);
        const float *As = f32_lds + b * BUF + (KMAJ_A ? (wi + fr) * LDA + ks * KW + hf * 4 : (ks * KW + hf * 4) * LDA + wi + fr);
        const float *Bs = f32_lds + b * BUF + A_WORDS + (KMAJ_B ? (wj + fr) * LDB + ks * KW + hf * 4 : (ks * KW + hf * 4) * LDB + wj + fr);
#pragma unroll
        for(int k = 0; k < KW; k += 8){
            float x[4], y[4];
            if constexpr(KMAJ_A){ const float4 v = *(const float4 *)(As + k); x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w; }
            else {
#pragma unroll
                for(int q = 0; q < 4; q++) x[q] = As[(k + q) * LDA];
            }
            if constexpr(KMAJ_B){ const float4 v = *(const float4 *)(Bs + k); y[0] = v.x; y[1] = v.y; y[2] = v.z; y[3] = v.w; }
            else {
#pragma unroll
                for(int q = 0; q < 4; q++) y[q] = Bs[(k + q) * LDB];
            }
#pragma unroll
            for(int q = 0; q < 4; q++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[q], y[q], acc, 0, 0, 0);
        }
        if(more) store(f32_lds + (b ^ 1) * BUF, f32_lds + (b ^ 1) * BUF + A_WORDS);
        __syncthreads();
    }

    /* ---- the lane holds column lane%32, rows (e/4)*8 + e%4 + 4*(lane/32) of its 32x32 outputs ---- */
    auto out = [&](int r, int c, float v){
        if(r < rows && c < cols){ float *o = P.C + (size_t)r * a.N + c; *o = P.beta != 0.0f ? *o + v : v; }
    };
    if constexpr(KS == 1){
#pragma unroll
        for(int e = 0; e < 16; e++) out(i0 + wi + (e >> 2) * 8 + (e & 3) + hf * 4, j0 + wj + fr, acc[e]);
    } else {
        float *red = f32_lds + ks * (BM * BN);
#pragma unroll
        for(int e = 0; e < 16; e++) red[(wi + (e >> 2) * 8 + (e & 3) + hf * 4) * BN + wj + fr] = acc[e];
        __syncthreads();
#pragma unroll
        for(int u = 0; u < BM * BN / NT; u++){
            const int x = u * NT + tid;
            float v = f32_lds[x];
#pragma unroll
            for(int q = 1; q < KS; q++) v += f32_lds[q * (BM * BN) + x];
            out(i0 + x / BN, j0 + x % BN, v);
        }
    }
}

template<int MODE, bool BF16, bool FAST, int WM, int WN, int KS>
static int launch_shape(const F32Args &args, const qlmx_gemm_prob *probs, int nprob, hipStream_t st){
    typedef F32Shape<WM, WN, KS> SH;
    F32Args a = args;
    ProbUpload up; int slot;
    int rc = qlmx_upload_problems(probs, nprob, MODE, a.K, a.N, SH::BM, SH::BN, st, &up, &slot); if(rc) return rc;
    if(up.ntiles == 0) return QLMX_OK;
    a.pr = up.dev; a.nprob = up.nprob; a.ntiles = up.ntiles;
    constexpr int LDA = MODE != GEMM_NT ? SH::BK + 4 : SH::BM + 8, LDB = MODE == GEMM_TN ? SH::BK + 4 : SH::BN + 8;
    constexpr int stage = 8 * ((MODE != GEMM_NT ? SH::BM : SH::BK) * LDA + (MODE == GEMM_TN ? SH::BN : SH::BK) * LDB);
    constexpr int red = KS > 1 ? 4 * KS * SH::BM * SH::BN : 0, lds = stage > red ? stage : red;
    static bool attr_set = false;
    if(!attr_set){
        QLMX_HIP(hipFuncSetAttribute((const void *)(k_gemm_f32<MODE, BF16, FAST, WM, WN, KS>), hipFuncAttributeMaxDynamicSharedMemorySize, lds), "fp32 gemm LDS size");
        attr_set = true;
    }
    hipLaunchKernelGGL((k_gemm_f32<MODE, BF16, FAST, WM, WN, KS>), dim3((up.ntiles + 7) & ~7), dim3(SH::NT), lds, st, a);
    QLMX_LAUNCH_CHECK("grouped gemm (fp32) launch");
    return qlmx_upload_done(slot, st);
}

/* Which shape: 64x64 outputs per workgroup (an operand value is fetched half as often) when there are several
 * rounds of them, else 32x32 with four wavefronts along the contraction (the launch is then four times as many,
 * four times as short pieces and ends evenly), and with sixteen when even those leave CUs without a workgroup. */
template<int MODE, bool BF16, bool FAST>
static int launch_f32(const F32Args &a, const qlmx_gemm_prob *probs, int nprob, hipStream_t st){
    long long t64 = 0, t32 = 0;
    for(int i = 0; i < nprob; i++){
        const long long r = MODE == GEMM_NT ? a.K : probs[i].M;
        if(probs[i].M <= 0) continue;
        t64 += ((r + 63) / 64) * ((a.N + 63) / 64);
        t32 += ((r + 31) / 32) * ((a.N + 31) / 32);
    }
    const int cus = qlmx_cu_count();
    if(t64 >= 6LL * cus) return launch_shape<MODE, BF16, FAST, 2, 2, 1>(a, probs, nprob, st);
    if(t32 >= cus)       return launch_shape<MODE, BF16, FAST, 1, 1, 4>(a, probs, nprob, st);
    return launch_shape<MODE, BF16, FAST, 1, 1, 16>(a, probs, nprob, st);
}

template<int MODE>
static int launch_mode(const F32Args &a, const qlmx_gemm_prob *probs, int nprob, int act_dtype, hipStream_t st){
    bool fast = a.K % 8 == 0 && a.N % 8 == 0 && (MODE == GEMM_NT || (a.group % 8 == 0 && ((uintptr_t)a.d & 3) == 0));
    for(int i = 0; i < nprob && fast; i++)
        fast = (((uintptr_t)probs[i].A | (MODE == GEMM_NT ? (uintptr_t)probs[i].B : 0)) & 15) == 0 && (MODE == GEMM_NT || probs[i].wq % 8 == 0);
    const bool b = act_dtype == QLMX_ACT_BF16;
    if(fast) return b ? launch_f32<MODE, true, true>(a, probs, nprob, st)  : launch_f32<MODE, false, true>(a, probs, nprob, st);
    return          b ? launch_f32<MODE, true, false>(a, probs, nprob, st) : launch_f32<MODE, false, false>(a, probs, nprob, st);
}

bool qlmx_gemm_f32s_takes(int mode, const signed char *d, int group, const qlmx_gemm_prob *probs, int nprob, int K, int N);
int qlmx_gemm_f32s_launch(int mode, const signed char *d, const float *s, int group, const qlmx_gemm_prob *probs, int nprob, int K, int N, hipStream_t st);

int qlmx_gemm_f32_dispatch(int mode, const signed char *d, const float *s, int group,
                           const qlmx_gemm_prob *probs, int nprob, int K, int N, int act_dtype, hipStream_t st){
    if(act_dtype == QLMX_ACT_F32 && qlmx_gemm_f32s_takes(mode, d, group, probs, nprob, K, N))
        return qlmx_gemm_f32s_launch(mode, d, s, group, probs, nprob, K, N, st);
    F32Args a; a.pr = nullptr; a.nprob = a.ntiles = 0; a.d = d; a.s = s; a.group = group; a.K = K; a.N = N;
    if(mode == GEMM_NN) return launch_mode<GEMM_NN>(a, probs, nprob, act_dtype, st);
    if(mode == GEMM_TN) return launch_mode<GEMM_TN>(a, probs, nprob, act_dtype, st);
    return launch_mode<GEMM_NT>(a, probs, nprob, act_dtype, st);
}
