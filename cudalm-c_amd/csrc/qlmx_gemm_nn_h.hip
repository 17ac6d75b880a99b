/* qlmx_gemm_nn_h.hip -- forward grouped GEMM (nn) on the fp16 matrix core: one MFMA per product.
 *
 * Y_e[M,N] = X_e[M,K] . W_e[K,N]   (mg_ab, cudalm.cu:3204-3256; call sites 4211-4225)
 *
 * W is packed 4-bit with its scale groups along N, so the scale differs for every contraction index and
 * cannot be taken out of the sum: the weight w = s*digit has to be one matrix-core operand. In bf16 (8
 * significant bits) that rounding alone costs 1.6e-3 of relative error, which is why the bf16 kernel
 * (qlmx_gemm_nn_lds.hip) splits w into hi + lo and spends two MFMAs per product. fp16 keeps 11 bits:
 * fp16(s*digit), rounded to nearest even, is within 2^-12 of w, about 2e-4 relative L2 on the output,
 * and one v_mfma_f32_32x32x16_f16 per product is enough. The activations arrive as bf16; every bf16 value
 * between 2^-14 and 65504 in magnitude is an fp16 value, so they are converted exactly on their way into LDS
 * (smaller ones become fp16 subnormals with an absolute error below 3e-8, larger ones saturate at 65504).
 * Weights are multiplied by 2^8 before the conversion and the accumulators by 2^-8 after the last step, which
 * moves the range in which fp16 keeps all 11 bits to 2.4e-7 <= |w| <= 255.
 *
 * Tiles of 256 x 256 (or less, nh_tiles), steps 64 deep, eight wavefronts with 128 x 64 outputs each, two LDS buffers per operand: 128 KB, one
 * workgroup per CU. Every operand passes through registers once: a thread loads 16 bytes of four activation rows and 32 weights per step,
 * converts them a step later and writes them into the buffer that is not being read. What bounds it is what the wavefronts do beside
 * the products: with the loads, conversions and LDS writes left out the gate|up launch of 3001 tokens (64 experts, top 4, 2048 x 1408) takes 137 of
 * its 190 us, without the loads alone 165, without the conversions 159; LDS reads and barriers are in the 137 (128 without them). So the tile is
 * as large as the registers allow -- a piece of activations or weights is prepared once for 256 columns or rows -- and the step is 64
 * deep: activation rows are read in whole lines of 128 bytes, weights and scales with half as many loads, and there are half as many barriers.
 * gate|up and down of those tokens, us: 228, 120 with 256 x 128 tiles on four wavefronts and steps of 32; 217, 110 with eight
 * wavefronts and 256 x 256; 199, 100 with steps of 64; 190, 97 with the operand reads spread over the first products of a slice. Loads one
 * step further ahead, wavefront priorities, buffer addressing or three LDS buffers change nothing.
 * What the larger tile costs: with a short contraction a tile is mostly its ends, which nothing covers with one workgroup per CU, where two of 192 x 128
 * on four wavefronts covered each other's. Against those over 2081 calls (sizes as at nh_tiles) these take 0.865 of the time in the mean, but more
 * than a twentieth longer in 81 of the 648 plain calls no deeper than 256 (2 of 645 with SwiGLU), at worst some 130 rows to an expert: 64 experts of
 * 130, 64 x 1408, 13.6 -> 16.6 us, 256 x 1408 20.0 -> 23.3; 128 of 130, 128 x 2048 36.2 -> 40.2; 64 of 190, 256 x 1408 22.8 -> 25.1.
 * In LDS activation rows are 128 bytes with the eight 16-byte pieces xor-swizzled by the row (conflict-free 128-bit operand
 * reads), weight rows in the matrix's own order with xor-swizzled 16-byte units, read through ds_read_b64_tr_b16.
 */
#include "qlmx_gemm.h"
#include <type_traits>

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float    f32x2 __attribute__((ext_vector_type(2)));
typedef float    f32x16 __attribute__((ext_vector_type(16)));
typedef int      i32x2 __attribute__((ext_vector_type(2)));
typedef int      i32x4 __attribute__((ext_vector_type(4)));

#define NH_BK 64
#define NH_BN(WN) (64 * (WN))                    /* columns of a tile: 256 or 128, 64 for each column of wavefronts */
#define NH_A_BYTES(ROWS) (NH_BK * (ROWS) * 2)
#define NH_B_BYTES(WN) (NH_BK * NH_BN(WN) * 2)   /* 32768, 16384 */
#define NH_LDS_BYTES(WN, ROWS) (2 * NH_B_BYTES(WN) + 2 * NH_A_BYTES(ROWS))
#define NH_THREADS 512
#define NH_WSCALE 4096.0f                       /* 16 (the digits come as digit/16) * 2^8 (range shift) */
#define NH_UNSCALE (1.0f / 256.0f)

/* Row plumbing of a launch (the MoE glue folded into the GEMM):
 *   NH_PLAIN    A and C of a problem are its own row-major buffers;
 *   NH_GATHER   k_gather in front (cudalm.cu:2536-2539, 4211): a problem's A field points at its row indices
 *               (const int *), row r of the problem is row idx[r] of `xsrc` (bf16 [tokens, K]), zeros where idx[r] < 0;
 *   NH_SCATTER  k_scatter_gate / k_scatter_add4 behind (cudalm.cu:2541-2545, 2564-2567, 4227): a problem's C field
 *               points at its row indices, out[idx[r], :] = out[idx[r], :] + gate[idx[r]] * y[r, :] (gate NULL: + y[r, :]),
 *               rows with idx[r] < 0 dropped. Within one launch every output row must be named at most once. */
enum { NH_PLAIN = 0, NH_GATHER = 1, NH_SCATTER = 2 };
struct NhArgs { const DevProb *pr; int nprob, ntiles, nfull, piece, rows; const signed char *d; const float *s; int gshift; int K, N;
                const char *xsrc; float *out; const float *gate; };

/* a row of zeros as long as the longest contraction a gathering launch accepts: what a dropped row reads */
#define NH_ZERO_BYTES 32768
static __device__ __align__(16) unsigned char nh_zero_row[NH_ZERO_BYTES];

__device__ __forceinline__ i32x4 nh_rd128(uint32_t addr, int off){
    i32x4 v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "i"(off));
    return v;
}
__device__ __forceinline__ i32x2 nh_tr(uint32_t addr, int off){
    i32x2 v;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "i"(off));
    return v;
}
__device__ __forceinline__ void nh_wr128(uint32_t addr, int off, i32x4 v){
    asm volatile("ds_write_b128 %0, %1 offset:%2" :: "v"(addr), "v"(v), "i"(off) : "memory");
}
/* Global loads are ordinary loads here: this kernel has no load-to-LDS instruction, so the compiler's own wait
 * counts are exact (it waits, with the right count, just before the first use of a loaded value, also when that
 * use is in the next iteration of the loop) and a tile's loads can stay in flight for a step and a half. */
typedef const __attribute__((address_space(1))) int   g_i32;
typedef const __attribute__((address_space(1))) i32x2 g_i32x2;
typedef const __attribute__((address_space(1))) i32x4 g_i32x4;
__device__ __forceinline__ int   nh_gld4(const void *p){ return *(g_i32 *)p; }
__device__ __forceinline__ i32x2 nh_gld8(const void *p){ return *(g_i32x2 *)p; }
__device__ __forceinline__ i32x4 nh_gld16(const void *p){ return *(g_i32x4 *)p; }
template<int NI> struct NhOps { i32x4 a[NI]; i32x2 b[2][2]; };
template<int NI> __device__ __forceinline__ void nh_wait_lds(NhOps<NI> &o){
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(o.b[0][0]), "+v"(o.b[0][1]), "+v"(o.b[1][0]), "+v"(o.b[1][1]) :: "memory");
#pragma unroll
    for(int i = 0; i < NI; i++) asm volatile("" : "+v"(o.a[i]));
}
__device__ __forceinline__ f16x8 nh_pack(const i32x2 lo, const i32x2 hi){
    const i32x4 v = {lo[0], lo[1], hi[0], hi[1]};
    return __builtin_bit_cast(f16x8, v);
}
/* two bf16 in a word -> the same two values as fp16 (exact inside fp16's normal range) */
__device__ __forceinline__ int nh_bf16x2_to_f16x2(int w){
    const float lo = __uint_as_float((uint32_t)w << 16), hi = __uint_as_float((uint32_t)w & 0xFFFF0000u);
    return __builtin_bit_cast(int, __builtin_amdgcn_cvt_pkrtz(lo, hi));
}
__device__ __forceinline__ int nh_pk(float lo, float hi){          /* round to nearest even: v_cvt_pk_f16_f32 */
    f32x2 v = {lo, hi};
    return __builtin_bit_cast(int, __builtin_convertvector(v, f16x2));
}

/* One output tile of WM*NI*32 rows and WN*64 columns on WM x WN wavefronts; the last tile of a problem takes the smallest NI that holds its rows. */
/* The second half of a gate|up problem (DUAL): the other weight matrix, its fp32 output, the SwiGLU output. The
 * tile's LDS columns are then [gate 0-31 | up 0-31 | gate 32-63 | up 32-63 | ...] of the problem's columns from
 * j0 on: a wavefront's first accumulator column holds gate and its second up of the same 32 columns. */
struct NhDual { unsigned long long wq, wg; float *C; unsigned short *act; };

template<int NI, int WN, int IO, bool DUAL = false>
__device__ __forceinline__ void nh_tile(const NhArgs &a, const DevProb &P, const NhDual &Q, int i0, int j0, unsigned char *lds){
    constexpr int WM = 8 / WN, NA = NI * WM / 2, DU = WN;         /* activation pieces and weight units (8 digits) of a thread and step */
    constexpr int BROW = NH_BN(WN) * 2, BB = NH_B_BYTES(WN), AB = NH_A_BYTES(WM * NI * 32);
    typedef std::conditional_t<WN == 4, i32x4, i32x2> digits_t;
    const int rows = P.M < i0 + a.rows ? P.M : i0 + a.rows;               /* a tile of 192 rows may be taken by wavefronts for 256 */
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = (wave / WN) * (NI * 32), wj = (wave % WN) * 64;
    const int fr = lane & 31, hf = lane >> 5;
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds;
    const int steps = a.K / NH_BK, blocks = a.K >> 5;             /* whole steps; blocks of 32 contraction indices */
    const bool half = a.K & 32, tiny = a.K == 32;

    /* ---- activations: position p = h*512 + tid of a buffer is row p/8, stored piece p%8 = ko ^ (row & 7) ---- */
    const char *srcA[NA];
#pragma unroll
    for(int h = 0; h < NA; h++){
        const int p = h * NH_THREADS + tid, r = p >> 3, ko = ((p & 7) ^ (r & 7)) & (tiny ? 3 : 7);
        const int rr = (i0 + r < rows) ? i0 + r : rows - 1;               /* clamp: feeds unstored rows only */
        if(IO == NH_GATHER){
            const int tok = ((const int *)P.A)[rr];
            srcA[h] = (tok >= 0 ? a.xsrc + (size_t)tok * a.K * 2 : (const char *)nh_zero_row) + ko * 16;
        } else srcA[h] = (const char *)P.A + ((size_t)rr * a.K + ko * 8) * 2;
    }
    /* ---- weights: thread = (contraction row kr, columns oc*8*DU .. +8*DU-1): one load of digits and one scale per
     * step. Unit u (8 columns) of row k is stored at u ^ f(k), f(k) = (k & 3) << 2 | (k >> 2 & 3): its upper bits part the
     * four rows of a transposing read, its lower ones the lanes of a write phase, which hold the same unit of
     * different rows; the lanes are dealt to (kr, oc) so that 16 of them hit 16 different units. ---- */
    const int oc = WN == 4 ? (lane & 3) | ((lane >> 2) & 4) : lane & 7;
    const int kr = WN == 4 ? (lane & 12) | (lane >> 5) | ((wave & 1) << 1) | ((wave >> 1) << 4)
                           : ((lane >> 1) & 4) | (lane >> 4) | (wave << 3);
    const bool second = DUAL && (WN == 4 ? oc & 1 : (oc >> 1) & 1);
    const int col0 = DUAL ? (WN == 4 ? (oc >> 1) * 32 : ((oc & 1) + ((oc >> 2) << 1)) * 16) : oc * (8 * DU);
    const size_t e0 = (size_t)(tiny ? kr & 31 : kr) * a.N + j0 + col0;
    const signed char *pw = a.d + (((second ? Q.wq : P.wq) + e0) >> 1);
    const float *ps = a.s + (second ? Q.wg : P.wg) + (e0 >> a.gshift);
    const size_t wblock = (size_t)32 * a.N >> 1, sblock = (size_t)32 * a.N >> a.gshift;
    /* first block of tile t: the tile behind the last whole one ends with the matrix, so that of half a tile the second half counts */
    auto block_of = [&](int t){ const int b = 2 * t < blocks - 2 ? 2 * t : blocks - 2; return (size_t)(b < 0 ? 0 : b); };
    digits_t wd; int wsc; i32x4 av[NA];
    auto load_wd = [&](int t){ if constexpr(WN == 4) wd = nh_gld16(pw + block_of(t) * wblock); else wd = nh_gld8(pw + block_of(t) * wblock); };
    auto load_ws = [&](int t){ wsc = nh_gld4(ps + block_of(t) * sblock); };
    auto load_a = [&](int t, int h){ av[h] = nh_gld16(srcA[h] + block_of(t) * 64); };

    /* ---- LDS addresses. Which of an operand's two buffers a step reads or writes is known at compile time (the
     * loop below is unrolled by two), so the buffer, the row tile, the k16 slice of the weights and the thread's piece
     * all go into the instructions' immediate offsets and the loop computes no LDS address at all. ---- */
    uint32_t ra[4];                                      /* [k16 slice] activations, 128-bit reads */
#pragma unroll
    for(int ks = 0; ks < 4; ks++) ra[ks] = lds_base + 2 * BB + (uint32_t)((wi + fr) * 128 + (((ks * 2 + hf) ^ (fr & 7)) << 4));
    uint32_t rb[2][2];                                   /* [column tile][rows 0-3, 4-7 of eight] weights, transposing reads */
    {
        const int g16 = lane >> 4, s16 = lane & 15, v = s16 >> 2, q = s16 & 3, khalf = g16 >> 1, chalf = g16 & 1;
#pragma unroll
        for(int j = 0; j < 2; j++)
#pragma unroll
            for(int e = 0; e < 2; e++){
                const int k = khalf * 8 + e * 4 + v, col = wj + j * 32 + chalf * 16 + q * 4, f = ((k & 3) << 2) | ((k >> 2) & 3);
                rb[j][e] = lds_base + (uint32_t)(k * BROW + (((col >> 3) ^ f) << 4) + (col & 7) * 2);
            }
    }
    const uint32_t wpa = lds_base + 2 * BB + (uint32_t)tid * 16;
    uint32_t wpb[DU];
#pragma unroll
    for(int u = 0; u < DU; u++) wpb[u] = lds_base + (uint32_t)(kr * BROW + (((oc * DU + u) ^ (((kr & 3) << 2) | ((kr >> 2) & 3))) << 4));

    f32x16 acc[NI][2];
#pragma unroll
    for(int i = 0; i < NI; i++)
#pragma unroll
        for(int j = 0; j < 2; j++) acc[i][j] = (f32x16)(0.0f);

    /* Everything a step does beside its products, cut into small items: per activation piece two conversions (the second
     * writes the piece) and the load of the tile after; per weight unit four pairs and the write; the weights' two loads. */
    constexpr int ITEMS = 3 * NA + 5 * DU + 2;
    i32x4 ah, wh; QxNibs dg; float sc = 0.0f;
    auto item = [&](auto WPARC, int k, int t){           /* tile t goes from the registers to its buffer, tile t+1 into the registers */
        constexpr int WA = decltype(WPARC)::value * AB, WB = decltype(WPARC)::value * BB;
        if(k < 3 * NA){
            const int h = k / 3, q = k % 3;
            if(q == 0){ ah[0] = nh_bf16x2_to_f16x2(av[h][0]); ah[1] = nh_bf16x2_to_f16x2(av[h][1]); }
            else if(q == 1){ ah[2] = nh_bf16x2_to_f16x2(av[h][2]); ah[3] = nh_bf16x2_to_f16x2(av[h][3]); nh_wr128(wpa, WA + h * (NH_THREADS * 16), ah); }
            else load_a(t + 1, h);
        } else if(k < 3 * NA + 5 * DU){
            const int u = (k - 3 * NA) / 5, q = (k - 3 * NA) % 5;
            if(k == 3 * NA) sc = __int_as_float(wsc) * NH_WSCALE;
            if(q == 0) dg = qx_nibs((uint32_t)wd[u]);
            if(q < 4) wh[q] = nh_pk(sc * qx_nib16(dg, 2 * q), sc * qx_nib16(dg, 2 * q + 1));
            else nh_wr128(wpb[u], WB, wh);
        } else if(k == 3 * NA + 5 * DU) load_wd(t + 1);
        else load_ws(t + 1);
    };
    typedef std::integral_constant<int, 0> P0; typedef std::integral_constant<int, 1> P1;

    /* ---- prologue: tile 0 into buffer 0, tile 1 into registers ---- */
    load_wd(0); load_ws(0);
#pragma unroll
    for(int h = 0; h < NA; h++) load_a(0, h);
#pragma unroll
    for(int k = 0; k < ITEMS; k++) item(P0(), k, 0);

    /* Main loop, two steps of 64 per iteration, a step in four slices of 16: the operands of a slice are read from LDS while the slice
     * before multiplies. Tile t+1 goes from the registers into the other buffer in the gaps between the products of tile t,
     * and each register is loaded again (tile t+2) right after its conversion, so a load has a whole step to arrive and needs
     * no second set of registers. One barrier per step stands in the middle of its last slice: the tile's own operands are all
     * read by then and the next tile is complete behind it, so its first operands arrive during the slice's other half.
     * A wavefront issues in order and an MFMA of this shape leaves room for a handful of vector-ALU instructions
     * behind it, so the items are dealt evenly into the gaps before the barrier (fences keep the compiler from gathering them). */
    constexpr int SLOTS = 7 * NI, PER = (4 + 3 * NI) / (2 * NI);       /* operand reads behind each of a slice's first products */
    NhOps<NI> o0, o1;
#define NH_READ(O, KS, RA, RB, Q)                                                                         \
        { if((Q) < 4) O.b[((Q) >> 1) & 1][(Q) & 1] = nh_tr(rb[((Q) >> 1) & 1][(Q) & 1], (RB) + KS * 16 * BROW); \
          else if((Q) < 4 + NI) O.a[((Q) - 4) % NI] = nh_rd128(ra[KS], (RA) + (((Q) - 4) % NI) * 4096); }
#define NH_MFMA(O, M)                                                                                     \
        acc[(M) >> 1][(M) & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, O.a[(M) >> 1]), nh_pack(O.b[(M) & 1][0], O.b[(M) & 1][1]), acc[(M) >> 1][(M) & 1], 0, 0, 0);
    /* products FROM .. TO-1 of slice KS from the operands O, with N reads of slice KS2's operands behind each */
#define NH_SLICE(KS, O, FROM, TO, N, O2, KS2, RA2, RB2)                                                   \
        _Pragma("unroll")                                                                                 \
        for(int m = FROM; m < TO; m++){                                                                   \
            const int slot = KS * NI * 2 + m;                                                             \
            NH_MFMA(O, m)                                                                                 \
            __builtin_amdgcn_sched_barrier(0);                                                            \
            _Pragma("unroll")                                                                             \
            for(int q = (m - FROM) * (N); q < (m - FROM + 1) * (N); q++) NH_READ(O2, KS2, RA2, RB2, q)    \
            if(slot < SLOTS){                                                                             \
                _Pragma("unroll")                                                                         \
                for(int k = slot * ITEMS / SLOTS; k < (slot + 1) * ITEMS / SLOTS; k++) item(std::integral_constant<int, 1 - PAR>(), k, t + 1); \
            }                                                                                             \
            __builtin_amdgcn_sched_barrier(0);                                                            \
        }
    auto step = [&](auto PARC, int t){
        constexpr int PAR = decltype(PARC)::value, RA = PAR * AB, RB = PAR * BB;
        NH_SLICE(0, o0, 0, 2 * NI, PER, o1, 1, RA, RB)
        nh_wait_lds(o1);
        NH_SLICE(1, o1, 0, 2 * NI, PER, o0, 2, RA, RB)
        nh_wait_lds(o0);
        NH_SLICE(2, o0, 0, 2 * NI, PER, o1, 3, RA, RB)
        nh_wait_lds(o1);
        NH_SLICE(3, o1, 0, NI, 0, o0, 0, 0, 0)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     /* this wavefront's writes */
        __builtin_amdgcn_s_barrier();
        NH_SLICE(3, o1, NI, 2 * NI, (4 + 2 * NI - 1) / NI, o0, 0, AB - RA, BB - RB)
        nh_wait_lds(o0);
    };
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for(int n = 0; n < 4 + NI; n++) NH_READ(o0, 0, 0, 0, n)
    nh_wait_lds(o0);
    for(int t = 0; t < steps;){
        step(P0(), t); if(++t >= steps) break;
        step(P1(), t); ++t;
    }
    if(half){                                              /* the last 32: the second half of the tile that ends with the matrix */
        const int odd = steps & 1;
#pragma unroll
        for(int ks = 2; ks < 4; ks++) ra[ks] += odd * AB;
#pragma unroll
        for(int j = 0; j < 2; j++)
#pragma unroll
            for(int e = 0; e < 2; e++) rb[j][e] += odd * BB;
#pragma unroll
        for(int n = 0; n < 4 + NI; n++){ NH_READ(o0, 2, 0, 0, n) NH_READ(o1, 3, 0, 0, n) }
        nh_wait_lds(o0); nh_wait_lds(o1);
#pragma unroll
        for(int m = 0; m < 2 * NI; m++){ NH_MFMA(o0, m) }
#pragma unroll
        for(int m = 0; m < 2 * NI; m++){ NH_MFMA(o1, m) }
    }
#undef NH_READ
#undef NH_MFMA
#undef NH_SLICE

    /* ---- epilogue: undo the range shift, then the lane holds column lane%32 of each 32x32 tile, four-row band lane/32 ---- */
#pragma unroll
    for(int i = 0; i < NI; i++)
#pragma unroll
        for(int j = 0; j < 2; j++) acc[i][j] = acc[i][j] * NH_UNSCALE;
    const int row = i0 + wi + hf * 4;
    if(DUAL){
        const size_t o = (size_t)(i0 + wi) * a.N + (j0 + (wj >> 1));
        __syncthreads();                                   /* the buffers become the wavefronts' strips */
        qx_store_swiglu<NI, true>(acc, (float *)lds + wave * QX_STRIP_FLOATS, P.C ? P.C + o : nullptr, Q.C + o, Q.act + o, rows - (i0 + wi), (size_t)a.N);
    } else if(IO == NH_SCATTER) qx_scatter_tiles<NI>(acc, (const int *)P.C, a.gate, a.out, row, rows, (size_t)a.N, j0 + wj + fr);
    else qx_store_tiles<NI, 2>(acc, P.C + (size_t)row * a.N + (j0 + wj + fr), row, i0 + wi, rows, (size_t)a.N, false);
}

/* the smallest NI that holds a tile's rows: 64 rows for each with four columns of wavefronts, 128 with two; a last tile
 * of 128 columns where the launch's tiles have 256 is one of two columns */
template<int WN, int BM, int IO, bool DUAL = false>
__device__ __forceinline__ void nh_rows(const NhArgs &a, const DevProb &P, const NhDual &Q, int i0, int j0, int left, unsigned char *lds){
    if(WN == 4 && j0 + NH_BN(4) / (DUAL ? 2 : 1) <= a.N){
        if(left > 192)      nh_tile<4, 4, IO, DUAL>(a, P, Q, i0, j0, lds);
        else if(left > 128) nh_tile<3, 4, IO, DUAL>(a, P, Q, i0, j0, lds);
        else if(left > 64)  nh_tile<2, 4, IO, DUAL>(a, P, Q, i0, j0, lds);
        else                nh_tile<1, 4, IO, DUAL>(a, P, Q, i0, j0, lds);
    } else if(BM == 256 && left > 128) nh_tile<2, 2, IO, DUAL>(a, P, Q, i0, j0, lds);
    else                               nh_tile<1, 2, IO, DUAL>(a, P, Q, i0, j0, lds);
}

template<int IO, int WN, int BM>
__global__ void __launch_bounds__(NH_THREADS, BM == 128 ? 4 : 2) k_gemm_nn_h(NhArgs a){
    __shared__ __attribute__((aligned(16))) unsigned char lds[NH_LDS_BYTES(WN, BM)];
    const int t = qx_lpt_tile(blockIdx.x, a.nfull, a.ntiles, a.piece);
    if(t >= a.ntiles) return;
    const DevProb P = a.pr[qx_find_problem(a.pr, a.nprob, t)];
    const int lt = t - P.tile0;
    const int ti = lt / P.tiles_n, tj = lt - ti * P.tiles_n;
    const int i0 = ti * a.rows, j0 = tj * NH_BN(WN), left = P.M - i0 < a.rows ? P.M - i0 : a.rows;
    const NhDual none = {0, 0, nullptr, nullptr};
    nh_rows<WN, BM, IO>(a, P, none, i0, j0, left, lds);
}

/* gate|up problems with the SwiGLU in the epilogue (mg_ab w1, mg_ab w3, e_swig; cudalm.cu:4211-4215): tiles of up to 256
 * rows x 128 columns of both matrices; the table entry after the problem's holds the second matrix, the up output
 * and the bf16 SwiGLU output. The fp32 gate / up outputs are skipped when the problem's C is NULL. */
template<int IO, int WN, int BM>
__global__ void __launch_bounds__(NH_THREADS, BM == 128 ? 4 : 2) k_gemm_nn_h_swiglu(NhArgs a){
    __shared__ __attribute__((aligned(16))) unsigned char lds[NH_LDS_BYTES(WN, BM)];
    const int t = qx_lpt_tile(blockIdx.x, a.nfull, a.ntiles, a.piece);
    if(t >= a.ntiles) return;
    const int pi = qx_find_problem(a.pr, a.nprob, t);
    const DevProb P = a.pr[pi];
    const DevProb P2 = a.pr[pi + 1];
    const NhDual Q = {P2.wq, P2.wg, P2.C, (unsigned short *)P2.B};
    const int lt = t - P.tile0;
    const int ti = lt / P.tiles_n, tj = lt - ti * P.tiles_n;
    const int i0 = ti * a.rows, j0 = tj * (NH_BN(WN) / 2), left = P.M - i0 < a.rows ? P.M - i0 : a.rows;
    nh_rows<WN, BM, IO, true>(a, P, Q, i0, j0, left, lds);
}

/* The loads of the compute units of an XCD while tiles are dealt to them, longest first, each to the least loaded one: groups of
 * units with the same load. */
#define NH_UNITS 48
struct NhLoads { int n; float load[NH_UNITS]; int units[NH_UNITS]; };
static void nh_deal(NhLoads &d, long long tiles, float cost){
    int total = 0;
    for(int k = 0; k < d.n; k++) total += d.units[k];
    if(tiles > 8LL * total){                               /* all but the last few rounds at once */
        const long long r = tiles / total - 4;
        for(int k = 0; k < d.n; k++) d.load[k] += r * cost;
        tiles -= r * total;
    }
    while(tiles > 0){
        int k = 0;
        for(int j = 1; j < d.n; j++) if(d.load[j] < d.load[k]) k = j;
        const int take = tiles < d.units[k] ? (int)tiles : d.units[k];
        const float l = d.load[k] + cost;
        tiles -= take; d.units[k] -= take;
        if(!d.units[k]){ d.n--; d.load[k] = d.load[d.n]; d.units[k] = d.units[d.n]; }
        int j = 0;
        while(j < d.n && d.load[j] != l) j++;
        if(j == d.n){ d.load[j] = l; d.units[j] = 0; d.n++; }
        d.units[j] += take;
    }
}
/* The tile of a launch: the shape whose tiles, dealt out as the launch deals them, end first. Costs in units of a whole 256 x 256 tile, by
 * height in 64 rows, from launches of whole rounds (256 compute units, contractions of 512 to 2048: 40, 33, 28 and 20 us for 256, 192, 128 and
 * 64 rows of 256 columns and 1024 deep, 24 and 18 for 256 and 128 rows of 128): a CU holds one such tile, or two of 128 x 128, which
 * share it (28 us for both) and overlap one's start and end with the other's loop, of use where the contraction is short: up to 384 such a tile
 * counts 0.29 instead of 0.36 (slower than the best of the five shapes by, in the mean over 3727 calls, with 0.29 / with 0.36: contractions of 256
 * 1.0 / 1.3 %, 384 0.9 / 1.0, 512 1.0 / 0.8, 640 1.2 / 0.8, 1024 1.2 / 0.6). Wide tiles do the
 * most products per weight and activation prepared and win wherever there are rounds enough; the others where the count is unlucky. us, chosen
 * <- 256 x 256 always: 12 experts of 530 rows, 640 x 640 gate|up 21 <- 24; 8 of 256, 768 x 2048 plain 16 <- 21 (256 x 128); 100 of
 * 120, 512 x 768 plain 24 <- 28 (128 x 128). Over those 3727 calls (4 to 128 experts of 70 to 400 rows, 64 to 1024 deep, 256 to 2048 wide, plain and
 * SwiGLU) the choice is within 0.9 % of the best of the five in the mean and more than 5 % behind it in 166. */
struct NhTiles { int rows, columns; };
static NhTiles nh_tiles(const qlmx_gemm_prob *probs, int nprob, int K, int columns){
    static const float wide[5] = {0.0f, 0.50f, 0.65f, 0.82f, 1.0f}, narrow[5] = {0.0f, 0.45f, 0.45f, 0.67f, 0.67f}, pair[3] = {0.0f, 0.36f, 0.36f}, pair_short[3] = {0.0f, 0.29f, 0.29f};
    NhTiles best = {256, 128};
    float least = 0.0f;
    long long full[3] = {0, 0, 0}, high[3][5] = {};                    /* tile rows, for tiles of 256, 192 and 128: whole ones, last ones by height */
    for(int i = 0; i < nprob; i++){
        const int m = probs[i].M, f[3] = {m / 256, m / 192, m / 128};
        for(int r = 0; r < 3; r++){ full[r] += f[r]; high[r][(m - f[r] * (256 - 64 * r) + 63) / 64]++; }
    }
    const int cus = qlmx_cu_count() / 8, units = cus < 1 ? 1 : cus < NH_UNITS ? cus : NH_UNITS - 1;
    for(int rows = 256; rows >= 128; rows -= 64)
        for(int cols = 256; cols >= 128; cols -= 128){
            if(cols > columns || (cols == 128 && rows == 192)) continue;
            const bool paired = rows == 128 && cols == 128;
            const float *thin = !paired ? narrow : K > 384 ? pair : pair_short;
            const int g_wide = cols == 256 ? columns / 256 : 0, g_thin = cols == 256 ? columns % 256 / 128 : columns / 128;
            const int r = (256 - rows) / 64;
            NhLoads ld; ld.n = 1; ld.load[0] = paired ? 0.11f : 0.0f; ld.units[0] = units;      /* a pair's last tile runs alone */
            nh_deal(ld, (full[r] * g_wide + 7) / 8, wide[rows / 64]); nh_deal(ld, (full[r] * g_thin + 7) / 8, thin[rows / 64]);
            for(int l = rows / 64; l > 0; l--){ nh_deal(ld, (high[r][l] * g_wide + 7) / 8, wide[l]); nh_deal(ld, (high[r][l] * g_thin + 7) / 8, thin[l]); }
            float t = 0.0f;
            for(int k = 0; k < ld.n; k++) if(ld.load[k] > t) t = ld.load[k];
            if(least == 0.0f || t < least){ least = t; best.rows = rows; best.columns = cols; }
        }
    return best;
}
/* How many tiles of a row of last tiles stay on one XCD: all of them (they read the same activations) where there are rows enough to go round;
 * fewer rows than that are dealt tile by tile, or a few XCDs get two rows and the others one: 3 experts of 700 rows, 2048 x 1408 gate|up 72 -> 38 us. */
static int nh_piece(const ProbUpload &up, int g){
    return (up.ntiles - up.nfull) / g >= 32 ? g : 1;
}
/* bf16 activations only; N % 128 == 0, K % 32 == 0, group a power of two >= 32 (checked by the caller).
 * io = NH_GATHER: xsrc is the bf16 token matrix and the problems' A fields are row-index lists;
 * io = NH_SCATTER: out (and gate, may be NULL) is the destination and the problems' C fields are row-index lists. */
int qlmx_gemm_nn_h_launch(const signed char *d, const float *s, int group, const qlmx_gemm_prob *probs, int nprob,
                          int K, int N, int io, const void *xsrc, float *out, const float *gate, hipStream_t st){
    QLMX_REQUIRE(io != NH_GATHER || (size_t)K * 2 <= NH_ZERO_BYTES, "grouped gemm nn with gather: K=%d exceeds %d", K, NH_ZERO_BYTES / 2);
    if(qlmx_small_rows(probs, nprob, GEMM_NN, K, N, 1, group)) return qlmx_gemm_nn_small_launch(d, s, group, probs, nprob, K, N, io, xsrc, out, gate, st);
    const NhTiles tl = nh_tiles(probs, nprob, K, N);
    const int bn = tl.columns;
    ProbUpload up; int slot;
    const RowBytes rb = {io == NH_GATHER ? sizeof(int) : (size_t)K * 2, io == NH_SCATTER ? sizeof(int) : (size_t)N * 4, 0, 0, 0};
    int rc = qlmx_upload_problems_split(probs, nullptr, nprob, GEMM_NN, K, N, tl.rows, bn, &rb, st, &up, &slot); if(rc) return rc;
    if(up.ntiles == 0) return QLMX_OK;
    NhArgs a; a.pr = up.dev; a.nprob = up.nprob; a.ntiles = up.ntiles; a.nfull = up.nfull; a.rows = tl.rows; a.piece = nh_piece(up, (N + bn - 1) / bn); a.d = d; a.s = s; a.K = K; a.N = N;
    a.xsrc = (const char *)xsrc; a.out = out; a.gate = gate;
    a.gshift = 0; while((1 << a.gshift) < group) a.gshift++;
    const int grid = qx_lpt_grid(up.nfull, up.ntiles, a.piece);
#define NH_LAUNCH(KERNEL, IO) do{ if(tl.columns == 256)            hipLaunchKernelGGL((KERNEL<IO, 4, 256>), dim3(grid), dim3(NH_THREADS), 0, st, a); \
                                  else if(tl.rows == 128) hipLaunchKernelGGL((KERNEL<IO, 2, 128>), dim3(grid), dim3(NH_THREADS), 0, st, a); \
                                  else                    hipLaunchKernelGGL((KERNEL<IO, 2, 256>), dim3(grid), dim3(NH_THREADS), 0, st, a); }while(0)
    if(io == NH_GATHER)       NH_LAUNCH(k_gemm_nn_h, NH_GATHER);
    else if(io == NH_SCATTER) NH_LAUNCH(k_gemm_nn_h, NH_SCATTER);
    else                      NH_LAUNCH(k_gemm_nn_h, NH_PLAIN);
    QLMX_LAUNCH_CHECK("grouped gemm nn (fp16 matrix core) launch");
    return qlmx_upload_done(slot, st);
}

/* gate|up pairs with the SwiGLU in the epilogue: N % 64 == 0, K % 32 == 0, group a power of two >= 64 (a tile's 64
 * columns of a matrix share a scale per contraction row). xsrc != NULL: the gate problems' A fields are row-index
 * lists into the bf16 token matrix xsrc (NH_GATHER). Problems whose gate C is NULL store the bf16 output only. */
int qlmx_gemm_nn_h_swiglu_launch(const signed char *d, const float *s, int group, const qlmx_gemm_prob *gate, const qlmx_gemm_prob *up_,
                                 int nprob, int K, int N, const void *xsrc, hipStream_t st){
    QLMX_REQUIRE(!xsrc || (size_t)K * 2 <= NH_ZERO_BYTES, "grouped gemm nn + swiglu with gather: K=%d exceeds %d", K, NH_ZERO_BYTES / 2);
    if(N % 128 == 0 && qlmx_small_rows(gate, nprob, GEMM_NN, K, N, 1, group)) return qlmx_gemm_nn_small_swiglu_launch(d, s, group, gate, up_, nprob, K, N, xsrc, st);
    const NhTiles tl = nh_tiles(gate, nprob, K, 2 * N);
    const int bn = tl.columns / 2;
    ProbUpload up; int slot;
    const RowBytes rb = {xsrc ? sizeof(int) : (size_t)K * 2, (size_t)N * 4, 0, (size_t)N * 2, (size_t)N * 4};
    int rc = qlmx_upload_problems_split(gate, up_, nprob, GEMM_NN, K, N, tl.rows, bn, &rb, st, &up, &slot); if(rc) return rc;
    if(up.ntiles == 0) return QLMX_OK;
    NhArgs a; a.pr = up.dev; a.nprob = up.nprob; a.ntiles = up.ntiles; a.nfull = up.nfull; a.rows = tl.rows; a.piece = nh_piece(up, (N + bn - 1) / bn); a.d = d; a.s = s; a.K = K; a.N = N;
    a.xsrc = (const char *)xsrc; a.out = nullptr; a.gate = nullptr;
    a.gshift = 0; while((1 << a.gshift) < group) a.gshift++;
    const int grid = qx_lpt_grid(up.nfull, up.ntiles, a.piece);
    if(xsrc) NH_LAUNCH(k_gemm_nn_h_swiglu, NH_GATHER);
    else     NH_LAUNCH(k_gemm_nn_h_swiglu, NH_PLAIN);
    QLMX_LAUNCH_CHECK("grouped gemm nn + swiglu (fp16 matrix core) launch");
    return qlmx_upload_done(slot, st);
}
