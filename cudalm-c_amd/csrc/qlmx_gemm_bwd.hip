/* qlmx_gemm_bwd.hip -- the input gradient and the weight gradient of one backward flush as ONE kernel launch.
 *
 * moe_backward flushes twice (cudalm.cu:4333-4335 and 4362-4366); each flush holds a weight gradient (mg_atb) and
 * an input gradient (mg_abt_b) that read the same operands and write different outputs. Launched one after the
 * other, each leaves compute units idle while its last round of tiles drains (a third of them at the sizes of a
 * training step), and two streams side by side pay a wait between hardware queues at the fork and at the join.
 * Here the two are one grid: the first workgroups are the tiles of the one, the rest the tiles of the other,
 * each running the code of its own kernel (qlmx_gemm_tn_body.h or, for few rows, qlmx_gemm_tn_small_body.h; qlmx_gemm_nt_body.h), so the second kind's
 * tiles take the compute units as the first kind's leave them. The results are bit-identical to the separate
 * launches: every tile does the same arithmetic in the same order.
 *
 * Use: qlmx_pair_begin(stream); the calls of the flush; qlmx_pair_end(stream). Between the two, the library
 * holds back at most one input-gradient launch and one weight-gradient launch of the kinds named below and
 * qlmx_pair_end issues them together. Everything else keeps its order on the stream: a second launch of a kind
 * already held, and any other library call, first issues what is held. */
#include "qlmx_gemm_tn_body.h"
#include "qlmx_gemm_nt_body.h"
#include "qlmx_gemm_tn_small_body.h"
#include <stdlib.h>

#define BWD_LDS_BYTES ((int)(Nt3Shape<128, 4>::LDS_BYTES) > TN3_LDS_BYTES ? (int)(Nt3Shape<128, 4>::LDS_BYTES) : TN3_LDS_BYTES)

/* workgroups [0, first) belong to the one kernel, the rest to the other; `first` is a multiple of 8, so that a
 * workgroup's index within its own kind keeps the XCD the hardware gave it (index % 8) */
template<bool TN_FIRST>
__global__ void __launch_bounds__(256, 2) k_gemm_bwd_pair(Tn3Args ta, Nt3Args na, unsigned first){
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const unsigned b = blockIdx.x;
    if((b < first) == TN_FIRST) tn3_block(ta, TN_FIRST ? b : b - first, lds);
    else                        nt3_block<128, 4>(na, TN_FIRST ? b - first : b);
}

/* The same with the input gradient of few rows, on tiles of 32 rows: 77 KB of LDS, so that two workgroups of either kind are on a CU. Both launches are
 * short and neither fills the chip: a training pass, us, launched apart / weight gradient first / input gradient first: 1000 tokens of 8 experts, 512 x 1536, 125.5 / 119.9 / 112.5,
 * 500 of 768 x 1024 106 / 101 / 99, 600 x 2 of 16, 1024 x 2048, 216 / 209 / 206, 1000 of 64, 1024 x 1408, 357 / - / 339. */
#define BWD_FEW_LDS_BYTES ((int)(Nt3Shape<128, 4>::LDS_BYTES) > SM_TLDS(2) ? (int)(Nt3Shape<128, 4>::LDS_BYTES) : SM_TLDS(2))
template<int IO>
__global__ void __launch_bounds__(256, 2) k_gemm_bwd_pair_few(SmArgs ta, Nt3Args na, unsigned first){
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const unsigned b = blockIdx.x;
    if(b < first) sm_tn_block<2, IO>(ta, (int)b, (int)first, lds);
    else          nt3_block<128, 4>(na, b - first);
}

struct PairState {
    bool open; hipStream_t st;
    bool has_tn, has_nt, few;                              /* few: the input gradient held is `small` */
    Tn3Args tn; int tn_grid, tn_slot;
    SmArgs small; int rt, io;                              /* rt: its height on its own, 16 or 32 rows */
    Nt3Args nt; int nt_grid, nt_slot; bool nt_units;
};
static PairState g_pair = {};
static int g_pair_tn_first = -1;

/* launch of a held input gradient alone: the kernels live in qlmx_gemm_tn_lds.hip and qlmx_gemm_small.hip, the weight gradient's in
 * qlmx_gemm_nt_lds.hip */
int qlmx_gemm_tn_lds_issue(const Tn3Args &a, int grid, int slot, hipStream_t st);
int qlmx_gemm_nt_lds_issue(const Nt3Args &a, int grid, int slot, bool units, hipStream_t st);
int qlmx_gemm_tn_small_issue(const SmArgs &a, int rt, int io, int slot, hipStream_t st);

template<int IO> static int launch_few(PairState &p){
    static bool attr_set = false;
    if(!attr_set){
        QLMX_HIP(hipFuncSetAttribute((const void *)k_gemm_bwd_pair_few<IO>, hipFuncAttributeMaxDynamicSharedMemorySize, BWD_FEW_LDS_BYTES), "backward pair (few rows) LDS size");
        attr_set = true;
    }
    const unsigned first = ((unsigned)p.small.ntiles + 7u) & ~7u;
    hipLaunchKernelGGL(k_gemm_bwd_pair_few<IO>, dim3(first + (unsigned)p.nt_grid), dim3(256), BWD_FEW_LDS_BYTES, p.st, p.small, p.nt, first);
    return QLMX_OK;
}
/* issues what is held, in one launch when both kinds are */
int qlmx_pair_flush(void){
    PairState &p = g_pair;
    if(!p.has_tn && !p.has_nt) return QLMX_OK;
    const bool tn = p.has_tn, nt = p.has_nt;
    p.has_tn = p.has_nt = false;
    if(tn && !nt) return p.few ? qlmx_gemm_tn_small_issue(p.small, p.rt, p.io, p.tn_slot, p.st) : qlmx_gemm_tn_lds_issue(p.tn, p.tn_grid, p.tn_slot, p.st);
    if(nt && !tn) return qlmx_gemm_nt_lds_issue(p.nt, p.nt_grid, p.nt_slot, p.nt_units, p.st);
    if(p.few){
        const int rc = p.io == SM_SCATTER ? launch_few<SM_SCATTER>(p) : p.io == SM_SWIGLU_BWD ? launch_few<SM_SWIGLU_BWD>(p) : launch_few<SM_PLAIN>(p);
        if(rc) return rc;
        QLMX_LAUNCH_CHECK("backward pair launch");
        const int done = qlmx_upload_done(p.tn_slot, p.st); if(done) return done;
        return p.nt_units ? qlmx_unit_done(p.nt_slot, p.st) : qlmx_upload_done(p.nt_slot, p.st);
    }
    static bool attr_set = false;
    if(!attr_set){
        QLMX_HIP(hipFuncSetAttribute((const void *)k_gemm_bwd_pair<true>, hipFuncAttributeMaxDynamicSharedMemorySize, BWD_LDS_BYTES), "backward pair LDS size");
        QLMX_HIP(hipFuncSetAttribute((const void *)k_gemm_bwd_pair<false>, hipFuncAttributeMaxDynamicSharedMemorySize, BWD_LDS_BYTES), "backward pair LDS size");
        attr_set = true;
    }
    if(g_pair_tn_first < 0){ const char *e = getenv("QLMX_PAIR_ORDER"); g_pair_tn_first = (e && e[0] == 'n') ? 0 : 1; }
    if(g_pair_tn_first){
        const unsigned first = ((unsigned)p.tn_grid + 7u) & ~7u;
        hipLaunchKernelGGL(k_gemm_bwd_pair<true>, dim3(first + (unsigned)p.nt_grid), dim3(256), BWD_LDS_BYTES, p.st, p.tn, p.nt, first);
    } else {
        const unsigned first = ((unsigned)p.nt_grid + 7u) & ~7u;
        hipLaunchKernelGGL(k_gemm_bwd_pair<false>, dim3(first + (unsigned)p.tn_grid), dim3(256), BWD_LDS_BYTES, p.st, p.tn, p.nt, first);
    }
    QLMX_LAUNCH_CHECK("backward pair launch");
    int rc = qlmx_upload_done(p.tn_slot, p.st); if(rc) return rc;
    return p.nt_units ? qlmx_unit_done(p.nt_slot, p.st) : qlmx_upload_done(p.nt_slot, p.st);
}

/* The launch functions of the two kernels call these with a launch ready to go: *held = true when it is kept
 * for qlmx_pair_end (the caller returns), false when the caller has to launch it. A launch of a kind already
 * held first issues what is held. */
int qlmx_pair_hold_tn(const Tn3Args &a, int grid, int slot, hipStream_t st, bool *held){
    PairState &p = g_pair;
    *held = false;
    if(!p.open || st != p.st) return QLMX_OK;
    if(p.has_tn){ const int rc = qlmx_pair_flush(); if(rc) return rc; }
    p.tn = a; p.tn_grid = grid; p.tn_slot = slot; p.has_tn = true; p.few = false; *held = true;
    return QLMX_OK;
}
/* a table of tiles of 16 rows (rt 1) is one of 32 too: no problem has more than 16 */
int qlmx_pair_hold_tn_few(const SmArgs &a, int rt, int io, int slot, hipStream_t st, bool *held){
    PairState &p = g_pair;
    *held = false;
    if(!p.open || st != p.st) return QLMX_OK;
    if(p.has_tn){ const int rc = qlmx_pair_flush(); if(rc) return rc; }
    p.small = a; p.rt = rt; p.io = io; p.tn_slot = slot; p.has_tn = true; p.few = true; *held = true;
    return QLMX_OK;
}
bool qlmx_pair_open(hipStream_t st){ return g_pair.open && g_pair.st == st; }
/* a weight gradient is held that has no input gradient yet */
bool qlmx_pair_waits(hipStream_t st){ return qlmx_pair_open(st) && g_pair.has_nt && !g_pair.has_tn; }
int qlmx_pair_hold_nt(const Nt3Args &a, int grid, int slot, bool units, hipStream_t st, bool *held){
    PairState &p = g_pair;
    *held = false;
    if(!p.open || st != p.st) return QLMX_OK;
    if(p.has_nt){ const int rc = qlmx_pair_flush(); if(rc) return rc; }
    p.nt = a; p.nt_grid = grid; p.nt_slot = slot; p.nt_units = units; p.has_nt = true; *held = true;
    return QLMX_OK;
}

extern "C" int qlmx_pair_begin(void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(!g_pair.open, "qlmx_pair_begin: a pair is already open (one at a time, like every call of the library from one thread)");
    g_pair.open = true; g_pair.st = (hipStream_t)stream; g_pair.has_tn = g_pair.has_nt = false;
    return QLMX_OK;
}
extern "C" int qlmx_pair_end(void *stream){
    QLMX_REQUIRE(g_pair.open, "qlmx_pair_end: no pair is open");
    QLMX_REQUIRE((hipStream_t)stream == g_pair.st, "qlmx_pair_end: not the stream of qlmx_pair_begin");
    const int rc = qlmx_pair_flush();
    g_pair.open = false;
    return rc;
}
