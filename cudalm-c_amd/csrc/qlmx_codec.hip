/* qlmx_codec.hip -- encode, render and scale servo of the nibble-packed 4-bit weight format.
 *
 * Replaces k_qlm_encode (qlm.cuh:136-167), k_qlm_render (qlm.cuh:170-178) and k_qlm_servo
 * (qlm.cuh:404-441); CPU twins cpu_kern.h:777-796, 857-873. Format: element i of d/r lives at
 * qi0+i; packed digits sit two per byte, even element in the low nibble, two's complement; one
 * fp32 scale per group of `group` consecutive elements of a span, the last group may be short.
 *
 * As in the optimizer kernel a group belongs to a team of W lanes: a DPP row of 16, or half of one for groups
 * of 64. With groups of 8 W, full and 8-element aligned, each lane handles 8 consecutive elements through
 * 128/64/32-bit accesses; everything else goes pair-per-lane so that a lane always owns whole bytes of packed digits
 * (which took 535 us for encode + servo + render of 64 M weights in groups of 64, against 152 in groups of 128).
 * All three are streaming kernels bound by HBM (encode: read 4 B, write 1.5 B per weight; render:
 * read 0.5 B, write 4 B; servo: read 1.5 B, write at most 1.5 B).
 */
#include "qlmx_dev.h"

struct GroupLoc { int n; uint64_t pof, qi0; };
__device__ __forceinline__ GroupLoc group_loc(const qlmx_span *sp, int si, int gi, int group){
    const qlmx_span S = sp[si];
    const uint64_t j0 = (uint64_t)(gi - S.gi0) * (uint64_t)group;
    const uint64_t left = S.n - j0;
    GroupLoc L;
    L.n = (int)((uint64_t)group < left ? (uint64_t)group : left);
    L.pof = S.pof + j0; L.qi0 = S.qi0 + j0;
    return L;
}
__device__ __forceinline__ int load_digit(const signed char *d, uint64_t qi, int packed){
    if(!packed) return (int)d[qi];
    const unsigned b = (unsigned char)d[qi >> 1];
    const int v = (qi & 1ULL) ? (int)(b >> 4) : (int)(b & 15u);
    return v >= 8 ? v - 16 : v;
}
/* digit and residual of t = value/scale (qlm.cuh:160-162, 434-436) */
__device__ __forceinline__ void quantize(float t, int dmax, int &dd, int &rr){
    dd = qx_clamp((int)rintf(t), -dmax, dmax);
    rr = qx_clamp((int)rintf((t - (float)dd) * 128.0f), -64, 64);
}

template<int W>
__global__ void __launch_bounds__(256) k_qlmx_encode(const float *P, signed char *d, signed char *r, float *s,
                                                     const qlmx_span *sp, int nspan, int group, int dmax,
                                                     int packed, int ngrp, int vec_ok){
    const int tl = threadIdx.x & (W - 1);
    const int gi = (int)((blockIdx.x * 256u + threadIdx.x) / W);
    const int si = qx_span_of_teams<64 / W>(sp, nspan, __builtin_amdgcn_readfirstlane(gi), (threadIdx.x & 63) / W);
    if(gi >= ngrp) return;
    const GroupLoc L = group_loc(sp, si, gi, group);
    const bool fast = vec_ok && group == 8 * W && packed && L.n == 8 * W && ((L.pof | L.qi0) & 7ULL) == 0;
    if(fast){
        const uint64_t e0 = (uint64_t)tl * 8;
        const float4 p0 = *(const float4 *)(P + L.pof + e0), p1 = *(const float4 *)(P + L.pof + e0 + 4);
        const float pv[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
        float amax = 0.0f;
#pragma unroll
        for(int k = 0; k < 8; k++) amax = fmaxf(amax, fabsf(pv[k]));
        amax = qx_team_max<W>(amax);
        float sg = amax / (float)dmax; if(!(sg > 0.0f)) sg = 1e-8f;
        if(tl == 0) s[gi] = sg;
        const GroupDiv div = qx_mkdiv(sg);                 /* 151 M weights, encode + servo + render: 333 -> 322 us */
        uint32_t dw = 0, r0 = 0, r1 = 0;
#pragma unroll
        for(int k = 0; k < 8; k++){
            int dd, rr; quantize(qx_gdiv(pv[k], div), dmax, dd, rr);
            dw |= ((uint32_t)dd & 15u) << (4 * k);
            if(k < 4) r0 |= ((uint32_t)rr & 0xFFu) << (8 * k); else r1 |= ((uint32_t)rr & 0xFFu) << (8 * (k - 4));
        }
        *(uint32_t *)(d + ((L.qi0 + e0) >> 1)) = dw;
        *(uint2 *)(r + L.qi0 + e0) = make_uint2(r0, r1);
    } else {
        float amax = 0.0f;
        for(int j = tl; j < L.n; j += W) amax = fmaxf(amax, fabsf(P[L.pof + j]));
        amax = qx_team_max<W>(amax);
        float sg = amax / (float)dmax; if(!(sg > 0.0f)) sg = 1e-8f;
        if(tl == 0) s[gi] = sg;
        for(int jb = 2 * tl; jb < L.n; jb += 2 * W){
            int dn[2] = {0, 0};
#pragma unroll
            for(int h = 0; h < 2; h++){
                const int j = jb + h;
                if(j < L.n){
                    int dd, rr; quantize(P[L.pof + j] / sg, dmax, dd, rr);
                    dn[h] = dd; r[L.qi0 + j] = (signed char)rr;
                    if(!packed) d[L.qi0 + j] = (signed char)dd;
                }
            }
            if(packed) d[(L.qi0 + jb) >> 1] = (signed char)(((dn[1] & 15) << 4) | (dn[0] & 15));
        }
    }
}

template<int W>
__global__ void __launch_bounds__(256) k_qlmx_render(float *P, const signed char *d, const float *s,
                                                     const qlmx_span *sp, int nspan, int group, int packed,
                                                     int gi_base, int ng, int vec_ok){
    const int tl = threadIdx.x & (W - 1);
    const int w = (int)((blockIdx.x * 256u + threadIdx.x) / W), gi = gi_base + w;
    const int si = qx_span_of_teams<64 / W>(sp, nspan, __builtin_amdgcn_readfirstlane(gi), (threadIdx.x & 63) / W);
    if(w >= ng) return;
    const GroupLoc L = group_loc(sp, si, gi, group);
    const float sg = s[gi];
    const bool fast = vec_ok && group == 8 * W && packed && L.n == 8 * W && ((L.pof | L.qi0) & 7ULL) == 0;
    if(fast){
        /* a lane renders elements 4*tl .. +3 and the same half a group further on: each of the two stores of
         * a team covers 16 W contiguous bytes of P, written past the caches */
        typedef float f4 __attribute__((ext_vector_type(4)));
        const uint64_t e0 = (uint64_t)tl * 4;
        const unsigned short *dh = (const unsigned short *)(d + (L.qi0 >> 1));
        const uint32_t w0 = dh[tl], w1 = dh[W + tl];
        f4 o0, o1;
        o0.x = sg * (float)qx_nib(w0, 0); o0.y = sg * (float)qx_nib(w0, 1);
        o0.z = sg * (float)qx_nib(w0, 2); o0.w = sg * (float)qx_nib(w0, 3);
        o1.x = sg * (float)qx_nib(w1, 0); o1.y = sg * (float)qx_nib(w1, 1);
        o1.z = sg * (float)qx_nib(w1, 2); o1.w = sg * (float)qx_nib(w1, 3);
        __builtin_nontemporal_store(o0, (f4 *)(P + L.pof + e0));
        __builtin_nontemporal_store(o1, (f4 *)(P + L.pof + e0 + 4 * W));
    } else {
        for(int j = tl; j < L.n; j += W) P[L.pof + j] = sg * (float)load_digit(d, L.qi0 + j, packed);
    }
}

/* the servo's new scale for a group with `railed` of n digits at their bound; the old one where it stays */
__device__ __forceinline__ float servo_scale(float sg, int railed, int n, float f_hi, float f_lo){
    const float f = (float)railed / (float)n;
    return f > f_hi ? sg * 1.09051f : f < f_lo ? sg / 1.09051f : sg;          /* 2^(1/8) */
}
/* any group: a pair of elements per lane and step */
template<int W>
__device__ void servo_pairs(const GroupLoc &L, int gi, int tl, signed char *d, signed char *r, float *s, int dmax, float f_hi, float f_lo, int packed){
    int railed = 0;
    for(int jb = 2 * tl; jb < L.n; jb += 2 * W)
        for(int h = 0; h < 2; h++){
            const int j = jb + h;
            if(j < L.n){ const int dd = load_digit(d, L.qi0 + j, packed); railed += (dd == dmax) | (dd == -dmax); }
        }
    railed = qx_team_sum<W>(railed);
    const float f = (float)railed / (float)L.n, sg = s[gi];
    if(!(f > f_hi || f < f_lo)) return;             /* uniform over the team */
    const float sn = servo_scale(sg, railed, L.n, f_hi, f_lo), conv = sg / sn;
    if(tl == 0) s[gi] = sn;
    for(int jb = 2 * tl; jb < L.n; jb += 2 * W){
        int dn[2] = {0, 0};
#pragma unroll
        for(int h = 0; h < 2; h++){
            const int j = jb + h;
            if(j < L.n){
                const uint64_t qi = L.qi0 + j;
                const float t = ((float)load_digit(d, qi, packed) + (float)r[qi] * (1.0f / 128.0f)) * conv;
                int dd, rr; quantize(t, dmax, dd, rr);
                dn[h] = dd; r[qi] = (signed char)rr;
                if(!packed) d[qi] = (signed char)dd;
            }
        }
        if(packed) d[(L.qi0 + jb) >> 1] = (signed char)(((dn[1] & 15) << 4) | (dn[0] & 15));
    }
}
/* adds to n how many of w's eight nibbles equal those of `up` or of `down` (which differ) */
__device__ __forceinline__ int nibbles_equal(uint32_t w, uint32_t up, uint32_t down, int n){
    uint32_t x = w ^ up, y = w ^ down;
    x |= x >> 2; y |= y >> 2;
    x |= x >> 1; y |= y >> 1;
    return n + __popc(~(x & y) & 0x11111111u);
}
/* Full aligned groups of 8 W are counted by Q lanes with one load of digits each, G groups per team with their loads side
 * by side. A workgroup lists the few groups that move; teams of W lanes then share the list and re-encode 8
 * consecutive elements per lane (160 instructions), in wavefronts full of moving groups, and take the groups of any other
 * shape a pair per lane. What bounds the kernel is the two round trips of a workgroup, not HBM. 151 M weights, 15 % of the
 * groups moving: 119 us with one group per row of 16 lanes from start to end, 77 with the list and four groups per row,
 * 44 with 16-byte loads (Q = W / 4) and two groups per team; below a million groups one (64 K groups, all three codec calls 24.5
 * against 26.4 us). Few groups leave most CUs empty that way, and there only the chain counts: Q = W and one group per team
 * (20 K groups 6.8 us, 7.5 to 8.7 the other way). */
template<int W, int Q, int G>
__global__ void __launch_bounds__(256) k_qlmx_servo(signed char *d, signed char *r, float *s,
                                                    const qlmx_span *sp, int nspan, int group, int dmax,
                                                    float f_hi, float f_lo, int packed, int ngrp, int vec_ok){
    constexpr int NW = W / Q, COUNTERS = 256 / Q, TEAMS = 256 / W;
    struct __attribute__((packed, aligned(4))) Words { uint32_t w[NW]; };
    __shared__ uint64_t at[COUNTERS * G];                  /* the moving groups: first element, old scale / new scale */
    __shared__ float conv[COUNTERS * G];
    __shared__ int other[COUNTERS * G];                    /* the groups of other shapes */
    __shared__ int moving, others;
    const int ql = threadIdx.x & (Q - 1), first = (int)blockIdx.x * (COUNTERS * G) + (int)threadIdx.x / Q;
    if(threadIdx.x == 0) moving = others = 0;
    const int s0 = qx_span_of_teams<64 / Q>(sp, nspan, __builtin_amdgcn_readfirstlane(first), (threadIdx.x & 63) / Q);
    __syncthreads();
    if(first < ngrp){
        qlmx_span S = sp[s0];
        uint64_t q0[G]; Words dw[G]; float sg[G]; bool fast[G];
#pragma unroll
        for(int q = 0; q < G; q++){
            const int gi = first + q * COUNTERS;
            fast[q] = false; dw[q] = Words{}; sg[q] = 0.0f; q0[q] = 0;
            if(gi >= ngrp) continue;
            if(gi >= S.gi0 + S.ngrp) S = sp[qx_span_of(sp, nspan, gi)];
            const uint64_t j0 = (uint64_t)(gi - S.gi0) * (uint64_t)group;
            fast[q] = vec_ok && group == 8 * W && packed && S.n - j0 >= 8 * W && ((S.qi0 + j0) & 7ULL) == 0;
            if(!fast[q]){ if(ql == 0) other[atomicAdd(&others, 1)] = gi; continue; }
            q0[q] = S.qi0 + j0;
            dw[q] = *(const Words *)(d + (q0[q] >> 1) + ql * (4 * NW));
            sg[q] = s[gi];
        }
        const uint32_t up = 0x11111111u * (uint32_t)(dmax & 15), down = 0x11111111u * (uint32_t)(-dmax & 15);
#pragma unroll
        for(int q = 0; q < G; q++){
            int railed = 0;
#pragma unroll
            for(int k = 0; k < NW; k++) railed = nibbles_equal(dw[q].w[k], up, down, railed);
            railed += qx_dpp_i<0xB1>(railed);
            if(Q >= 4) railed += qx_dpp_i<0x4E>(railed);
            if(Q >= 8) railed += qx_dpp_i<0x141>(railed);
            if(Q >= 16) railed += qx_dpp_i<0x140>(railed);
            const float f = (float)railed * (1.0f / (8 * W));
            if(fast[q] && ql == 0 && (f > f_hi || f < f_lo)){
                const float sn = servo_scale(sg[q], railed, 8 * W, f_hi, f_lo);
                const int k = atomicAdd(&moving, 1);
                at[k] = q0[q]; conv[k] = sg[q] / sn;
                s[first + q * COUNTERS] = sn;
            }
        }
    }
    __syncthreads();
    const int tl = threadIdx.x & (W - 1), team = threadIdx.x / W;
    for(int k = team; k < moving; k += TEAMS){
        const uint64_t e0 = at[k] + (uint64_t)tl * 8;
        const uint32_t dw = *(const uint32_t *)(d + (e0 >> 1));
        const uint2 rw = *(const uint2 *)(r + e0);
        const float cv = conv[k];
        uint32_t dn = 0, r0 = 0, r1 = 0;
#pragma unroll
        for(int k8 = 0; k8 < 8; k8++){
            const int rb = (int)(signed char)(((k8 < 4 ? rw.x : rw.y) >> (8 * (k8 & 3))) & 0xFFu);
            const float t = ((float)qx_nib(dw, k8) + (float)rb * (1.0f / 128.0f)) * cv;
            int dd, rr; quantize(t, dmax, dd, rr);
            dn |= ((uint32_t)dd & 15u) << (4 * k8);
            if(k8 < 4) r0 |= ((uint32_t)rr & 0xFFu) << (8 * k8); else r1 |= ((uint32_t)rr & 0xFFu) << (8 * (k8 - 4));
        }
        *(uint32_t *)(d + (e0 >> 1)) = dn;
        *(uint2 *)(r + e0) = make_uint2(r0, r1);
    }
    for(int k = team; k < others; k += TEAMS){
        const int gi = other[k];
        servo_pairs<W>(group_loc(sp, qx_span_of(sp, nspan, gi), gi, group), gi, tl, d, r, s, dmax, f_hi, f_lo, packed);
    }
}

static int codec_args_ok(const char *who, int nspan, int group, int dmax, int packed){
    QLMX_REQUIRE(nspan > 0, "%s: nspan %d", who, nspan);
    QLMX_REQUIRE(group >= 2 && group <= 256, "%s: group %d outside [2,256]", who, group);
    QLMX_REQUIRE(dmax >= 1 && dmax <= 127, "%s: dmax %d", who, dmax);
    QLMX_REQUIRE(!packed || (dmax <= 7 && (group & 1) == 0), "%s: packed digits need dmax<=7 and an even group", who);
    return QLMX_OK;
}

extern "C" int qlmx_encode(const float *P, signed char *d, signed char *r, float *s,
                           const qlmx_span *sp, int nspan, int group, int dmax, int packed, int ngrp,
                           void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(P && d && r && s && sp, "qlmx_encode: NULL buffer");
    rc = codec_args_ok("qlmx_encode", nspan, group, dmax, packed); if(rc) return rc;
    if(ngrp <= 0) return QLMX_OK;
    const int vec_ok = ((uintptr_t)P & 15) == 0 && ((uintptr_t)r & 7) == 0 && ((uintptr_t)d & 3) == 0;
    if(group == 64) hipLaunchKernelGGL(k_qlmx_encode<8>, dim3((unsigned)((ngrp + 31) / 32)), dim3(256), 0, (hipStream_t)stream,
                                       P, d, r, s, sp, nspan, group, dmax, packed, ngrp, vec_ok);
    else hipLaunchKernelGGL(k_qlmx_encode<16>, dim3((unsigned)((ngrp + 15) / 16)), dim3(256), 0, (hipStream_t)stream,
                            P, d, r, s, sp, nspan, group, dmax, packed, ngrp, vec_ok);
    QLMX_LAUNCH_CHECK("qlmx_encode launch");
    return QLMX_OK;
}

extern "C" int qlmx_render(float *P, const signed char *d, const float *s,
                           const qlmx_span *sp, int nspan, int group, int packed, int gi_base, int ng,
                           void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(P && d && s && sp, "qlmx_render: NULL buffer");
    rc = codec_args_ok("qlmx_render", nspan, group, packed ? 7 : 127, packed); if(rc) return rc;
    QLMX_REQUIRE(gi_base >= 0, "qlmx_render: gi_base %d", gi_base);
    if(ng <= 0) return QLMX_OK;
    const int vec_ok = ((uintptr_t)P & 15) == 0 && ((uintptr_t)d & 3) == 0;
    if(group == 64) hipLaunchKernelGGL(k_qlmx_render<8>, dim3((unsigned)((ng + 31) / 32)), dim3(256), 0, (hipStream_t)stream,
                                       P, d, s, sp, nspan, group, packed, gi_base, ng, vec_ok);
    else hipLaunchKernelGGL(k_qlmx_render<16>, dim3((unsigned)((ng + 15) / 16)), dim3(256), 0, (hipStream_t)stream,
                            P, d, s, sp, nspan, group, packed, gi_base, ng, vec_ok);
    QLMX_LAUNCH_CHECK("qlmx_render launch");
    return QLMX_OK;
}

extern "C" int qlmx_servo(signed char *d, signed char *r, float *s,
                          const qlmx_span *sp, int nspan, int group, int dmax,
                          float f_hi, float f_lo, int packed, int ngrp, void *stream){
    int rc = qlmx_check_ready(); if(rc) return rc;
    QLMX_REQUIRE(d && r && s && sp, "qlmx_servo: NULL buffer");
    rc = codec_args_ok("qlmx_servo", nspan, group, dmax, packed); if(rc) return rc;
    if(ngrp <= 0) return QLMX_OK;
    const int vec_ok = ((uintptr_t)r & 7) == 0 && ((uintptr_t)d & 3) == 0;
    const bool few = ngrp < 49152, many = ngrp >= 1000000;
#define SERVO(W, Q, G) hipLaunchKernelGGL((k_qlmx_servo<W, Q, G>), dim3((unsigned)((ngrp + 256 / Q * G - 1) / (256 / Q * G))), dim3(256), 0, (hipStream_t)stream, \
                                          d, r, s, sp, nspan, group, dmax, f_hi, f_lo, packed, ngrp, vec_ok)
    if(group == 64){ if(few) SERVO(8, 8, 1); else if(many) SERVO(8, 2, 2); else SERVO(8, 2, 1); }
    else           { if(few) SERVO(16, 16, 1); else if(many) SERVO(16, 4, 2); else SERVO(16, 4, 1); }
#undef SERVO
    QLMX_LAUNCH_CHECK("qlmx_servo launch");
    return QLMX_OK;
}
