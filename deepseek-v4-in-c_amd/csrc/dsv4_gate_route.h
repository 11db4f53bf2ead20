/* SPDX-License-Identifier: Apache-2.0 */
/* dsv4_gate_route.h - device code of the router shared by its own launches
 * (dsv4_route.hip, which states the algorithm) and the launch that runs the
 * shared expert's gate/up beside the fused gate + router
 * (dsv4_decode_mx.hip). */
#ifndef DSV4_GATE_ROUTE_H
#define DSV4_GATE_ROUTE_H

#include "dsv4_internal.h"
#include "dsv4_bf16.h"
#include "dsv4_route_math.h"

namespace dsv4 {

namespace {

constexpr int RT_MAXJ = GATE_ROUTE_MAX_EXPERTS / 64;   /* experts per lane, at most */
constexpr int RT_GROUPS = GATE_ROUTE_GROUPS;           /* arrival counters below the top one */
constexpr int RT_LINE_WORDS = 32;                      /* one 128-byte line per counter */

template <int CTRL, int ROWMASK = 0xF>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t old, uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, ROWMASK, 0xF, false);
}

__device__ __forceinline__ uint64_t max64(uint64_t a, uint64_t b) { return a > b ? a : b; }

__device__ __forceinline__ uint32_t min32(uint32_t a, uint32_t b) { return a < b ? a : b; }
__device__ __forceinline__ uint32_t max32(uint32_t a, uint32_t b) { return a > b ? a : b; }

/* Largest 32-bit value over the wave (each step one DPP-fused max). */
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v)
{
    v = max32(v, dpp_u32<DPP_QUAD_1032>(v, v));
    v = max32(v, dpp_u32<DPP_QUAD_2301>(v, v));
    v = max32(v, dpp_u32<DPP_ROW_HALF_MIRROR>(v, v));
    v = max32(v, dpp_u32<DPP_ROW_MIRROR>(v, v));
    v = max32(v, dpp_u32<DPP_ROW_BCAST15, 0xA>(v, v));
    v = max32(v, dpp_u32<DPP_ROW_BCAST31, 0xC>(v, v));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

/* The largest 64-bit key over the wave: the largest upper half first (one
 * 32-bit reduction), then, among the lanes that hold it (almost always
 * one), the largest lower half. */
__device__ __forceinline__ uint64_t wave_max_key(uint64_t v)
{
    const uint32_t hi = wave_max_u32((uint32_t)(v >> 32));
    const uint64_t at = __builtin_amdgcn_ballot_w64((uint32_t)(v >> 32) == hi);
    uint32_t lo;
    if (__builtin_popcountll(at) == 1)
        lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, (int)__builtin_ctzll(at));
    else
        lo = wave_max_u32((uint32_t)(v >> 32) == hi ? (uint32_t)v : 0u);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v)
{
    v = min32(v, dpp_u32<DPP_QUAD_1032>(v, v));
    v = min32(v, dpp_u32<DPP_QUAD_2301>(v, v));
    v = min32(v, dpp_u32<DPP_ROW_HALF_MIRROR>(v, v));
    v = min32(v, dpp_u32<DPP_ROW_MIRROR>(v, v));
    v = min32(v, dpp_u32<DPP_ROW_BCAST15, 0xA>(v, v));
    v = min32(v, dpp_u32<DPP_ROW_BCAST31, 0xC>(v, v));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

/* sqrt(softplus(x)) bit for bit as the reference's host libm computes it */
__device__ __forceinline__ float route_orig(float x) { return dsv4_route::route_orig(x); }

/* Order-preserving key of a non-NaN score (-0 as +0) over the complemented
 * expert id: the larger key is the reference's preferred pick. */
__device__ __forceinline__ uint64_t pick_key(float v, int e)
{
    uint32_t u = __float_as_uint(v);
    u = u == 0x80000000u ? 0u : u;
    const uint32_t o = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return ((uint64_t)o << 32) | (uint32_t)~(uint32_t)e;
}

/* Element j of a lane's register array, for a wave-uniform j. */
template <int NJ>
__device__ __forceinline__ float lane_elem(const float (&a)[NJ], int j)
{
    float r = a[0];
#pragma unroll
    for (int i = 1; i < NJ; i++) r = j == i ? a[i] : r;
    return r;
}

/* The router's picks and weights for one token, by one wavefront. og / bs:
 * the lane's orig and biased scores of experts lane + 64 j, j < NJ. hash:
 * the token's table row (topk ids), or NULL; hash_bad: a token id outside
 * the table. Lane k < topk holds pick k and its orig; the k loop stays
 * rolled so that no per-k value lives in scalar registers. */
template <int NJ>
__device__ __forceinline__ void route_wave(const float (&og)[NJ], const float (&bs)[NJ], int ne,
                                           int topk, const int64_t *hash, bool hash_bad,
                                           float route_scale, int *idx, float *w,
                                           unsigned *status, int lane)
{
    int my_pick = -1;
    float my_o = 0.0f;
    if (hash || hash_bad) {
        if (lane < topk && !hash_bad) my_pick = (int)hash[lane];
    } else {
        bool nan = false;
#pragma unroll
        for (int j = 0; j < NJ; j++) nan |= lane + 64 * j < ne && bs[j] != bs[j];
        const bool any_nan = __builtin_amdgcn_ballot_w64(nan) != 0;
        /* the keys of the lane's non-NaN experts; 0 marks none or taken */
        uint64_t key[NJ];
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int e = lane + 64 * j;
            key[j] = e < ne && bs[j] == bs[j] ? pick_key(bs[j], e) : 0;
        }
        uint32_t taken = 0;
#pragma clang loop unroll(disable)
        for (int k = 0; k < topk; k++) {
            uint64_t best = key[0];
#pragma unroll
            for (int j = 1; j < NJ; j++) best = max64(best, key[j]);
            best = wave_max_key(best);
            int p = (int)~(uint32_t)best;
            if (any_nan) {
                /* a NaN first candidate is never replaced in the reference's scan */
                uint32_t first = 0xFFFFFFFFu;
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    const int e = lane + 64 * j;
                    first = e < ne && !((taken >> j) & 1u) ? min32(first, (uint32_t)e) : first;
                }
                const uint32_t f = wave_min_u32(first);
                const float fv = __int_as_float(__builtin_amdgcn_readlane(
                    __float_as_int(lane_elem(bs, (int)(f >> 6))), (int)(f & 63u)));
                if (best == 0 || fv != fv) p = (int)f;
            }
            p = __builtin_amdgcn_readfirstlane(p);
            my_pick = lane == k ? p : my_pick;
            const bool mine = (p & 63) == lane;
            taken |= mine ? 1u << (p >> 6) : 0u;
#pragma unroll
            for (int j = 0; j < NJ; j++) key[j] = mine && (p >> 6) == j ? 0 : key[j];
        }
    }
    /* each pick's orig, from the lane that holds it, in k order */
    bool bad = false;
    double sum = 0.0;
#pragma clang loop unroll(disable)
    for (int k = 0; k < topk; k++) {
        const int p = __builtin_amdgcn_readlane(my_pick, k);
        if (p < 0 || p >= ne) { bad = true; continue; }
        const float o = __int_as_float(__builtin_amdgcn_readlane(
            __float_as_int(lane_elem(og, p >> 6)), p & 63));
        my_o = lane == k ? o : my_o;
        sum += (double)o;
    }
    const float inv = sum != 0.0 ? (float)(1.0 / sum) : 0.0f;
    if (lane < topk) {
        idx[lane] = my_pick;
        w[lane] = bad ? __builtin_nanf("") : my_o * inv * route_scale;
    }
    if (bad && lane == 0) atomicOr(status, ST_BAD_EXPERT_ID);
}

/* The token's hash-table row, or NULL with *bad set for a token id outside
 * the table. */
__device__ __forceinline__ const int64_t *hash_row(const GateRouteArgs &a, int tok, bool *bad)
{
    *bad = false;
    if (!a.tid2eid) return nullptr;
    if (tok < 0 || tok >= a.n_vocab) { *bad = true; return nullptr; }
    return a.tid2eid + (int64_t)tok * a.topk;
}

/* Device-scope 32-bit store: written through the XCD's L2, so another
 * XCD's device-scope load sees it. */
__device__ __forceinline__ void st_dev(float *p, float v)
{
    __hip_atomic_store((uint32_t *)p, __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* Device-scope loads through a buffer resource (sc1: past the CU's L1 and the
 * XCD's L2), issued together rather than one atomic load at a time; bytes
 * beyond the resource read as zero. */
constexpr int RT_CPOL_SC1 = 16;
__device__ __forceinline__ float ld_dev(__amdgpu_buffer_rsrc_t r, int byte_off)
{
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, byte_off, 0, RT_CPOL_SC1));
}

/* The decode step's gate matvec and router in one launch: workgroup r of
 * nblk computes gate rows 4 r .. 4 r + 3; the last to finish routes the token.
 * Four waves; lds: b4_lds_bytes(1, a.cols). */
template <int NJ>
__device__ __forceinline__ void gate_route_group(const GateRouteArgs &a, unsigned nblk, uint8_t *lds)
{
    const int ne = a.n_experts;
    const int lane = threadIdx.x & 63;
    const double acc = bf16_dot4(lds, a.gate_w, 4 * blockIdx.x, ne, a.x, 0, 1, a.cols);
    const int r = 4 * blockIdx.x + (lane >> 4);
    if (threadIdx.x < 64 && (lane & 15) == 0 && r < ne) {
        const float s = (float)acc;
        const float o = route_orig(s);
        st_dev(a.ws_orig + r, o);
        st_dev(a.ws_biased + r, a.bias ? o + a.bias[r] : o);
        if (a.scores_out) a.scores_out[r] = s;
        if (a.orig) a.orig[r] = o;
    }
    if (threadIdx.x >= 64) return;                 /* the first wave stored the rows */
    /* The workgroup's rows stored and acknowledged, then one add to its
     * group's counter; the last of a group adds one to the top counter, and
     * the last of those is the last workgroup. Adds to one word serialise
     * (one per row cost 3 us, one per workgroup 1.3 us). */
    __builtin_amdgcn_s_waitcnt(0x0F70);            /* vmcnt(0) */
    asm volatile("" ::: "memory");
    unsigned last = 0;
    if (lane == 0) {
        const unsigned grp = blockIdx.x % RT_GROUPS;
        const unsigned in_grp = (nblk - grp + RT_GROUPS - 1) / RT_GROUPS;
        const unsigned groups = nblk < RT_GROUPS ? nblk : RT_GROUPS;
        if (__hip_atomic_fetch_add(a.counter + grp * RT_LINE_WORDS, 1u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT) == in_grp - 1)
            last = __hip_atomic_fetch_add(a.counter + RT_GROUPS * RT_LINE_WORDS, 1u, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT) == groups - 1;
    }
    if (!__builtin_amdgcn_readfirstlane((int)last)) return;
    /* the last workgroup: every other row's stores were acknowledged before
     * its workgroup's add */
    asm volatile("" ::: "memory");
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(a.ws_orig, (short)0, 4 * ne, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(a.ws_biased, (short)0, 4 * ne, 0x00020000);
    float og[NJ], bs[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        og[j] = ld_dev(ro, 4 * (lane + 64 * j));
        bs[j] = ld_dev(rb, 4 * (lane + 64 * j));
    }
    if (lane <= RT_GROUPS)
        __hip_atomic_store(a.counter + lane * RT_LINE_WORDS, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    bool hbad;
    const int64_t *hrow = hash_row(a, a.token_id, &hbad);
    route_wave<NJ>(og, bs, ne, a.topk, hrow, hbad, a.route_scale, a.idx, a.w, a.status, lane);
}

} // namespace

} // namespace dsv4

#endif /* DSV4_GATE_ROUTE_H */
