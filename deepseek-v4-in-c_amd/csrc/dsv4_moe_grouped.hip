/* SPDX-License-Identifier: Apache-2.0 */
/* dsv4_moe_grouped.hip - MoE over many tokens at once: batched decode and
 * the prefill MoE layer.
 *
 * What it replaces, in the reference:
 *   - the permutation of (token, k) pairs by expert
 *     (src/80_prefill/dsv4_prefill_union.c:30-66),
 *   - the per-expert bucket: gather, w1 / w3 GEMMs, SwiGLU, w2 GEMM, scatter
 *     (src/80_prefill/dsv4_prefill_experts.c:23-77; its GPU leg, the fused
 *     Vulkan expert, src/80_prefill/dsv4_prefill_vk_expert.c:45-172),
 *   - the combine: per token, out = sum_k w_k * acc_k in k order, then the
 *     shared expert's output added unweighted
 *     (src/80_prefill/dsv4_prefill_union_run.c:109-121).
 * The CPU/GPU bucket scheduler (src/80_prefill/dsv4_prefill_union_sched.c)
 * has no counterpart: every bucket runs in one device-resident pass.
 *
 * PIPELINE (one stream, no host round trip)
 *   k_moe_route     counting sort by expert: first row of each expert's
 *                   bucket (grp_off), prefix of its token tiles (tile_pre),
 *                   each tile's bucket, first row and rows (tile_rec),
 *                   each pair's row (pos) and each row's token (row_tok);
 *                   one launch, each workgroup placing its own chunks of
 *                   1024 pairs after counting all of them.
 *   k_to_f16_rows   x -> fp16 (round to nearest even) after scaling each
 *                   row by the power of two that puts its largest magnitude
 *                   in [2^14, 2^15); the GEMM epilogues undo it exactly.
 *   k_grouped       one wave = one work item: an expert, a slab of output
 *                   features (64 for gate/up with both w1 and w3 rows, 128 for
 *                   down) and a tile of up to 16*TT of its rows, read from
 *                   the tile's record; the grid is an upper bound and
 *                   surplus waves exit.
 *   k_moe_combine   out[t] = sum_k w[t][k] * Y[pos(t, k)] (k order) + shared[t].
 *
 * NUMERICS
 *   v_mfma_f32_16x16x32_f16, fp32 accumulation. Weights are decoded into the
 *   MFMA operand with v_cvt_scalef32_pk_f16_{fp4,fp8}: e2m1 * 2^e is exact in
 *   fp16 for E8M0 scale bytes 104..140 (checked on every block: outside it
 *   the status word gets ST_SCALE_RANGE); e4m3 values enter unscaled (exact)
 *   and the 128x128 block scale, E8M0 or fp32, multiplies each 128-K chunk's
 *   partial sum in fp32, as the reference's fp8_n applies it per block. The
 *   activations (row-scaled by a power of two, so no finite value overflows
 *   and values down to 2^-28 of the row maximum stay normal) and the SwiGLU
 *   output enter the MFMA rounded to fp16 (relative error at most 2^-11
 *   each); a SwiGLU output beyond the fp16 range raises ST_F16_RANGE.
 *   Everything else is fp32.
 *
 * MFMA OPERANDS (gfx950, measured): lane l supplies row l % 16 of A and of B
 *   with 8 consecutive reduction indices, lane group l / 16 selecting which 8;
 *   accumulator element e of lane l is row 4 (l / 16) + e, column l % 16.
 *   Weights are A (rows = output features), tokens are B. The reduction index
 *   may be permuted freely as long as A and B agree: each lane loads 16
 *   contiguous weight bytes per 128-K chunk (FP4: 32 values, one E8M0 block)
 *   and the B side is fetched in the same order (kmap).
 *
 * Bound: HBM (weights) for small buckets, MFMA for large ones.
 */
#include "dsv4_internal.h"

namespace dsv4 {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int KC = 128;           /* reduction chunk */
template <int N> struct IC { static constexpr int value = N; };
constexpr int RB = 8;             /* 16-row weight blocks per item */
constexpr int MAX_ROUTE_EXPERTS = 1024;

/* first reduction index (within a 128-K chunk) of MFMA step j for lane
 * group gq; FP4 lanes hold 32 contiguous values, FP8 lanes two runs of 16 */
template <int WF>
__device__ __forceinline__ int kmap(int gq, int j)
{
    if constexpr (WF == FMT_FP4_E8M0) return 32 * gq + 8 * j;
    else return 64 * (j >> 1) + 16 * gq + 8 * (j & 1);
}

__device__ __forceinline__ uint32_t pk_f16_fp4(uint32_t w, float sc, int sel)
{
    return __builtin_bit_cast(uint32_t, sel == 0 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, sc, 0)
                                       : sel == 1 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, sc, 1)
                                       : sel == 2 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, sc, 2)
                                                  : __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, sc, 3));
}

template <bool HI>
__device__ __forceinline__ uint32_t pk_f16_fp8(uint32_t w, float sc)
{
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, sc, HI));
}

/* A operand of step j from one lane's raw weight bytes (whole-word bit casts
 * only: extracting one half of a packed convert result is not reliable) */
template <int WF>
__device__ __forceinline__ h8 a_operand(const u32x4 (&w)[2], float sc, int j)
{
    u32x4 v;
    if constexpr (WF == FMT_FP4_E8M0) {
        const uint32_t d = j == 0 ? w[0].x : j == 1 ? w[0].y : j == 2 ? w[0].z : w[0].w;
        v.x = pk_f16_fp4(d, sc, 0);
        v.y = pk_f16_fp4(d, sc, 1);
        v.z = pk_f16_fp4(d, sc, 2);
        v.w = pk_f16_fp4(d, sc, 3);
    } else {
        const u32x4 &h = w[j >> 1];
        const uint32_t d0 = (j & 1) ? h.z : h.x, d1 = (j & 1) ? h.w : h.y;
        v.x = pk_f16_fp8<false>(d0, sc);
        v.y = pk_f16_fp8<true>(d0, sc);
        v.z = pk_f16_fp8<false>(d1, sc);
        v.w = pk_f16_fp8<true>(d1, sc);
    }
    return __builtin_bit_cast(h8, v);
}

__device__ __forceinline__ f4v mfma16(const h8 &a, const h8 &b, const f4v &c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t f16_bits(float v)
{
    return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v);
}

/* The power of two that output row r's B row carries (0 without bexp). */
__device__ __forceinline__ int b_row_exp(const GroupedArgs &a, int r)
{
    if (!a.bexp) return 0;
    return a.bexp[a.row_tok ? a.row_tok[r] : r];
}

/* Four fp32 results of a row that carries 2^ex, brought back to scale
 * (exact: a power-of-two multiply). */
__device__ __forceinline__ f4v unscale4(f4v v, int ex)
{
    if (ex == 0) return v;
    return f4v{ldexpf(v.x, -ex), ldexpf(v.y, -ex), ldexpf(v.z, -ex), ldexpf(v.w, -ex)};
}

/* SwiGLU of four (gate, up) pairs of a row that carries 2^ex, packed as four
 * fp16; a finite result beyond the fp16 range raises ST_F16_RANGE in bad. */
__device__ __forceinline__ uint2 swiglu_f16x4(const f4v &g, const f4v &u, int ex, float limit,
                                              unsigned &bad)
{
    const f4v gs = unscale4(g, ex), us = unscale4(u, ex);
    float m[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        m[e] = dev_swiglu(gs[e], us[e], limit);
        if (__builtin_isfinite(m[e]) && __builtin_fabsf(m[e]) >= 65520.0f) bad |= ST_F16_RANGE;
    }
    uint2 pk;
    pk.x = f16_bits(m[0]) | (f16_bits(m[1]) << 16);
    pk.y = f16_bits(m[2]) | (f16_bits(m[3]) << 16);
    return pk;
}

template <int WF>
__device__ __forceinline__ bool qmat_matches(const DSV4QMat &m, int rows, int cols)
{
    if (m.rows != rows || m.cols != cols || !m.w || !m.s) return false;
    if constexpr (WF == FMT_FP4_E8M0) return m.wdt == DSV4_WFP4 && m.blk_r == 1 && m.blk_c == 32;
    else if constexpr (WF == FMT_FP8_E8M0) return m.wdt == DSV4_WFP8 && m.blk_r == 128 && m.blk_c == 128;
    else return m.wdt == DSV4_WFP8_F32S && m.blk_r == 128 && m.blk_c == 128;
}

/* what buffer loads need of their bases */
__device__ __forceinline__ bool dword_aligned(const DSV4QMat &m)
{
    return (((uintptr_t)m.w | (uintptr_t)m.s) & 3) == 0;
}

} // namespace

/* ----------------------------------------------------- rows to fp16 --- */

/* One workgroup of NTHR threads converts a row: the row's largest finite
 * magnitude (a fixed-order max, order does not matter), then 8 floats -> 8
 * fp16 per thread and unit, each multiplied by the row's power of two first
 * (exact). The second pass re-reads the row from cache. */
__device__ __forceinline__ float finite_abs(float v)
{
    const float m = __builtin_fabsf(v);
    return __builtin_isfinite(m) ? m : 0.0f;
}

template <int NTHR>
__device__ __forceinline__ void row_to_f16(uint16_t *o, int *ex, const float *x, int row, int cols, float *wmax)
{
    const float *xr = x + (size_t)row * cols;
    uint16_t *orow = o + (size_t)row * cols;
    const int units = cols / 8;
    float m = 0.0f;
    for (int u = threadIdx.x; u < units; u += NTHR) {
        const f32x4 a = *(const f32x4 *)(xr + 8 * u), b = *(const f32x4 *)(xr + 8 * u + 4);
        m = fmaxf(m, fmaxf(fmaxf(finite_abs(a.x), finite_abs(a.y)), fmaxf(finite_abs(a.z), finite_abs(a.w))));
        m = fmaxf(m, fmaxf(fmaxf(finite_abs(b.x), finite_abs(b.y)), fmaxf(finite_abs(b.z), finite_abs(b.w))));
    }
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) m = fmaxf(m, __shfl_xor(m, s, 64));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
    __syncthreads();
    m = wmax[0];
#pragma unroll
    for (int w = 1; w < NTHR / 64; w++) m = fmaxf(m, wmax[w]);
    const int e = m > 0.0f ? 14 - ilogbf(m) : 0;       /* m * 2^e in [2^14, 2^15) */
    if (threadIdx.x == 0) ex[row] = e;
    for (int u = threadIdx.x; u < units; u += NTHR) {
        const f32x4 a = *(const f32x4 *)(xr + 8 * u), b = *(const f32x4 *)(xr + 8 * u + 4);
        u32x4 v;
        v.x = f16_bits(ldexpf(a.x, e)) | (f16_bits(ldexpf(a.y, e)) << 16);
        v.y = f16_bits(ldexpf(a.z, e)) | (f16_bits(ldexpf(a.w, e)) << 16);
        v.z = f16_bits(ldexpf(b.x, e)) | (f16_bits(ldexpf(b.y, e)) << 16);
        v.w = f16_bits(ldexpf(b.z, e)) | (f16_bits(ldexpf(b.w, e)) << 16);
        *(u32x4 *)(orow + 8 * u) = v;
    }
}

__global__ __launch_bounds__(256) void k_to_f16_rows(uint16_t *o, int *ex, const float *x, int cols)
{
    __shared__ float wmax[4];
    row_to_f16<256>(o, ex, x, blockIdx.x, cols, wmax);
}

/* ------------------------------------------------------------ routing --- */

/* Chunks of 1024 pairs whose routing ids a thread holds in registers at
 * once: their loads are all issued before the first is used, so a pass over
 * them waits out one memory latency instead of one per chunk. */
constexpr int ROUTE_BATCH = 32;
constexpr int ROUTE_MAX_BLOCKS = 256;

__device__ __forceinline__ void route_load(int (&ev)[ROUTE_BATCH], const RouteArgs &a, int c0, int nch,
                                           int tid)
{
#pragma unroll
    for (int i = 0; i < ROUTE_BATCH; i++) {
        const int p = (c0 + i) * 1024 + tid;
        ev[i] = (c0 + i < nch && p < a.npairs) ? a.idx[p] : -1;
    }
}

/* The lanes of the wave whose routing id equals this lane's; ids outside
 * [0, E) (bad ids and pairs past the end) all count as one id of their own:
 * one ballot per bit of the key id + 1 (E <= 1024, so 11 bits). */
__device__ __forceinline__ uint64_t same_id_lanes(int e, int E)
{
    const unsigned key = (unsigned)e < (unsigned)E ? (unsigned)e + 1u : 0u;
    uint64_t peers = ~0ull;
#pragma unroll
    for (int b = 0; b < 11; b++) {
        const bool bit = (key >> b) & 1u;
        const uint64_t m = __ballot(bit);
        peers &= bit ? m : ~m;
    }
    return peers;
}

/* The wave's count of this lane's expert when this lane is the highest of
 * that expert's lanes, else 0: one LDS add per expert and wave rather than
 * one per pair, so a popular expert's counter is not hammered by every lane.
 * Called by every lane of the wave (it ballots). */
__device__ __forceinline__ int route_leader_count(int e, int E, uint64_t below)
{
    const uint64_t peers = same_id_lanes(e, E);
    const int n = __popcll(peers);
    return ((unsigned)e < (unsigned)E && __popcll(peers & below) == n - 1) ? n : 0;
}

/* Pass one of the two-launch form: workgroup c counts chunk c's pairs per
 * expert into chist[c][E] (and reports bad ids). The workgroups from nch on
 * convert a row of x each. */
__global__ __launch_bounds__(1024) void k_moe_route_count(RouteArgs a, int nch, RowsF16Args x16)
{
    __shared__ int hist[MAX_ROUTE_EXPERTS];
    const int tid = threadIdx.x, E = a.n_experts, c = blockIdx.x;
    if (c >= nch) {
        row_to_f16<1024>(x16.o, x16.ex, x16.x, c - nch, x16.cols, (float *)hist);
        return;
    }
    const int lane = tid & 63;
    const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;
    const int p = c * 1024 + tid;
    const int e = p < a.npairs ? a.idx[p] : -1;
    hist[tid] = 0;
    __syncthreads();
    const int n = route_leader_count(e, E, below);
    if (n) atomicAdd(&hist[e], n);
    else if ((unsigned)e >= (unsigned)E && p < a.npairs) atomicOr(a.status, ST_BAD_EXPERT_ID);
    __syncthreads();
    if (tid < E) a.chist[(size_t)c * E + tid] = hist[tid];
}

/* Stable counting sort of the pairs by expert. Pairs go in chunks of 1024;
 * workgroup b places chunks [b * cpb, (b + 1) * cpb). It needs the bucket
 * sizes and how many pairs of each expert precede its first chunk: with
 * PRECOUNT it sums them from the per-chunk counts k_moe_route_count wrote
 * (two launches); without, every workgroup counts every pair itself (one
 * launch, no workgroup waits for another: the form for a few chunks).
 * Workgroup 0 also writes grp_off and tile_pre, every workgroup a share
 * of the tile records (with a.fat_rows two lists of them); bad ids are
 * reported by workgroup 0 (one launch) or by the counting pass. The
 * workgroups from nblk on convert a row of x each (one launch). */
template <bool PRECOUNT>
__global__ __launch_bounds__(1024) void k_moe_route(RouteArgs a, int cpb, int nblk, RowsF16Args x16)
{
    __shared__ int hist[MAX_ROUTE_EXPERTS], before[MAX_ROUTE_EXPERTS];
    __shared__ int cur[MAX_ROUTE_EXPERTS];
    __shared__ int scan_r[MAX_ROUTE_EXPERTS], scan_t[MAX_ROUTE_EXPERTS];
    __shared__ unsigned short wcnt[16][MAX_ROUTE_EXPERTS];
    const int tid = threadIdx.x;
    const int E = a.n_experts;
    if (!PRECOUNT && (int)blockIdx.x >= nblk) {
        row_to_f16<1024>(x16.o, x16.ex, x16.x, blockIdx.x - nblk, x16.cols, (float *)hist);
        return;
    }
    const int nch = (a.npairs + 1023) / 1024;
    const int c_lo = blockIdx.x * cpb, c_hi = min(nch, c_lo + cpb);
    int ev[ROUTE_BATCH];
    /* the first batch of routing ids is in flight while the tables clear */
    if (!PRECOUNT) route_load(ev, a, 0, nch, tid);
    if (tid < E) {
        hist[tid] = 0;
        before[tid] = 0;
        for (int w = 0; w < 16; w++) wcnt[w][tid] = 0;
    }
    __syncthreads();
    unsigned bad = 0;
    const int lane = tid & 63, wv = tid >> 6;
    const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;
    if constexpr (PRECOUNT) {
        /* expert tid's count in every chunk: sixteen loads in flight per
         * round, summed in chunk order (integers: any order gives the same) */
        if (tid < E) {
            int tot = 0, bef = 0;
            for (int c0 = 0; c0 < nch; c0 += 16) {
                int v[16];
#pragma unroll
                for (int i = 0; i < 16; i++) v[i] = c0 + i < nch ? a.chist[(size_t)(c0 + i) * E + tid] : 0;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    tot += v[i];
                    if (c0 + i < c_lo) bef += v[i];
                }
            }
            hist[tid] = tot;
            before[tid] = bef;
        }
    } else
    for (int c0 = 0; c0 < nch; c0 += ROUTE_BATCH) {
        if (c0) route_load(ev, a, c0, nch, tid);
#pragma unroll
        for (int i = 0; i < ROUTE_BATCH; i++) {
            if (c0 + i >= nch) break;                              /* uniform */
            const int p = (c0 + i) * 1024 + tid;
            const int n = route_leader_count(ev[i], E, below);
            if (n) {
                atomicAdd(&hist[ev[i]], n);
                if (c0 + i < c_lo) atomicAdd(&before[ev[i]], n);
            } else if ((unsigned)ev[i] >= (unsigned)E && p < a.npairs) {
                bad = ST_BAD_EXPERT_ID;
            }
        }
    }
    __syncthreads();
    /* inclusive scans of the bucket sizes and tile counts, one expert per
     * thread (E <= 1024): within each wave by shuffles, then the totals of
     * the lower waves added (two barriers) */
    const int cnt = tid < E ? hist[tid] : 0;
    const bool fat = a.fat_rows && cnt > a.fat_min;
    const int rows = fat ? a.fat_rows : a.tile_rows;
    const int tls = (cnt + rows - 1) / rows << (fat ? 16 : 0);
    {
        /* only the waves that hold experts scan (E / 64 rounded up) */
        __shared__ int wsum[2][16];
        const bool live = wv * 64 < E;
        int ir = cnt, it = tls;
        if (live) {
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int xr = __shfl_up(ir, d, 64), xt = __shfl_up(it, d, 64);
                if (lane >= d) {
                    ir += xr;
                    it += xt;
                }
            }
            if (lane == 63) {
                wsum[0][wv] = ir;
                wsum[1][wv] = it;
            }
        }
        __syncthreads();
        if (live) {
            for (int w = 0; w < wv; w++) {
                ir += wsum[0][w];
                it += wsum[1][w];
            }
            scan_r[tid] = ir;
            scan_t[tid] = it;
        }
        __syncthreads();
    }
    /* each tile's bucket: the first expert whose inclusive tile prefix
     * exceeds it, tiles spread over every workgroup's threads; with the
     * bucket's first row and the tile's rows. With fat_rows the upper half
     * words count the tiles of the large buckets, which follow the others. */
    const int fat_shift = a.fat_rows ? 16 : 0, thin_mask = a.fat_rows ? 0xFFFF : -1;
    const int nthin = scan_t[E - 1] & thin_mask, nfat = a.fat_rows ? scan_t[E - 1] >> 16 : 0;
    for (int i = blockIdx.x * 1024 + tid; i < nthin + nfat; i += nblk * 1024) {
        const bool f = i >= nthin;
        const int t = f ? i - nthin : i, trows = f ? a.fat_rows : a.tile_rows;
        const int shift = f ? fat_shift : 0, mask = f ? 0xFFFF : thin_mask;
        int lo = 0, hi = E - 1;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (((scan_t[mid] >> shift) & mask) > t) hi = mid;
            else lo = mid + 1;
        }
        const int go = lo > 0 ? scan_r[lo - 1] : 0, tp = lo > 0 ? (scan_t[lo - 1] >> shift) & mask : 0;
        const int r0 = go + (t - tp) * trows;
        TileRec rec;
        rec.grp = lo;
        rec.r0 = r0;
        rec.ntok = min(trows, scan_r[lo] - r0);
        rec.bucket = scan_r[lo] - go;
        a.tile_rec[f ? a.fat_base + t : t] = rec;
    }
    if (tid < E) {
        const int o = scan_r[tid] - cnt;
        cur[tid] = o + before[tid];
        if (blockIdx.x == 0) {
            a.grp_off[tid] = o;
            a.tile_pre[tid] = (scan_t[tid] - tls) & thin_mask;
            if (tid == E - 1) {
                a.grp_off[E] = scan_r[tid];
                a.tile_pre[E] = nthin;
                if (a.fat_rows) a.tile_pre[E + 1] = nfat;
            }
        }
    }
    __syncthreads();
    /* Rows inside a bucket in pair order (token-major, k-minor), as the
     * reference's counting sort places them: a pair's row is its bucket's
     * start, plus the pairs of the same expert in earlier chunks, plus those
     * in lower waves of its chunk (each expert's per-wave counts turned into
     * exclusive prefixes in place), plus those in lower lanes of its wave.
     * A workgroup that counted every chunk in one batch already holds its
     * routing ids. */
    const bool have_ids = !PRECOUNT && c_lo == 0 && c_hi == nch && nch <= ROUTE_BATCH;
    for (int c0 = c_lo; c0 < c_hi; c0 += ROUTE_BATCH) {
        if (!have_ids) route_load(ev, a, c0, c_hi, tid);
#pragma unroll
        for (int i = 0; i < ROUTE_BATCH; i++) {
            if (c0 + i >= c_hi) break;                             /* uniform */
            const int p = (c0 + i) * 1024 + tid;
            const int e = ev[i];
            const bool ok = (unsigned)e < (unsigned)E;
            const uint64_t peers = same_id_lanes(e, E);
            const int rank = __popcll(peers & below);
            if (ok && rank == __popcll(peers) - 1) wcnt[wv][e] = (unsigned short)(rank + 1);
            __syncthreads();
            int tot = 0;
            if (tid < E) {
                unsigned short c[16];
#pragma unroll
                for (int w = 0; w < 16; w++) c[w] = wcnt[w][tid];
#pragma unroll
                for (int w = 0; w < 16; w++) {
                    wcnt[w][tid] = (unsigned short)tot;
                    tot += c[w];
                }
            }
            __syncthreads();
            if (ok) {
                const int r = cur[e] + wcnt[wv][e] + rank;
                a.pos[p] = r;
                a.row_tok[r] = p / a.topk;
                if (a.row_k) a.row_k[r] = p - (p / a.topk) * a.topk;
            } else if (p < a.npairs) {
                a.pos[p] = -1;
            }
            __syncthreads();
            if (tid < E) {
                cur[tid] += tot;
#pragma unroll
                for (int w = 0; w < 16; w++) wcnt[w][tid] = 0;
            }
            __syncthreads();
        }
    }
    if (!PRECOUNT && bad && blockIdx.x == 0) atomicOr(a.status, bad);
}

/* --------------------------------------------------------- grouped GEMM --- */

template <int WF, bool SWIGLU, int TT>
__global__ __launch_bounds__(256) void k_grouped(GroupedArgs a)
{
    constexpr int FEAT = SWIGLU ? 64 : 128;       /* output features per item */
    constexpr int TROWS = 16 * TT;                /* rows per tile           */
    constexpr bool FP4 = WF == FMT_FP4_E8M0;
    const int lane = threadIdx.x & 63;
    const int rr = lane & 15, gq = lane >> 4;
    const int item = blockIdx.x * 4 + wave_in_group();
    const int nslab = a.N / FEAT;
    const int tile = item / nslab, slab = item - tile * nslab;

    int r0, ntok;
    DSV4QMat m1, m3;
    if (a.table) {
        const int E = a.n_experts;
        const int ntiles = ld_uniform(a.tile_pre, E);
        const TileRec tr = ld_uniform(a.tile_rec, tile);  /* read beside the count: one round trip */
        if ((tile >= ntiles) | (tr.ntok <= 0)) return;
        r0 = tr.r0;
        ntok = tr.ntok;
        const DSV4ExpertW e = ld_uniform(a.table, tr.grp);
        m1 = SWIGLU ? e.w1 : e.w2;
        m3 = e.w3;
    } else {
        r0 = tile * TROWS;
        if (r0 >= a.nrows) return;
        ntok = min(TROWS, a.nrows - r0);
        m1 = a.m1;
        m3 = a.m3;
    }
    const int ntt = (ntok + 15) >> 4;              /* live 16-row tiles */
    const int f0 = slab * FEAT;
    const int K = a.K, N = a.N;

    if (!qmat_matches<WF>(m1, N, K) || (SWIGLU && !qmat_matches<WF>(m3, N, K))) {
        if (lane == 0) atomicOr(a.status, ST_BAD_DESCRIPTOR);
        const float nan = __builtin_nanf("");
        for (int t = 0; t < ntok; t++)
            for (int f = lane; f < FEAT; f += 64) {
                const size_t o = (size_t)(r0 + t) * N + f0 + f;
                if constexpr (SWIGLU) ((uint16_t *)a.out)[o] = (uint16_t)f16_bits(nan);
                else ((float *)a.out)[o] = nan;
            }
        return;
    }

    /* this lane's weight rows: SwiGLU items take w1 rows in blocks 0-3 and
     * the matching w3 rows in blocks 4-7 */
    const int rowb = FP4 ? K / 2 : K;              /* bytes per weight row */
    /* 32-bit per-lane offsets from the wave-uniform matrix bases (a matrix is
     * below 4 GiB): the weight byte of block rb is base(rb) + wofs[rb], its
     * FP4 scale row base_s(rb) + sofs[rb] */
    const uint8_t *wb1 = (const uint8_t *)m1.w, *wb3 = (const uint8_t *)m3.w;
    const uint8_t *sb1 = (const uint8_t *)m1.s, *sb3 = (const uint8_t *)m3.s;
    uint32_t wofs[RB], sofs[RB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        const int row = f0 + 16 * (SWIGLU ? (rb & 3) : rb) + rr;
        wofs[rb] = (uint32_t)row * (uint32_t)rowb + 16u * (uint32_t)gq;
        sofs[rb] = (uint32_t)row * (uint32_t)(K / 32);
    }
    /* FP8: one scale per (128-row block, 128-K chunk) per matrix */
    const int nb = f0 / 128, kbn = K / 128;

    /* this lane's B rows (tokens); rows past the tile's end repeat row r0 */
    const uint16_t *brow[TT];
#pragma unroll
    for (int tt = 0; tt < TT; tt++) {
        const int t = 16 * tt + rr;
        const int r = t < ntok ? r0 + t : r0;
        const int src = a.row_tok ? a.row_tok[r] : r;
        brow[tt] = a.B + (size_t)src * K;
    }

    f4v acc[RB][TT];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int tt = 0; tt < TT; tt++) acc[rb][tt] = f4v{0.0f, 0.0f, 0.0f, 0.0f};

    unsigned scale_bad = 0;
    const int nchunk = K / KC;
    /* Raw weights of the next PF chunks are in flight while one multiplies:
     * with 16-row tiles the item is a weight stream and needs several chunks
     * in flight to cover HBM latency; with 64-row tiles one chunk of compute
     * covers it. The B operands (tokens, from L2) are fetched one chunk
     * ahead. */
    constexpr int PF = (TT == 1 && FP4) ? 3 : 1;
    constexpr int CB = FP4 ? 64 : 128;             /* weight bytes per row per chunk */
    struct WChunk {
        u32x4 w[RB][2];
        uint32_t s[RB];                            /* FP4: the lane's 4 E8M0 bytes  */
        float fs[2];                               /* FP8: chunk scale of m1, m3    */
    };
    auto load_w = [&](int c, WChunk &o) {
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            const bool up = SWIGLU && rb >= 4;
            const uint8_t *p = (up ? wb3 : wb1) + (wofs[rb] + (uint32_t)(c * CB));
            o.w[rb][0] = ld_stream16(p);
            if constexpr (!FP4) o.w[rb][1] = ld_stream16(p + 64);
            if constexpr (FP4)
                o.s[rb] = *gptr((const uint32_t *)((up ? sb3 : sb1) + (sofs[rb] + 4u * (uint32_t)c)));
        }
        if constexpr (WF == FMT_FP8_E8M0) {
            o.fs[0] = dev_e8m0(ld_u8(m1.s, (size_t)nb * kbn + c));
            o.fs[1] = SWIGLU ? dev_e8m0(ld_u8(m3.s, (size_t)nb * kbn + c)) : 0.0f;
        } else if constexpr (WF == FMT_FP8_F32S) {
            o.fs[0] = ld_f32(m1.s, (size_t)nb * kbn + c);
            o.fs[1] = SWIGLU ? ld_f32(m3.s, (size_t)nb * kbn + c) : 0.0f;
        } else {
            o.fs[0] = o.fs[1] = 1.0f;
        }
    };
    auto load_b = [&](int c, h8 (&b)[TT][4]) {
#pragma unroll
        for (int tt = 0; tt < TT; tt++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                b[tt][j] = *gptr((const h8 *)(brow[tt] + c * KC + kmap<WF>(gq, j)));
    };
    auto compute = [&](const WChunk &wc, const h8 (&bop)[TT][4]) {
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            float cvt_scale = 1.0f;                /* FP8: raw e4m3, exact in fp16 */
            if constexpr (FP4) {
                const uint32_t b = (wc.s[rb] >> (8 * gq)) & 0xFFu;
                scale_bad |= (b - 104u) > 36u;
                cvt_scale = dev_e8m0(b);
            }
            if constexpr (!FP4) {
                f4v part[TT];
#pragma unroll
                for (int tt = 0; tt < TT; tt++) part[tt] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const h8 av = a_operand<WF>(wc.w[rb], cvt_scale, j);
#pragma unroll
                    for (int tt = 0; tt < TT; tt++)
                        if (tt < ntt) part[tt] = mfma16(av, bop[tt][j], part[tt]);
                }
                const float sc = (SWIGLU && rb >= 4) ? wc.fs[1] : wc.fs[0];
#pragma unroll
                for (int tt = 0; tt < TT; tt++)
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[rb][tt][e] = fmaf(part[tt][e], sc, acc[rb][tt][e]);
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const h8 av = a_operand<WF>(wc.w[rb], cvt_scale, j);
#pragma unroll
                    for (int tt = 0; tt < TT; tt++)
                        if (tt < ntt) acc[rb][tt] = mfma16(av, bop[tt][j], acc[rb][tt]);
                }
            }
        }
    };

    /* Loads are issued unconditionally (past the end they repeat the last
     * chunk, an L2 hit): a load behind a branch makes the wait-count pass
     * drain every outstanding load at the join, prefetches included. */
    const int last = nchunk - 1;
    WChunk ring[PF];
#pragma unroll
    for (int i = 0; i < PF; i++) load_w(min(i, last), ring[i]);
    h8 bnext[TT][4];
    load_b(0, bnext);
    int c = 0;
    for (; c + PF <= nchunk; c += PF) {
#pragma unroll
        for (int i = 0; i < PF; i++) {
            const WChunk wc = ring[i];
            load_w(min(c + i + PF, last), ring[i]);
            h8 bop[TT][4];
#pragma unroll
            for (int tt = 0; tt < TT; tt++)
#pragma unroll
                for (int j = 0; j < 4; j++) bop[tt][j] = bnext[tt][j];
            load_b(min(c + i + 1, last), bnext);
            compute(wc, bop);
        }
    }
    /* at most PF - 1 chunks remain; they are already in the ring */
#pragma unroll
    for (int i = 0; i + 1 < PF; i++) {
        if (c + i < nchunk) {
            h8 bop[TT][4];
#pragma unroll
            for (int tt = 0; tt < TT; tt++)
#pragma unroll
                for (int j = 0; j < 4; j++) bop[tt][j] = bnext[tt][j];
            load_b(min(c + i + 1, last), bnext);
            compute(ring[i], bop);
        }
    }
    if (scale_bad) atomicOr(a.status, ST_SCALE_RANGE);

    /* epilogue: lane holds token rr of each tile, features 4 gq .. 4 gq + 3
     * of each 16-row block */
    unsigned range_bad = 0;
#pragma unroll
    for (int tt = 0; tt < TT; tt++) {
        const int t = 16 * tt + rr;
        if (t >= ntok) continue;
        const size_t orow = (size_t)(r0 + t) * N;
        const int ex = b_row_exp(a, r0 + t);
        if constexpr (SWIGLU) {
#pragma unroll
            for (int rb = 0; rb < 4; rb++)
                *(uint2 *)((uint16_t *)a.out + orow + f0 + 16 * rb + 4 * gq) =
                    swiglu_f16x4(acc[rb][tt], acc[rb + 4][tt], ex, a.limit, range_bad);
        } else {
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
                *(f4v *)((float *)a.out + orow + f0 + 16 * rb + 4 * gq) = unscale4(acc[rb][tt], ex);
        }
    }
    if (range_bad) atomicOr(a.status, range_bad);
}

/* ------------------------------------------- LDS-staged grouped GEMM --- */

/* The same work as k_grouped, for K a multiple of 256, with a workgroup per
 * item and every operand staged through LDS by direct loads. Direct global
 * loads in the MFMA layout make each instruction touch 16 rows (64 B each)
 * and keep the texture-address units ~85 % busy; here every 1 KiB load
 * instruction covers whole 128-byte lines of at most 8 rows.
 *
 * Workgroup: 128 weight rows (gate/up: 64 w1 rows + the matching 64 w3 rows;
 * down: 128 w2 rows) x TOK = 16*TT token rows. TT = 1 (a weight stream): 4
 * waves of 32 rows each. TT = 4: 8 waves, 4 x 32 rows by 2 x 32 tokens, two
 * waves per SIMD, so that one wave's LDS operand reads (~27 B/clk each) and
 * conversions overlap the other's MFMAs. A stage is 256 reduction indices: weights (FP4 128 B
 * or FP8 256 B per row), the FP4 rows' eight E8M0 bytes, and the token rows
 * (fp16, 512 B each), in NST ring buffers; stage s+NST-1 is loaded while s
 * multiplies. 16-byte chunks are XOR-swizzled so the operand reads of 16
 * rows hit distinct banks. */
namespace {

typedef __attribute__((address_space(3))) void lds_void;
constexpr int KS = 256;

__device__ __forceinline__ void dma16(const void *src, uint8_t *dst)
{
    __builtin_amdgcn_global_load_lds(gptr(src), (lds_void *)dst, 16, 0, 0);
}
__device__ __forceinline__ void dma4(const void *src, uint8_t *dst)
{
    __builtin_amdgcn_global_load_lds(gptr(src), (lds_void *)dst, 4, 0, 0);
}

/* Default ring depth: FP4 16-row tiles two stages (2 x 25 KiB, three
 * workgroups per CU overlap each other's pipeline ramp), FP8 16-row tiles
 * three (3 x 40 KiB), 64-row tiles FP4 three, FP8 two. */
template <int WF, int TT>
constexpr int g2_stages() { return TT == 1 ? (WF == FMT_FP4_E8M0 ? 2 : 3) : (WF == FMT_FP4_E8M0 ? 3 : 2); }

template <int WF, int TT, int STAGES = g2_stages<WF, TT>()>
struct G2 {
    static constexpr bool FP4 = WF == FMT_FP4_E8M0;
    static constexpr int WB = FP4 ? KS / 2 : KS;         /* weight bytes per row per stage */
    static constexpr int ROWS = 128;
    static constexpr int TOK = 16 * TT;
    static constexpr int NWAVE = TT == 1 ? 4 : 8;        /* 64-row tiles: 2 waves / SIMD */
    static constexpr int WR = 4;                         /* waves along rows           */
    static constexpr int WT = NWAVE / WR;                /* waves along tokens         */
    static constexpr int RBW = 8 / WR;                   /* 16-row blocks per wave     */
    static constexpr int TTW = TT / WT;                  /* 16-token tiles per wave    */
    static constexpr int OFF_S = ROWS * WB;
    static constexpr int OFF_PAD = OFF_S + (FP4 ? ROWS * 8 : 0);   /* scale loads of waves 4+ */
    static constexpr int OFF_B = OFF_PAD + (FP4 && NWAVE > 4 ? 256 : 0);
    static constexpr int STAGE = OFF_B + TOK * KS * 2;
    static constexpr int NST = STAGES;
    static constexpr int LDS = NST * STAGE;
    static constexpr int NW = ROWS * WB / 1024 / NWAVE;  /* weight loads per wave per stage */
    static constexpr int NS = FP4 ? 1 : 0;               /* scale loads                */
    static constexpr int NB = TOK * KS * 2 / 1024 / NWAVE;   /* token-row loads        */
    static_assert(NW * NWAVE * 1024 == ROWS * WB && NB * NWAVE * 1024 == TOK * KS * 2, "load split");
    static constexpr int VM = NW + NS + NB;
    static_assert(LDS <= 160 * 1024, "LDS ring exceeds 160 KiB");
    static_assert((NST - 2) * VM <= 63, "vmcnt range");
};

/* physical 16-byte slot of logical chunk c in staged row r */
__device__ __forceinline__ int swz_w4(int r, int c) { return c ^ ((r >> 1) & 7); }   /* 8 slots   */
__device__ __forceinline__ int swz_w8(int r, int c) { return c ^ (r & 15); }         /* 16 slots  */
__device__ __forceinline__ int swz_b(int r, int c) { return c ^ (r & 15); }          /* 32 slots  */

/* B chunk (8 halves) of MFMA step sg (0..7) for lane group gq: the token side
 * of the reduction order the weight side is read in */
template <int WF>
__device__ __forceinline__ int bchunk(int gq, int sg)
{
    if constexpr (WF == FMT_FP4_E8M0) return 16 * (sg >> 2) + 4 * gq + (sg & 3);
    else return 8 * (sg >> 1) + 2 * gq + (sg & 1);
}

} // namespace

template <int WF, bool SWIGLU, int TT, int NS>
__global__ __launch_bounds__(512) void k_grouped2(GroupedArgs a)
{
    using C = G2<WF, TT, NS>;
    constexpr bool FP4 = C::FP4;
    constexpr int FEAT = SWIGLU ? 64 : 128;
    extern __shared__ __align__(16) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = wave_in_group();
    const int rr = lane & 15, gq = lane >> 4;
    const int nslab = a.N / FEAT;
    const int tile = blockIdx.x / nslab, slab = blockIdx.x - tile * nslab;

    int r0, ntok;
    DSV4QMat m1, m3;
    if (a.table) {
        const int E = a.n_experts;
        const int ntiles = ld_uniform(a.tile_pre, E);
        const TileRec tr = ld_uniform(a.tile_rec, tile);  /* read beside the count: one round trip */
        if ((tile >= ntiles) | (tr.ntok <= 0)) return;   /* whole workgroup */
        r0 = tr.r0;
        ntok = tr.ntok;
        const DSV4ExpertW e = ld_uniform(a.table, tr.grp);
        m1 = SWIGLU ? e.w1 : e.w2;
        m3 = e.w3;
    } else {
        r0 = tile * C::TOK;
        if (r0 >= a.nrows) return;
        ntok = min(C::TOK, a.nrows - r0);
        m1 = a.m1;
        m3 = a.m3;
    }
    const int f0 = slab * FEAT;
    const int K = a.K, N = a.N;
    if (!qmat_matches<WF>(m1, N, K) || (SWIGLU && !qmat_matches<WF>(m3, N, K))) {
        if (threadIdx.x == 0) atomicOr(a.status, ST_BAD_DESCRIPTOR);
        const float nan = __builtin_nanf("");
        for (int i = threadIdx.x; i < ntok * FEAT; i += 64 * C::NWAVE) {
            const size_t o = (size_t)(r0 + i / FEAT) * N + f0 + i % FEAT;
            if constexpr (SWIGLU) ((uint16_t *)a.out)[o] = (uint16_t)f16_bits(nan);
            else ((float *)a.out)[o] = nan;
        }
        return;
    }

    /* ---- load plan: per-lane source offsets of this wave's loads ---- */
    const int rowb = FP4 ? K / 2 : K;
    const int nst = K / KS, last = nst - 1;
    const uint8_t *wbase[C::NW];
    int wdst[C::NW];
#pragma unroll
    for (int i = 0; i < C::NW; i++) {
        const int j = wave * C::NW + i;                    /* 1 KiB instruction index */
        const int rpi = 1024 / C::WB;                      /* rows per instruction    */
        const int r = j * rpi + lane / (C::WB / 16);
        const int p = lane % (C::WB / 16);
        const bool up = SWIGLU && r >= 64;
        const int row = f0 + (SWIGLU ? (r & 63) : r);
        const int c = FP4 ? swz_w4(r, p) : swz_w8(r, p);
        wbase[i] = (const uint8_t *)(up ? m3.w : m1.w) + (size_t)row * rowb + 16 * c;
        wdst[i] = 1024 * j;
    }
    const uint8_t *sbase = nullptr;
    if constexpr (FP4) {
        const int r = 32 * (wave & 3) + lane / 2;          /* waves 4+ repeat rows into the pad */
        const bool up = SWIGLU && r >= 64;
        const int row = f0 + (SWIGLU ? (r & 63) : r);
        sbase = (const uint8_t *)(up ? m3.s : m1.s) + (size_t)row * (K / 32) + 4 * (lane & 1);
    }
    const uint16_t *bbase[C::NB];
#pragma unroll
    for (int i = 0; i < C::NB; i++) {
        const int j = wave * C::NB + i;
        const int t = 2 * j + lane / 32, p = lane & 31;
        const int r = t < ntok ? r0 + t : r0;
        const int src = a.row_tok ? a.row_tok[r] : r;
        bbase[i] = a.B + (size_t)src * K + 8 * swz_b(t, p);
    }
    auto issue = [&](int stg, uint8_t *buf) {
#pragma unroll
        for (int i = 0; i < C::NW; i++) dma16(wbase[i] + (size_t)stg * C::WB, buf + wdst[i]);
        if constexpr (FP4)
            dma4(sbase + (size_t)stg * 8, buf + (wave < 4 ? C::OFF_S + 256 * wave : C::OFF_PAD));
#pragma unroll
        for (int i = 0; i < C::NB; i++)
            dma16(bbase[i] + (size_t)stg * KS, buf + C::OFF_B + 1024 * (wave * C::NB + i));
    };

    /* ---- this wave's share ---- */
    const int wr = wave % C::WR, wt = wave / C::WR;
    int blk[C::RBW];
#pragma unroll
    for (int i = 0; i < C::RBW; i++) {
        constexpr int H = C::RBW / 2;
        blk[i] = SWIGLU ? (i < H ? H * wr + i : 4 + H * wr + (i - H)) : C::RBW * wr + i;
    }
    int ntw = 0;                                           /* live tiles of this wave */
#pragma unroll
    for (int u = 0; u < C::TTW; u++) ntw += 16 * (wt * C::TTW + u) < ntok ? 1 : 0;

    f4v acc[C::RBW][C::TTW];
#pragma unroll
    for (int i = 0; i < C::RBW; i++)
#pragma unroll
        for (int u = 0; u < C::TTW; u++) acc[i][u] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
    unsigned scale_bad = 0;

#pragma unroll
    for (int s0 = 0; s0 < C::NST - 1; s0++) issue(min(s0, last), lds + s0 * C::STAGE);

    /* The main loop, instantiated per count NT of this wave's live 16-token
     * tiles so that the MFMA sequence of a stage is straight-line code (a
     * branch per MFMA splits it into blocks the scheduler cannot overlap). */
    auto run = [&](auto ntc) {
        constexpr int NT = decltype(ntc)::value;
        for (int st = 0; st < nst; st++) {
            __builtin_amdgcn_s_waitcnt(0x0F70 | ((C::NST - 2) * C::VM & 15) | ((((C::NST - 2) * C::VM) >> 4) << 14));
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            {
                int nb = st + C::NST - 1;
                nb = nb >= C::NST ? nb - C::NST * (nb / C::NST) : nb;
                issue(min(st + C::NST - 1, last), lds + nb * C::STAGE);
            }
            if constexpr (NT > 0) {
                const uint8_t *buf = lds + (st % C::NST) * C::STAGE;

                /* token operands of this wave's live tiles, all 8 steps */
                h8 bop[NT][8];
#pragma unroll
                for (int u = 0; u < NT; u++) {
                    const int t = 16 * (wt * C::TTW + u) + rr;
                    const uint8_t *brow = buf + C::OFF_B + t * (KS * 2);
#pragma unroll
                    for (int sg = 0; sg < 8; sg++)
                        bop[u][sg] = *(const h8 *)(brow + 16 * swz_b(t, bchunk<WF>(gq, sg)));
                }
                /* FP8 chunk scales: 2 blocks of 128 per stage, per matrix */
                float fs[2][2] = {{1.0f, 1.0f}, {1.0f, 1.0f}};
                if constexpr (!FP4) {
                    const int nb = f0 / 128, kbn = K / 128;
#pragma unroll
                    for (int b = 0; b < 2; b++) {
                        const size_t si = (size_t)nb * kbn + 2 * st + b;
                        if constexpr (WF == FMT_FP8_E8M0) {
                            fs[0][b] = dev_e8m0(ld_u8(m1.s, si));
                            fs[1][b] = SWIGLU ? dev_e8m0(ld_u8(m3.s, si)) : 1.0f;
                        } else {
                            fs[0][b] = ld_f32(m1.s, si);
                            fs[1][b] = SWIGLU ? ld_f32(m3.s, si) : 1.0f;
                        }
                    }
                }
#pragma unroll
                for (int i = 0; i < C::RBW; i++) {
                    const int r = 16 * blk[i] + rr;            /* staged row */
                    if constexpr (FP4) {
                        const uint2 sc8 = *(const uint2 *)(buf + C::OFF_S + r * 8);
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            const int c = 4 * h + gq;
                            const u32x4 w16 = *(const u32x4 *)(buf + r * C::WB + 16 * swz_w4(r, c));
                            const uint32_t sb = ((c < 4 ? sc8.x : sc8.y) >> (8 * (c & 3))) & 0xFFu;
                            scale_bad |= (sb - 104u) > 36u;
                            const float cs = dev_e8m0(sb);
                            const u32x4 wv[2] = {w16, w16};
#pragma unroll
                            for (int s = 0; s < 4; s++) {
                                const h8 av = a_operand<WF>(wv, cs, s);
#pragma unroll
                                for (int u = 0; u < NT; u++) acc[i][u] = mfma16(av, bop[u][4 * h + s], acc[i][u]);
                            }
                        }
                    } else {
                        const float *fsm = fs[(SWIGLU && blk[i] >= 4) ? 1 : 0];
#pragma unroll
                        for (int b = 0; b < 2; b++) {          /* 128-K block of the stage */
                            f4v part[NT];
#pragma unroll
                            for (int u = 0; u < NT; u++) part[u] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                            for (int q2 = 0; q2 < 2; q2++) {
                                const int q = 2 * b + q2;
                                const int c = 4 * q + gq;
                                const u32x4 w16 = *(const u32x4 *)(buf + r * C::WB + 16 * swz_w8(r, c));
                                const u32x4 wv[2] = {w16, w16};
#pragma unroll
                                for (int s = 0; s < 2; s++) {
                                    const h8 av = a_operand<WF>(wv, 1.0f, s);   /* dwords 2s, 2s+1 */
#pragma unroll
                                    for (int u = 0; u < NT; u++) part[u] = mfma16(av, bop[u][2 * q + s], part[u]);
                                }
                            }
#pragma unroll
                            for (int u = 0; u < NT; u++)
#pragma unroll
                                for (int e = 0; e < 4; e++) acc[i][u][e] = fmaf(part[u][e], fsm[b], acc[i][u][e]);
                        }
                    }
                }
            }
        }
    };
    if (ntw >= C::TTW) run(IC<C::TTW>{});
    else if constexpr (C::TTW > 1) {
        if (ntw == 1) run(IC<1>{});
        else run(IC<0>{});
    } else run(IC<0>{});
    __builtin_amdgcn_s_waitcnt(0x0F70);     /* trailing repeat loads drain before exit */
    if (scale_bad) atomicOr(a.status, ST_SCALE_RANGE);

    unsigned range_bad = 0;
#pragma unroll
    for (int u = 0; u < C::TTW; u++) {
        const int t = 16 * (wt * C::TTW + u) + rr;
        if (t >= ntok) continue;
        const size_t orow = (size_t)(r0 + t) * N;
        const int ex = b_row_exp(a, r0 + t);
        if constexpr (SWIGLU) {
            constexpr int H = C::RBW / 2;
#pragma unroll
            for (int i = 0; i < H; i++)
                *(uint2 *)((uint16_t *)a.out + orow + f0 + 16 * blk[i] + 4 * gq) =
                    swiglu_f16x4(acc[i][u], acc[i + H][u], ex, a.limit, range_bad);
        } else {
#pragma unroll
            for (int i = 0; i < C::RBW; i++)
                *(f4v *)((float *)a.out + orow + f0 + 16 * blk[i] + 4 * gq) = unscale4(acc[i][u], ex);
        }
    }
    if (range_bad) atomicOr(a.status, range_bad);
}

/* ------------------------------------------- 128-token FP4 tiles (prefill) --- */

/* For buckets of many tokens (the prefill MoE layer). Workgroup: 8 waves,
 * 256 FP4 weight rows (gate/up: 128 w1 rows + the matching 128 w3 rows;
 * down: 256 w2 rows) x 128 token rows; each wave owns 64 rows x 64 tokens
 * (4 x 4 MFMA tiles), so one converted weight operand feeds 4 MFMAs and one
 * token operand 4 more, which keeps both the conversions (VALU) and the LDS
 * operand reads below the MFMA time.
 *
 * A stage is 128 reduction indices: 256 x 64 weight bytes, the rows' four
 * E8M0 bytes, and 128 x 256 bytes of fp16 token rows; three stages in flight.
 * Every operand arrives by buffer loads straight into LDS; token rows past
 * the end of the bucket use an offset beyond the buffer, which the hardware
 * answers with zeros and no memory traffic. Chunks are XOR-swizzled so that
 * the 16 rows of an MFMA operand read hit distinct banks:
 *   weight row r (64 B):  chunk c at slot c ^ ((r >> 2) & 3)
 *   token row t (256 B):  chunk c at slot c ^ (t & 15)
 * Reduction order: lane group gq's 16 weight bytes of a row (32 values, one
 * E8M0 block) feed MFMA steps s = 0..3, 8 values each; the token side reads
 * the same 8 indices, chunk 4 gq + s of the row. */
namespace {

struct G3 {
    static constexpr int KS = 128;
    static constexpr int ROWS = 256, TOK = 128, NWAVE = 8;
    static constexpr int WB = KS / 2;                        /* FP4 bytes per row per stage */
    static constexpr int OFF_S = ROWS * WB;                  /* E8M0: 256 B per wave        */
    static constexpr int OFF_B = OFF_S + NWAVE * 256;
    static constexpr int STAGE = OFF_B + TOK * KS * 2;
    static constexpr int NST = 3;
    static constexpr int LDS = NST * STAGE;
    static constexpr int NW = ROWS * WB / 1024 / NWAVE;      /* 16-row weight loads per wave */
    static constexpr int NB = TOK * KS * 2 / 1024 / NWAVE;   /* 4-row token loads per wave   */
    static constexpr int VM = NW + 1 + NB;
    static_assert(LDS <= 160 * 1024, "LDS ring exceeds 160 KiB");
    static_assert(NW * NWAVE * 1024 == ROWS * WB && NB * NWAVE * 1024 == TOK * KS * 2, "load split");
};

constexpr uint32_t RSRC_WORD3 = 0x00020000u;      /* raw dword buffer, gfx9 */
constexpr uint32_t OOB_OFFSET = 0x80000000u;      /* beyond every buffer    */

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void *p, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, (int)RSRC_WORD3);
}
__device__ __forceinline__ void bdma16(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff, uint8_t *dst)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)dst, 16, (int)voff, soff, 0, 0);
}
__device__ __forceinline__ void bdma4(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff, uint8_t *dst)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)dst, 4, (int)voff, soff, 0, 0);
}

/* 8 e2m1 values (one dword, low nibble first) times 2^e -> fp16 operand */
__device__ __forceinline__ h8 fp4_h8(uint32_t d, float sc)
{
    u32x4 v;
    v.x = pk_f16_fp4(d, sc, 0);
    v.y = pk_f16_fp4(d, sc, 1);
    v.z = pk_f16_fp4(d, sc, 2);
    v.w = pk_f16_fp4(d, sc, 3);
    return __builtin_bit_cast(h8, v);
}

} // namespace

template <bool SWIGLU>
__global__ __launch_bounds__(512) void k_grouped3(GroupedArgs a)
{
    using C = G3;
    constexpr int FEAT = SWIGLU ? 128 : 256;
    extern __shared__ __align__(16) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = wave_in_group();
    const int rr = lane & 15, gq = lane >> 4;
    const int nslab = a.N / FEAT;
    const int tile = blockIdx.x / nslab, slab = blockIdx.x - tile * nslab;

    int r0, ntok;
    DSV4QMat m1, m3;
    if (a.table) {
        const int E = a.n_experts;
        const int ntiles = ld_uniform(a.tile_pre, E);
        const TileRec tr = ld_uniform(a.tile_rec, tile);  /* read beside the count: one round trip */
        if ((tile >= ntiles) | (tr.ntok <= 0)) return;   /* whole workgroup */
        r0 = tr.r0;
        ntok = tr.ntok;
        const DSV4ExpertW e = ld_uniform(a.table, tr.grp);
        m1 = SWIGLU ? e.w1 : e.w2;
        m3 = e.w3;
    } else {
        r0 = tile * C::TOK;
        if (r0 >= a.nrows) return;
        ntok = min(C::TOK, a.nrows - r0);
        m1 = a.m1;
        m3 = a.m3;
    }
    const int f0 = slab * FEAT;
    const int K = a.K, N = a.N;
    if (!qmat_matches<FMT_FP4_E8M0>(m1, N, K) || (SWIGLU && !qmat_matches<FMT_FP4_E8M0>(m3, N, K)) ||
        !dword_aligned(m1) || (SWIGLU && !dword_aligned(m3))) {
        if (threadIdx.x == 0) atomicOr(a.status, ST_BAD_DESCRIPTOR);
        const float nan = __builtin_nanf("");
        for (int i = threadIdx.x; i < ntok * FEAT; i += 64 * C::NWAVE) {
            const size_t o = (size_t)(r0 + i / FEAT) * N + f0 + i % FEAT;
            if constexpr (SWIGLU) ((uint16_t *)a.out)[o] = (uint16_t)f16_bits(nan);
            else ((float *)a.out)[o] = nan;
        }
        return;
    }

    /* ---- load plan: per-lane byte offsets into the buffers ---- */
    const uint32_t rowb = (uint32_t)K / 2, srow = (uint32_t)K / 32;
    const int nst = K / C::KS, last = nst - 1;
    const __amdgpu_buffer_rsrc_t rw1 = buf_rsrc(m1.w, (uint32_t)N * rowb);
    const __amdgpu_buffer_rsrc_t rs1 = buf_rsrc(m1.s, (uint32_t)N * srow);
    const __amdgpu_buffer_rsrc_t rw3 = SWIGLU ? buf_rsrc(m3.w, (uint32_t)N * rowb) : rw1;
    const __amdgpu_buffer_rsrc_t rs3 = SWIGLU ? buf_rsrc(m3.s, (uint32_t)N * srow) : rs1;
    const __amdgpu_buffer_rsrc_t rb = buf_rsrc(a.B, (uint32_t)a.nrows * (uint32_t)K * 2u);
    uint32_t wofs[C::NW];
#pragma unroll
    for (int i = 0; i < C::NW; i++) {
        const int j = wave * C::NW + i;                 /* rows 16 j .. 16 j + 15 */
        const int r = 16 * j + lane / 4;
        const int c = (lane & 3) ^ ((r >> 2) & 3);
        const int row = f0 + (SWIGLU ? (r & 127) : r);
        wofs[i] = (uint32_t)row * rowb + 16u * c;
    }
    uint32_t sofs;
    {
        const int r = 32 * wave + (lane & 31);           /* lanes 32..63 repeat 0..31 */
        const int row = f0 + (SWIGLU ? (r & 127) : r);
        sofs = (uint32_t)row * srow;
    }
    uint32_t bofs[C::NB];
#pragma unroll
    for (int i = 0; i < C::NB; i++) {
        const int j = wave * C::NB + i;                 /* token rows 4 j .. 4 j + 3 */
        const int t = 4 * j + lane / 16;
        const int c = (lane & 15) ^ (t & 15);
        if (t < ntok) {
            const int src = a.row_tok ? a.row_tok[r0 + t] : r0 + t;
            bofs[i] = (uint32_t)src * (uint32_t)K * 2u + 16u * c;
        } else {
            bofs[i] = OOB_OFFSET;
        }
    }
    /* wave-uniform: which matrix each weight load and the scale load read */
    const bool up_s = SWIGLU && wave >= 4;
    auto issue = [&](int stg, uint8_t *buf) {
#pragma unroll
        for (int i = 0; i < C::NW; i++) {
            const bool up = SWIGLU && (wave * C::NW + i) >= 8;
            bdma16(up ? rw3 : rw1, wofs[i], stg * C::WB, buf + 1024 * (wave * C::NW + i));
        }
        bdma4(up_s ? rs3 : rs1, sofs, stg * (C::KS / 32), buf + C::OFF_S + 256 * wave);
#pragma unroll
        for (int i = 0; i < C::NB; i++)
            bdma16(rb, bofs[i], stg * C::KS * 2, buf + C::OFF_B + 1024 * (wave * C::NB + i));
    };

    /* ---- this wave's share: 4 row blocks x 4 token tiles ---- */
    const int wr = wave & 3, wt = wave >> 2;
    int blk[4];
#pragma unroll
    for (int i = 0; i < 4; i++) blk[i] = SWIGLU ? (i < 2 ? 2 * wr + i : 8 + 2 * wr + (i - 2)) : 4 * wr + i;
    int ntw = 0;
#pragma unroll
    for (int u = 0; u < 4; u++) ntw += 64 * wt + 16 * u < ntok ? 1 : 0;

    f4v acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int u = 0; u < 4; u++) acc[i][u] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
    unsigned scale_bad = 0;

#pragma unroll
    for (int s0 = 0; s0 < C::NST - 1; s0++) issue(min(s0, last), lds + s0 * C::STAGE);

    auto run = [&](auto ntc) {
        constexpr int NT = decltype(ntc)::value;
        for (int st = 0; st < nst; st++) {
            __builtin_amdgcn_s_waitcnt(0x0F70 | ((C::NST - 2) * C::VM & 15) | ((((C::NST - 2) * C::VM) >> 4) << 14));
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            {
                int nb = st + C::NST - 1;
                nb = nb >= C::NST ? nb - C::NST * (nb / C::NST) : nb;
                issue(min(st + C::NST - 1, last), lds + nb * C::STAGE);
            }
            if constexpr (NT > 0) {
                const uint8_t *buf = lds + (st % C::NST) * C::STAGE;
                u32x4 wraw[4];
                float cs[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int r = 16 * blk[i] + rr;
                    wraw[i] = *(const u32x4 *)(buf + r * C::WB + 16 * (gq ^ ((r >> 2) & 3)));
                    const uint32_t sw = *(const uint32_t *)(buf + C::OFF_S + (r >> 5) * 256 + (r & 31) * 4);
                    const uint32_t sb = (sw >> (8 * gq)) & 0xFFu;
                    scale_bad |= (sb - 104u) > 36u;
                    cs[i] = dev_e8m0(sb);
                }
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    h8 bop[NT];
#pragma unroll
                    for (int u = 0; u < NT; u++) {
                        const int t = 64 * wt + 16 * u + rr;
                        bop[u] = *(const h8 *)(buf + C::OFF_B + t * (C::KS * 2) + 16 * ((4 * gq + s) ^ rr));
                    }
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const uint32_t d = s == 0 ? wraw[i].x : s == 1 ? wraw[i].y : s == 2 ? wraw[i].z : wraw[i].w;
                        const h8 av = fp4_h8(d, cs[i]);
#pragma unroll
                        for (int u = 0; u < NT; u++) acc[i][u] = mfma16(av, bop[u], acc[i][u]);
                    }
                }
            }
        }
    };
    switch (ntw) {
    case 4: run(IC<4>{}); break;
    case 3: run(IC<3>{}); break;
    case 2: run(IC<2>{}); break;
    case 1: run(IC<1>{}); break;
    default: run(IC<0>{}); break;
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);     /* trailing repeat loads drain before exit */
    if (scale_bad) atomicOr(a.status, ST_SCALE_RANGE);

    unsigned range_bad = 0;
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int t = 64 * wt + 16 * u + rr;
        if (t >= ntok) continue;
        const size_t orow = (size_t)(r0 + t) * N;
        const int ex = b_row_exp(a, r0 + t);
        if constexpr (SWIGLU) {
#pragma unroll
            for (int i = 0; i < 2; i++)
                *(uint2 *)((uint16_t *)a.out + orow + f0 + 16 * blk[i] + 4 * gq) =
                    swiglu_f16x4(acc[i][u], acc[i + 2][u], ex, a.limit, range_bad);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                *(f4v *)((float *)a.out + orow + f0 + 16 * blk[i] + 4 * gq) = unscale4(acc[i][u], ex);
        }
    }
    if (range_bad) atomicOr(a.status, range_bad);
}

/* -------------------------------- FP4 weights streamed to registers --- */

/* For buckets of up to a few dozen tokens, where an expert's weights are used
 * so few times that streaming them is the bound (the batched decode, short
 * prompts). Workgroup: four waves, a tile of 16 token rows. Each wave owns 16
 * rows of each of two 64-row halves (gate/up: the w1 rows and the matching w3
 * rows; down: rows f0 .. f0 + 63 and f0 + 64 .. f0 + 127) over all of K. A
 * step is 256 reduction indices (128 bytes of a row), a group two steps: two
 * groups of weights are in flight straight to registers, and the tile's token
 * rows (fp16) of the same steps pass through four LDS slots, every wave
 * loading its share in the same order as its weights, so that one counted
 * wait covers both.
 *
 * A load instruction reads whole 128-byte lines of eight rows: lane
 * 16 g + 2 r + h takes bytes 64 h + 16 g of row 2 r + j (j the instruction),
 * and a lane-pair exchange forms the MFMA operands of rows 2 r + h. The
 * reduction order, and so the bits, are k_grouped2's. The rows' E8M0 bytes
 * go to LDS once, 8-byte pieces (a step's) XOR-swizzled by the row so that
 * the 16 rows of a read start in distinct banks.
 *
 * Measured, 64 tokens x top-6 of 256 experts (Zipf), hidden 4096, inter 2048:
 * gate/up 217 -> 172 us (6.1 TB/s), down 108 -> 92 us against k_grouped2,
 * which passes the weights through LDS a step at a time. What decided: 256
 * contiguous bytes of a row asked for together (one step at a time: 210 and
 * 105), three workgroups a CU (113 registers, 48 KB of LDS; two: 352 against
 * 322 us for the call), weights that nothing else reads loaded non-temporal,
 * and few vector operations per weight (scale bytes shifted into place and
 * checked once at the end). */
namespace {

constexpr int GW_G = 2;                            /* steps per group                     */
constexpr int GW_XI = 2;                           /* token load instructions, wave, step */
constexpr int GW_VM = GW_G * (4 + GW_XI);          /* loads per wave and group            */
constexpr int GW_SLOT = 16 * KS * 2;               /* a step's 16 token rows              */
constexpr int GW_KMAX = 8192;
static_assert(GW_VM <= 15, "the wait below encodes vmcnt in four bits");
constexpr int gw_lds(int K) { return 2 * GW_G * GW_SLOT + 128 * (K / 32); }

constexpr int CPOL_NT = 2;                         /* non-temporal */
template <int CPOL>
__device__ __forceinline__ u32x4 bload16(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff)
{
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, soff, CPOL));
}

/* whether one of four E8M0 bytes lies outside 104..140 */
__device__ __forceinline__ bool scales_bad(uint32_t s)
{
    bool bad = false;
#pragma unroll
    for (int b = 0; b < 4; b++) bad |= ((s >> (8 * b)) & 0xFFu) - 104u > 36u;
    return bad;
}

} // namespace

template <bool SWIGLU>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_grouped_w(GroupedArgs a)
{
    constexpr int FEAT = SWIGLU ? 64 : 128;
    extern __shared__ __align__(16) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = wave_in_group();
    const int rr = lane & 15, gq = lane >> 4;
    const int nslab = a.N / FEAT;
    const int tile = blockIdx.x / nslab, slab = blockIdx.x - tile * nslab;
    const int ntiles = ld_uniform(a.tile_pre, a.n_experts);
    const TileRec tr = ld_uniform(a.tile_rec, tile);      /* read beside the count: one round trip */
    if ((tile >= ntiles) | (tr.ntok <= 0)) return;        /* whole workgroup */
    const int r0 = tr.r0, ntok = tr.ntok;
    const DSV4ExpertW e = ld_uniform(a.table, tr.grp);
    const DSV4QMat m1 = SWIGLU ? e.w1 : e.w2, m3 = e.w3;
    const int f0 = slab * FEAT;
    const int K = a.K, N = a.N;
    if (!qmat_matches<FMT_FP4_E8M0>(m1, N, K) || (SWIGLU && !qmat_matches<FMT_FP4_E8M0>(m3, N, K)) ||
        !dword_aligned(m1) || (SWIGLU && !dword_aligned(m3))) {
        if (threadIdx.x == 0) atomicOr(a.status, ST_BAD_DESCRIPTOR);
        const float nan = __builtin_nanf("");
        for (int i = threadIdx.x; i < ntok * FEAT; i += 256) {
            const size_t o = (size_t)(r0 + i / FEAT) * N + f0 + i % FEAT;
            if constexpr (SWIGLU) ((uint16_t *)a.out)[o] = (uint16_t)f16_bits(nan);
            else ((float *)a.out)[o] = nan;
        }
        return;
    }
    /* groups rounded up to an even count: steps past the end multiply zeros */
    const int nst = K / KS, ngr = (nst + 2 * GW_G - 1) / (2 * GW_G) * 2;
    /* the two halves' rows: f0 .. f0 + 63 of m1 and of m3, or the next 64 of m1 */
    const uint32_t rowb = (uint32_t)K / 2, srow = (uint32_t)K / 32;
    const uint8_t *wb[2] = {(const uint8_t *)m1.w + (size_t)f0 * rowb,
                            SWIGLU ? (const uint8_t *)m3.w + (size_t)f0 * rowb
                                   : (const uint8_t *)m1.w + (size_t)(f0 + 64) * rowb};
    const uint8_t *sb[2] = {(const uint8_t *)m1.s + (size_t)f0 * srow,
                            SWIGLU ? (const uint8_t *)m3.s + (size_t)f0 * srow
                                   : (const uint8_t *)m1.s + (size_t)(f0 + 64) * srow};
    uint8_t *ssc = lds + 2 * GW_G * GW_SLOT;
    const int npair = (int)srow / 8;
    const int smask = (npair & (npair - 1)) ? 0 : min(npair - 1, 15);
    {
        /* LDS dword d of a half is dword c = d % sd of row d / sd, whose
         * 8-byte piece c / 2 holds the step (c / 2) ^ (row & smask); wave w
         * loads half w / 2, alternate instructions of the two waves */
        const __amdgpu_buffer_rsrc_t rs = buf_rsrc(wave < 2 ? sb[0] : sb[1], 64u * srow);
        const uint32_t sd = srow / 4, inv = (1u << 20) / sd + 1;    /* exact for d < 64 sd, sd <= 64 */
        uint8_t *dst = ssc + (wave >> 1) * 64 * srow;
        for (uint32_t i = wave & 1; i < sd; i += 2) {
            const uint32_t d = 64 * i + lane, row = (d * inv) >> 20, c = d - row * sd;
            bdma4(rs, row * srow + 8 * ((c >> 1) ^ (row & (uint32_t)smask)) + 4 * (c & 1), 0, dst + 256 * i);
        }
    }
    /* this wave's loads: token rows (rows past the tile's end answer with
     * zeros) and weights; steps past the end read nothing but are counted */
    const __amdgpu_buffer_rsrc_t rb = buf_rsrc(a.B, (uint32_t)a.nrows * (uint32_t)K * 2u);
    const __amdgpu_buffer_rsrc_t rw[2] = {buf_rsrc(wb[0], 64u * rowb), buf_rsrc(wb[1], 64u * rowb)};
    const __amdgpu_buffer_rsrc_t none = buf_rsrc(wb[0], 0);
    uint32_t xofs[GW_XI];
#pragma unroll
    for (int i = 0; i < GW_XI; i++) {
        const int t = 2 * (wave * GW_XI + i) + lane / 32;
        const int src = t < ntok ? (a.row_tok ? a.row_tok[r0 + t] : r0 + t) : 0;
        xofs[i] = t < ntok ? (uint32_t)src * (uint32_t)K * 2u + 16u * (uint32_t)swz_b(t, lane & 31) : OOB_OFFSET;
    }
    const uint32_t wofs0 = (uint32_t)(16 * wave + (lane & 14)) * rowb + 64u * (lane & 1) + 16u * gq;
    const uint32_t wofs1 = wofs0 + rowb;
    struct W { u32x4 v[GW_G][2][2]; };             /* [step][half][instruction] */
    auto load = [&](W &w, int g, auto cpol) {
        asm volatile("" ::: "memory");
        uint8_t *slot = lds + (g & 1) * (GW_G * GW_SLOT);
#pragma unroll
        for (int k = 0; k < GW_G; k++)
#pragma unroll
            for (int i = 0; i < GW_XI; i++)
                bdma16(g * GW_G + k < nst ? rb : none, xofs[i], (g * GW_G + k) * (KS * 2),
                       slot + k * GW_SLOT + 1024 * (wave * GW_XI + i));
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int k = 0; k < GW_G; k++)
                    w.v[k][m][j] = bload16<decltype(cpol)::value>(g * GW_G + k < nst ? rw[m] : none,
                                                                  j ? wofs1 : wofs0, (g * GW_G + k) * (KS / 2));
        asm volatile("" ::: "memory");
    };
    f4v acc[2] = {f4v{0.0f, 0.0f, 0.0f, 0.0f}, f4v{0.0f, 0.0f, 0.0f, 0.0f}};
    const bool odd = lane & 1;
    const uint8_t *sp = ssc + (16 * wave + rr) * srow;
    const int sx = (16 * wave + rr) & smask;
    auto compute = [&](const u32x4 (&v)[2][2], int g, int k) {
        const int st = min(g * GW_G + k, nst - 1);  /* for the scales; the weights past the end are zeros */
        const uint8_t *brow = lds + ((g & 1) * GW_G + k) * GW_SLOT + rr * (KS * 2);
        float sc[2][2];
        u32x4 op[2][2];                            /* [matrix half][128-index half of the step] */
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const uint2 s8 = *(const uint2 *)(sp + m * 64 * srow + 8 * (st ^ sx));
            /* as fp32 exponents: exact for the bytes 104..140 this path decodes */
            sc[m][0] = __uint_as_float(((s8.x >> (8 * gq)) & 0xFFu) << 23);
            sc[m][1] = __uint_as_float(((s8.y >> (8 * gq)) & 0xFFu) << 23);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t x0 = v[m][0][i], x1 = v[m][1][i];
                const uint32_t p0 = (uint32_t)__builtin_amdgcn_mov_dpp((int)x0, DPP_QUAD_1032, 0xF, 0xF, false);
                const uint32_t p1 = (uint32_t)__builtin_amdgcn_mov_dpp((int)x1, DPP_QUAD_1032, 0xF, 0xF, false);
                op[m][0][i] = odd ? p1 : x0;       /* row 2 r + h: half 0, then half 1 */
                op[m][1][i] = odd ? x1 : p0;
            }
        }
        /* token operands one MFMA step ahead of their use */
        h8 bop[2];
        auto read_b = [&](int i) { return *(const h8 *)(brow + 16 * swz_b(rr, 16 * (i >> 2) + 4 * gq + (i & 3))); };
        bop[0] = read_b(0);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            if (i < 7) bop[(i + 1) & 1] = read_b(i + 1);
            asm volatile("" ::: "memory");
#pragma unroll
            for (int m = 0; m < 2; m++)
                acc[m] = mfma16(fp4_h8(op[m][i >> 2][i & 3], sc[m][i >> 2]), bop[i & 1], acc[m]);
        }
    };
    auto run = [&](auto cpol) {
        W ring[2];
        load(ring[0], 0, cpol);
        load(ring[1], 1, cpol);
        for (int g = 0; g < ngr; g += 2) {
#pragma unroll
            for (int d = 0; d < 2; d++) {
                /* this group's tokens and weights (and, before the first, the
                 * scales) have landed: only the next group's are outstanding */
                __builtin_amdgcn_s_waitcnt(0x0F70 | GW_VM);
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
#pragma unroll
                for (int k = 0; k < GW_G; k++) {
                    compute(ring[d].v[k], g + d, k);
                    /* nothing of a later step moves up: its first use of a
                     * weight register would wait for that register's load */
                    __builtin_amdgcn_sched_barrier(0);
                }
                __builtin_amdgcn_s_waitcnt(0xC07F);    /* lgkmcnt(0): its slots have been read */
                __builtin_amdgcn_s_barrier();
                load(ring[d], g + d + 2, cpol);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    /* a bucket of one tile reads its weights once; with more, the tiles run
     * side by side and the later ones find the weights in the L2 (non-temporal
     * throughout: 1,000 tokens 1,267 against 1,100 us) */
    if (tr.bucket <= 16) run(IC<CPOL_NT>{});
    else run(IC<0>{});
    __builtin_amdgcn_s_waitcnt(0x0F70);            /* the counted loads past the end */
    bool scale_bad = false;                        /* this wave's 32 rows */
    for (int m = 0; m < 2; m++)
        for (int i = lane; i < 4 * (int)srow; i += 64)
            scale_bad |= scales_bad(*(const uint32_t *)(ssc + (m * 64 + 16 * wave) * srow + 4 * i));
    if (scale_bad) atomicOr(a.status, ST_SCALE_RANGE);

    if (rr >= ntok) return;
    unsigned range_bad = 0;
    const size_t orow = (size_t)(r0 + rr) * N + f0 + 16 * wave + 4 * gq;
    const int ex = b_row_exp(a, r0 + rr);
    if constexpr (SWIGLU) {
        *(uint2 *)((uint16_t *)a.out + orow) = swiglu_f16x4(acc[0], acc[1], ex, a.limit, range_bad);
        if (range_bad) atomicOr(a.status, range_bad);
    } else {
        *(f4v *)((float *)a.out + orow) = unscale4(acc[0], ex);
        *(f4v *)((float *)a.out + orow + 64) = unscale4(acc[1], ex);
    }
}

/* ------------------------------------------------ dense FP8 (many tokens) --- */

/* One FP8 matrix (or the shared expert's w1 and w3) against many tokens: the
 * dense form in tiles of 128 weight rows x 16 T tokens. Products, order and
 * so bits are k_grouped2's.
 *
 * Four waves along the rows, 32 each (gate/up: 16 w1 rows and the w3 rows of
 * the same features), by one over all 16 T tokens (T = 1 .. 3) or two over 8 T
 * each (T = 4, 6). A stage is one 128-wide reduction block, rows and tokens by
 * buffer loads straight to LDS, NST stages in a ring. A wave
 * reads its operands of the next stage while it multiplies one, a read to
 * two MFMAs and a load between them, so that the barrier between stages waits
 * for no read. A row block's scales sit in one register, one block per lane.
 *
 * Bound: the LDS path of a wave (32 clk per 16-byte read, 16 clk per MFMA; no
 * reads: 6 of 19 us gone at 4096 x 4096, 333 tokens, T = 3) and the loads' L2
 * traffic (no loads: 5). Reads and MFMAs of one wave hardly overlap, so waves
 * per SIMD count: T = 6 30.6 us in eight waves, 37.7 in four. 4096 x 4096, the
 * call: 333 tokens 38.0 -> 25.3 us, 700 tokens 70.0 -> 35.9; 1024 x 4096, 64
 * tokens 22.8 -> 16.1, 1,300 tokens 61.4 -> 28.0 (k_grouped2 and the seam
 * GEMM). */
namespace {

constexpr int D8_KMAX = 64 * KC;
constexpr int D8_W = 128 * KC;                         /* weight bytes of a stage */

template <int T> struct D8 {
    static constexpr int WT = T >= 4 ? 2 : 1, NWAVE = 4 * WT;      /* 4 waves along rows, WT along tokens */
    static constexpr int U = T / WT;                   /* 16-token groups of a wave */
    static constexpr int STAGE = D8_W + 16 * T * KC * 2;
    static constexpr int NST = T == 1 ? 4 : T == 2 ? 3 : T == 3 ? 5 : 4;
    static constexpr int LDS = NST * STAGE;
    static constexpr int LW = 16 / NWAVE, LX = 4 * T / NWAVE;      /* a wave's loads a stage  */
    static constexpr int VM = LW + LX;
    static_assert(LDS <= 160 * 1024 && (NST - 1) * VM < 64 && T % WT == 0, "ring");
};

template <int N>
__device__ __forceinline__ void d8_wait()
{
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

} // namespace

template <bool SWIGLU, bool WF32S, int T>
__global__ __launch_bounds__(64 * D8<T>::NWAVE) void k_dense8(GroupedArgs a)
{
    using C = D8<T>;
    constexpr int FEAT = SWIGLU ? 64 : 128;
    extern __shared__ __align__(16) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = wave_in_group();
    const int rr = lane & 15, gq = lane >> 4, wr = wave & 3, wt = wave >> 2;
    constexpr int U = C::U;
    const int K = a.K, N = a.N, M = a.nrows;
    const int mt = (M + 16 * T - 1) / (16 * T), nslab = N / FEAT, nst = K / KC;
    /* the slabs of one XCD (workgroups go round the eight) side by side, each
     * with all its token tiles: W is then fetched into one L2 only */
    int lin = blockIdx.x;
    if (nslab % 8 == 0) lin = (lin % 8) * (nslab / 8 * mt) + lin / 8;
    const int f0 = lin / mt * FEAT, m0 = lin % mt * (16 * T);

    const bool w_up = SWIGLU && wave >= C::NWAVE / 2;             /* staged rows 64 .. 127 are w3's */
    const __amdgpu_buffer_rsrc_t rw = buf_rsrc(w_up ? a.m3.w : a.m1.w, (uint32_t)N * (uint32_t)K);
    const __amdgpu_buffer_rsrc_t rx = buf_rsrc(a.B, (uint32_t)M * (uint32_t)K * 2u);
    uint32_t wo[C::LW], xo[C::LX];
#pragma unroll
    for (int i = 0; i < C::LW; i++) {
        const int r = 8 * (C::LW * wave + i) + lane / 8;
        wo[i] = (uint32_t)(f0 + (SWIGLU ? r & 63 : r)) * (uint32_t)K + 16u * (uint32_t)swz_w4(r, lane & 7);
    }
#pragma unroll
    for (int i = 0; i < C::LX; i++) {
        const int r = 4 * (C::LX * wave + i) + lane / 16;
        xo[i] = m0 + r < M ? (uint32_t)(m0 + r) * (uint32_t)K * 2u + 16u * (uint32_t)swz_b(r, lane & 15) : OOB_OFFSET;
    }
    /* load i of a wave's share of stage st; past the end zeros, no traffic */
    auto issue = [&](int st, int slot, int i) {
        const uint32_t oob = st < nst ? 0u : OOB_OFFSET;
        uint8_t *buf = lds + slot * C::STAGE;
        if (i < C::LW) bdma16(rw, wo[min(i, C::LW - 1)] | oob, st * KC, buf + 1024 * (C::LW * wave + i));
        else bdma16(rx, xo[max(i - C::LW, 0)] | oob, st * KC * 2, buf + D8_W + 1024 * (C::LX * wave + i - C::LW));
    };
    uint32_t wsc[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const void *s = SWIGLU && i ? a.m3.s : a.m1.s;
        const size_t si = (size_t)(f0 / 128) * nst + min(lane, nst - 1);
        wsc[i] = WF32S ? __float_as_uint(ld_f32(s, si)) : __float_as_uint(dev_e8m0(ld_u8(s, si)));
    }
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("" : "+v"(wsc[0]), "+v"(wsc[1]));     /* their wait before the ring's loads */
#endif
#pragma unroll
    for (int s = 0; s < C::NST; s++)
#pragma unroll
        for (int i = 0; i < C::VM; i++) issue(s, s, i);

    /* this wave's operands of a stage */
    struct Op { u32x4 w[2][2]; h8 x[4][U]; };
    const int wrow[2] = {SWIGLU ? 16 * wr + rr : 32 * wr + rr, SWIGLU ? 64 + 16 * wr + rr : 32 * wr + 16 + rr};
    auto read_w = [&](Op &o, const uint8_t *buf, int h, int i) {
        o.w[h][i] = *(const u32x4 *)(buf + wrow[i] * KC + 16 * swz_w4(wrow[i], 4 * h + gq));
    };
    auto read_x = [&](Op &o, const uint8_t *buf, int j, int u) {
        const int t = 16 * (U * wt + u) + rr;
        o.x[j][u] = *(const h8 *)(buf + D8_W + t * (2 * KC) + 16 * swz_b(t, 8 * (j >> 1) + 2 * gq + (j & 1)));
    };
    auto decode = [&](h8 (&av)[2], const Op &o, int j) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const u32x4 wv[2] = {o.w[j >> 1][i], o.w[j >> 1][i]};
            av[i] = a_operand<FMT_FP8_E8M0>(wv, 1.0f, j & 1);
        }
    };
    f4v acc[2][U], part[2][U];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int u = 0; u < U; u++) acc[i][u] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
    int slot = 0;                                      /* of the stage multiplied next */
    auto step = [&](const Op &cur, Op &nxt, int st) {
        /* this stage's operands are in registers, and this wave's loads of
         * the next stage have landed; after the barrier every wave's */
        __builtin_amdgcn_s_waitcnt(0xC07F);
        d8_wait<(C::NST - 2) * C::VM>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int free = slot;
        slot = slot + 1 == C::NST ? 0 : slot + 1;
        const uint8_t *buf = lds + slot * C::STAGE;
        h8 av[2][2];                                   /* decoded a step ahead */
        decode(av[0], cur, 0);
#pragma unroll
        for (int j = 0; j < 4; j++) {
#pragma unroll
            for (int u = 0; u < U; u++) {
#pragma unroll
                for (int i = 0; i < C::VM; i++)
                    if (1 + i * (4 * U - 1) / C::VM == U * j + u) issue(st + C::NST, free, i);
                read_x(nxt, buf, j, u);
                if ((j & 1) == 0 && u == 0) read_w(nxt, buf, j >> 1, 0);
                if ((j & 1) == 0 && u == U - 1) read_w(nxt, buf, j >> 1, 1);
                part[0][u] = mfma16(av[j & 1][0], cur.x[j][u], j == 0 ? f4v{0.0f, 0.0f, 0.0f, 0.0f} : part[0][u]);
                if (u == 0 && j < 3) decode(av[(j + 1) & 1], cur, j + 1);
                part[1][u] = mfma16(av[j & 1][1], cur.x[j][u], j == 0 ? f4v{0.0f, 0.0f, 0.0f, 0.0f} : part[1][u]);
                DSV4_ORDER();
            }
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const float sw = st < nst ? __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)wsc[i], st)) : 0.0f;
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[i][u][e] = fmaf(part[i][u][e], sw, acc[i][u][e]);
        }
        DSV4_ORDER();
    };

    d8_wait<(C::NST - 1) * C::VM>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    Op o0, o1;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (j < 2) { read_w(o0, lds, j, 0); read_w(o0, lds, j, 1); }
#pragma unroll
        for (int u = 0; u < U; u++) read_x(o0, lds, j, u);
    }
    for (int st = 0; st < nst; st += 2) {
        step(o0, o1, st);
        step(o1, o0, st + 1);
    }
    d8_wait<0>();                                      /* the loads past the end */

    unsigned range_bad = 0;
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int m = m0 + 16 * (U * wt + u) + rr;
        if (m >= M) continue;
        const int ex = a.bexp ? a.bexp[m] : 0;
        if constexpr (SWIGLU) {
            *(uint2 *)((uint16_t *)a.out + (size_t)m * N + f0 + 16 * wr + 4 * gq) =
                swiglu_f16x4(acc[0][u], acc[1][u], ex, a.limit, range_bad);
        } else {
#pragma unroll
            for (int i = 0; i < 2; i++)
                *(f4v *)((float *)a.out + (size_t)m * N + f0 + 32 * wr + 16 * i + 4 * gq) = unscale4(acc[i][u], ex);
        }
    }
    if (range_bad) atomicOr(a.status, range_bad);
}

/* ------------------------------------------------------------- combine --- */

/* 4 consecutive outputs of one token per thread. The positions and weights
 * of all k (topk <= 16) are read first and every Y load is issued before the
 * first is used, so a thread waits one memory latency rather than topk
 * dependent pairs of them; the sum stays in k order. */
__global__ __launch_bounds__(256) void k_moe_combine(CombineArgs a)
{
    constexpr int KMAX = 16;
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int q = a.hidden / 4;
    if (i >= (size_t)a.n * q) return;
    const int t = (int)(i / q), c = (int)(i - (size_t)t * q) * 4;
    const int topk = a.topk;
    int p[KMAX];
    float wk[KMAX];
#pragma unroll
    for (int k = 0; k < KMAX; k++) {
        p[k] = k < topk ? a.pos[(size_t)t * topk + k] : -1;
        wk[k] = k < topk ? a.w[(size_t)t * topk + k] : 0.0f;
    }
    f32x4 v[KMAX];
    const float nan = __builtin_nanf("");
#pragma unroll
    for (int k = 0; k < KMAX; k++) {
        if (k < topk && p[k] >= 0) v[k] = *(const f32x4 *)(a.Y + (size_t)p[k] * a.hidden + c);
        else v[k] = f32x4{nan, nan, nan, nan};
    }
    f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
    if (a.YS) s = *(const f32x4 *)(a.YS + (size_t)t * a.hidden + c);
    f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < KMAX; k++) {
        if (k < topk) {
            o.x = __fadd_rn(o.x, __fmul_rn(wk[k], v[k].x));
            o.y = __fadd_rn(o.y, __fmul_rn(wk[k], v[k].y));
            o.z = __fadd_rn(o.z, __fmul_rn(wk[k], v[k].z));
            o.w = __fadd_rn(o.w, __fmul_rn(wk[k], v[k].w));
        }
    }
    if (a.YS) {
        o.x = __fadd_rn(o.x, s.x);
        o.y = __fadd_rn(o.y, s.y);
        o.z = __fadd_rn(o.z, s.z);
        o.w = __fadd_rn(o.w, s.w);
    }
    *(f32x4 *)(a.out + (size_t)t * a.hidden + c) = o;
}

/* ------------------------------------------------------------ launchers --- */

hipError_t moe_route_launch(const RouteArgs &a, const RowsF16Args &x16, hipStream_t st)
{
    if (a.n_experts < 1 || a.n_experts > MAX_ROUTE_EXPERTS) return hipErrorInvalidValue;
    const int nch = (a.npairs + 1023) / 1024;
    const int cpb = nch > ROUTE_MAX_BLOCKS ? (nch + ROUTE_MAX_BLOCKS - 1) / ROUTE_MAX_BLOCKS : 1;
    const int blocks = nch > 0 ? (nch + cpb - 1) / cpb : 1;
    if (a.chist && nch >= ROUTE_PRECOUNT_CHUNKS) {
        hipLaunchKernelGGL(k_moe_route_count, dim3(nch + x16.rows), dim3(1024), 0, st, a, nch, x16);
        hipLaunchKernelGGL(k_moe_route<true>, dim3(blocks), dim3(1024), 0, st, a, cpb, blocks, x16);
    } else {
        hipLaunchKernelGGL(k_moe_route<false>, dim3(blocks + x16.rows), dim3(1024), 0, st, a, cpb, blocks, x16);
    }
    return hipGetLastError();
}

hipError_t to_f16_rows_launch(uint16_t *o, int *ex, const float *x, int rows, int cols,
                              hipStream_t st)
{
    if (rows <= 0 || cols <= 0 || cols % 8) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_to_f16_rows, dim3((unsigned)rows), dim3(256), 0, st, o, ex, x, cols);
    return hipGetLastError();
}

int grouped_rows_per_tile(int tt) { return tt == GROUPED_STREAM ? 16 : 16 * tt; }

template <int WF, bool SW, int TT, int NS>
static hipError_t grouped2_ns(const GroupedArgs &a, long items, hipStream_t st)
{
    static bool attr_done = false;
    if (!attr_done) {
        const hipError_t e = hipFuncSetAttribute((const void *)k_grouped2<WF, SW, TT, NS>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 G2<WF, TT, NS>::LDS);
        if (e != hipSuccess) return e;
        attr_done = true;
    }
    constexpr int lds_bytes = G2<WF, TT, NS>::LDS, threads = 64 * G2<WF, TT, NS>::NWAVE;
    hipLaunchKernelGGL((k_grouped2<WF, SW, TT, NS>), dim3((unsigned)items), dim3(threads), lds_bytes, st, a);
    return hipGetLastError();
}

/* FP8 16-row tiles (a shared expert of up to 64 tokens): when the grid
 * outnumbers the CUs, two stages (2 x 40 KiB) so two workgroups share a CU
 * (hidden 4096, inter 6144, 64 tokens, the call 94 -> 80 us, inter 8192 122 ->
 * 105); up to one workgroup per CU the three-stage ring keeps more of a lone
 * workgroup's loads in flight (7168 x 4608, 34 tokens 81.5 against 85.5 us). */
template <int WF, bool SW, int TT>
static hipError_t grouped2(const GroupedArgs &a, long items, hipStream_t st)
{
    if constexpr (WF != FMT_FP4_E8M0 && TT == 1) {
        if (items > CUS) return grouped2_ns<WF, SW, TT, 2>(a, items, st);
    }
    return grouped2_ns<WF, SW, TT, g2_stages<WF, TT>()>(a, items, st);
}

template <bool SW, bool WS, int T>
static hipError_t dense8_t(const GroupedArgs &a, hipStream_t st)
{
    static bool attr_done = false;
    if (!attr_done) {
        const hipError_t e = hipFuncSetAttribute((const void *)k_dense8<SW, WS, T>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, D8<T>::LDS);
        if (e != hipSuccess) return e;
        attr_done = true;
    }
    const long items = (long)((a.nrows + 16 * T - 1) / (16 * T)) * (a.N / (SW ? 64 : 128));
    constexpr int lds_bytes = D8<T>::LDS;
    hipLaunchKernelGGL((k_dense8<SW, WS, T>), dim3((unsigned)items), dim3(64 * D8<T>::NWAVE), lds_bytes, st, a);
    return hipGetLastError();
}

/* k_dense8 takes rows of up to its scale register's 64 blocks, weights on
 * 16-byte boundaries and 31-bit offsets; what its callers' other forms flag
 * in the kernel goes to those. */
bool grouped_dense_ok(const GroupedArgs &a, int fmt, bool swiglu)
{
    auto ok = [&](const DSV4QMat &m) {
        return m.rows == a.N && m.cols == a.K && m.w && m.s && ((uintptr_t)m.w & 15) == 0 && m.blk_r == 128 &&
               m.blk_c == 128 && m.wdt == (fmt == FMT_FP8_F32S ? DSV4_WFP8_F32S : DSV4_WFP8);
    };
    return !a.table && (fmt == FMT_FP8_E8M0 || fmt == FMT_FP8_F32S) && a.K % KC == 0 && a.K <= D8_KMAX &&
           a.N % 128 == 0 && a.nrows > 0 && ok(a.m1) && (!swiglu || ok(a.m3)) &&
           (size_t)a.nrows * a.K * 2 < (1u << 31) && (size_t)a.N * a.K < (1u << 31);
}

template <bool WS, bool SW>
static hipError_t dense8(const GroupedArgs &a, hipStream_t st)
{
    long cost;
    switch (dense8_tile(a.nrows, a.N / (SW ? 64 : 128), &cost)) {
    case 1: return dense8_t<SW, WS, 1>(a, st);
    case 2: return dense8_t<SW, WS, 2>(a, st);
    case 3: return dense8_t<SW, WS, 3>(a, st);
    case 4: return dense8_t<SW, WS, 4>(a, st);
    default: return dense8_t<SW, WS, 6>(a, st);
    }
}

template <int WF, bool SW>
static hipError_t grouped_tt(const GroupedArgs &a, int tt, long items, hipStream_t st)
{
    if (a.K % KS == 0) {        /* LDS-staged form: one workgroup per item */
        return tt == 1 ? grouped2<WF, SW, 1>(a, items, st) : grouped2<WF, SW, 4>(a, items, st);
    }
    const dim3 grid((unsigned)((items + 3) / 4)), block(256);
    if (tt == 1) hipLaunchKernelGGL((k_grouped<WF, SW, 1>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((k_grouped<WF, SW, 4>), grid, block, 0, st, a);
    return hipGetLastError();
}

template <bool SW>
static hipError_t grouped3(const GroupedArgs &a, long items, hipStream_t st)
{
    static bool attr_done = false;
    if (!attr_done) {
        const hipError_t e = hipFuncSetAttribute((const void *)k_grouped3<SW>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, G3::LDS);
        if (e != hipSuccess) return e;
        attr_done = true;
    }
    constexpr int lds_bytes = G3::LDS, threads = 64 * G3::NWAVE;
    hipLaunchKernelGGL((k_grouped3<SW>), dim3((unsigned)items), dim3(threads), lds_bytes, st, a);
    return hipGetLastError();
}

template <bool SW>
static hipError_t grouped_w(const GroupedArgs &a, long items, hipStream_t st)
{
    static bool attr_done = false;
    if (!attr_done) {
        const hipError_t e = hipFuncSetAttribute((const void *)k_grouped_w<SW>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, gw_lds(GW_KMAX));
        if (e != hipSuccess) return e;
        attr_done = true;
    }
    hipLaunchKernelGGL((k_grouped_w<SW>), dim3((unsigned)items), dim3(256), gw_lds(a.K), st, a);
    return hipGetLastError();
}

bool grouped_stream_ok(long nrows, int K, int N)
{
    return K % KS == 0 && K <= GW_KMAX && N % 128 == 0 && (size_t)nrows * K * 2 < (1u << 31);
}

hipError_t grouped_launch(int fmt, bool swiglu, int tt, const GroupedArgs &a, long max_tiles,
                          hipStream_t st)
{
    if (tt == GROUPED_STREAM) {
        if (fmt != FMT_FP4_E8M0 || !a.table || max_tiles <= 0 || a.nrows <= 0 || !grouped_stream_ok(a.nrows, a.K, a.N))
            return hipErrorInvalidValue;
        const long items = max_tiles * (a.N / (swiglu ? 64 : 128));
        return swiglu ? grouped_w<true>(a, items, st) : grouped_w<false>(a, items, st);
    }
    if (tt == GROUPED_DENSE) {
        if (!grouped_dense_ok(a, fmt, swiglu)) return hipErrorInvalidValue;
        if (fmt == FMT_FP8_F32S) return swiglu ? dense8<true, true>(a, st) : dense8<true, false>(a, st);
        return swiglu ? dense8<false, true>(a, st) : dense8<false, false>(a, st);
    }
    if (tt == 8) {
        /* 128-token tiles: FP4 only; byte offsets of every buffer fit 31 bits */
        const int feat = swiglu ? 128 : 256;
        if (fmt != FMT_FP4_E8M0 || a.N % feat || a.K % G3::KS || max_tiles <= 0 || a.nrows <= 0 ||
            (size_t)a.nrows * a.K * 2 >= (1u << 31) || (size_t)a.N * a.K / 2 >= (1u << 31))
            return hipErrorInvalidValue;
        const long items = max_tiles * (a.N / feat);
        return swiglu ? grouped3<true>(a, items, st) : grouped3<false>(a, items, st);
    }
    const int feat = swiglu ? 64 : 128;
    if (a.N % feat || a.K % KC || (tt != 1 && tt != 4) || max_tiles <= 0) return hipErrorInvalidValue;
    const long items = max_tiles * (a.N / feat);
    switch (fmt) {
    case FMT_FP4_E8M0:
        return swiglu ? grouped_tt<FMT_FP4_E8M0, true>(a, tt, items, st)
                      : grouped_tt<FMT_FP4_E8M0, false>(a, tt, items, st);
    case FMT_FP8_E8M0:
        return swiglu ? grouped_tt<FMT_FP8_E8M0, true>(a, tt, items, st)
                      : grouped_tt<FMT_FP8_E8M0, false>(a, tt, items, st);
    case FMT_FP8_F32S:
        return swiglu ? grouped_tt<FMT_FP8_F32S, true>(a, tt, items, st)
                      : grouped_tt<FMT_FP8_F32S, false>(a, tt, items, st);
    default:
        return hipErrorInvalidValue;
    }
}

hipError_t moe_combine_launch(const CombineArgs &a, hipStream_t st)
{
    if (a.hidden % 4) return hipErrorInvalidValue;
    const size_t threads = (size_t)a.n * (a.hidden / 4);
    hipLaunchKernelGGL(k_moe_combine, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, a);
    return hipGetLastError();
}

} // namespace dsv4
