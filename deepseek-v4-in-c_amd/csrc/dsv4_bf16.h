/* SPDX-License-Identifier: Apache-2.0 */
/* dsv4_bf16.h - the BF16 row dot product of bf16_n on the GPU, shared by the
 * BF16 matvec (dsv4_gemv.hip) and the fused gate + router (dsv4_route.hip). */
#ifndef DSV4_BF16_H
#define DSV4_BF16_H

#include "dsv4_choose.h"
#include "dsv4_dev.h"

namespace dsv4 {

/* Replaces bf16_n (src/10_compute/dsv4_matmul.c:88-113) bit for bit. Its row
 * dot product (BLOCK_DOT_V, src/10_compute/dsv4_dec_common.h:45-61) runs 16
 * fp64 FMA chains over the n - n % 16 leading columns, chain c taking columns
 * c, c + 16, c + 32, ... in increasing order from +0; then
 *   bb[j] = (chain j + chain 4 + j) + (chain 8 + j + chain 12 + j),
 *   acc = (bb[0] + bb[1]) + (bb[2] + bb[3]),
 * the n % 16 trailing columns are added to acc one FMA each, and y = (float)
 * acc. Every product of a bf16 weight and an fp32 activation is exact in
 * fp64 and an fp64 FMA is correctly rounded on both sides, so the same order
 * gives the same bits.
 *
 * The chains run on the fp64 MFMA: its four reduction steps are four fp64
 * FMAs in order k = 0..3, each rounded (measured bit for bit against fma()
 * on 5e5 random sums, both instructions used), so one MFMA takes four
 * consecutive steps of a chain and the accumulator carries the chain to the
 * next. A step of the code below is 64 columns: lane group k = lane / 16
 * holds columns 16 k .. 16 k + 15, one of each chain, contiguous in memory.
 * Columns past the last whole 16 enter as 0 x 0, which leaves a chain that
 * started at +0 unchanged. */
__device__ __forceinline__ double bf16_of(uint16_t h) { return (double)__uint_as_float((uint32_t)h << 16); }

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void bf_lds_t;

/* element q of packed bf16 weights */
template <class V>
__device__ __forceinline__ double bf16_elem(const V &w, int q)
{
    const uint32_t d = w[q >> 1];
    return (double)__uint_as_float((q & 1) ? d & 0xFFFF0000u : d << 16);
}

/* Many rows: the row dot products of one wave on v_mfma_f64_4x4x4 (four
 * 4 x 4 x 4 blocks, 16 cycles), RG groups of eight rows times up to four
 * tokens. The four blocks are two halves of the chains times two halves of
 * the rows: lane i + 4 b + 16 k supplies row 4 (b / 2) + i, token i and
 * chains 8 (b % 2) .. + 7, so its eight weights are contiguous and one load
 * instruction reads whole 128-byte lines of eight rows. Result of lane
 * j + 4 b + 16 i': token j, row 4 (b / 2) + i'. Tokens past nt repeat the
 * last, rows past the end too. */
template <int RG>
struct Bf16Tile {
    static constexpr int ROWS = 8;                   /* rows per group */
    const DSV4_GLOBAL u32x4 *wp[RG];                 /* the lane's weights, step 0 */
    const DSV4_GLOBAL f32x4 *xp;                     /* the lane's activations     */
    double acc[RG][8];

    static __device__ __forceinline__ int out_row(int lane) { return ((lane >> 1) & 4) + (lane >> 4); }

    __device__ __forceinline__ void init(const uint16_t *W, int row0, int rows, const float *x, int x_ld, int nt,
                                         int cols, int lane)
    {
        const int col = 16 * (lane >> 4) + 8 * ((lane >> 2) & 1);
#pragma unroll
        for (int r = 0; r < RG; r++) {
            const int row = min(row0 + ROWS * r + ((lane >> 1) & 4) + (lane & 3), rows - 1);
            wp[r] = gptr((const u32x4 *)(W + (size_t)row * cols + col));
        }
        xp = gptr((const f32x4 *)(x + (size_t)min(lane & 3, nt - 1) * x_ld + col));
#pragma unroll
        for (int r = 0; r < RG; r++)
#pragma unroll
            for (int q = 0; q < 8; q++) acc[r][q] = 0.0;
    }

    struct Step {
        u32x4 w[RG];
        f32x4 x[2];
    };
    __device__ __forceinline__ void load(Step &s, int step) const
    {
        s.x[0] = xp[16 * step];
        s.x[1] = xp[16 * step + 1];
#pragma unroll
        for (int r = 0; r < RG; r++) s.w[r] = __builtin_nontemporal_load(wp[r] + 8 * step);
    }
    __device__ __forceinline__ void mac(const Step &s)
    {
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const double b = (double)s.x[q >> 2][q & 3];
#pragma unroll
            for (int r = 0; r < RG; r++)
                acc[r][q] = __builtin_amdgcn_mfma_f64_4x4x4f64(bf16_elem(s.w[r], q), b, acc[r][q], 0, 0, 0);
        }
    }
    /* every step of the row: D of them in flight ahead of the one computed */
    template <int D>
    __device__ __forceinline__ void chains(int cols, int lane)
    {
        const int full = cols / 64;
        const int ring = full / D * D;
        if (ring) {
            Step s[D];
#pragma unroll
            for (int d = 0; d < D; d++) load(s[d], d);
            for (int c = D; c < ring; c += D) {
#pragma unroll
                for (int d = 0; d < D; d++) {
                    mac(s[d]);
                    load(s[d], c + d);
                }
            }
#pragma unroll
            for (int d = 0; d < D; d++) mac(s[d]);
        }
        for (int c = ring; c < full; c++) {
            Step s;
            load(s, c);
            mac(s);
        }
        if (cols / 16 * 16 > 64 * full) {            /* the last one to three 16-column groups */
            Step s;
            if (64 * full + 16 * (lane >> 4) + 16 <= cols) {
                load(s, full);
            } else {
#pragma unroll
                for (int r = 0; r < RG; r++) s.w[r] = u32x4{};
                s.x[0] = s.x[1] = f32x4{};
            }
            mac(s);
        }
    }
    /* The chains of row group r combined in the reference's order and the
     * trailing columns added: the lane's row row0 + 8 r + out_row(lane),
     * token lane % 4, alike in the lanes of both chain halves. wrow and xrow:
     * that row and that token. */
    __device__ __forceinline__ double finish(int r, const uint16_t *wrow, const float *xrow, int cols) const
    {
        double bb[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const double p = acc[r][j] + acc[r][4 + j];
            bb[j] = p + __shfl_xor(p, 4, 64);
        }
        double v = (bb[0] + bb[1]) + (bb[2] + bb[3]);
        for (int e = cols / 16 * 16; e < cols; e++) v = fma(bf16_of(wrow[e]), (double)xrow[e], v);
        return v;
    }
};

/* Few rows: four rows times up to four tokens by a workgroup of four waves.
 * All of the rows and tokens (B4_COLS columns at a time) go to LDS by direct
 * loads first, so the call waits out one memory latency, then every wave
 * runs four of the chains, one MFMA a step: lane i + 4 b + 16 k supplies row
 * i, token i of chain 4 b + w for wave w. */
/* Returns the dot product of row row0 + lane / 16 and token t0 + lane % 4 in
 * wave 0's lanes with (lane & 12) == 0. lds: b4_lds_bytes(min(ntok, 4), cols). Rows
 * past the end repeat the last, tokens past the end give no result. */
__device__ __forceinline__ double bf16_dot4(uint8_t *lds, const uint16_t *W, int row0, int rows, const float *x,
                                            int x_ld, int ntok, int cols)
{
    __shared__ double part[4][16];
    const int lane = threadIdx.x & 63, wv = wave_in_group();
    const int cols16 = cols / 16 * 16;
    const int i = lane & 3, b = (lane >> 2) & 3, k = lane >> 4;
    const int w_ld = b4_w_ld(cols), x_ldb = b4_x_ld(cols);
    uint8_t *xl = lds + 4 * w_ld;
    double acc = 0.0;
    for (int c0 = 0; c0 < cols16; c0 += B4_COLS) {
        const int nc = min(B4_COLS, cols16 - c0);    /* columns of this part */
        if (c0) __syncthreads();
        /* wave w: row w, token w; 1 KiB per instruction, zeros past nc */
        const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(W + (size_t)min(row0 + wv, rows - 1) * cols + c0), (short)0, 2 * nc, 0x00020000);
        for (int m = 0; m < (nc + 511) / 512; m++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (bf_lds_t *)(lds + wv * w_ld + 1024 * m), 16,
                                                     1024 * m + 16 * lane, 0, 0, 0);
        /* the tokens' pieces dealt to the waves */
        const int xm = (nc + 255) / 256;
        for (int m = wv; m < ntok * xm; m += 4) {
            const int t = m / xm, p = m - t * xm;
            const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
                (void *)(x + (size_t)t * x_ld + c0), (short)0, 4 * nc, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (bf_lds_t *)(xl + t * x_ldb + 1024 * p), 16,
                                                     1024 * p + 16 * lane, 0, 0, 0);
        }
        __syncthreads();                             /* everything has landed */
        const uint16_t *wl = (const uint16_t *)(lds + i * w_ld) + 16 * k + 4 * b + wv;
        const float *xr = (const float *)(xl + (i < ntok ? i : 0) * x_ldb) + 16 * k + 4 * b + wv;
        /* eight steps' reads issued before the eight before them multiply;
         * columns past nc were loaded as zeros up to whole 512s (rows) and
         * 256s (tokens), both at least the last step's end */
        const int steps = (nc + 63) / 64;
        uint16_t w[8];
        float xv[8];
#pragma unroll
        for (int d = 0; d < 8; d++) { w[d] = wl[64 * min(d, steps - 1)]; xv[d] = xr[64 * min(d, steps - 1)]; }
        int s = 0;
        for (; s + 8 <= steps; s += 8) {
            uint16_t wn[8];
            float xn[8];
#pragma unroll
            for (int d = 0; d < 8; d++) {
                const int c = min(s + 8 + d, steps - 1);
                wn[d] = wl[64 * c];
                xn[d] = xr[64 * c];
            }
#pragma unroll
            for (int d = 0; d < 8; d++)
                acc = __builtin_amdgcn_mfma_f64_4x4x4f64(bf16_of(w[d]), (double)xv[d], acc, 0, 0, 0);
#pragma unroll
            for (int d = 0; d < 8; d++) { w[d] = wn[d]; xv[d] = xn[d]; }
        }
#pragma unroll
        for (int d = 0; d < 8; d++)
            if (s + d < steps)
                acc = __builtin_amdgcn_mfma_f64_4x4x4f64(bf16_of(w[d]), (double)xv[d], acc, 0, 0, 0);
    }
    /* block b of wave w ran chain 4 b + w: bb[w] = (b0 + b1) + (b2 + b3) */
    double p = acc + __shfl_xor(acc, 4, 64);
    p = p + __shfl_xor(p, 8, 64);
    if (b == 0) part[wv][4 * k + i] = p;
    __syncthreads();
    if (wv != 0 || b != 0) return 0.0;
    double v = (part[0][4 * k + i] + part[1][4 * k + i]) + (part[2][4 * k + i] + part[3][4 * k + i]);
    if (i < ntok) {
        const uint16_t *wr = W + (size_t)min(row0 + k, rows - 1) * cols;
        for (int e = cols16; e < cols; e++) v = fma(bf16_of(wr[e]), (double)x[(size_t)i * x_ld + e], v);
    }
    return v;
}

/* One wave, four rows, a token at a time: lane 16 r + c runs chain c of row r
 * as its FMAs, over rows and token in LDS. */
constexpr int bfw_row_ld(int kch) { return 1024 * kch + 64; }            /* bank offset */
constexpr int bfw_lds_bytes(int kch) { return 4 * bfw_row_ld(kch) + 2048 * kch; }

/* rows row0 .. row0 + 3 (the last repeated) of `rows` into LDS, KCH KiB each;
 * the caller waits */
template <int KCH>
__device__ __forceinline__ void bfw_rows_to_lds(uint8_t *lds, const uint16_t *W, int row0, int rows, int cols, int lane)
{
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(W + (size_t)min(row0 + r, rows - 1) * cols), (short)0, 2 * cols, 0x00020000);
#pragma unroll
        for (int k = 0; k < KCH; k++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (bf_lds_t *)(lds + r * bfw_row_ld(KCH) + 1024 * k), 16,
                                                     1024 * k + 16 * lane, 0, 0, 0);
    }
}

/* the token into LDS behind the rows; the caller waits */
template <int KCH>
__device__ __forceinline__ void bfw_x_to_lds(uint8_t *lds, const float *x, int cols, int lane)
{
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)x, (short)0, 4 * cols, 0x00020000);
#pragma unroll
    for (int k = 0; k < 2 * KCH; k++)
        if (256 * k < cols)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (bf_lds_t *)(lds + 4 * bfw_row_ld(KCH) + 1024 * k), 16,
                                                     1024 * k + 16 * lane, 0, 0, 0);
}

/* The dot product of row lane / 16 and the token, in that group's first lane.
 * The next eight steps' reads are issued before the eight before them add. */
template <int KCH>
__device__ __forceinline__ double bfw_dot(const uint8_t *lds, int cols, int lane)
{
    const int steps = cols / 16;
    const uint16_t *wr = (const uint16_t *)(lds + (lane >> 4) * bfw_row_ld(KCH));
    const float *xr = (const float *)(lds + 4 * bfw_row_ld(KCH));
    const uint16_t *wl = wr + (lane & 15);
    const float *xl = xr + (lane & 15);
    double acc = 0.0;
    uint16_t w[8];
    float xv[8];
    int s = 0;
    if (steps >= 8) {
#pragma unroll
        for (int i = 0; i < 8; i++) { w[i] = wl[16 * i]; xv[i] = xl[16 * i]; }
        for (; s + 8 <= steps; s += 8) {
            uint16_t wn[8];
            float xn[8];
            const int sn = s + 16 <= steps ? s + 8 : s;     /* the last round re-reads its own */
#pragma unroll
            for (int i = 0; i < 8; i++) { wn[i] = wl[16 * (sn + i)]; xn[i] = xl[16 * (sn + i)]; }
#pragma unroll
            for (int i = 0; i < 8; i++) acc = fma(bf16_of(w[i]), (double)xv[i], acc);
#pragma unroll
            for (int i = 0; i < 8; i++) { w[i] = wn[i]; xv[i] = xn[i]; }
        }
    }
    for (; s < steps; s++) acc = fma(bf16_of(wl[16 * s]), (double)xl[16 * s], acc);
    acc = acc + __shfl_down(acc, 4, 16);       /* lanes 0..3, 8..11: chain c + chain c + 4 */
    acc = acc + __shfl_down(acc, 8, 16);       /* lanes 0..3: bb[c]                        */
    acc = acc + __shfl_down(acc, 1, 16);       /* lanes 0, 2: bb[0] + bb[1], bb[2] + bb[3] */
    acc = acc + __shfl_down(acc, 2, 16);
    for (int e = 16 * steps; e < cols; e++) acc = fma(bf16_of(wr[e]), (double)xr[e], acc);
    return acc;
}

} // namespace dsv4

#endif /* DSV4_BF16_H */
