/* SPDX-License-Identifier: Apache-2.0 */
/* dsv4_gemv.hip - decode matvec for packed FP8 / FP4 weights on gfx950.
 *
 * Replaces the nt == 1 bodies of fp8_n (src/10_compute/dsv4_matmul_fp8.c:55-100)
 * and fp4_n (src/10_compute/dsv4_matmul_fp4.c:51-86): y[o] = sum_c W[o,c] x[c]
 * with W decoded in registers and its block scale applied once per block.
 *
 * LAYOUT AND SCHEDULE
 *   A wavefront owns ROWS consecutive output rows. Lane L reads the 16 bytes at
 *   row byte offset 16 L + 1024 j (j = 0..KCH-1): one 128-bit load per lane,
 *   1 KiB contiguous per row per wave instruction. 16 bytes are 16 e4m3
 *   columns (inside one 128-wide FP8 scale block) or 32 e2m1 columns (exactly
 *   one 1x32 FP4 scale block), so every lane applies ONE scale per load.
 *   Load order is the schedule: the lane's x slice first (an L2 hit shared by
 *   every wave), then the block scales, then all ROWS x KCH weight chunks of
 *   the wave. Loads complete in issue order, so the first row's arithmetic
 *   starts as soon as its own chunks land while the later rows are still in
 *   flight, and x never waits behind weight traffic.
 *   Each row's lane partials are summed with a fixed DPP tree; lane r keeps
 *   row r's sum so the wave writes its ROWS outputs with one store.
 *
 * Bound: HBM. Algorithmic bytes per row = row bytes + its scales; the x
 * vector and y are read/written once per call.
 */
#include "dsv4_internal.h"
#include "dsv4_bf16.h"

namespace dsv4 {

/* One token's pass over the wave's ROWS rows: y[t*y_ld + o] for o in
 * [r0, r0+ROWS). W row pitch = row_bytes; scale grid row pitch = sc_cols
 * entries, scale block height blk_r, width 128 (FP8) or 32 (FP4) columns.
 * The weight loads sit inside the pass on purpose: for t = 0 they stream from
 * HBM, later tokens of the same call find them in cache, and the compiler
 * never holds a decoded copy of every chunk at once. */
template <int FMT, int KCH, int ROWS, bool FULL>
__device__ __forceinline__ void gemv_pass(const GemvArgs &a, int t, int lane, int r0)
{
    constexpr bool FP4 = FMT == FMT_FP4_E8M0;
    constexpr bool F32S = FMT == FMT_FP8_F32S;
    constexpr int CPL = FP4 ? 32 : 16;
    constexpr int BLK_C = FP4 ? 32 : 128;

    float xs[KCH][CPL];
    load_x_slice<FP4, KCH, FULL>(xs, a.x + (size_t)t * a.x_ld, lane, a.row_bytes);
    DSV4_ORDER();
    uint32_t sraw[ROWS][KCH];
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        const int row = r0 + r < a.rows ? r0 + r : a.rows - 1;
        const size_t srow = (size_t)(row / a.blk_r) * a.sc_cols;
#pragma unroll
        for (int j = 0; j < KCH; j++) {
            const int b = chunk_byte(lane, j);
            const bool in = FULL || b < a.row_bytes;
            sraw[r][j] = ld_scale_raw<F32S>(a.S, srow + (in ? (FP4 ? 2 * b : b) / BLK_C : 0));
        }
    }
    DSV4_ORDER();
    u32x4 w[ROWS][KCH];
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        const int row = r0 + r < a.rows ? r0 + r : a.rows - 1;
        load_w_row<KCH, FULL>(w[r], a.W + (size_t)row * a.row_bytes, lane, a.row_bytes);
    }
    DSV4_ORDER();
    if (!dsv4_opaque_true()) return;
    float keep = 0.0f;
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j < KCH; j++) {
            float sc = scale_from_raw<F32S>(sraw[r][j]);
            if (!FULL && chunk_byte(lane, j) >= a.row_bytes) sc = 0.0f;
            acc = fmaf(dot16<FP4>(w[r][j], xs[j]), sc, acc);
        }
        const float s = wave_sum(acc);
        if (lane == r) keep = s;
    }
    if (lane < ROWS && r0 + lane < a.rows) a.y[(size_t)t * a.y_ld + r0 + lane] = keep;
}

template <int FMT, int KCH, int ROWS, bool FULL>
__global__ __launch_bounds__(256) void k_gemv(GemvArgs a)
{
    const int lane = threadIdx.x & 63;
    const int r0 = wave_id() * ROWS;
    if (r0 >= a.rows) return;
    for (int t = 0; t < a.nt; t++) gemv_pass<FMT, KCH, ROWS, FULL>(a, t, lane, r0);
}

/* Rows per wave so that a wave keeps sixteen 16-byte chunks per lane (16 KiB)
 * in flight: ROWS x KCH = 16. */
template <int FMT, int KCH>
static hipError_t launch_k(const GemvArgs &a, hipStream_t st)
{
    constexpr int ROWS = 16 / KCH;
    constexpr int WAVES_PER_BLOCK = 4;
    const int waves = (a.rows + ROWS - 1) / ROWS;
    const int blocks = (waves + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
    if (a.row_bytes == KCH * 1024)
        hipLaunchKernelGGL((k_gemv<FMT, KCH, ROWS, true>), dim3(blocks),
                           dim3(64 * WAVES_PER_BLOCK), 0, st, a);
    else
        hipLaunchKernelGGL((k_gemv<FMT, KCH, ROWS, false>), dim3(blocks),
                           dim3(64 * WAVES_PER_BLOCK), 0, st, a);
    return hipGetLastError();
}

template <int FMT>
static hipError_t launch_fmt(const GemvArgs &a, hipStream_t st)
{
    const int kch = (a.row_bytes + 1023) / 1024;
    switch (kch) {
    case 1: return launch_k<FMT, 1>(a, st);
    case 2: return launch_k<FMT, 2>(a, st);
    case 3: return launch_k<FMT, 3>(a, st);
    case 4: return launch_k<FMT, 4>(a, st);
    case 5: case 6: return launch_k<FMT, 6>(a, st);
    case 7: case 8: return launch_k<FMT, 8>(a, st);
    default: return hipErrorInvalidValue;
    }
}

/* ------------------------------------------------------------- BF16 --- */

/* One to four tokens, many rows: a wave's 8 RG rows straight from memory to
 * registers, D steps of 64 columns in flight. Waves are independent. Bound by
 * HBM: the [129280 x 4096] head, one token, 284 -> 178 us (3.7 -> 6.0 TB/s)
 * against a wave that staged its rows and x in LDS and ran each chain as
 * dependent fp64 FMAs. RG = 2 halves the x loads per weight (RG = 1: 222 us;
 * RG = 4, with half the waves, 226), D = 2 / 4 / 8: 182 / 179 / 177. */
template <int RG, int D>
__global__ __launch_bounds__(256) void k_gemv_bf16(GemvBf16Args a)
{
    typedef Bf16Tile<RG> Tile;
    const int lane = threadIdx.x & 63;
    const int r0 = wave_id() * (Tile::ROWS * RG);
    if (r0 >= a.rows) return;
    Tile tile;
    tile.init(a.W, r0, a.rows, a.x, a.x_ld, a.nt, a.cols, lane);
    tile.template chains<D>(a.cols, lane);
    const int tok = lane & 3;
    const float *xrow = a.x + (size_t)min(tok, a.nt - 1) * a.x_ld;
#pragma unroll
    for (int r = 0; r < RG; r++) {
        const int row = r0 + Tile::ROWS * r + Tile::out_row(lane);
        const double v = tile.finish(r, a.W + (size_t)min(row, a.rows - 1) * a.cols, xrow, a.cols);
        if (!(lane & 4) && row < a.rows && tok < a.nt) a.y[(size_t)tok * a.y_ld + row] = (float)v;
    }
}

/* One or two tokens of short rows: a wave per four rows. Bound by latency, and
 * by HBM with very many rows ([100000 x 1024], one token: 31 us, 6.5 TB/s; in the
 * form above 37). */
template <int KCH>
__global__ __launch_bounds__(64) void k_gemv_wave_bf16(GemvBf16Args a)
{
    __shared__ __align__(16) uint8_t lds[bfw_lds_bytes(KCH)];
    const int lane = threadIdx.x, r0 = 4 * blockIdx.x, row = r0 + (lane >> 4);
    bfw_rows_to_lds<KCH>(lds, a.W, r0, a.rows, a.cols, lane);
    for (int t = 0; t < a.nt; t++) {
        /* a single wave: its reads of the token before are done */
        bfw_x_to_lds<KCH>(lds, a.x + (size_t)t * a.x_ld, a.cols, lane);
        __builtin_amdgcn_s_waitcnt(0x0F70);          /* vmcnt(0): rows and token landed */
        asm volatile("" ::: "memory");
        const double v = bfw_dot<KCH>(lds, a.cols, lane);
        if ((lane & 15) == 0 && row < a.rows) a.y[(size_t)t * a.y_ld + row] = (float)v;
    }
}

/* Few tokens, few rows: four rows and four tokens per workgroup. Bound by
 * latency: the [256 x 4096] gate, 8 tokens, 42.3 -> 6.8 us. */
__global__ __launch_bounds__(256) void k_gemv4_bf16(GemvBf16Args a)
{
    extern __shared__ __align__(16) uint8_t b4_lds[];
    const int r0 = 4 * blockIdx.x, t0 = 4 * blockIdx.y;
    const double v = bf16_dot4(b4_lds, a.W, r0, a.rows, a.x + (size_t)t0 * a.x_ld, a.x_ld, min(4, a.nt - t0), a.cols);
    const int tid = threadIdx.x, row = r0 + (tid >> 4), tok = t0 + (tid & 3);
    if (tid < 64 && !(tid & 12) && row < a.rows && tok < a.nt) a.y[(size_t)tok * a.y_ld + row] = (float)v;
}

/* Many tokens: 16 rows x 16 tokens per workgroup on v_mfma_f64_16x16x4 (64
 * cycles), wave w of four running chains 4 w .. 4 w + 3. 256 columns of the
 * rows and the tokens at a time go through LDS (two stages, direct loads);
 * the chains meet in LDS at the end. Bound by the fp64 matrix rate with many
 * tokens (the gate [256 x 4096], 701 tokens: 3,890 -> 34 us, 19 us of it MFMA
 * issue at 2.4 GHz), by the 16 stages' latency with few (15 us). */
constexpr int BFG_COLS = 256;
constexpr int BFG_A_LD = 1024 + 16;                /* two rows of 512 bytes, then a bank offset */
constexpr int BFG_B_LD = 1024 + 16;                /* one token of 1024 bytes                    */
constexpr int BFG_STAGE = 8 * BFG_A_LD + 16 * BFG_B_LD;
typedef double f64x4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void k_gemm_bf16(GemvBf16Args a)
{
    __shared__ __align__(16) uint8_t lds[2 * BFG_STAGE];
    static_assert(2 * BFG_STAGE >= 4 * 16 * 64 * 8, "the chains' exchange");
    const int lane = threadIdx.x & 63, wv = wave_in_group();
    const int lr = lane & 15, lk = lane >> 4;
    const int nrb = (a.rows + 15) / 16;
    const int t0 = blockIdx.x / nrb * 16, r0 = blockIdx.x % nrb * 16;
    const int cols16 = a.cols / 16 * 16;
    const int nstage = (cols16 + BFG_COLS - 1) / BFG_COLS;
    const int nr = min(16, a.rows - r0), nt = min(16, a.nt - t0);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a.W + (size_t)r0 * a.cols), (short)0, nr * a.cols * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a.x + (size_t)t0 * a.x_ld), (short)0, ((nt - 1) * a.x_ld + a.cols) * 4, 0x00020000);
    /* columns past cols16 answer with zeros (an offset past the resource);
     * rows and tokens past the end repeat the last */
    const int none = 0x7FFFFFF0;
    auto load = [&](int st) {
        uint8_t *base = lds + (st & 1) * BFG_STAGE;
        const int c0 = st * BFG_COLS;
#pragma unroll
        for (int i = 0; i < 2; i++) {              /* row pairs wv and wv + 4 */
            const int p = wv + 4 * i, row = min(2 * p + (lane >> 5), nr - 1), c = c0 + 8 * (lane & 31);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (bf_lds_t *)(base + p * BFG_A_LD), 16,
                                                     c < cols16 ? (row * a.cols + c) * 2 : none, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {              /* tokens wv + 4 i */
            const int p = wv + 4 * i, tok = min(p, nt - 1), c = c0 + 4 * lane;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (bf_lds_t *)(base + 8 * BFG_A_LD + p * BFG_B_LD), 16,
                                                     c < cols16 ? (tok * a.x_ld + c) * 4 : none, 0, 0, 0);
        }
    };
    f64x4 acc[4];
#pragma unroll
    for (int q = 0; q < 4; q++) acc[q] = f64x4{0.0, 0.0, 0.0, 0.0};
    load(0);
    __syncthreads();
    for (int st = 0; st < nstage; st++) {
        if (st + 1 < nstage) load(st + 1);
        const uint8_t *base = lds + (st & 1) * BFG_STAGE;
        const uint8_t *pa = base + (lr >> 1) * BFG_A_LD + (lr & 1) * 512 + 2 * (16 * lk + 4 * wv);
        const uint8_t *pb = base + 8 * BFG_A_LD + lr * BFG_B_LD + 4 * (16 * lk + 4 * wv);
#pragma unroll
        for (int s = 0; s < BFG_COLS / 64; s++) {
            const u32x2 w = *(const u32x2 *)(pa + 128 * s);
            const f32x4 x = *(const f32x4 *)(pb + 256 * s);
#pragma unroll
            for (int q = 0; q < 4; q++)
                acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(bf16_elem(w, q), (double)x[q], acc[q], 0, 0, 0);
        }
        __syncthreads();                           /* the next stage has landed, this one is free */
    }
    /* element e of chain q, lane l: row 4 e + l / 16, token l % 16. Wave w
     * combines the elements e = w: chain j is wave j / 4's q = j % 4. */
    double *xc = (double *)lds;
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
        for (int e = 0; e < 4; e++) xc[((wv * 4 + q) * 4 + e) * 64 + lane] = acc[q][e];
    __syncthreads();
    double bb[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        double c[4];
#pragma unroll
        for (int w = 0; w < 4; w++) c[w] = xc[((w * 4 + q) * 4 + wv) * 64 + lane];
        bb[q] = (c[0] + c[1]) + (c[2] + c[3]);
    }
    double v = (bb[0] + bb[1]) + (bb[2] + bb[3]);
    const int row = 4 * wv + lk;
    if (row >= nr || lr >= nt) return;
    const uint16_t *wr = a.W + (size_t)(r0 + row) * a.cols;
    const float *xr = a.x + (size_t)(t0 + lr) * a.x_ld;
    for (int e = cols16; e < a.cols; e++) v = fma(bf16_of(wr[e]), (double)xr[e], v);
    a.y[(size_t)(t0 + lr) * a.y_ld + r0 + row] = (float)v;
}

hipError_t gemv_bf16_launch(const GemvBf16Args &a, hipStream_t st)
{
    if (a.rows <= 0 || a.cols <= 0 || a.cols % 8 || a.nt <= 0) return hipErrorInvalidValue;
    static_assert(BF16_WAVE_COLS == 4 * 512, "the longest rows of k_gemv_wave_bf16<4>");
    const Bf16Form form = bf16_form(a.rows, a.cols, a.nt);
    if (form == BF16_ROWS) {
        constexpr int RG = 2;
        const int waves = (a.rows + 8 * RG - 1) / (8 * RG);
        const dim3 grid((unsigned)((waves + 3) / 4));
        if (bf16_rows_depth(a.rows, a.cols) == 4) hipLaunchKernelGGL((k_gemv_bf16<RG, 4>), grid, dim3(256), 0, st, a);
        else hipLaunchKernelGGL((k_gemv_bf16<RG, 8>), grid, dim3(256), 0, st, a);
        return hipGetLastError();
    }
    if (form == BF16_WAVE) {
        const dim3 grid((unsigned)((a.rows + 3) / 4));
        if (a.cols <= 512) hipLaunchKernelGGL(k_gemv_wave_bf16<1>, grid, dim3(64), 0, st, a);
        else if (a.cols <= 1024) hipLaunchKernelGGL(k_gemv_wave_bf16<2>, grid, dim3(64), 0, st, a);
        else hipLaunchKernelGGL(k_gemv_wave_bf16<4>, grid, dim3(64), 0, st, a);
        return hipGetLastError();
    }
    if (form == BF16_SMALL) {
        static bool attr_done = false;             /* not again inside a stream capture of a later call */
        if (!attr_done) {
            const hipError_t e = hipFuncSetAttribute((const void *)k_gemv4_bf16,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, b4_lds_bytes(4, B4_COLS));
            if (e != hipSuccess) return e;
            attr_done = true;
        }
        hipLaunchKernelGGL(k_gemv4_bf16, dim3((unsigned)((a.rows + 3) / 4), (unsigned)((a.nt + 3) / 4)), dim3(256),
                           b4_lds_bytes(a.nt < 4 ? a.nt : 4, a.cols), st, a);
        return hipGetLastError();
    }
    const long grid = (((long)a.nt + 15) / 16) * (((long)a.rows + 15) / 16);
    if (grid > 0x7FFFFFFF) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_gemm_bf16, dim3((unsigned)grid), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t gemv_launch(int fmt, const GemvArgs &a, hipStream_t st)
{
    switch (fmt) {
    case FMT_FP8_E8M0: return launch_fmt<FMT_FP8_E8M0>(a, st);
    case FMT_FP8_F32S: return launch_fmt<FMT_FP8_F32S>(a, st);
    case FMT_FP4_E8M0: return launch_fmt<FMT_FP4_E8M0>(a, st);
    default: return hipErrorInvalidValue;
    }
}

/* ------------------------------------------------- generic geometry --- */

/* Any block geometry (blk_r >= 1 rows x blk_c >= 1 columns per scale, any
 * column count, rows of any width): the reference's generic bodies of fp8_n
 * and fp4_n (src/10_compute/dsv4_matmul_fp8.c:158-176,
 * src/10_compute/dsv4_matmul_fp4.c:143-162), which only fixtures and rows
 * wider than the fast kernels' limits reach. One wave per output row: for
 * each block of blk_c columns the lanes' products are summed (lane order
 * over the block, then a butterfly), the block sum times its scale is added
 * to the row's total in block order. */
template <int FMT>
__global__ __launch_bounds__(256) void k_gemv_generic(GemvGenArgs a)
{
    const int lane = threadIdx.x & 63;
    const int o = blockIdx.x * 4 + wave_in_group();
    if (o >= a.rows) return;
    const int scg = (a.cols + a.blk_c - 1) / a.blk_c;
    const size_t srow = (size_t)(o / a.blk_r) * (size_t)scg;
    const size_t rb = FMT == FMT_GEN_FP4 ? (size_t)a.cols / 2 : (size_t)a.cols;
    const uint8_t *wr = a.W + (size_t)o * rb;
    for (int t = 0; t < a.nt; t++) {
        const float *xt = a.x + (size_t)t * a.cols;
        float total = 0.0f;
        int bi = 0;
        for (int c0 = 0; c0 < a.cols; c0 += a.blk_c, bi++) {
            const int n = min(a.blk_c, a.cols - c0);
            float d = 0.0f;
            for (int i = lane; i < n; i += 64) {
                const int c = c0 + i;
                float w;
                if constexpr (FMT == FMT_GEN_FP4) {
                    const f32x2 p = dev_e2m1x2<0>((uint32_t)wr[c >> 1]);
                    w = (c & 1) ? p.y : p.x;
                } else {
                    w = dev_e4m3x2<false>((uint32_t)wr[c]).x;
                }
                d = fmaf(w, xt[c], d);
            }
#pragma unroll
            for (int sh = 32; sh >= 1; sh >>= 1) d += __shfl_xor(d, sh, 64);
            const float sc = FMT == FMT_GEN_FP8F ? ld_f32(a.S, srow + bi) : dev_e8m0(ld_u8(a.S, srow + bi));
            total = total + d * sc;
        }
        if (lane == 0) a.y[(size_t)t * a.rows + o] = total;
    }
}

hipError_t gemv_generic_launch(int fmt, const GemvGenArgs &a, hipStream_t st)
{
    if (a.rows <= 0 || a.cols <= 0 || a.blk_r <= 0 || a.blk_c <= 0 || a.nt <= 0 ||
        (fmt == FMT_GEN_FP4 && a.cols % 2))
        return hipErrorInvalidValue;
    const dim3 grid((unsigned)((a.rows + 3) / 4)), block(256);
    switch (fmt) {
    case FMT_GEN_FP8: hipLaunchKernelGGL(k_gemv_generic<FMT_GEN_FP8>, grid, block, 0, st, a); break;
    case FMT_GEN_FP8F: hipLaunchKernelGGL(k_gemv_generic<FMT_GEN_FP8F>, grid, block, 0, st, a); break;
    case FMT_GEN_FP4: hipLaunchKernelGGL(k_gemv_generic<FMT_GEN_FP4>, grid, block, 0, st, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

} // namespace dsv4
