/* SPDX-License-Identifier: Apache-2.0 */
/* dsv4_choose.h - which form a call's sizes take: the rules of the dispatch as
 * plain arithmetic on the host, with nothing of HIP, so that the CPU tests
 * compile and ask them (tests/test_choice.py). Costs are in the unit that each
 * rule names, rounds are of CUS workgroups. */
#ifndef DSV4_CHOOSE_H
#define DSV4_CHOOSE_H

#include <stddef.h>

namespace dsv4 {

constexpr long CUS = 256;                              /* compute units of an MI355X */

inline long ceil_div(long a, long b) { return (a + b - 1) / b; }
inline long rounds(long workgroups) { return ceil_div(workgroups, CUS); }

/* ---- FP8 and MXFP8 GEMMs (dsv4_gemm.hip, dsv4_gemm_mid.hip) ---- */

/* The k_gemm_mid tile of 16 t tokens (t = 2, 4, 8) of least cost, 0 for the 128
 * x 256 tiles: a round of 256 workgroups takes 11, 15 or 23 us with T = 2, 4 or
 * 8 at 4,096 columns, of the 128 x 256 tiles 30. us of the call
 * with T = 2 / 4 / 8 / 128 x 256, MXFP8: 4096 x 4096 300 tokens 20.2 / 18.2 /
 * 22.7 / 30.0, 700 tokens 32.8 / 28.8 / 26.4 / 32.1, 1,500 tokens 57.6 / 46.5 /
 * 48.1 / 38.1; 2048 x 7168 700 tokens 36.2 / 29.1 / 35.3 / 48.0. The loads
 * address A, W and Sa with 31-bit byte offsets, and a row block's scales fit
 * one register. */
constexpr int GEMM_MID_KMAX = 64 * 128;
inline int gemm_mid_tile(int M, int N, int K)
{
    if (M <= 0 || N % 128 || K % 128 || K > GEMM_MID_KMAX || (size_t)M * K >= (1u << 31) ||
        (size_t)M * N / 1024 >= (1u << 31))
        return 0;
    const int t[3] = {2, 4, 8}, c[3] = {11, 15, 23};
    int best = 0;
    long cost = 30 * rounds(ceil_div(M, 128) * ceil_div(N, 256));
    for (int i = 0; i < 3; i++) {
        const long v = c[i] * rounds(ceil_div(M, 16 * t[i]) * (N / 128));
        if (best ? v < cost : v <= cost) {
            best = t[i];
            cost = v;
        }
    }
    return best;
}

/* ---- FP8 matrices over many tokens (k_dense8, the seam GEMM) ---- */

/* The 16-token groups T of a k_dense8 tile with the least cost: a round of 256
 * workgroups takes 8, 11, 16, 19 or 26 us with T = 1, 2, 3, 4 or 6 for 4,096
 * columns (tiles smaller than their share re-read the weights, larger ones
 * leave CUs idle). 4096 x 4096, us of the call with T = 1 / 2 / 3 / 4 / 6: 77
 * tokens 16.5 / 19.9 / 21.9 / 23.6 / 27.3, 333 tokens 33.4 / 28.6 / 25.3 / 26.6
 * / 30.6, 700 tokens 56.6 / 44.4 / 45.3 / 48.1 / 35.9. slabs: 128-row blocks of
 * the matrix (gate/up: 64 rows of each). */
inline int dense8_tile(int M, long slabs, long *cost)
{
    const int t[5] = {1, 2, 3, 4, 6}, c[5] = {8, 11, 16, 19, 26};
    int best = 0;
    for (int i = 0; i < 5; i++) {
        const long v = c[i] * rounds(ceil_div(M, 16 * t[i]) * slabs);
        if (!best || v < *cost) {
            best = t[i];
            *cost = v;
        }
    }
    return best;
}

/* Whether an FP8 matrix of rows x cols against nt tokens takes the seam GEMM
 * (128 x 256 tiles) rather than k_dense8 (dense) or, for operands that k_dense8
 * does not address, the grouped form. A unit of dense8_tile's costs takes a time
 * that grows as 620 + cols, a round of the seam GEMM as 12,000 + 59 cols (its
 * epilogue is the smaller part of a long row), a tenth of it as the round's
 * tiles. us of dense / seam: 4096 x 4096,
 * 1,500 tokens 70 / 74, 2,000 tokens 113 / 79; 15360 x 4096, 500 tokens 94 / 71;
 * 512 x 4096, 4,000 tokens 47 / 75; 1280 x 384, 3,708 tokens 23.7 / 16.6; 15360 x
 * 640, 1,751 tokens 87 / 67; 1280 x 128, 2,000 tokens both 11.4. Of 246 shapes the
 * choice is within 9 % of the better one, on average 0.1 %. */
constexpr int MMQ_SEAM_GEMM_MIN_TOKENS = 1280;
inline bool mmq_takes_seam(int nt, int rows, int cols, bool dense)
{
    if (!dense) return nt >= MMQ_SEAM_GEMM_MIN_TOKENS;
    long units = 0;
    dense8_tile(nt, rows / 128, &units);
    const long tiles = ceil_div(nt, 128) * ceil_div(rows, 256), past = tiles > CUS ? tiles : CUS;
    return (9 * CUS * rounds(tiles) + past) * (12000 + 59L * cols) < 10 * CUS * units * (620 + cols);
}

/* ---- routed FP4 experts (dsv4_moe_grouped.hip) ---- */

/* Tiles of the grouped GEMMs: 1, 4 or 8 times 16 rows, the 16-row tiles that
 * stream the weights to registers, or the dense tiles of one FP8 matrix. */
constexpr int GROUPED_STREAM = 5, GROUPED_DENSE = 6;

/* The form of the routed experts' GEMMs, by the mean bucket. Up to 28 rows an
 * expert the weight stream is the bound: the 16-row tiles that stream to
 * registers (4096 x 2048, 256 experts: 7 tokens 135 against 161 us of the
 * LDS-staged 16-row tiles, 64 tokens 297 / 356, 701 tokens 870 / 1,005 and
 * 1,128 of the 128-row tiles; at 33 rows an expert 1,233 / 1,374 / 1,193).
 * With fewer than four steps of 256 to a row its setup costs more than it
 * saves (inter 512: 62 against 59 us at 60 tokens): there the LDS-staged
 * tiles, 16 rows up to 32 rows an expert (16 beyond GROUPED_FEW_PAIRS), else
 * 128 rows, which use the weights again across a tile. us of 16 / 128 rows with
 * weights that no cache holds, as between a model's layers, and an FP8 shared
 * expert: hidden 4096, inter 512, 64 experts, 17 rows each 120 / 132, 24 rows
 * 134 / 140, 36 rows 156 / 156, 60 rows 208 / 183; 2048 x 512, 128 experts, 17
 * rows 114 / 121. stream: the geometry is one that the streaming tiles take.
 *
 * Few experts make few 128-row tiles, and a workgroup of those takes its time
 * however many CUs stay idle: up to 4,096 pairs, where they do not fill the
 * device once, they have to be the cheaper ones (us of 16 / 128 rows, hidden
 * 4096, inter 2048: one expert, 100 tokens 36 / 85, 560 tokens 84 / 98, 1,600
 * tokens 194 / 131; eight experts, 140 rows each, 138 / 106; 2048 x 512, one
 * expert, 800 tokens 36 / 59). In units of a 16-row tile's multiplications, one
 * per weight: a 128-row workgroup's latency grows with its K and, by 0.3 + 0.7
 * rows / 128, with the tile's rows; 45 and 1.5 fit 390 measured calls of 1 to 64
 * experts (7168 x 2048 to 512 x 512) within 10 % of the better form. */
constexpr long GROUPED_FEW_PAIRS = 4096;
inline int grouped_form(long pairs, int n_experts, int hidden, int inter, bool stream)
{
    const int form16 = stream && hidden >= 1024 && inter >= 1024 ? GROUPED_STREAM : 1;
    const long mean = form16 == GROUPED_STREAM ? 28 : pairs <= GROUPED_FEW_PAIRS ? 32 : 16;
    if (pairs <= mean * n_experts) return form16;
    const double buckets = (double)(pairs < n_experts ? pairs : n_experts), rows = (double)pairs / buckets;
    const double tiles16 = (double)pairs / 16 + buckets / 2;
    const double tiles128 = rows > 64 ? (double)pairs / 128 + buckets / 2 : buckets;
    if (pairs > GROUPED_FEW_PAIRS || tiles128 * inter / 128 >= (double)CUS) return 8;
    const double weights = (double)hidden * inter;
    const double latency = 45.0 * 1024.0 * (hidden + inter) * (0.3 + 0.7 * (rows < 128 ? rows / 128 : 1.0));
    return latency + 1.5 * tiles128 * weights < tiles16 * weights ? 8 : form16;
}

/* The mean bucket says nothing about tokens that gather on few experts, whose
 * weights the 16-row tiles would read and decode once per 16 of them: above
 * GROUPED_FEW_PAIRS pairs the buckets of more than GROUPED_FAT_MIN rows go to
 * 128-row tiles in launches of their own, ahead of the others on the stream
 * (where there are none, two launches of empty workgroups, 3 to 6 us). 256
 * experts of 4096 x 2048, top-6, us without / with: 1,000 tokens on 8 of them
 * 578 / 359, on 64 660 / 435, Zipf 974 / 883, even routing 942 / 949; 701
 * tokens, Zipf, 819 / 784; of 2048 x 1024, 1,000 tokens on 8 175 / 140, Zipf 285
 * / 297. Smaller experts are read again from the caches and keep one form (1024
 * x 1024: on 8 109 / 91, but Zipf 163 / 173, even 166 / 171). Fat from 96 rows:
 * 4096 x 2048, 64 experts used 586, Zipf 880; the others on a second stream
 * beside them: Zipf 863, even routing 962 against 955. Below GROUPED_FEW_PAIRS
 * 16-row tiles alone are no slower (680 tokens on 8 experts: 390). */
constexpr int GROUPED_FAT_ROWS = 128, GROUPED_FAT_MIN = 64;
constexpr long GROUPED_FAT_WEIGHTS = 1L << 21;
inline bool grouped_splits(long pairs, int form, int hidden, int inter)
{
    return pairs > GROUPED_FEW_PAIRS && form != 8 && (long)hidden * inter >= GROUPED_FAT_WEIGHTS;
}
/* their number at most: such a bucket's tiles hold 64.5 rows each or more */
inline long grouped_fat_tiles(long pairs) { return 2 * pairs / (GROUPED_FAT_ROWS + 1); }

/* ---- routed MXFP8 experts (dsv4_moe_mx.hip) ---- */

/* Whether rows of K columns take mx_tile_wide (else mx_tile, the same bits):
 * whole groups of four stages, and enough of them for its longer start. us of
 * the call, mx_tile / mx_tile_wide in both launches: 512 x 512, 16 experts,
 * 2,000 tokens x 4 80.4 / 83.1; 1024 x 1024 118.8 / 119.0; 1536 x 1536 145.4 /
 * 146.3; 32 experts, 4,000 tokens: 2048 x 2048 352 / 347, 3072 x 3072 637 / 603,
 * 4096 x 2048 547 / 526. */
constexpr int MX_WIDE_MIN_K = 2048;
constexpr bool mx_wide_k(int K) { return K % 512 == 0 && K >= MX_WIDE_MIN_K; }

/* ---- BF16 matvecs (dsv4_gemv.hip) ---- */

/* LDS of k_gemv4_bf16: four rows and up to four tokens of b4_cols(cols) columns
 * at a time (whole load instructions of the rows), a bank offset behind each. */
constexpr int B4_COLS = 4096;
constexpr int b4_cols(int cols) { return cols < B4_COLS ? (cols + 511) / 512 * 512 : B4_COLS; }
constexpr int b4_w_ld(int cols) { return 2 * b4_cols(cols) + 64; }
constexpr int b4_x_ld(int cols) { return 4 * b4_cols(cols) + 16; }
constexpr int b4_lds_bytes(int ntok, int cols) { return 4 * b4_w_ld(cols) + ntok * b4_x_ld(cols); }

/* Which form, all with the same bits. us at 4096 columns for (small /
 * rows / GEMM), measured: 1 token: 1024 rows 6.4 / 20 / 15, 8192 rows 18.8 /
 * 22 / 25, 16384 rows 37 / 25 / 45; 4 tokens: 256 rows 6.7 / - / 15, 4096
 * rows 20 / 31 / 16, 8192 rows 37 / 31 / 26, 32768 rows 147 / 61 / 88; 32
 * tokens: 256 rows 10.1 / - / 15, 1024 rows 36 / - / 15. So: the rows form
 * for a few tokens of a large matrix, the small form while its workgroups
 * run in at most three rounds of what LDS lets the device hold at once (rows of
 * 4096 columns), else the GEMM.
 *
 * One token of short rows, and two of a middling number of them, leave most of
 * an MFMA's columns and a workgroup's latency unused: a wave of its own for
 * four rows. us of (wave / small / rows): 1 token 8192 x 440 3.8 / 5.6 / 6.6,
 * 16384 x 1024 6.9 / 10.5 / 8.5, 100000 x 232 13.4 / 33 / 16, 4096 x 2024 5.7 /
 * 7.0 / 14, but 16384 x 2024 18.7 / 19.8 / 16.3 and 4096 x 4096 15.2 / 10.0 /
 * 21; 2 tokens 12000 x 768 6.8 / 7.8 / 7.6, but 16384 x 768 9.7 / 9.5 / 7.8 and
 * 4096 x 440 5.0 / 4.6. Rows of up to 128 columns: 3 tokens, 12000 rows 4.1 /
 * 5.9 / 3.5. */
enum Bf16Form { BF16_SMALL = 1, BF16_ROWS, BF16_GEMM, BF16_WAVE };
constexpr int BF16_WAVE_COLS = 2048;
inline Bf16Form bf16_form(int rows, int cols, int nt)
{
    if (nt == 1 && cols > 64 && cols <= 1024 && rows >= 2048) return BF16_WAVE;
    if (nt == 1 && cols <= BF16_WAVE_COLS && rows >= 3072 && rows < 8192) return BF16_WAVE;
    if (nt == 2 && cols > 128 && cols <= 1024 && rows >= 5120 && rows < 14336) return BF16_WAVE;
    if (nt <= 4 && rows >= (nt == 1 ? 9216 : cols <= 128 ? 4096 : 12288)) return BF16_ROWS;
    const int lds = b4_lds_bytes(nt < 4 ? nt : 4, B4_COLS);
    return ceil_div(rows, 4) * ceil_div(nt, 4) <= 3 * CUS * (160 * 1024 / lds) ? BF16_SMALL : BF16_GEMM;
}
/* Steps of 64 columns that the rows form has in flight: fewer where a row is
 * hardly longer than eight and the waves many. 2 tokens, 4 / 8 steps, us: 100000
 * rows of 256 columns 13.2 / 16.9, 960 39.0 / 48.0 (2024, one token: 93.5 /
 * 91.4), 60000 of 256 10.4 / 9.8. */
constexpr int bf16_rows_depth(int rows, int cols) { return cols < 1024 && rows >= 65536 ? 4 : 8; }

} // namespace dsv4

#endif /* DSV4_CHOOSE_H */
