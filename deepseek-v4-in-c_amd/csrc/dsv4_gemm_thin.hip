/* SPDX-License-Identifier: Apache-2.0 */
/* dsv4_gemm_thin.hip - the FP8 GEMMs of dsv4_gemm.hip in small tiles, for
 * shapes whose 128 x 256 tiles leave most of the device idle: few tokens, or
 * a matrix of few rows.
 *
 * Two forms of C[m][n] = sum_k A[m][k] W[n][k], each with the products, the
 * reduction order and so the bits of its large-tile kernel:
 *   T_FP8   e4m3 tokens with fp32 1 x 128 scales, fp32 or E8M0 weight blocks,
 *           every 128-wide block's product folded into fp32 (k_gemm_fp8)
 *   T_MX    MXFP8 tokens, E8M0 weight blocks, both in the MFMA's scale
 *           operands (k_gemm_mx)
 *
 * SCHEDULE
 *   A workgroup of four waves owns 64 features x 16 NT tokens; wave w the 16
 *   weight rows 16 w .. 16 w + 15, over all of K. K advances in groups of
 *   four 128-wide blocks, two groups in flight: the weights straight to
 *   registers (a load instruction reads whole 128-byte lines of eight rows;
 *   lanes i and i ^ 8 of a row of 16 then trade halves to form the operand),
 *   the token rows and their scales to LDS, wave w loading block w of the
 *   group. All of a wave's loads complete in order, so one counted wait and
 *   one barrier hand a group over and one barrier frees its slots. The 64
 *   weight scales of a row block sit in one register, one per lane.
 *   The loads past the end of K read nothing and multiply as zeros.
 *
 * Bound: the launch (an empty grid of the same size takes all but 3 us of the
 * smallest calls) and, with several workgroups to a CU, the L2 reads through
 * registers. 1024 x 4096 MXFP8, 300 tokens: 24.8 -> 11.5 us (the large tiles
 * are 12 workgroups there). Three or four groups in flight are slower (14.2
 * against 13.5 us at 8 tokens), starting workgroups at different blocks of K
 * changes nothing.
 */
#include "dsv4_internal.h"

namespace dsv4 {

namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

enum { T_FP8 = 0, T_MX = 1 };

constexpr int TB = 128;                            /* reduction block           */
constexpr int TG = 4;                              /* blocks per group, a wave each */
constexpr int TN = 64;                             /* features per workgroup    */
constexpr int T_KMAX = 64 * TB;
constexpr uint32_t T_OOB = 0x80000000u;            /* beyond every buffer       */
constexpr int T_E8M0_ONE = 127;

template <int NT> struct Thin {
    static constexpr int XI = 16 * NT * TB / 1024;                 /* token loads per block   */
    static constexpr int XBLK = 1024 * XI + 256;                   /* LDS of a block          */
    static constexpr int LDS = 2 * TG * XBLK;
    static constexpr int VM = 2 * TG + XI + 1;                     /* a wave's loads a group  */
    static_assert(VM <= 63, "vmcnt range");
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t t_rsrc(const void *p, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
}

__device__ __forceinline__ void t_dma16(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff, uint8_t *dst)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)dst, 16, (int)voff, soff, 0, 0);
}
__device__ __forceinline__ void t_dma4(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff, uint8_t *dst)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)dst, 4, (int)voff, soff, 0, 0);
}
__device__ __forceinline__ u32x4 t_load16(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff)
{
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, soff, 0));
}

__device__ __forceinline__ uint32_t t_bf16(float f)
{
    const uint32_t u = __float_as_uint(f);
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (u >> 16) | 0x40u;   /* quiet NaN */
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

} // namespace

/* one call's operands in any of the forms */
struct ThinArgs {
    const void *A;            /* e4m3 tokens [M][K]                               */
    const void *Sa;           /* token scales (a dword per token and block)       */
    const uint8_t *W;
    const void *Sw;
    void *C;
    int M, N, K;
    int sa_tok, sa_kb;        /* dword strides of Sa                              */
};

template <int MODE, bool WF32S, bool OUT_BF16, int NT>
__global__ __launch_bounds__(256) void k_gemm_thin(ThinArgs a)
{
    using C = Thin<NT>;
    extern __shared__ __align__(16) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = wave_in_group();
    const int rr = lane & 15, gq = lane >> 4;
    /* feature tiles of one XCD (workgroups go round the eight) side by side,
     * each with all its token tiles, when they divide: W is then fetched into
     * one L2 only */
    const int mt = (a.M + 16 * NT - 1) / (16 * NT), ft = a.N / TN;
    int lin = blockIdx.x;
    if (ft % 8 == 0) lin = (lin % 8) * (ft / 8 * mt) + lin / 8;
    const int n0 = lin / mt * TN, m0 = lin % mt * (16 * NT);
    const int nkb = a.K / TB, ngr = (nkb + 2 * TG - 1) / (2 * TG) * 2;

    const __amdgpu_buffer_rsrc_t rx = t_rsrc(a.A, (uint32_t)a.M * (uint32_t)a.K);
    const __amdgpu_buffer_rsrc_t rw = t_rsrc(a.W + (size_t)n0 * a.K, (uint32_t)TN * (uint32_t)a.K);
    const __amdgpu_buffer_rsrc_t none = t_rsrc(a.W, 0);
    const __amdgpu_buffer_rsrc_t rs = t_rsrc(
        a.Sa, 4u * ((uint32_t)(nkb - 1) * (uint32_t)a.sa_kb + (uint32_t)(a.M - 1) * (uint32_t)a.sa_tok + 1u));
    /* token row r of a block holds chunk c at slot swx(r, c) */
    auto swx = [](int r, int c) { return c ^ ((r >> 1) & 7); };
    uint32_t xofs[C::XI];
#pragma unroll
    for (int i = 0; i < C::XI; i++) {
        const int r = 8 * i + lane / 8, c = swx(r, lane & 7);
        xofs[i] = m0 + r < a.M ? (uint32_t)(m0 + r) * (uint32_t)a.K + 16u * (uint32_t)c : T_OOB;
    }
    const int mlane = m0 + (lane & (16 * NT - 1));
    const uint32_t sofs = lane < 16 * NT && mlane < a.M ? 4u * (uint32_t)mlane * (uint32_t)a.sa_tok : T_OOB;
    /* load j of a block: lanes i < 8 the low 64-byte half's 16 bytes of row
     * 8 j + i, lanes i >= 8 the high half's of row 8 j + i - 8 */
    const uint32_t wofs = (uint32_t)(16 * wave + (lane & 7)) * (uint32_t)a.K + 64u * ((lane >> 3) & 1) + 16u * gq;
    const uint32_t wofs1 = wofs + 8u * (uint32_t)a.K;

    struct G { u32x4 w[TG][2]; };
    auto load = [&](G &w, int g) {
        asm volatile("" ::: "memory");
        const int kb = g * TG + wave;              /* this wave's block of tokens */
        uint8_t *dst = lds + ((g & 1) * TG + wave) * C::XBLK;
#pragma unroll
        for (int i = 0; i < C::XI; i++)
            t_dma16(kb < nkb ? rx : none, xofs[i], kb * TB, dst + 1024 * i);
        t_dma4(kb < nkb ? rs : none, sofs, 4 * kb * a.sa_kb, dst + 1024 * C::XI);
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int k = 0; k < TG; k++)
                w.w[k][j] = t_load16(g * TG + k < nkb ? rw : none, j ? wofs1 : wofs, (g * TG + k) * TB);
        asm volatile("" ::: "memory");
    };
    /* lane kb: the weight scale of block kb (nkb <= 64) */
    uint32_t wsc;
    {
        const size_t i = (size_t)(n0 / 128) * nkb + min(lane, nkb - 1);
        if constexpr (WF32S) wsc = __float_as_uint(ld_f32(a.Sw, i));
        else if constexpr (MODE == T_MX) wsc = ld_u8(a.Sw, i);
        else wsc = __float_as_uint(dev_e8m0(ld_u8(a.Sw, i)));
    }
    G ring[2];
    load(ring[0], 0);
    load(ring[1], 1);
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("" : "+v"(wsc));                  /* its wait here, not inside the first group */
#endif

    v4f acc[NT];
#pragma unroll
    for (int u = 0; u < NT; u++) acc[u] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    const bool lo8 = !(lane & 8);
    auto compute = [&](const u32x4 (&q)[2], const uint8_t *blk, int kb) {
        u32x4 lo, hi;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t s0 = (uint32_t)__builtin_amdgcn_mov_dpp((int)q[0][e], DPP_ROW_ROR8, 0xF, 0xF, false);
            const uint32_t s1 = (uint32_t)__builtin_amdgcn_mov_dpp((int)q[1][e], DPP_ROW_ROR8, 0xF, 0xF, false);
            lo[e] = lo8 ? q[0][e] : s1;
            hi[e] = lo8 ? s0 : q[1][e];
        }
        const uint32_t sw = (uint32_t)__builtin_amdgcn_readlane((int)wsc, min(kb, nkb - 1));
        const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
        v8i w;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            w[e] = (int)lo[e];
            w[4 + e] = (int)hi[e];
        }
#pragma unroll
        for (int u = 0; u < NT; u++) {
            const int t = 16 * u + rr;
            const u32x4 b0 = *(const u32x4 *)(blk + t * TB + 16 * swx(t, gq));
            const u32x4 b1 = *(const u32x4 *)(blk + t * TB + 16 * swx(t, gq + 4));
            const uint32_t ts = *(const uint32_t *)(blk + 1024 * C::XI + 4 * t);
            v8i b;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                b[e] = (int)b0[e];
                b[4 + e] = (int)b1[e];
            }
            if constexpr (MODE == T_MX) {
                acc[u] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, b, acc[u], 0, 0, 0, (int)sw, 0,
                                                                         (int)((ts >> (8 * gq)) & 0xFFu));
            } else {
                const v4f p = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, b, zero, 0, 0, 0, T_E8M0_ONE,
                                                                              0, T_E8M0_ONE);
                const float cs = __uint_as_float(ts) * __uint_as_float(sw);
#pragma unroll
                for (int e = 0; e < 4; e++) acc[u][e] = fmaf(p[e], cs, acc[u][e]);
            }
        }
    };
    for (int g = 0; g < ngr; g += 2) {
#pragma unroll
        for (int d = 0; d < 2; d++) {
            /* this group has landed (only the next one's loads outstanding) */
            __builtin_amdgcn_s_waitcnt(0x0F70 | (C::VM & 15) | ((C::VM >> 4) << 14));
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
#pragma unroll
            for (int k = 0; k < TG; k++) {
                compute(ring[d].w[k], lds + (d * TG + k) * C::XBLK, (g + d) * TG + k);
                if constexpr (NT == 1) __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0xC07F);    /* lgkmcnt(0): its slots have been read */
            __builtin_amdgcn_s_barrier();
            load(ring[d], g + d + 2);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);            /* the counted loads past the end */
#pragma unroll
    for (int u = 0; u < NT; u++) {
        const int m = m0 + 16 * u + rr;
        if (m >= a.M) continue;
        const size_t o = (size_t)m * a.N + n0 + 16 * wave + 4 * gq;
        const v4f v = acc[u];
        if constexpr (OUT_BF16) {
            uint2 pk;
            pk.x = t_bf16(v[0]) | (t_bf16(v[1]) << 16);
            pk.y = t_bf16(v[2]) | (t_bf16(v[3]) << 16);
            *(uint2 *)((uint16_t *)a.C + o) = pk;
        } else {
            *(f32x4 *)((float *)a.C + o) = f32x4{v[0], v[1], v[2], v[3]};
        }
    }
}

template <int MODE, bool WS, bool OB, int NT>
static hipError_t thin_launch(const ThinArgs &a, hipStream_t st)
{
    using C = Thin<NT>;
    static bool attr_done = false;
    if (!attr_done) {
        const hipError_t e = hipFuncSetAttribute((const void *)k_gemm_thin<MODE, WS, OB, NT>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
        if (e != hipSuccess) return e;
        attr_done = true;
    }
    const long tiles = (long)((a.M + 16 * NT - 1) / (16 * NT)) * (a.N / TN);
    hipLaunchKernelGGL((k_gemm_thin<MODE, WS, OB, NT>), dim3((unsigned)tiles), dim3(256), C::LDS, st, a);
    return hipGetLastError();
}

/* the loads address A, W and Sa with 31-bit byte offsets, and a row block's
 * scales fit one register */
static bool thin_ok(int M, int N, int K)
{
    return M > 0 && N % 128 == 0 && K % TB == 0 && K <= T_KMAX && (size_t)M * K < (1u << 31) &&
           (size_t)M * N / 1024 < (1u << 31);
}

template <int MODE, bool WS>
static hipError_t thin_nt(const ThinArgs &a, bool out_bf16, int nt, hipStream_t st)
{
    switch (nt) {
    case 1: return out_bf16 ? thin_launch<MODE, WS, true, 1>(a, st) : thin_launch<MODE, WS, false, 1>(a, st);
    case 2: return out_bf16 ? thin_launch<MODE, WS, true, 2>(a, st) : thin_launch<MODE, WS, false, 2>(a, st);
    default: return out_bf16 ? thin_launch<MODE, WS, true, 4>(a, st) : thin_launch<MODE, WS, false, 4>(a, st);
    }
}

static ThinArgs thin_args(const GemmArgs &g)
{
    ThinArgs a;
    a.A = g.Aq; a.Sa = g.Sa; a.W = g.W; a.Sw = g.Sw; a.C = g.C;
    a.M = g.M; a.N = g.N; a.K = g.K; a.sa_tok = g.sa_tok; a.sa_kb = g.sa_kb;
    return a;
}

hipError_t gemm_thin_fp8_launch(const GemmArgs &g, bool w_f32s, bool out_bf16, int nt, hipStream_t st)
{
    const ThinArgs a = thin_args(g);
    return w_f32s ? thin_nt<T_FP8, true>(a, out_bf16, nt, st) : thin_nt<T_FP8, false>(a, out_bf16, nt, st);
}

hipError_t gemm_thin_mx_launch(const GemmArgs &g, bool out_bf16, int nt, hipStream_t st)
{
    return thin_nt<T_MX, false>(thin_args(g), out_bf16, nt, st);
}

/* workgroups of nt 16-token groups a tile */
static long thin_wgs(int M, int N, int nt) { return ((long)M + 16 * nt - 1) / (16 * nt) * (N / TN); }

/* The widest spread that still fits one workgroup to a CU. us of the call,
 * quantization included, thin tiles against the 128 x 256 ones: 1024 x 4096
 * 8 tokens 13.5 / 26.6, 64 tokens 13.8 / 27.5, 300 tokens (nt 2) 16.6 / 30.0,
 * 700 tokens (nt 4) 23.6 / 32.6; 4096 x 4096 64 tokens 13.9 / 27.7; past 256
 * workgroups of nt = 4 the large tiles win (1024 x 4096, 1,300 tokens 34.2 /
 * 33.2; 4096 x 4096, 300 tokens 30.3 / 30.1): the small ones read W once per
 * token tile, through registers. */
int gemm_thin_nt(int M, int N, int K)
{
    if (!thin_ok(M, N, K)) return 0;
    for (int nt = 1; nt <= 4; nt *= 2)
        if (thin_wgs(M, N, nt) <= 256) return nt;
    return 0;
}

} // namespace dsv4
