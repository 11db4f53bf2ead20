/* SPDX-License-Identifier: Apache-2.0 */
/* dsv4_gemm_mid.hip - the FP8 GEMMs of dsv4_gemm.hip in tiles of 128 features
 * x 32, 64 or 128 tokens, for shapes whose 128 x 256 tiles leave most of the
 * device idle: few tokens, or a matrix of few rows.
 *
 * Two forms of C[m][n] = sum_k A[m][k] W[n][k], each with the products, the
 * reduction order and so the bits of its large-tile kernel:
 *   T_FP8   e4m3 tokens with fp32 1 x 128 scales, fp32 or E8M0 weight blocks,
 *           every 128-wide block's product folded into fp32 (k_gemm_fp8)
 *   T_MX    MXFP8 tokens, E8M0 weight blocks, both in the MFMA's scale
 *           operands (k_gemm_mx)
 *
 * SCHEDULE
 *   Waves: 4 x 32 features by one (T = 2) or two along the 16 T tokens. A
 *   stage is one 128-wide block: features, tokens and each wave's own tokens'
 *   scales by buffer loads straight to LDS, NST stages in a ring (two
 *   workgroups a CU for T <= 4). A wave reads its operands of the next stage
 *   while it multiplies one, a read and a load between the MFMAs, so that the
 *   barrier between stages waits for no read. The 64 weight scales of a row
 *   block sit in one register, one per lane. Loads past the end of K read
 *   nothing and multiply as zeros.
 *
 * Bound: one round of workgroups and its loads (a stage's 22 to 35 KB per CU
 * from L2). us of the call, quantization included, against the 128 x 256
 * tiles: MXFP8 1024 x 4096 8 tokens 26.8 -> 13.5, 300 tokens 29.7 -> 15.8,
 * 1,300 tokens 33.8 -> 23.1; 4096 x 4096 150 tokens 28.7 -> 14.7, 300 tokens
 * 30.0 -> 18.2, 1,000 tokens 33.2 -> 30.2. 64-feature tiles with the weights
 * straight to registers: 13.9 at 64 tokens as well, 29.8 at 4096 x 4096, 300
 * tokens (L2 reads through registers, once per token tile).
 */
#include "dsv4_internal.h"

namespace dsv4 {

namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

enum { T_FP8 = 0, T_MX = 1 };

constexpr int TB = 128;                            /* reduction block           */
static_assert(GEMM_MID_KMAX == 64 * TB, "one lane to a weight scale");
constexpr uint32_t T_OOB = 0x80000000u;            /* beyond every buffer       */
constexpr int T_E8M0_ONE = 127;

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
__device__ __forceinline__ uint32_t t_bf16(float f)
{
    const uint32_t u = __float_as_uint(f);
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (u >> 16) | 0x40u;   /* quiet NaN */
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

} // namespace

/* one call's operands in any of the forms */
struct MidArgs {
    const void *A;            /* e4m3 tokens [M][K]                               */
    const void *Sa;           /* token scales (a dword per token and block)       */
    const uint8_t *W;
    const void *Sw;
    void *C;
    int M, N, K;
    int sa_tok, sa_kb;        /* dword strides of Sa                              */
};

template <int T> struct Mid {
    static constexpr int WT = T >= 4 ? 2 : 1, NWAVE = 4 * WT, U = T / WT;
    static constexpr int OFF_X = 128 * TB, OFF_S = OFF_X + 16 * T * TB;
    static constexpr int STAGE = OFF_S + 256 * NWAVE;
    static constexpr int NST = T <= 4 ? 3 : 4;
    static constexpr int LDS = NST * STAGE;
    static constexpr int LW = 16 / NWAVE, LX = 2 * T / NWAVE, VM = LW + LX + 1;
    static_assert(LX * NWAVE == 2 * T && (NST - 1) * VM < 64 && LDS <= 160 * 1024, "ring");
    static_assert(U >= 2, "a stage's two weight operands are read beside the first two token groups");
};

template <int N>
__device__ __forceinline__ void t_wait()
{
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

template <int MODE, bool WF32S, bool OUT_BF16, int T>
__global__ __launch_bounds__(64 * Mid<T>::NWAVE) void k_gemm_mid(MidArgs a)
{
    using C = Mid<T>;
    constexpr int U = C::U;
    extern __shared__ __align__(16) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = wave_in_group();
    const int rr = lane & 15, gq = lane >> 4, wr = wave & 3, wt = wave >> 2;
    const int mt = (a.M + 16 * T - 1) / (16 * T), ft = a.N / 128, nst = a.K / TB;
    int lin = blockIdx.x;
    /* feature tiles of one XCD (workgroups go round the eight) side by side,
     * each with all its token tiles, when they divide: W is then fetched into
     * one L2 only */
    if (ft % 8 == 0) lin = (lin % 8) * (ft / 8 * mt) + lin / 8;
    const int n0 = lin / mt * 128, m0 = lin % mt * (16 * T);

    const __amdgpu_buffer_rsrc_t rx = t_rsrc(a.A, (uint32_t)a.M * (uint32_t)a.K);
    const __amdgpu_buffer_rsrc_t rw = t_rsrc(a.W + (size_t)n0 * a.K, 128u * (uint32_t)a.K);
    const __amdgpu_buffer_rsrc_t rs = t_rsrc(
        a.Sa, 4u * ((uint32_t)(nst - 1) * (uint32_t)a.sa_kb + (uint32_t)(a.M - 1) * (uint32_t)a.sa_tok + 1u));
    auto swz = [](int r, int c) { return c ^ ((r >> 1) & 7); };
    uint32_t wo[C::LW], xo[C::LX];
#pragma unroll
    for (int i = 0; i < C::LW; i++) {
        const int r = 8 * (C::LW * wave + i) + lane / 8;
        wo[i] = (uint32_t)r * (uint32_t)a.K + 16u * (uint32_t)swz(r, lane & 7);
    }
#pragma unroll
    for (int i = 0; i < C::LX; i++) {
        const int r = 8 * (C::LX * wave + i) + lane / 8;
        xo[i] = m0 + r < a.M ? (uint32_t)(m0 + r) * (uint32_t)a.K + 16u * (uint32_t)swz(r, lane & 7) : T_OOB;
    }
    const int ms = m0 + 16 * U * wt + lane;
    const uint32_t so = lane < 16 * U && ms < a.M ? 4u * (uint32_t)ms * (uint32_t)a.sa_tok : T_OOB;
    /* load i of a wave's share of stage st; past the end zeros, no traffic */
    auto issue = [&](int st, int slot, int i) {
        const uint32_t oob = st < nst ? 0u : T_OOB;
        const int sc = min(st, nst - 1);
        uint8_t *buf = lds + slot * C::STAGE;
        if (i < C::LW) t_dma16(rw, wo[min(i, C::LW - 1)] | oob, sc * TB, buf + 1024 * (C::LW * wave + i));
        else if (i < C::LW + C::LX)
            t_dma16(rx, xo[max(0, min(i - C::LW, C::LX - 1))] | oob, sc * TB,
                    buf + C::OFF_X + 1024 * (C::LX * wave + i - C::LW));
        else t_dma4(rs, so | oob, 4 * sc * a.sa_kb, buf + C::OFF_S + 256 * wave);
    };
    uint32_t wsc;                                  /* lane kb: the weight scale of block kb */
    {
        const size_t i = (size_t)(n0 / 128) * nst + min(lane, nst - 1);
        if constexpr (WF32S) wsc = __float_as_uint(ld_f32(a.Sw, i));
        else if constexpr (MODE == T_MX) wsc = ld_u8(a.Sw, i);
        else wsc = __float_as_uint(dev_e8m0(ld_u8(a.Sw, i)));
    }
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("" : "+v"(wsc));
#endif
#pragma unroll
    for (int s = 0; s < C::NST; s++)
#pragma unroll
        for (int i = 0; i < C::VM; i++) issue(s, s, i);

    struct Op { v8i w[2], x[U]; uint32_t ts[U]; };
    auto op16 = [&](v8i &o, const uint8_t *rows, int r) {
        const u32x4 lo = *(const u32x4 *)(rows + r * TB + 16 * swz(r, gq));
        const u32x4 hi = *(const u32x4 *)(rows + r * TB + 16 * swz(r, gq + 4));
#pragma unroll
        for (int e = 0; e < 4; e++) {
            o[e] = (int)lo[e];
            o[4 + e] = (int)hi[e];
        }
    };
    auto read_w = [&](Op &o, const uint8_t *buf, int i) { op16(o.w[i], buf, 32 * wr + 16 * i + rr); };
    auto read_x = [&](Op &o, const uint8_t *buf, int u) {
        op16(o.x[u], buf + C::OFF_X, 16 * (U * wt + u) + rr);
        o.ts[u] = *(const uint32_t *)(buf + C::OFF_S + 256 * wave + 4 * (16 * u + rr));
    };
    v4f acc[2][U], part[2][U];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int u = 0; u < U; u++) acc[i][u] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    int slot = 0;
    auto step = [&](const Op &cur, Op &nxt, int st) {
        __builtin_amdgcn_s_waitcnt(0xC07F);        /* this stage's operands are in registers */
        t_wait<(C::NST - 2) * C::VM>();            /* the wave's loads of the next have landed */
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int free = slot;
        slot = slot + 1 == C::NST ? 0 : slot + 1;
        const uint8_t *buf = lds + slot * C::STAGE;
        const uint32_t swv = (uint32_t)__builtin_amdgcn_readlane((int)wsc, min(st, nst - 1));
        auto fold = [&](int i, int u) {
            const float cs = st < nst ? __uint_as_float(cur.ts[u]) * __uint_as_float(swv) : 0.0f;
#pragma unroll
            for (int e = 0; e < 4; e++) acc[i][u][e] = fmaf(part[i][u][e], cs, acc[i][u][e]);
        };
#pragma unroll
        for (int q = 0; q < 2 * U; q++) {
            const int u = q >> 1, i = q & 1;
            if (i == 0) read_x(nxt, buf, u);
            else if (u < 2) read_w(nxt, buf, u);
            if constexpr (MODE == T_MX) {
                acc[i][u] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                    cur.w[i], cur.x[u], acc[i][u], 0, 0, 0, (int)swv, 0, (int)((cur.ts[u] >> (8 * gq)) & 0xFFu));
            } else {
                part[i][u] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                    cur.w[i], cur.x[u], v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0, T_E8M0_ONE, 0, T_E8M0_ONE);
                if (q >= 2) fold(i, u - 1);
            }
#pragma unroll
            for (int l = 0; l < C::VM; l++)
                if (l * 2 * U / C::VM == q) issue(st + C::NST, free, l);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (MODE != T_MX) {
            fold(0, U - 1);
            fold(1, U - 1);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    t_wait<(C::NST - 1) * C::VM>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    Op o0, o1;
#pragma unroll
    for (int i = 0; i < 2; i++) read_w(o0, lds, i);
#pragma unroll
    for (int u = 0; u < U; u++) read_x(o0, lds, u);
    for (int st = 0; st < nst; st += 2) {
        step(o0, o1, st);
        step(o1, o0, st + 1);
    }
    t_wait<0>();                                   /* the loads past the end */
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int m = m0 + 16 * (U * wt + u) + rr;
        if (m >= a.M) continue;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const size_t o = (size_t)m * a.N + n0 + 32 * wr + 16 * i + 4 * gq;
            const v4f v = acc[i][u];
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
}

template <int MODE, bool WS, bool OB, int T>
static hipError_t mid_launch(const MidArgs &a, hipStream_t st)
{
    using C = Mid<T>;
    static bool attr_done = false;
    if (!attr_done) {
        const hipError_t e = hipFuncSetAttribute((const void *)k_gemm_mid<MODE, WS, OB, T>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
        if (e != hipSuccess) return e;
        attr_done = true;
    }
    const long tiles = (long)((a.M + 16 * T - 1) / (16 * T)) * (a.N / 128);
    constexpr int lds_bytes = C::LDS;
    hipLaunchKernelGGL((k_gemm_mid<MODE, WS, OB, T>), dim3((unsigned)tiles), dim3(64 * C::NWAVE), lds_bytes, st, a);
    return hipGetLastError();
}

template <int MODE, bool WS>
static hipError_t mid_t(const MidArgs &a, bool out_bf16, int t, hipStream_t st)
{
    switch (t) {
    case 2: return out_bf16 ? mid_launch<MODE, WS, true, 2>(a, st) : mid_launch<MODE, WS, false, 2>(a, st);
    case 4: return out_bf16 ? mid_launch<MODE, WS, true, 4>(a, st) : mid_launch<MODE, WS, false, 4>(a, st);
    default: return out_bf16 ? mid_launch<MODE, WS, true, 8>(a, st) : mid_launch<MODE, WS, false, 8>(a, st);
    }
}

static MidArgs mid_args(const GemmArgs &g)
{
    MidArgs a;
    a.A = g.Aq; a.Sa = g.Sa; a.W = g.W; a.Sw = g.Sw; a.C = g.C;
    a.M = g.M; a.N = g.N; a.K = g.K; a.sa_tok = g.sa_tok; a.sa_kb = g.sa_kb;
    return a;
}

hipError_t gemm_mid_fp8_launch(const GemmArgs &g, bool w_f32s, bool out_bf16, int t, hipStream_t st)
{
    const MidArgs a = mid_args(g);
    return w_f32s ? mid_t<T_FP8, true>(a, out_bf16, t, st) : mid_t<T_FP8, false>(a, out_bf16, t, st);
}

hipError_t gemm_mid_mx_launch(const GemmArgs &g, bool out_bf16, int t, hipStream_t st)
{
    return mid_t<T_MX, false>(mid_args(g), out_bf16, t, st);
}

} // namespace dsv4
