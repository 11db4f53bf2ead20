/* SPDX-License-Identifier: Apache-2.0 */
/* dsv4_route.hip - the MoE router on the device.
 *
 * Replaces dsv4_route (src/10_compute/dsv4_ops.c:117-157), and, fused with
 * the BF16 gate matvec in front of it (dsv4_mmq at
 * src/70_decode/dsv4_layer.c:52), the decode step's router, so that no host
 * round trip separates the gate from the experts:
 *   orig[e]   = sqrt(softplus(scores[e]))   softplus(x) = x for x > 20
 *   biased[e] = orig[e] + bias[e]            (orig[e] without a bias)
 *   idx       = tid2eid[token] (hash routing), or the topk largest biased
 *               scores, descending, ties to the lower expert id
 *   w[k]      = orig[idx[k]] * inv * route_scale,  inv = (float)(1 / sum_k
 *               (double) orig[idx[k]]), 0 when that sum is 0
 * The bias steers the selection only; the weights come from orig.
 *
 * Selection, one wavefront per token. The reference's loop picks, for each
 * k, the first untaken expert and replaces it by every later untaken one
 * whose biased score is strictly greater. As a closed form: if the first
 * untaken score is NaN it stays; otherwise the pick is the largest non-NaN
 * untaken score, the lowest id among equals (+0 and -0 compare equal, as in
 * the loop). Lane l holds experts l, l + 64, ...; each pick is one wave
 * maximum of 64-bit keys (order-preserving bits of the score above, the
 * complemented id below) over DPP lane moves, with no LDS and no barrier;
 * the first-untaken minimum is taken only when the token has a NaN.
 *
 * orig is the reference's bits: sqrtf, log1pf and expf restated from the
 * host library's algorithms (dsv4_route_math.h; identical to the host's libm
 * on every fp32 input of [-104, 20]), so the picks are the reference's ids.
 *
 * A hash-routed id outside [0, n_experts), or a token id outside [0, n_vocab)
 * (whose ids are then -1), raises ST_BAD_EXPERT_ID; every weight of that
 * token is NaN, and the ids are written as they are so that the experts' own
 * range check catches them too.
 *
 * The fused gate + router (k_gate_route_bf16): a workgroup computes the fp64
 * dot products of four gate rows in bf16_n's order (dsv4_bf16.h: the bits of
 * dsv4_mmq on the host, src/10_compute/dsv4_matmul.c:88-113), their orig and
 * biased scores, and stores them device-scope (written through its XCD's
 * L2); once the stores are acknowledged it adds one to a counter. The
 * workgroup whose add completes the count is the last of the launch: every
 * other row's stores are visible to its device-scope loads, so its first
 * wave runs the selection, then sets the counter back to zero for the next
 * launch. Nothing waits on another workgroup. 256 rows of 4096: 12.7 -> 10.4
 * us with the chains on the fp64 MFMA instead of 256 dependent FMAs a lane
 * (one wave per row).
 *
 * Bound: launch latency; the gate's bytes (n_experts x hidden x 2) are read
 * once, by n_experts / 4 workgroups.
 */
#include "dsv4_gate_route.h"

namespace dsv4 {

namespace {

/* dsv4_route for n tokens given their scores: a workgroup per token, an expert
 * per thread (and every 256 beyond), so that the scores, the biases and the
 * exp tables of a token's experts are one latency each; then the first wave
 * selects. One wave per token with its experts one after another waited them
 * out NJ times (256 experts: 7 tokens 11.9 -> 5.4 us, 701 tokens 20.4 -> 9.1). */
template <int NJ>
__global__ __launch_bounds__(256) void k_route(GateRouteArgs a)
{
    __shared__ float so[64 * NJ], sbias[64 * NJ];
    const int t = blockIdx.x;
    const int lane = threadIdx.x & 63;
    const int ne = a.n_experts;
    const float *sc = a.scores + (size_t)t * a.scores_ld;
    constexpr int NE = (64 * NJ + 255) / 256;          /* experts of a thread */
    float v[NE], bv[NE];
#pragma unroll
    for (int j = 0; j < NE; j++) {
        const int e = min((int)threadIdx.x + 256 * j, ne - 1);
        v[j] = sc[e];
        bv[j] = a.bias ? a.bias[e] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < NE; j++) {
        const int e = threadIdx.x + 256 * j;
        if (e >= ne) continue;
        const float o = route_orig(v[j]);
        so[e] = o;
        sbias[e] = a.bias ? o + bv[j] : o;
        if (a.orig) a.orig[(size_t)t * ne + e] = o;
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    float og[NJ], bs[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int e = lane + 64 * j;
        og[j] = e < ne ? so[e] : 0.0f;
        bs[j] = e < ne ? sbias[e] : 0.0f;
    }
    bool hbad;
    const int64_t *hrow = hash_row(a, a.token_ids ? a.token_ids[t] : a.token_id, &hbad);
    route_wave<NJ>(og, bs, ne, a.topk, hrow, hbad, a.route_scale, a.idx + (size_t)t * a.topk,
                   a.w + (size_t)t * a.topk, a.status, lane);
}

template <int NJ>
__global__ __launch_bounds__(256) void k_gate_route_bf16(GateRouteArgs a)
{
    __shared__ __align__(16) uint8_t lds[b4_lds_bytes(1, B4_COLS)];
    gate_route_group<NJ>(a, gridDim.x, lds);
}

template <int NJ>
hipError_t launch_route_nj(const GateRouteArgs &a, hipStream_t st)
{
    if (a.gate_w) {
        hipLaunchKernelGGL(k_gate_route_bf16<NJ>, dim3((unsigned)((a.n_experts + 3) / 4)), dim3(256), 0, st, a);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_route<NJ>, dim3((unsigned)a.n), dim3(256), 0, st, a);
    return hipGetLastError();
}

} // namespace

bool gate_route_ok(const GateRouteArgs &a)
{
    if (a.n <= 0 || a.n_experts < 1 || a.n_experts > GATE_ROUTE_MAX_EXPERTS || a.topk < 1 ||
        a.topk > GATE_ROUTE_MAX_TOPK || a.topk > a.n_experts)
        return false;
    if (!a.gate_w) return a.scores_ld >= a.n_experts;
    return a.n == 1 && a.cols > 0 && a.cols % 8 == 0 && a.cols <= 4096 && a.counter && a.ws_orig && a.ws_biased;
}

hipError_t gate_route_launch(const GateRouteArgs &a, hipStream_t st)
{
    if (!gate_route_ok(a)) return hipErrorInvalidValue;
    const int nj = (a.n_experts + 63) / 64;
    if (nj <= 1) return launch_route_nj<1>(a, st);
    if (nj <= 2) return launch_route_nj<2>(a, st);
    if (nj <= 4) return launch_route_nj<4>(a, st);
    if (nj <= 8) return launch_route_nj<8>(a, st);
    return launch_route_nj<RT_MAXJ>(a, st);
}

} // namespace dsv4
