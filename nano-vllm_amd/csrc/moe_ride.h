// moe_ride.h -- a mixture's router and choices, and their sorting, beside the shared expert's products of hundreds of tokens: workgroups on
// the CUs that the tiles leave idle (RouteRider; gemm_wide.h, gemm_waves.h).
#pragma once

#include "gemm_common.h"
#include "moe_route.h"

namespace nvllm {

namespace {

constexpr int ROUTER_LD = 68, ROUTER_NB = 4;   // floats between a token's logits in LDS; row blocks of the widest router
constexpr int ROUTER_TB = 4;                   // token blocks at a time
constexpr int ROUTER_CHAINS = 8;               // sums of a logit's K: as many as the router's own launch has waves
constexpr int ROUTER_RIDE_LDS = ROUTER_TB * (2 * ROUTER_CHAINS * 1024 + 16 * ROUTER_LD * 4);

// Logits and choices of the activations (and their norm) that the tiles multiply: a workgroup's token blocks, ROUTER_TB at a time, in pairs of the
// router's row blocks, K dealt to the waves as in gemm_waves.h.  Sums in the order of the router's own launch (gemm_tile of eight waves), so that a
// mixture gives the same bits whether it rides or not -- a last bit moves the choice of a near tie: every eighth step is a chain of its own (even and odd
// steps of four waves), chains are added one after the other, and squares are summed in that launch's parts (RouteRider::ss_parts).
// What bounds it: the bytes into its CU (a token block per wave and all of K, where every wave reads the whole router, held the launch up: 33.8 us
// without riders, 44.6; so 34.8 with chains and squares summed in pairs, 35.5 in this order).
// Simivik-1.2B, prompts of 200, 256, 400, 700, 1,029, 1,500 tokens (router 8.7, choice and sorting 8 to 17 us a layer apart, 0.3 to 2 so):
// 3,008 -> 2,903, 3,427 -> 3,157, 3,519 -> 3,326, 4,130 -> 3,969, 4,912 -> 4,756, 5,774 -> 5,641 us a pass.
template <int WAVES>
__device__ __forceinline__ void router_ride(const GemmArgs& p, int wave, int lane, unsigned char* lds) {
    constexpr int RB = ROUTER_TB, RING = 4, MINE = (RB + WAVES - 1) / WAVES;   // MINE: token blocks that a wave finishes
    constexpr int CH = ROUTER_CHAINS / WAVES;                                   // chains of a wave
    static_assert(CH * WAVES == ROUTER_CHAINS && RING % CH == 0);
    const RouteRider& r = p.route;
    const int group = (int)blockIdx.x - p.ride_from, groups = (int)gridDim.x - p.ride_from, part = lane >> 4, cols = p.e.ss_tiles;
    f4_t* sums = reinterpret_cast<f4_t*>(lds);   // [RB][2][chain][64]
    float* rows = reinterpret_cast<float*>(lds + RB * 2 * ROUTER_CHAINS * 1024);   // [RB][16][ROUTER_LD]
    const int steps = wave < p.Kb ? (p.Kb - wave + WAVES - 1) / WAVES : 0;
    const bool parts32 = r.ss_parts == 32;   // (else 16)
    for (int tb0 = group * RB; tb0 < p.Tb; tb0 += groups * RB) {
        float rinv[MINE];
#pragma unroll
        for (int m = 0; m < MINE; m++) {
            rinv[m] = 1.f;
            if (!p.e.ss_in) continue;
            const float* sp = p.e.ss_in + (size_t)min((tb0 + wave + m * WAVES) * 16 + (lane & 15), p.T - 1) * cols;
            float of[8] = {};   // squares' part 4 u + (lane's row)
            for (int j0 = 0; j0 < cols; j0 += 64) {   // (all of a lane's requested together)
                float v[16];
#pragma unroll
                for (int k = 0; k < 16; k++) v[k] = sp[min(j0 + 4 * k + part, cols - 1)];
#pragma unroll
                for (int k = 0; k < 16; k++) {
                    if (j0 + 4 * k + part >= cols) v[k] = 0.f;
                    if (k & 4 && parts32) of[4 + (k & 3)] += v[k];
                    else of[k & 3] += v[k];
                }
            }
            float sum = 0.f;
#pragma unroll
            for (int q = 0; q < 32; q++) {
                const float v = __shfl(of[q >> 2], (lane & 15) + 16 * (q & 3), 64);
                if (q < 16 || parts32) sum += v;
            }
            rinv[m] = __fdiv_rn(1.0f, sqrtf(__fadd_rn(__fdiv_rn(sum, (float)p.e.d_in), p.e.eps)));
        }
        for (int f0 = 0; f0 < r.NB; f0 += 2) {
            const h8_t* w0 = reinterpret_cast<const h8_t*>(r.W + (size_t)f0 * p.Kb * TILE_HALVES) + lane;
            const h8_t* a0 = reinterpret_cast<const h8_t*>(p.A + (size_t)tb0 * p.Kb * TILE_HALVES) + lane;
            const int next = f0 + 1 < r.NB ? p.Kb * 64 : 0;
            int of[RB];
#pragma unroll
            for (int j = 0; j < RB; j++) of[j] = min(j, p.Tb - 1 - tb0) * p.Kb * 64;
            h8_t a[RING][RB], w[RING][2];
            f4_t acc[CH][RB][2];   // of this wave's chains: wave, wave + 4
            auto load = [&](int s, int i) {   // step i of this wave's into slot s (past the last: the last again, not multiplied)
                const int at = (wave + min(i, max(steps - 1, 0)) * WAVES) * 64;
                const bool any = wave < p.Kb;
                w[s][0] = w0[any ? at : 0];
                w[s][1] = w0[any ? at + next : 0];
#pragma unroll
                for (int j = 0; j < RB; j++) a[s][j] = a0[any ? at + of[j] : 0];
            };
            auto step = [&](int s) {
#pragma unroll
                for (int j = 0; j < RB; j++)
#pragma unroll
                    for (int f = 0; f < 2; f++) acc[s % CH][j][f] = OpBf16::mfma(w[s][f], a[s][j], acc[s % CH][j][f]);
            };
#pragma unroll
            for (int c = 0; c < CH; c++)
#pragma unroll
                for (int j = 0; j < RB; j++) acc[c][j][0] = acc[c][j][1] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < RING; s++) load(s, s);
            int i = 0;
            for (; i + RING <= steps; i += RING)
#pragma unroll
                for (int s = 0; s < RING; s++) {
                    step(s);
                    load(s, i + RING + s);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
            for (int s = 0; s < RING - 1; s++)
                if (i + s < steps) step(s);
            __syncthreads();   // (the sums of the pair before have been read)
#pragma unroll
            for (int c = 0; c < CH; c++)
#pragma unroll
                for (int j = 0; j < RB; j++)
#pragma unroll
                    for (int f = 0; f < 2; f++) sums[((j * 2 + f) * ROUTER_CHAINS + wave + WAVES * c) * 64 + lane] = acc[c][j][f];
            __syncthreads();
#pragma unroll
            for (int m = 0; m < MINE; m++) {
                const int j = wave + m * WAVES, t = (tb0 + j) * 16 + (lane & 15);
                if (j >= RB) continue;
#pragma unroll
                for (int f = 0; f < 2; f++) {
                    f4_t chain[ROUTER_CHAINS];
#pragma unroll
                    for (int u = 0; u < ROUTER_CHAINS; u++) chain[u] = sums[((j * 2 + f) * ROUTER_CHAINS + u) * 64 + lane];
                    f4_t sum = chain[0];
#pragma unroll
                    for (int u = 1; u < ROUTER_CHAINS; u++) sum += chain[u];
                    const int n = (f0 + f) * 16 + 4 * part;
                    const float4 y = make_float4(sum[0] * rinv[m], sum[1] * rinv[m], sum[2] * rinv[m], sum[3] * rinv[m]);
                    if (f0 + f < r.NB) {
                        *reinterpret_cast<float4*>(rows + (j * 16 + (lane & 15)) * ROUTER_LD + n) = y;
                        if (t < p.T) *reinterpret_cast<float4*>(r.z + (size_t)t * r.ldz + n) = y;
                    }
                }
            }
        }
        // (a wave chooses for the tokens whose logits it has formed)
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (int j = wave; j < RB; j += WAVES)
            for (int t4 = 0; t4 < 16; t4 += 4) {
                const int t = (tb0 + j) * 16 + t4;
                if (t >= p.T) break;
                float v[4];
#pragma unroll
                for (int u = 0; u < 4; u++) v[u] = lane < r.plan.E ? rows[(j * 16 + t4 + u) * ROUTER_LD + lane] : -INFINITY;
                choose_four(v, r.plan.E, r.plan.top, lane, [&](int u, int k, int e, float score) {
                    if (t + u < p.T) {
                        r.plan.choice[(size_t)(t + u) * r.plan.top + k] = e;
                        r.plan.score[(size_t)(t + u) * r.plan.top + k] = score;
                    }
                });
            }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): else the compiler waits inside the tiles' loop for what flies here
}

// Riders beside `tiles` workgroups, of which a CU holds one: on free CUs only, and only what is done about when the tiles are: up to two passes of the
// router over a workgroup's blocks, of which a wave chooses for 16 tokens, and up to 4,096 choices to sort (256 threads; the launch of its own has 1,024).
// In us: a pass over the blocks, a step of four tokens' choices, the tiles at 900 TFLOP/s; and what the launches of router, choice and sorting take that
// are saved.  Those launches and both products together, riding and apart, pairs of 2,816 features over 2,048 k: 2 of 16 experts, 400 and 1,029 tokens 31
// and 50, 57 and 68; 8 of 63, 256, 700, 1,500 tokens 55 and 91, 71 and 68, 99 and 103; over 1,024 k 4 of 31, 400, 1,029 (two trips of a rider), 1,500
// tokens 33 and 41, 65 and 56, 54 and 63; 8 of 63 256, 700, 1,500 46 and 85, 63 and 53, 80 and 76; of 768 features over 288 k 39 and 73, 50 and 35, 61 and 50.
inline int route_groups(const GemmArgs& a, int tiles) {
    const RoutePlan& r = a.route.plan;
    const int spare = rt().num_cus - tiles;
    if (r.T == 0 || spare <= 0) return 0;
    if (a.e.kind == GemmEpilogue::F32) return (long)r.T * r.top <= 4096 && r.E <= 1024 ? 1 : 0;
    if (a.e.kind != GemmEpilogue::SWIGLU_A16 || a.route.NB > ROUTER_NB || r.E > 64 || !router_parts(a.Tb, a.route.NB)) return 0;
    const int groups = std::min(cdiv(a.Tb, ROUTER_TB), spare), trips = cdiv(a.Tb, groups * ROUTER_TB), passes = cdiv(a.route.NB, 2);
    if (trips * passes > 2) return 0;
    const double rider = 2.0 + trips * (passes * (2.0 + 0.065 * a.Kb) + 4.0 * r.top * 0.87), tiled = 5.0 + 1024.0 * r.T * a.Kb * a.NB / 9.0e8;
    const double saved = 7.5 + 0.06 * a.Kb + (r.T <= ROUTE_ONE ? 1.0 + route_us(r.T, r.E, r.top, 16) : 3.0 + 0.5 * r.top);
    return rider <= tiled + saved ? groups : 0;
}

}  // namespace

}  // namespace nvllm
