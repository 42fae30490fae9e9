// gemm_f32.hip -- out[T, N] = act[T, K] x W[N, K]^T with everything in fp32, on v_mfma_f32_16x16x4_f32 (an exact fma
// chain), and the element-wise work around a projection in the same launch: the RMS norm in front (x * gain enters the
// product, 1/rms scales its sums -- a scalar per token commutes with the projection), and behind it SwiGLU of a gated
// pair, the residual add, rotation and cache rows.
//
// A workgroup owns NB 16-row blocks of W (of both matrices of a pair) x TB 16-token blocks; its KS waves take the K-steps of
// 32 round-robin and meet in LDS, so nothing is cut across workgroups and a launch needs no second one.
// Operands go from global memory into MFMA registers as they lie: lane (row x, group g) reads 4 consecutive k at
// 4g (+16 for the step's second half), product i of a quad takes element i of every lane, and the same rule on both
// sides makes the four products one 16-deep step.  No LDS staging: at 2 x 4 blocks a step of 32 multiplies (1,024
// matrix-core cycles per SIMD) needs 6 KiB per wave, 24 bytes per cycle and CU, well below what L2 delivers.
//
// What bounds it: few tokens -- bytes of W, and below ~10 MB the launch itself; hundreds of tokens -- the fp32 matrix
// rate (157 TFLOP/s).  These products occupy the vector unit: an addition of four registers between them costs half of one.
// A launch of few tokens is a chain of trips to memory (a dependent launch that reads and writes one value: 1.6 us), so every trip
// that depends on nothing starts at once: the arguments' lines, the tile's segment without a loop over them, and positions, cache rows,
// angles and residual values with the first steps instead of behind the last (tiles of four blocks and more: behind it).  us a launch before and
// with that: stories15M, one row, q/k/v 5.1 -> 4.6, gate/up 5.6 -> 5.2, wo and w_down 4.9 -> 4.4; Simivik-0.4B, 80 tokens, 64 x 3 tiles of 1 x 2 blocks
// 11.9 -> 11.4.  A pass 217 -> 204 (with the ids out of the classifier's blocks) and 1,657 -> 1,598.
#include <algorithm>
#include <climits>

#include "gemm_common.h"
#include "gemm_f32_tail.h"
#include "moe_route.h"

namespace nvllm {

constexpr int F32_STEP = 32;   // k per step: 128 bytes, a cache line, of every row
// waves per SIMD the registers are dealt for: two workgroups of eight waves share a CU where the tiles allow it
constexpr int f32_occupancy(int tiles, bool norm) { return tiles >= 6 ? 2 : tiles == 4 && norm ? 3 : 4; }

// AMAX: the classifier's, which leaves pairs (F32Gemm::amax_pairs)
template <int NB, int TB, int KS, bool PAIR, bool NORM, bool AMAX = false>
__global__ __launch_bounds__(KS * 64, f32_occupancy((PAIR ? 2 : 1) * NB * TB, NORM)) void k_gemm_f32(F32Gemm p) {
    constexpr int NT = PAIR ? 2 * NB : NB;   // weight blocks per step: all of the first matrix, then all of the second
    constexpr int RING = NT * TB == 1 ? (NORM ? 3 : 4) : 2;
    constexpr int ITEMS = NB * TB * 64;   // results, four features of a token each
    constexpr int FPT = (ITEMS + KS * 64 - 1) / (KS * 64);
    request_arguments<sizeof(F32Gemm)>();
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_f32[];
    f4_t(*s_red)[NT * TB][64] = reinterpret_cast<f4_t(*)[NT * TB][64]>(lds_f32);                     // [wave]
    float(*s_ss)[TB * 16] = reinterpret_cast<float(*)[TB * 16]>(lds_f32 + KS * NT * TB * 1024);   // NORM: [wave]
    if constexpr (PAIR && NORM) {
        if ((int)blockIdx.x >= p.route_from) {
            if (blockIdx.y == 0) route_sort<true, KS * 64>(p.route, p.z, p.ldz, reinterpret_cast<int*>(lds_f32));
            return;
        }
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = lane & 15, g = lane >> 4;
    const int tile = (int)blockIdx.x;
    const F32Segment& sg = p.seg[f32_segment(p, tile)];
    const int nb0 = (tile - sg.first) * NB, tb0 = (int)blockIdx.y * TB;
    const int K = p.K, T = p.T, N = sg.N;
    const float *W = sg.W, *W2 = sg.W2;
    if (p.block_expert) {   // (TB = 1: a workgroup's rows are of one expert)
        const int e = __builtin_amdgcn_readfirstlane(p.block_expert[tb0]);
        if (e < 0) return;   // fewer rows than the launch has room for
        W += (size_t)e * p.expert_stride;
        if (PAIR) W2 += (size_t)e * p.expert_stride;
    }
    const float* wp[NT];
#pragma unroll
    for (int i = 0; i < NB; i++) {
        const size_t row = (size_t)min((nb0 + i) * 16 + x, N - 1) * K + 4 * g;   // rows past the last are read again and not stored
        wp[i] = W + row;
        if constexpr (PAIR) wp[NB + i] = W2 + row;
    }
    const float* ap[TB];
#pragma unroll
    for (int j = 0; j < TB; j++) {
        int t = min((tb0 + j) * 16 + x, T - 1);
        if (p.in_rows) {
            t = p.in_rows[t];
            asm volatile("" ::"v"(t));   // (waited for here, and not where launches without these rows meet)
        }
        ap[j] = p.in + (size_t)t * K + 4 * g;
    }
    const float* gp = NORM ? p.gain + 4 * g : nullptr;

    // What the epilogue needs beside the sums travels with the first steps, and angles behind their positions; with four blocks or more it is
    // asked for behind the last: their products hide less of a wait for it in front of them than the meeting of the waves' sums hides behind, and
    // 2 x 2 blocks at four waves a SIMD have no registers for it.  us a launch with the first steps -> behind the last, q/k/v: 2 x 2 blocks of
    // stories42M, 150 tokens 9.6 -> 8.7, of stories15M, 240 tokens 7.3 -> 6.6; 2 x 3 of stories42M, 480 tokens 17.1 -> 16.7; 2 x 4, 301 tokens 13.1 -> 12.0,
    // 900 tokens 29.4 -> 28.4 (w_down 12.3 -> 11.6); the other way 1 x 1 blocks of stories15M, one row 4.6 against 5.1.
    constexpr bool EARLY = PAIR || NT * TB < 4;
    const bool turns = !PAIR && !AMAX && f32_turns(sg), adds = !PAIR && sg.kind == F32Out::ADD;
    int at[FPT], row[FPT];
    f4_t side[FPT];   // angles, or what is added to
    auto item = [&](int q, int& t, int& n) {
        const int e = min((int)threadIdx.x + q * KS * 64, ITEMS - 1), l = e & 63;
        t = min((tb0 + (e >> 6) % TB) * 16 + (l & 15), T - 1);
        n = (nb0 + (e >> 6) / TB) * 16 + 4 * (l >> 4);
    };
    auto request_positions = [&] {
#pragma unroll
        for (int q = 0; q < FPT; q++) {
            int t, n;
            item(q, t, n);
            at[q] = turns ? p.pos[t] : 0;
        }
    };
    if constexpr (EARLY) request_positions();
    auto request_side = [&] {
        if constexpr (AMAX) return;   // (its rows are stored as they are)
        if constexpr (!EARLY) request_positions();
#pragma unroll
        for (int q = 0; q < FPT; q++) {
            int t, n;
            item(q, t, n);
            row[q] = PAIR ? -1 : f32_row(p, sg, t);
            if (turns) side[q] = f32_angles(p, at[q], n);
            else if (adds) side[q] = f32_old(sg, t, n);
            else side[q] = f4_t{0.f, 0.f, 0.f, 0.f};
        }
    };

    f4_t w[RING][NT][2], a[RING][TB][2], gv[RING][NORM ? 2 : 1];
    const f4_t zero = {0.f, 0.f, 0.f, 0.f};
    auto load = [&](int r, int i) {
        const int k = (wave + i * KS) * F32_STEP;
        __builtin_amdgcn_sched_barrier(0);   // requests stay in the order of their use: waits count what is younger
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int n = 0; n < NT; n++) w[r][n][h] = *reinterpret_cast<const f4_t*>(wp[n] + k + 16 * h);
#pragma unroll
            for (int j = 0; j < TB; j++) a[r][j][h] = *reinterpret_cast<const f4_t*>(ap[j] + k + 16 * h);
            if constexpr (NORM) gv[r][h] = *reinterpret_cast<const f4_t*>(gp + k + 16 * h);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // Short chains keep the error that of pairwise sums.  One block by eight waves keeps the eight products of a step apart, each
    // in a chain of its own over the wave's steps: 64 chains of K / 64, no addition between products.  Larger tiles have no
    // registers for that, four waves too few chains: they sum chains of eight (two products of four k) over every step, a tile's
    // behind the next one's first products.  Error against 64 bits in 1e-8, K = 288 / 512 / 1,024: 64 chains 7.8 / 8.6 / 10, chains
    // of eight 8.2 / 8.7 / 9.5, of 16 9.9 / 10 / 10.5; chains of four 7.9 / 8.4 / 9.2, but a pass of 301 tokens takes 7 % longer.
    constexpr int TILES = NT * TB;
    constexpr bool APART = TILES == 1 && KS == 8;
    static_assert(TILES == 1 || TILES % 2 == 0, "two sets of chains in turn, from one step's last tile to the next one's first");
    f4_t acc[NT][TB], chain[APART ? 1 : 2][APART ? 8 : 4];
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int j = 0; j < TB; j++) acc[n][j] = zero;
#pragma unroll
    for (int t = 0; t < (APART ? 1 : 2); t++)
#pragma unroll
        for (int q = 0; q < (APART ? 8 : 4); q++) chain[t][q] = zero;
    float ss[TB];
#pragma unroll
    for (int j = 0; j < TB; j++) ss[j] = 0.f;
    auto multiply = [&](int r) {
        if constexpr (NORM) {
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int j = 0; j < TB; j++) {
                    f4_t& v = a[r][j][h];
                    float sq = v[0] * v[0];
#pragma unroll
                    for (int e = 1; e < 4; e++) sq = fmaf(v[e], v[e], sq);
                    ss[j] += sq;
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] *= gv[r][h][e];
                }
        }
        auto product = [&](int t, int q, const f4_t& sum) {
            return __builtin_amdgcn_mfma_f32_16x16x4f32(w[r][t / TB][q >> 2][q & 3], a[r][t % TB][q >> 2][q & 3], sum, 0, 0, 0);
        };
        if constexpr (APART) {
#pragma unroll
            for (int q = 0; q < 8; q++) chain[0][q] = product(0, q, chain[0][q]);
        } else if constexpr (TILES == 1) {
            f4_t(&c)[4] = chain[0];
#pragma unroll
            for (int q = 0; q < 4; q++) c[q] = product(0, 2 * q, zero);
#pragma unroll
            for (int q = 0; q < 4; q++) c[q] = product(0, 2 * q + 1, c[q]);
            acc[0][0] += (c[0] + c[1]) + (c[2] + c[3]);
        } else {
#pragma unroll
            for (int t = 0; t < TILES; t++) {
                f4_t(&c)[4] = chain[t & 1];
                f4_t(&old)[4] = chain[(t & 1) ^ 1];   // the tile before (at first: the last tile of the step before)
                f4_t& to = acc[(t + TILES - 1) % TILES / TB][(t + TILES - 1) % TILES % TB];
#pragma unroll
                for (int q = 0; q < 4; q++) c[q] = product(t, 2 * q, zero);
                __builtin_amdgcn_sched_barrier(0);
                to += (old[0] + old[1]) + (old[2] + old[3]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = 0; q < 4; q++) c[q] = product(t, 2 * q + 1, c[q]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // Whole steps: the steady loop requests without a condition (where paths with and without requests meet, the compiler
    // waits for all of them); what is left of it is at most RING conditional requests.
    const int whole = K / F32_STEP;
    const int mine = wave < whole ? (whole - wave + KS - 1) / KS : 0;
    if (mine < RING) {
#pragma unroll
        for (int r = 0; r + 1 < RING; r++)
            if (r < mine) load(r, r);
        if constexpr (EARLY) request_side();
#pragma unroll
        for (int r = 0; r + 1 < RING; r++)
            if (r < mine) multiply(r);
    } else {
#pragma unroll
        for (int r = 0; r < RING; r++) load(r, r);
        if constexpr (EARLY) request_side();
        int i0 = 0;
        for (; i0 + 2 * RING <= mine; i0 += RING) {
#pragma unroll
            for (int r = 0; r < RING; r++) {
                multiply(r);
                load(r, i0 + r + RING);
            }
        }
#pragma unroll
        for (int r = 0; r < RING; r++) {
            if (i0 + r < mine) multiply(r);
            if (i0 + r + RING < mine) load(r, i0 + r + RING);
        }
#pragma unroll
        for (int r = 0; r < RING; r++)
            if (i0 + r + RING < mine) multiply(r);
    }
    if (whole * F32_STEP < K && whole % KS == wave) {   // the rest of K (K % 4 == 0: a lane's four are in or out together)
        const int k = whole * F32_STEP;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const bool in = k + 16 * h + 4 * g < K;
#pragma unroll
            for (int n = 0; n < NT; n++) w[0][n][h] = in ? *reinterpret_cast<const f4_t*>(wp[n] + k + 16 * h) : zero;
#pragma unroll
            for (int j = 0; j < TB; j++) a[0][j][h] = in ? *reinterpret_cast<const f4_t*>(ap[j] + k + 16 * h) : zero;
            if constexpr (NORM) gv[0][h] = in ? *reinterpret_cast<const f4_t*>(gp + k + 16 * h) : zero;
        }
        multiply(0);
    }
    if constexpr (APART) {
        const f4_t(&c)[8] = chain[0];
        acc[0][0] = ((c[0] + c[1]) + (c[2] + c[3])) + ((c[4] + c[5]) + (c[6] + c[7]));
    } else if constexpr (TILES > 1) {
        acc[NT - 1][TB - 1] += (chain[1][0] + chain[1][1]) + (chain[1][2] + chain[1][3]);
    }
    auto rinv_of = [&](float sum) { return __fdiv_rn(1.0f, sqrtf(__fadd_rn(__fdiv_rn(sum, (float)K), p.eps))); };
    if constexpr (NORM) {
#pragma unroll
        for (int j = 0; j < TB; j++) {
            ss[j] += __shfl_xor(ss[j], 16, 64);
            ss[j] += __shfl_xor(ss[j], 32, 64);
        }
    }
    auto finish = [&](int t, int n, f4_t y, f4_t u, float sum, f4_t side, int row) {
        const bool live = t < T && n < N;
        if (!AMAX && !live) return;
        float scale = NORM ? rinv_of(sum) : 1.f;
        if (p.row_weight) scale *= p.row_weight[AMAX ? min(t, T - 1) : t];
        if (NORM || p.row_weight) {
            y *= scale;
            if constexpr (PAIR) u *= scale;
        }
        if (live) f32_finish<PAIR>(p, sg, t, n, y, u, side, row);
        if constexpr (AMAX) f32_pairs(p, N, n >> 4, n, t, (n & 15) == 0 && live, y);
    };
    if constexpr (!EARLY) request_side();
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int j = 0; j < TB; j++) s_red[wave][n * TB + j][lane] = acc[n][j];
    if constexpr (NORM) {
#pragma unroll
        for (int j = 0; j < TB; j++)
            if (g == 0) s_ss[wave][j * 16 + x] = ss[j];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < FPT; q++) {
        const int e = (int)threadIdx.x + q * KS * 64;
        if (e >= ITEMS) break;
        const int l = e & 63, j = (e >> 6) % TB, i = (e >> 6) / TB;
        auto waves = [&](int block) {
            f4_t z[KS];
#pragma unroll
            for (int v = 0; v < KS; v++) z[v] = s_red[v][block][l];
#pragma unroll
            for (int d = 1; d < KS; d <<= 1)
#pragma unroll
                for (int v = 0; v + d < KS; v += 2 * d) z[v] += z[v + d];
            return z[0];
        };
        const f4_t y = waves(i * TB + j), u = PAIR ? waves((NB + i) * TB + j) : zero;
        float sum = 0.f;
        if constexpr (NORM) {
#pragma unroll
            for (int v = 0; v < KS; v++) sum += s_ss[v][j * 16 + (l & 15)];
        }
        finish((tb0 + j) * 16 + (l & 15), (nb0 + i) * 16 + 4 * (l >> 4), y, u, sum, AMAX ? zero : side[q], AMAX ? -1 : row[q]);
    }
}

template <int NB, int TB, int KS, bool PAIR, bool NORM, bool AMAX = false>
void launch_f32(const F32Gemm& a, dim3 grid) {
    constexpr int LDS = KS * ((PAIR ? 2 : 1) * NB * TB * 1024 + (NORM ? TB * 64 : 0));
    const int lds = (int)grid.x > a.route_from ? std::max(LDS, (int)route_sort_lds(a.route.T, a.route.E, a.route.top)) : LDS;
    static bool enabled = false;
    if (LDS > 64 * 1024 && !enabled) {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_f32<NB, TB, KS, PAIR, NORM, AMAX>), hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        enabled = true;
    }
    NVLLM_LAUNCH((k_gemm_f32<NB, TB, KS, PAIR, NORM, AMAX>), grid, dim3(KS * 64), lds, a);
}

// Rows that are no multiples of 16 bytes (K % 4 != 0, or a caller's odd pointer): a wave sums four features of four tokens,
// its lanes striding over k.
template <bool PAIR>
__global__ __launch_bounds__(256) void k_gemm_f32_any(F32Gemm p) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const F32Segment& sg = p.seg[f32_segment(p, (int)blockIdx.x)];
    const int n = (((int)blockIdx.x - sg.first) * 4 + wave) * 4;
    int t0 = (int)blockIdx.y * 4;
    const int K = p.K, T = p.T, N = sg.N;
    if (n >= N) return;
    for (; t0 < T; t0 += (int)gridDim.y * 4) {
        const float *W = sg.W, *W2 = sg.W2;
        if (p.block_expert) {
            const int e = p.block_expert[t0 >> 4];
            if (e < 0) continue;
            W += (size_t)e * p.expert_stride;
            if (PAIR) W2 += (size_t)e * p.expert_stride;
        }
        float acc[4][4] = {}, acc2[4][4] = {}, ss[4] = {};   // [token][feature]
        const float* ap[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int t = min(t0 + j, T - 1);
            ap[j] = p.in + (size_t)(p.in_rows ? p.in_rows[t] : t) * K;
        }
        for (int k = lane; k < K; k += 64) {
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                v[j] = ap[j][k];
                if (p.gain) {
                    ss[j] = fmaf(v[j], v[j], ss[j]);
                    v[j] *= p.gain[k];
                }
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const size_t at = (size_t)min(n + i, N - 1) * K + k;
                const float w = W[at], w2 = PAIR ? W2[at] : 0.f;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    acc[j][i] = fmaf(v[j], w, acc[j][i]);
                    if (PAIR) acc2[j][i] = fmaf(v[j], w2, acc2[j][i]);
                }
            }
        }
        auto total = [](float v) {
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
            return v;
        };
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float scale = 1.f;
            if (p.gain) scale = __fdiv_rn(1.0f, sqrtf(__fadd_rn(__fdiv_rn(total(ss[j]), (float)K), p.eps)));
            if (p.row_weight) scale *= p.row_weight[min(t0 + j, T - 1)];
            f4_t y, u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                y[i] = total(acc[j][i]) * scale;
                if (PAIR) u[i] = total(acc2[j][i]) * scale;
            }
            const int t = t0 + j;
            if (lane == 0 && t < T) {
                const f4_t side = PAIR ? u : sg.kind == F32Out::ADD ? f32_old(sg, t, n) : f32_turns(sg) ? f32_angles(p, p.pos[t], n) : u;
                f32_finish<PAIR>(p, sg, t, n, y, u, side, f32_row(p, sg, t));
            }
        }
    }
}

static bool launch_products(const F32Gemm& g, int prof_cls, bool* has_pairs) {
    F32Gemm a = g;
    const bool pair = a.seg[0].W2 != nullptr;
    double weights = 0, outs = 0;
    int blocks = 0;   // 16-row blocks of W (of each matrix of a pair)
    auto aligned = [](const void* q) { return (reinterpret_cast<size_t>(q) & 15) == 0; };
    bool rows16 = a.K % 4 == 0 && aligned(a.in) && aligned(a.gain);
    for (int s = 0; s < a.n_segs; s++) {
        F32Segment& q = a.seg[s];
        if (pair != (q.W2 != nullptr) || q.N <= 0) NVLLM_FATAL("fp32 projection: segment %d of %d", s, a.n_segs);
        rows16 = rows16 && aligned(q.W) && aligned(q.W2) && a.expert_stride % 4 == 0;
        q.vec = q.N % 4 == 0 && q.ldo % 4 == 0 && aligned(q.out);
        weights += (double)q.N * a.K * (pair ? 2 : 1);
        outs += q.N;
        blocks += cdiv(q.N, 16);
    }
    // Blocks per wave.  A launch takes about what its busiest CU has to fetch (64 bytes per block and k, at about 20 bytes
    // per cycle of the mix of weights and activations) and to multiply (8 cycles per product and quad of k on four SIMDs):
    // larger tiles fetch less per product, smaller ones reach more CUs.  K = 512 at 301 tokens: 2 x 2 blocks of a 512-wide
    // output 8 us, 1 x 1 10 us; 2 x 4 of a 1,536-wide one 13.6 us against 17.0 in 2 x 2.  Three token blocks where two and four fill
    // their last round worse: 2,816 features x 1,024 k at 80 tokens (176 tiles of 2 x 3; 880 of 1 x 1) 19.9 -> 15.5, 1,024 x 1,024 at
    // 300 15.9 -> 14.4, 864 x 288 at 301 11.6 -> 7.9; pairs 2 x 768 x 288 at 200 10.9 -> 7.9, 2 x 2,816 x 1,024 at 170 38.0 -> 32.3.  (1 x 3 of a
    // plain one fetches as much per CU as 2 x 2: 13.6 -> 13.1 at best.)  With a short K in one round only: a second one has too few steps to hide its
    // start (K = 288, pairs of 768 at 690 tokens 18.1 -> 20.3, 864 features at 600 11.0 -> 12.7).
    const int Tb = cdiv(a.T, 16), cus = rt().num_cus;
    static const int shapes[][2] = {{1, 1}, {1, 2}, {2, 2}, {2, 3}, {2, 4}}, pair_shapes[][2] = {{1, 1}, {1, 2}, {1, 3}, {1, 4}};
    int NB = 1, TB = 1;
    long tiles_all = (long)blocks * Tb;
    double best = 0;   // cycles per k
    if (!a.block_expert && rows16) {
        for (int i = 0; i < (pair ? 4 : 5); i++) {
            const int nb = pair ? pair_shapes[i][0] : shapes[i][0], tb = pair ? pair_shapes[i][1] : shapes[i][1], nt = pair ? 2 * nb : nb;
            const long tiles = (long)cdiv(blocks, nb) * cdiv(Tb, tb);
            if (tb == 3 && tiles > cus && a.K < 512) continue;
            const double cost = (double)cdiv((int)std::min(tiles, 1L << 30), cus) * ((nt + tb) * 64.0 / 20.0 + nt * tb * 2.0);
            if (i == 0 || cost < best) best = cost, NB = nb, TB = tb, tiles_all = tiles;
        }
    }
    // Thousands of tiles (a classifier): two row blocks share a workgroup's start and its activations, 32,000 x 1,024 for one
    // token 31.4 -> 28.1 us.  Slices of K: eight until every SIMD has two waves; of the large tiles in one round only, and of 2 x 4 blocks
    // where eight waves request all of K at once (1,536 features x 512 at 301 tokens 12.3 -> 11.7; 1,024 x 2,816 at 400 34.0 -> 36.0).
    if (!pair && NB == 1 && TB == 1 && !a.block_expert && tiles_all >= 4L * cus) {
        NB = 2;
        tiles_all = (long)cdiv(blocks, 2) * Tb;
    }
    const int KS = TB > 2 ? (tiles_all <= cus && (TB == 3 || a.K <= 512) ? 8 : 4) : tiles_all * 4 < (a.block_expert ? 16L : 8L) * cus ? 8 : 4;   // (a grid of experts is an upper bound)
    int tiles = 0;
    for (int s = 0; s < a.n_segs; s++) {
        a.seg[s].first = tiles;
        tiles += cdiv(cdiv(a.seg[s].N, 16), NB);
    }
    for (int s = a.n_segs; s < F32_SEGMENTS; s++) a.seg[s].first = INT_MAX;
    ProfScope ps(prof_cls, 4.0 * (weights * a.touched + (double)a.live * (a.K + outs)), 2.0 * a.live * weights);
    if (!rows16) {   // (its maxima are found in the rows)
        const dim3 grid(tiles, std::min(cdiv(a.T, 4), 32768));
        if (pair) NVLLM_LAUNCH(k_gemm_f32_any<true>, grid, dim3(256), 0, a);
        else NVLLM_LAUNCH(k_gemm_f32_any<false>, grid, dim3(256), 0, a);
        *has_pairs = false;
        return false;
    }
    // Choices of few tokens and their sorting, by one workgroup more (route_rides)
    a.route_from = tiles;
    const bool rides = a.route.T > 0 && pair && a.gain && route_rides(a.route, KS, 3.0 + best * a.K / 2600.0) && route_sort_lds(a.route.T, a.route.E, a.route.top) <= 64 * 1024;
    if (rides) ps.add(choice_bytes(a.route), 0);
    const dim3 grid(tiles + rides, cdiv(Tb, TB));
#define NVLLM_GEMM_F32(nb, tb, ks, pr)                                                                    \
    do {                                                                                                  \
        if (!pr && a.gain && a.amax_out) launch_f32<nb, tb, ks, pr, true, !pr>(a, grid);                  \
        else if (a.gain) launch_f32<nb, tb, ks, pr, true>(a, grid);                                       \
        else launch_f32<nb, tb, ks, pr, false>(a, grid);                                                  \
    } while (0)
#define NVLLM_GEMM_F32_4_8(nb, tb, pr)                                                                    \
    do {                                                                                                  \
        if (KS == 8) NVLLM_GEMM_F32(nb, tb, 8, pr);                                                       \
        else NVLLM_GEMM_F32(nb, tb, 4, pr);                                                               \
    } while (0)
    if (pair) {
        if (TB == 1) NVLLM_GEMM_F32_4_8(1, 1, true);
        else if (TB == 2) NVLLM_GEMM_F32_4_8(1, 2, true);
        else if (TB == 3) NVLLM_GEMM_F32_4_8(1, 3, true);
        else NVLLM_GEMM_F32_4_8(1, 4, true);
    } else if (TB == 1) {
        if (NB == 1) NVLLM_GEMM_F32_4_8(1, 1, false);
        else NVLLM_GEMM_F32_4_8(2, 1, false);
    } else if (TB == 2) {
        if (NB == 1) NVLLM_GEMM_F32_4_8(1, 2, false);
        else NVLLM_GEMM_F32_4_8(2, 2, false);
    } else if (TB == 3) {
        NVLLM_GEMM_F32_4_8(2, 3, false);
    } else {
        NVLLM_GEMM_F32_4_8(2, 4, false);
    }
#undef NVLLM_GEMM_F32_4_8
#undef NVLLM_GEMM_F32
    return rides;
}

bool launch_gemm_f32(const F32Gemm& g, int prof_cls) {
    if (g.T <= 0 || g.n_segs == 0) return false;
    if (g.amax_out && (!g.amax_pairs || g.amax_ld < g.T)) NVLLM_FATAL("fused arg-max needs a pair buffer of at least %d rows per block", g.T);
    // Pairs from products behind a norm, of as many outputs as fp32 has whole numbers for (a pair's index is one); else the rows are scanned
    bool has_pairs = g.amax_out && g.gain && !g.seg[0].W2 && g.seg[0].N <= 1 << 24;
    F32Gemm a = g;
    if (!has_pairs) a.amax_out = nullptr;
    const bool rides = launch_products(a, prof_cls, &has_pairs);
    // us a launch for one row of 32,000, 64 and 128 of them: scanned 7.2, 8.1, 8.9, pairs merged 6.0, 7.5, 9.0 (and the classifier no slower for leaving them)
    if (has_pairs) launch_argmax_tiles(g.amax_out, g.amax_pairs, cdiv(g.seg[0].N, 16), g.T, g.amax_ld, g.amax_out_host);
    else if (g.amax_out) launch_argmax_ld(g.amax_out, g.seg[0].out, g.T, g.seg[0].N, g.seg[0].ldo, g.amax_out_host);
    return rides;
}

}  // namespace nvllm
