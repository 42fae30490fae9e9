// gemm_thin.hip -- projections of fp16 weights for up to 6 tokens: the layers of a model that serves one user or a few.
//
// The weights are all there is to read (2 bytes each, against 4 bytes per token and k of activations), so a launch is as
// fast as its CUs can fetch: about 50 GB/s each from HBM, 128 CUs saturate it.  A workgroup therefore owns ONE 16-row block
// (2,048 rows: 128 workgroups of 64 KiB), and its KS waves take the tiles of K round-robin, four tiles in flight each, and
// meet in LDS: no K split across workgroups, whose close costs about 5 us.  Activations are plain fp32 rows, 32 bytes per
// lane and tile (tile order would bring 16 rows where one is alive): the RMS norm in front (gain and sum of squares), the
// split into fp16 hi + lo and the element-wise work behind the product happen here, and the next launch reads rows again.
//
// TinyLlama shape, one token, us per launch, 64-row tiles of gemm.hip (K cut over workgroups) and here: wo and w_down
// together 18.2 and 15.5, gate/up 13.2 and 13.9, q/k/v 8.6 and 7.2; the pass 1,217 and 1,168.  The activations, read by every
// workgroup, weigh more with every token: a pass of 4 tokens 1,134 and 1,104, of 6 1,136 and 1,126, of 7 1,137 and 1,142, of
// 8 1,145 and 1,164.  So up to 6; passes of 6 and (tiles) 7 tokens at other widths: stories42M 303 and 352, four layers of
// Llama-2-7B 522 and 551.
// Eight rows to a workgroup instead of 16 (256 of them for wo and w_down) and six tiles in flight measured the same or
// slower: it is the start of a launch, two dependent trips to memory, that is left.  (With every trip that depends on nothing
// started at once, as in gemm_f32.hip, a pass of one token 1,055 -> 1,035.)
#include <climits>

#include "gemm_f32_tail.h"
#include "gemm_tile.h"

namespace nvllm {

// tiles in flight per wave, as many as 128 registers hold (16 waves per CU)
constexpr int thin_ring(int NT, bool norm) { return NT == 1 ? 4 : NT == 2 ? (norm ? 3 : 4) : 2; }

// What follows the complete sums of features n0 .. n0 + 3 of token x.
template <bool PAIR>
__device__ __forceinline__ void thin_finish(const F32Gemm& p, const F32Segment& sg, int x, int g, int nb, int n0, const f4_t& y, const f4_t& u, const f4_t& side, int row) {
    const int T = p.T, N = sg.N;
    if (x < T && n0 < N) f32_finish<PAIR>(p, sg, x, n0, y, u, side, row);
    if (!PAIR && p.amax_pairs != nullptr) f32_pairs(p, N, nb, n0, x, g == 0 && x < T, y);
}

// The same with the activations in LDS, where every workgroup lays them out once, in operand order: [k tile][group of 8 k][token], the hi
// plane and then the lo plane.  From memory a wave asks for 2 KiB of them beside each KiB of weights, and for 2 of gains where there is a
// norm (every lane its operand, whichever of the 16 columns is alive).  The activations are asked for first (loads return in order), the ring of
// weights behind them.  w_down of TinyLlama at one token: the products are done 5.9 us after the first workgroup's start instead of 7.8, the
// launch after 8.0 instead of 8.9; what is left is its 23 MB, 4.6 us of them, behind a start of 1.1, the slowest wave's issue and layout, and two meetings.
constexpr int thin_lds_ring(int NT) { return NT == 1 ? 8 : 6; }
template <int NT, int KS>
constexpr int thin_lds_bytes(int K, int T, bool norm) { return KS * NT * 1024 + K * T * 4 + (norm ? T * (K / 32) * 4 : 0); }
constexpr int THIN_LAP = 4;   // activations: items of four k of a token that a thread requests together
constexpr int THIN_LDS_MOST = 84 * 1024;   // what launch_thin's rule comes to: 16 waves' sums, a lap of 16,384 values and their sums of squares
template <int KS, bool PAIR, bool NORM>
__global__ __launch_bounds__(KS * 64) void k_gemm_thin_lds(F32Gemm p) {   // a block, or one of either matrix, a workgroup
    constexpr int NT = PAIR ? 2 : 1, RING = thin_lds_ring(NT), THREADS = KS * 64, LAP = THIN_LAP;
    request_arguments<sizeof(F32Gemm)>();
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_thin[];
    f4_t(*s_red)[NT][64] = reinterpret_cast<f4_t(*)[NT][64]>(lds_thin);   // [wave]
    __half* s_act = reinterpret_cast<__half*>(lds_thin + KS * NT * 1024);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = lane & 15, g = lane >> 4;
    const F32Segment& sg = p.seg[f32_segment(p, (int)blockIdx.x)];
    const int nb = (int)blockIdx.x - sg.first;
    const int K = p.K, T = p.T, Kb = K >> 5, K4 = K >> 2;
    float* s_sq = reinterpret_cast<float*>(s_act + 2 * (size_t)K * T);   // NORM: [token][32 k]
    const int tx = min(x, T - 1);   // columns past the last token compute it again and are not stored
    const int n0 = nb * 16 + 4 * g;
    const bool finishes = wave == 0, turns = !PAIR && finishes && f32_turns(sg), adds = !PAIR && finishes && sg.kind == F32Out::ADD;
    const int at = turns ? p.pos[tx] : 0;

    // activations: item i is four k of a token, LAP of a thread at a time
    const int items = T * K4;
    f4_t v[LAP], gn[NORM ? LAP : 1];
    auto place = [&](int i, int& t, int& k4) {
        t = 0;
        k4 = min(i, items - 1);
#pragma unroll
        for (int u = 1; u < THIN_TOKENS; u++)
            if (k4 >= K4) {
                k4 -= K4;
                t++;
            }
    };
    auto request = [&](int i0) {
#pragma unroll
        for (int u = 0; u < LAP; u++) {
            if (u * THREADS + i0 - (int)threadIdx.x >= items) continue;   // (uniform: nobody's)
            int t, k4;
            place(i0 + u * THREADS, t, k4);
            if (p.in_rows) {
                t = p.in_rows[t];
                asm volatile("" ::"v"(t));
            }
            v[u] = *reinterpret_cast<const f4_t*>(p.in + (size_t)t * K + 4 * k4);
            if constexpr (NORM) gn[u] = *reinterpret_cast<const f4_t*>(p.gain + 4 * k4);
        }
    };
    auto lay_out = [&](int i0) {
#pragma unroll
        for (int u = 0; u < LAP; u++) {
            const int i = i0 + u * THREADS;
            if (i >= items) continue;
            int t, k4;
            place(i, t, k4);
            f4_t a = v[u];
            if constexpr (NORM) {
                float sq = a[0] * a[0];
#pragma unroll
                for (int e = 1; e < 4; e++) sq = fmaf(a[e], a[e], sq);
                // (K4 is a multiple of eight: eight lanes side by side have a token's 32 k)
                sq += __shfl_xor(sq, 1, 64);
                sq += __shfl_xor(sq, 2, 64);
                sq += __shfl_xor(sq, 4, 64);
                if ((k4 & 7) == 0) s_sq[t * Kb + (k4 >> 3)] = sq;
                a *= gn[u];
            }
            alignas(8) _Float16 hi[4], lo[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float c = fminf(fmaxf(a[e], -65504.f), 65504.f);
                hi[e] = (_Float16)c;
                lo[e] = (_Float16)(c - (float)hi[e]);
            }
            __half* to = s_act + ((size_t)(k4 >> 1) * T + t) * 8 + 4 * (k4 & 1);
            *reinterpret_cast<uint2*>(to) = *reinterpret_cast<uint2*>(hi);
            *reinterpret_cast<uint2*>(to + (size_t)K * T) = *reinterpret_cast<uint2*>(lo);
        }
    };
    request((int)threadIdx.x);

    // weights: a step past the wave's last is requested through a descriptor of length zero: no traffic, and no branch around a request
    const int mine = wave < Kb ? (Kb - wave + KS - 1) / KS : 0;
    h8_t w[RING][NT];
    const __half* W = reinterpret_cast<const __half*>(sg.W) + (size_t)nb * sg.nb_stride;
    const __half* W2 = PAIR ? reinterpret_cast<const __half*>(sg.W2) + (size_t)nb * sg.nb_stride : nullptr;
    auto load = [&](int r, int i) {
        const int bytes = i < mine ? 0x7fffffff : 0;
        const auto from = __builtin_amdgcn_make_buffer_rsrc(const_cast<__half*>(W), 0, bytes, 0x00020000);
        const auto from2 = __builtin_amdgcn_make_buffer_rsrc(const_cast<__half*>(PAIR ? W2 : W), 0, bytes, 0x00020000);
        const unsigned step = (unsigned)(wave + i * KS) * 1024u;
        __builtin_amdgcn_sched_barrier(0);   // requests stay in the order of their use: waits count what is younger
#pragma unroll
        for (int n = 0; n < NT; n++)
            w[r][n] = __builtin_bit_cast(h8_t, __builtin_amdgcn_raw_buffer_load_b128(n == 1 ? from2 : from, lane * 16, step, /*nt*/ 2));
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int r = 0; r < RING; r++) load(r, r);
    lay_out((int)threadIdx.x);
    for (int i0 = (int)threadIdx.x + LAP * THREADS; i0 - (int)threadIdx.x < items; i0 += LAP * THREADS) {
        request(i0);
        lay_out(i0);
    }
    // what the epilogue needs beside the sums travels with the first tiles
    f4_t side = {0.f, 0.f, 0.f, 0.f};   // angles, or what is added to
    int row = -1;
    if (!PAIR && finishes) row = f32_row(p, sg, tx);
    if (turns) side = f32_angles(p, at, n0);
    else if (adds) side = f32_old(sg, tx, n0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (not for the weights in flight)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");

    const f4_t zero = {0.f, 0.f, 0.f, 0.f};
    f4_t hi[NT], lo[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) hi[n] = lo[n] = zero;
    const h8_t* acts = reinterpret_cast<const h8_t*>(s_act) + (size_t)g * T + tx;
    const int plane = K / 8 * T;
    for (int i0 = 0; i0 < mine; i0 += RING) {
#pragma unroll
        for (int r = 0; r < RING; r++) {
            if (i0 + r < mine) {
                const h8_t* a = acts + (size_t)(wave + (i0 + r) * KS) * 4 * T;
                const h8_t vh = a[0], vl = a[plane];
#pragma unroll
                for (int n = 0; n < NT; n++) {
                    hi[n] = OpF16x2::mfma(w[r][n], vh, hi[n]);
                    lo[n] = OpF16x2::mfma(w[r][n], vl, lo[n]);
                }
            }
            load(r, i0 + r + RING);
        }
    }
#pragma unroll
    for (int n = 0; n < NT; n++) s_red[wave][n][lane] = hi[n] + lo[n];
    __syncthreads();
    if (!finishes) return;
    f4_t y = s_red[0][0][lane], u = zero;
#pragma unroll
    for (int q = 1; q < KS; q++) y += s_red[q][0][lane];
    if constexpr (PAIR) {
        u = s_red[0][1][lane];
#pragma unroll
        for (int q = 1; q < KS; q++) u += s_red[q][1][lane];
    }
    if constexpr (NORM) {
        float sum = 0.f;
#pragma unroll 4
        for (int j = g; j < Kb; j += 4) sum += s_sq[tx * Kb + j];
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        const float rinv = __fdiv_rn(1.0f, sqrtf(__fadd_rn(__fdiv_rn(sum, (float)K), p.eps)));
        y *= rinv;
        if constexpr (PAIR) u *= rinv;
    }
    thin_finish<PAIR>(p, sg, x, g, nb, n0, y, u, side, row);
}

template <int NB, int KS, bool PAIR, bool NORM>
__global__ __launch_bounds__(KS * 64) void k_gemm_thin(F32Gemm p) {
    static_assert(!PAIR || NB == 1, "a pair is one block of either matrix");
    static_assert(NB <= KS, "a wave finishes a block");
    constexpr int NT = PAIR ? 2 : NB, RING = thin_ring(NT, NORM);
    request_arguments<sizeof(F32Gemm)>();
    __shared__ f4_t s_red[KS][NT][64];
    __shared__ float s_ss[KS][16];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = lane & 15, g = lane >> 4;
    const F32Segment& sg = p.seg[f32_segment(p, (int)blockIdx.x)];
    const int nb0 = ((int)blockIdx.x - sg.first) * NB;
    const int K = p.K, T = p.T, N = sg.N, blocks = (N + 15) >> 4;
    const h8_t* wp[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) {
        const float* W = PAIR && n == 1 ? sg.W2 : sg.W;
        wp[n] = reinterpret_cast<const h8_t*>(reinterpret_cast<const __half*>(W) + (size_t)(PAIR ? nb0 : min(nb0 + n, blocks - 1)) * sg.nb_stride) + lane;
    }
    const int tx = min(x, T - 1);   // columns past the last token compute it again and are not stored
    int from = tx;
    if (p.in_rows) {
        from = p.in_rows[tx];
        asm volatile("" ::"v"(from));   // (waited for here, and not where launches without these rows meet)
    }
    const float* ap = p.in + (size_t)from * K + 8 * g;
    const float* gp = NORM ? p.gain + 8 * g : nullptr;
    // what the epilogue needs beside the sums travels with the first tiles, and angles behind their positions
    const int nb = nb0 + (PAIR ? 0 : wave), n0 = nb * 16 + 4 * g;   // of the block this wave finishes
    const bool turns = !PAIR && wave < NB && f32_turns(sg), adds = !PAIR && wave < NB && sg.kind == F32Out::ADD;
    f4_t side = {0.f, 0.f, 0.f, 0.f};   // angles, or what is added to
    int row = -1;
    const int at = turns ? p.pos[tx] : 0;
    auto request_side = [&] {
        if (!PAIR && wave < NB) row = f32_row(p, sg, tx);
        if (turns) side = f32_angles(p, at, n0);
        else if (adds) side = f32_old(sg, tx, n0);
    };
    h8_t w[RING][NT];
    f4_t a[RING][2], gv[RING][NORM ? 2 : 1];
    auto load = [&](int r, int i) {
        const int kb = wave + i * KS;
        __builtin_amdgcn_sched_barrier(0);   // requests stay in the order of their use: waits count what is younger
#pragma unroll
        for (int h = 0; h < 2; h++) {
            a[r][h] = *reinterpret_cast<const f4_t*>(ap + kb * 32 + 4 * h);
            if constexpr (NORM) gv[r][h] = *reinterpret_cast<const f4_t*>(gp + kb * 32 + 4 * h);
        }
#pragma unroll
        for (int n = 0; n < NT; n++) w[r][n] = NVLLM_WLOAD(wp[n] + (size_t)kb * 64);
        __builtin_amdgcn_sched_barrier(0);
    };
    const f4_t zero = {0.f, 0.f, 0.f, 0.f};
    f4_t hi[NT], lo[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) hi[n] = lo[n] = zero;
    float ss = 0.f;
    auto multiply = [&](int r) {
        h8_t vh, vl;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            f4_t v = a[r][h];
            if constexpr (NORM) {
                float sq = v[0] * v[0];
#pragma unroll
                for (int e = 1; e < 4; e++) sq = fmaf(v[e], v[e], sq);
                ss += sq;
                v *= gv[r][h];
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float c = fminf(fmaxf(v[e], -65504.f), 65504.f);
                vh[4 * h + e] = (_Float16)c;
                vl[4 * h + e] = (_Float16)(c - (float)vh[4 * h + e]);
            }
        }
#pragma unroll
        for (int n = 0; n < NT; n++) {
            hi[n] = OpF16x2::mfma(w[r][n], vh, hi[n]);
            lo[n] = OpF16x2::mfma(w[r][n], vl, lo[n]);
        }
    };
    // (as in gemm_f32.hip: the steady loop requests without a condition)
    const int Kb = K >> 5, mine = wave < Kb ? (Kb - wave + KS - 1) / KS : 0;
    if (mine < RING) {
#pragma unroll
        for (int r = 0; r + 1 < RING; r++)
            if (r < mine) load(r, r);
        request_side();
#pragma unroll
        for (int r = 0; r + 1 < RING; r++)
            if (r < mine) multiply(r);
    } else {
#pragma unroll
        for (int r = 0; r < RING; r++) load(r, r);
        request_side();
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
#pragma unroll
    for (int n = 0; n < NT; n++) s_red[wave][n][lane] = hi[n] + lo[n];
    if constexpr (NORM) {
        ss += __shfl_xor(ss, 16, 64);
        ss += __shfl_xor(ss, 32, 64);
        if (g == 0) s_ss[wave][x] = ss;
    }
    __syncthreads();
    if (wave >= NB || nb >= blocks) return;
    f4_t y = s_red[0][PAIR ? 0 : wave][lane], u = zero;
#pragma unroll
    for (int v = 1; v < KS; v++) y += s_red[v][PAIR ? 0 : wave][lane];
    if constexpr (PAIR) {
        u = s_red[0][1][lane];
#pragma unroll
        for (int v = 1; v < KS; v++) u += s_red[v][1][lane];
    }
    if constexpr (NORM) {
        float sum = 0.f;
#pragma unroll
        for (int v = 0; v < KS; v++) sum += s_ss[v][x];
        const float rinv = __fdiv_rn(1.0f, sqrtf(__fadd_rn(__fdiv_rn(sum, (float)K), p.eps)));
        y *= rinv;
        if constexpr (PAIR) u *= rinv;
    }
    thin_finish<PAIR>(p, sg, x, g, nb, n0, y, u, side, row);
}

template <int NB, int KS, bool PAIR, bool NORM>
static void launch_thin(const F32Gemm& a, int tiles) {
    if constexpr (NB == 1) {
        constexpr int NT = PAIR ? 2 : 1;
        const int lds = thin_lds_bytes<NT, KS>(a.K, a.T, NORM), Kb = a.K / 32;
        // One or two tokens, and enough steps a wave to make up for the way over LDS.  With 8 waves (more workgroups than CUs) eight, as long as
        // two workgroups share a CU; with 16 the more the fuller the chip, whose rate is the bound then, and activations in one lap (a
        // second one returns behind the weights in flight).  us a launch as lanes read them and this way, one and two tokens:
        //   8 waves, q/k/v        K 2,560 12.9 -> 10.9, 13.2 -> 11.3; 4,096 25.5 -> 21.7, 25.6 -> 22.5; 5,120 39.5 -> 28.1, 39.8 -> 29.3
        //   8 waves, gate/up      K 2,048 13.9 -> 13.6, 14.0 -> 14.0; 3,584 28.9 -> 27.0, 29.0 -> 28.4; 4,096 (688 workgroups) 34.0 -> 33.8, 33.8 -> 34.2,
        //                         (512) 24.9 -> 26.4 both, (352) 22.8 -> 21.4, 22.7 -> 22.4; 5,120 52.2 -> 47.5, 52.1 -> 49.6
        //   8 waves, wo, w_down   K 5,120 14.8 -> 12.7, 14.8 -> 13.2; 13,824 35.5 -> 28.4, 35.6 -> 37.5 (118 KB)
        //   16 waves, steps       64 workgroups, 16: 12.0 -> 9.4, 12.2 -> 10.4; 128, 8: 5.6 -> 5.6 (K 4,096: 7.5 -> 7.1, 7.5 -> 7.4), 9: 8.2 -> 8.5, 8.2 -> 8.8,
        //                         10: 9.1 -> 8.3, 9.2 -> 8.7, 11: 9.9 -> 8.9, 10.0 -> 9.3; 192, 10: 9.4 -> 9.6, 9.3 -> 9.9, 16: 12.6 -> 11.9, 12.7 -> 12.6;
        //                         224, 19: 15.7 -> 14.4, 15.8 -> 15.3; 256, 8: 8.2 -> 9.4, 8.2 -> 9.5, 16: 13.7 -> 13.9, 13.8 -> 14.3, 21: 17.7 -> 17.2, 17.8 -> 18.1
        // Three tokens are more to lay out than lanes read twice (TinyLlama, all of its long projections: 1,063 -> 1,076 a pass), and the classifier's four
        // blocks already share one reading (K 4,096 45.4 -> 47.1, 46.3 -> 47.8; 2,048 25.5 -> 25.3, 27.7 -> 27.4).
        const bool pays = KS == 8 ? Kb >= 8 * KS && lds <= 80 * 1024 : Kb >= KS * (2 + tiles / 16) && (long)a.T * a.K <= 4L * THIN_LAP * KS * 64;
        if (a.T <= 2 && pays) {
            static bool enabled = false;
            if (!enabled) {
                HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_thin_lds<KS, PAIR, NORM>), hipFuncAttributeMaxDynamicSharedMemorySize, THIN_LDS_MOST));
                enabled = true;
            }
            NVLLM_LAUNCH((k_gemm_thin_lds<KS, PAIR, NORM>), dim3(tiles), dim3(KS * 64), lds, a);
            return;
        }
    }
    NVLLM_LAUNCH((k_gemm_thin<NB, KS, PAIR, NORM>), dim3(tiles), dim3(KS * 64), 0, a);
}

void launch_gemm_thin(const F32Gemm& g, int prof_cls) {
    if (g.T <= 0 || g.n_segs == 0) return;
    if (g.T > THIN_TOKENS || g.K % 32) NVLLM_FATAL("thin projection: %d tokens of %d values", g.T, g.K);
    F32Gemm a = g;
    const bool pair = a.seg[0].W2 != nullptr;
    double weights = 0, outs = 0;
    int blocks = 0;
    for (int s = 0; s < a.n_segs; s++) {
        F32Segment& q = a.seg[s];
        if (pair != (q.W2 != nullptr)) NVLLM_FATAL("thin projection: pairs and single matrices in one launch");
        q.vec = q.N % 4 == 0 && q.ldo % 4 == 0 && (reinterpret_cast<size_t>(q.out) & 15) == 0;
        weights += (double)q.N * a.K * (pair ? 2 : 1);
        outs += q.N;
        blocks += cdiv(q.N, 16);
    }
    // One block per workgroup, and as many waves as keep a CU's fetch path busy: 16 where a CU has one workgroup, 8 where
    // it has two.  Thousands of blocks (the classifier): four to a workgroup, which then reads the activations once for all.
    const int cus = rt().num_cus, NB = !pair && blocks > 4 * cus ? 4 : 1;
    int tiles = 0;
    for (int s = 0; s < a.n_segs; s++) {
        a.seg[s].first = tiles;
        tiles += cdiv(cdiv(a.seg[s].N, 16), NB);
    }
    for (int s = a.n_segs; s < F32_SEGMENTS; s++) a.seg[s].first = INT_MAX;
    ProfScope ps(prof_cls, 2.0 * weights + 4.0 * a.T * (a.K + outs), 2.0 * a.T * weights);
#define NVLLM_GEMM_THIN(nb, ks, pair_)                                                                             \
    do {                                                                                                         \
        if (a.gain) launch_thin<nb, ks, pair_, true>(a, tiles);                                                 \
        else launch_thin<nb, ks, pair_, false>(a, tiles);                                                       \
    } while (0)
    if (NB == 4) NVLLM_GEMM_THIN(4, 8, false);
    else if (pair) NVLLM_GEMM_THIN(1, 8, true);
    else if (tiles <= cus) NVLLM_GEMM_THIN(1, 16, false);
    else NVLLM_GEMM_THIN(1, 8, false);
#undef NVLLM_GEMM_THIN
}

}  // namespace nvllm
