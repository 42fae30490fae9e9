// gemm_wide.h -- projections of hundreds of tokens in tiles of 256 features: out[T, N] = act[T, K] x W[N, K]^T.
//
// What bounds a dense tile here is not the matrix cores but the bytes that feed them: about 45 bytes a cycle into a CU
// from L2, 128 out of its LDS.  A workgroup of four waves owns 256 features x 16 TBN tokens; wave w has features
// 64 w .. 64 w + 63 and ALL the tokens, so a K-step of 32 costs
//     (16 + PL TBN) KiB into the CU and 4 (4 + PL TBN) KiB out of LDS per 64 PL TBN matrix-core cycles
// (PL activation planes), e.g. fp16 hi + lo at 96 tokens 28 KiB and 64 KiB per 768 cycles, where the tiles of 128 x 96 in
// gemm_prefill_tile.h (2 x 2 waves) take 40 and 112 for the same products.  One wave per SIMD then has the register file to
// itself: accumulators for up to nine token blocks with hi + lo planes of
// activations (ten with one bf16 plane), and operands that are replaced as they are used, so that the LDS reads
// of step s + 1 and the copies of step s + RING - 1 are issued between the products of step s.  Copies go global -> LDS
// directly (one 1-KiB tile per wave instruction, both operands are stored in operand order) through a ring of RING stages
// with counted waits; one barrier a step publishes step s + 1 and frees the buffer of step s - 1, whose operands are in
// registers by then.  TinyLlama-1.1B's gate/up of 1,548 tokens: 175 us in the smaller tiles, 140 here (512 TFLOP/s of
// products, twice that in the matrix cores: hi + lo; large library products of this type reach 1,096).
//
// The epilogues are those of gemm_prefill_tile.h.
#pragma once

#include <climits>

#include "gemm_prefill_tile.h"
#include "moe_ride.h"

namespace nvllm {

namespace {

// WT: 1, four waves with all the tokens; 2, eight waves, two groups of four with half the tokens each
template <int TBN, int PL, int WT>
struct WideGeom {
    static constexpr int FB = 16;                          // 16-row blocks of W per tile, four per wave
    static constexpr int TILES = FB + PL * TBN;            // 1-KiB tiles per stage
    static constexpr int WAVES = 4 * WT;
    static constexpr int CPW = (TILES + WAVES - 1) / WAVES;   // copies per wave and stage (the last tile is copied by several waves when there are fewer)
    static constexpr int RING = TILES <= 22 ? 7 : TILES <= 24 ? 6 : TILES <= 30 ? 5 : TILES <= 39 ? 4 : 3;
    static constexpr int RINV_BYTES = 1024;                // 1/rms of up to 256 tokens in front of the ring
    static constexpr int LDS = RINV_BYTES + RING * TILES * 1024;
    static_assert(LDS <= 160 * 1024, "the ring must fit the CU's LDS");
};

// One 1-KiB tile global -> LDS: lane l's 16 bytes at (wave-uniform) `src` + `offset` land at LDS byte `dst` + `buf` + 16 l.
__device__ __forceinline__ void wide_copy(const __half* src, unsigned offset, unsigned dst, unsigned buf) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(offset), "s"(src), "s"(dst), "s"(buf) : "memory", "scc");
}
template <int N>
__device__ __forceinline__ void wide_wait() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// EXP: rows sorted by expert, every tile's of one (ExpertRows)
template <int TBN, int WT, int EPI, typename KVT, typename OP, bool EXP = false>
__global__ __launch_bounds__(256 * WT, 1) void k_gemm_wide(GemmArgs p, int tiles_n, int tiles_t, int panel) {
    request_arguments<sizeof(GemmArgs)>();
    constexpr int PL = OP::PLANES;
    using G = WideGeom<TBN, PL, WT>;
    constexpr int RING = G::RING, CPW = G::CPW, WAVES = G::WAVES, TBW = TBN / WT;   // TBW: token blocks of a wave
    static_assert(TBN % WT == 0);
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_wide[];
    float* s_rinv = reinterpret_cast<float*>(lds_wide);
    const h8_t* ring = reinterpret_cast<const h8_t*>(lds_wide + G::RINV_BYTES);

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wf = wave & 3, wt = wave >> 2;   // this wave's features and tokens inside the tile
    if constexpr (EPI == GemmEpilogue::LATENT_Q) {
        if ((int)blockIdx.x >= p.ride_from) {
            ride_along(p, WAVES, wave, lane);
            return;
        }
    }
    if constexpr (EPI == GemmEpilogue::SWIGLU_A16 && PL == 1 && !EXP) {
        if ((int)blockIdx.x >= p.ride_from) {
            router_ride<WAVES>(p, wave, lane, lds_wide);
            return;
        }
    }
    // every XCD a contiguous range of tiles, panel after panel: what runs together behind one L2 shares weights and activations
    const int total = tiles_n * tiles_t;
    int id;
    {
        const int xcd = (int)blockIdx.x & 7, slot = (int)blockIdx.x >> 3, q = total >> 3, r = total & 7;
        id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + slot;
    }
    // a panel: `panel` feature tiles, whose token tiles follow each other, of each all its features
    const int first = id / (panel * tiles_t) * panel, width = min(panel, tiles_n - first), at = id - first * tiles_t;
    const int nb0 = (first + at % width) * G::FB, tb0 = at / width * TBN;
    const __half* W = p.W;
    if constexpr (EXP) {
        const int e = __builtin_amdgcn_readfirstlane(p.block_expert[tb0]);
        if (e < 0) return;   // fewer rows than the launch has room for
        W += (size_t)e * p.expert_stride;
    }
    // wave w copies tiles w, w + WAVES, ...: weight blocks, then the planes of each token block (past the last: the last again, the
    // same bytes to the same place, so that no branch parts the loop)
    const __half* src[CPW];
    unsigned dst[CPW];
#pragma unroll
    for (int u = 0; u < CPW; u++) {
        const int q = min(wave + WAVES * u, G::TILES - 1);
        dst[u] = (unsigned)(size_t)(lds_void*)lds_wide + G::RINV_BYTES + q * 1024;
        src[u] = q < G::FB ? W + (size_t)min(nb0 + q, p.NB - 1) * p.nb_stride
                           : p.A + ((size_t)min(tb0 + (q - G::FB) / PL, p.Tb - 1) * p.Kb * PL + (q - G::FB) % PL) * TILE_HALVES;
    }
    unsigned at_w = lane * 16, at_a = lane * 16;   // bytes from a source's start: its k-tile, this lane's piece
    auto copy = [&](int u, unsigned buf) {   // (whether a copy brings weights or activations depends on u alone: FB is a multiple of WAVES)
        wide_copy(src[u], WAVES * u < G::FB ? at_w : at_a, dst[u], buf);
    };
    auto copied = [&]() {   // a stage's copies are out
        at_w += 1024;
        at_a += PL * 1024;
    };
    auto wait_but = [&](auto stages) { wide_wait<decltype(stages)::value * CPW>(); };   // at most that many stages of this wave's copies still fly

    const int n = p.Kb;   // stages; n > RING (the launcher's rule)
#pragma unroll
    for (int s = 0; s + 1 < RING; s++) {
#pragma unroll
        for (int u = 0; u < CPW; u++) copy(u, s * G::TILES * 1024);
        copied();
    }
    if (p.e.ss_in != nullptr) tile_rinv<16 * TBN, 64 * WAVES>(p, tb0, s_rinv);

    f4_t acc[4][TBW];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < TBW; j++) acc[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};
    h8_t wa[4], wb[4], af[PL * TBW];   // weights of this stage and the next, in turn; activations: a block's are replaced as soon as it is done
    const h8_t* mine = ring + (size_t)wf * 4 * 64 + lane;
    const h8_t* acts = ring + (size_t)(G::FB + wt * PL * TBW) * 64 + lane;
    int rb = 0;   // buffer of stage s
    // The products of a stage; between them the reads of the next one's operands and, with COPY, the copies of stage
    // s + RING - 1 into the buffer of stage s - 1.
    auto phase = [&](h8_t (&wf)[4], h8_t (&wn)[4], auto with_copy, auto with_read) {
        constexpr bool COPY = decltype(with_copy)::value, READ = decltype(with_read)::value;
        constexpr int GROUP = 4 * PL;                 // products of a token block
        const int nx = rb + 1 == RING ? 0 : rb + 1, behind = rb == 0 ? RING - 1 : rb - 1;
        const h8_t *next_w = mine + nx * G::TILES * 64, *next_a = acts + nx * G::TILES * 64;
        const unsigned to = __builtin_amdgcn_readfirstlane(behind * G::TILES * 1024);
        // A wave issues an instruction every four cycles and a product takes sixteen: up to three others fit behind one, and
        // more of them in a row leave the matrix cores idle.  So one read or one copy behind a product, in places of their own.
#pragma unroll
        for (int j = 0; j < TBW; j++) {
#pragma unroll
            for (int m = 0; m < GROUP; m++) {
                const int i = m & 3, pl = m >> 2;
                acc[i][j] = OP::mfma(wf[i], af[PL * j + pl], acc[i][j]);
                if (READ && i == 3) af[PL * j + pl] = next_a[(PL * j + pl) * 64];
                if (READ && m == 1 && j < 4) wn[j] = next_w[j * 64];
                if (COPY && m == GROUP - 2 && j < CPW) copy(j, to);
                if (COPY && m == 0 && TBW + j < CPW) copy(TBW + j, to);
                if (COPY && m == 2 && PL == 2 && 2 * TBW + j < CPW) copy(2 * TBW + j, to);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        static_assert(CPW <= (PL == 2 ? 3 : 2) * TBW && TBW >= 4, "a place for every copy and every read");
        if (COPY) copied();
        rb = nx;
    };
    // Everybody's copies of the stage to be read have landed; everybody holds the operands of stage s - 1, whose buffer is free.
    auto meet = [&]() {
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    wait_but(std::integral_constant<int, RING - 2>{});
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the 1/rms written above)
    meet();
#pragma unroll
    for (int f = 0; f < 4; f++) wa[f] = mine[f * 64];
#pragma unroll
    for (int f = 0; f < PL * TBW; f++) af[f] = acts[f * 64];
    int s = 0;
    using yes = std::true_type;
    using no = std::false_type;
    auto next = [&](auto in_flight) {
        wait_but(in_flight);
        meet();
    };
    // stages s + 1 .. s + RING - 2 fly at the wait, of which the first has to have landed; two stages a turn
    for (; s + RING < n; s += 2) {
        next(std::integral_constant<int, RING - 3>{});
        phase(wa, wb, yes{}, yes{});
        next(std::integral_constant<int, RING - 3>{});
        phase(wb, wa, yes{}, yes{});
    }
    if (s + RING - 1 < n) {
        next(std::integral_constant<int, RING - 3>{});
        phase(wa, wb, yes{}, yes{});
        s++;
#pragma unroll
        for (int i = 0; i < 4; i++) wa[i] = wb[i];
    }
    wait_but(std::integral_constant<int, 0>{});   // the last stages: nothing more to copy
    for (; s + 1 < n; s++) {
        meet();
        phase(wa, wb, no{}, yes{});
#pragma unroll
        for (int i = 0; i < 4; i++) wa[i] = wb[i];
    }
    phase(wa, wb, no{}, no{});

    pf_epilogue<4, TBW, EPI, KVT, OP>(p, acc, nb0 + wf * 4, wt * TBW, tb0, s_rinv, lane, p.NB);
}

// Feature tiles of a panel: those with which the tiles that an XCD works on at a time, a contiguous range of its CUs' number, bring the
// fewest bytes into its L2 (`w` KiB a feature tile and step, `a` a token tile).  One, which is token tiles fastest, has all activations enter every
// L2: TinyLlama-1.1B's w_down and wo, 200 tiles of 64 tokens, 55.7 us on average, in panels of three (which this picks) 53.2, of four 52.9; its gate/up 125.5 and 124.1; with one plane of
// activations no difference.
inline int wide_panel(int tiles_n, int tiles_t, int w, int a) {
    const int range = std::min(cdiv(tiles_n * tiles_t, 8), rt().num_cus / 8);
    int best = 1;
    long least = LONG_MAX;
    for (int panel = 1; panel <= std::min(tiles_n, range); panel++) {
        const int tokens = std::min(tiles_t, cdiv(range, panel));
        const long bytes = (long)cdiv(range, tokens) * w + (long)tokens * a;
        if (bytes < least) least = bytes, best = panel;
    }
    return best;
}

template <int TBN, int EPI, typename KVT, typename OP, int WT = 1, bool EXP = false>
bool launch_wide(GemmArgs a, int tiles_n, int tiles_t) {   // whether a.route rode
    using G = WideGeom<TBN, OP::PLANES, WT>;
    constexpr bool CARRIES = EPI == GemmEpilogue::SWIGLU_A16 && OP::PLANES == 1 && !EXP;   // a router (moe_ride.h)
    static bool enabled = false;
    if (!enabled) {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_wide<TBN, WT, EPI, KVT, OP, EXP>), hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS));
        enabled = true;
    }
    a.ride_from = tiles_n * tiles_t;
    const int route = CARRIES ? route_groups(a, a.ride_from) : 0;
    static_assert(!CARRIES || ROUTER_RIDE_LDS <= G::LDS);
    NVLLM_LAUNCH((k_gemm_wide<TBN, WT, EPI, KVT, OP, EXP>), dim3(a.ride_from + rider_groups(a, a.ride_from, G::WAVES) + route), dim3(64 * G::WAVES), G::LDS, a, tiles_n, tiles_t,
                 OP::PLANES == 1 ? 1 : wide_panel(tiles_n, tiles_t, G::FB, OP::PLANES * TBN));
    return route > 0;
}

// Microseconds a launch takes in tiles of TBN token blocks: rounds of one workgroup per CU, each a start and an end beside its
// Kb steps.  Fitted to fp16 launches of 64 and 176 steps on a full chip (a round of 4, 6 and 9 blocks: 36, 45 and 60 us; 92,
// 120 and 140 us).
inline double wide_us(int tiles, int Kb, int TBN, int PL, int cus) {
    return (double)cdiv(tiles, cus) * (5.0 + 0.8 * TBN + Kb * (0.23 + 0.027 * PL * TBN));
}

}  // namespace

}  // namespace nvllm
