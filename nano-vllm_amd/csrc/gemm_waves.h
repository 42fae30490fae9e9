// gemm_waves.h -- projections of hundreds of tokens whose tiles fit the chip in one round: out[T, N] = act[T, K] x W[N, K]^T,
// K dealt to the waves.
//
// A workgroup of four waves owns 128 features x 16 TBN tokens and every wave multiplies ALL of it, over K-steps wave,
// wave + 4, ...: operands go from global memory straight into the registers that feed the matrix cores (both are stored
// in operand order), nothing is shared through LDS and no barrier stands in the loop.  A byte still enters the CU once,
// because no two waves want the same one.  One wave per SIMD has 512 registers: up to 224 hold the sums, the rest two to
// four K-steps, 144 to 216 KiB per CU, of which 80 to 144 are on their way while a step is multiplied.  The waves' sums meet in LDS once, at the end; wave w finishes row
// blocks 2 w and 2 w + 1 of the tile.
//
// What bounds it: the bytes into a CU, (8 + PL TBN) KiB a step (PL activation planes).  2,048 features x 5,632 k at 1,029
// tokens in bf16, 208 tiles of 80 tokens: 75 GB/s into each CU, 38 us a launch where the LDS tiles of
// gemm_prefill_tile.h (272 of 64 tokens: sixteen CUs with two, one workgroup's 36 KiB in flight on the others) take 48; with
// weights that already lie in L2 34, without the products 37.  More steps in flight, loads spread evenly between the
// products, padded strides and other cache policies measured the same or worse.
#pragma once

#include "gemm_prefill_tile.h"
#include "moe_ride.h"

namespace nvllm {

namespace {

constexpr int WAVES_FB = 8;   // 16-row blocks of W per tile
// K-steps in flight per wave: what 512 registers hold beside the sums
constexpr int waves_ring(int planes, int TBN) {
    return planes == 1 ? (TBN <= 3 ? 4 : 3) : (TBN <= 2 ? 4 : TBN <= 5 ? 3 : 2);
}

// A router beside the gated pairs, its sorting beside plain rows (moe_ride.h).  Not the router beside seven blocks: they fill the
// registers, and the compiler waits in their loop for loads of the other branch.
constexpr bool waves_carry_route(int TBN, int EPI, int planes) {
    return planes == 1 && (EPI == GemmEpilogue::F32 || (EPI == GemmEpilogue::SWIGLU_A16 && TBN <= 6));
}

template <int TBN, int EPI, typename KVT, typename OP>
__global__ __launch_bounds__(256, 1) void k_gemm_waves(GemmArgs p, int tiles_n, int tiles_t) {
    request_arguments<sizeof(GemmArgs)>();
    constexpr int FB = WAVES_FB, PL = OP::PLANES, NA = PL * TBN, RING = waves_ring(PL, TBN);
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_waves[];
    float* s_rinv = reinterpret_cast<float*>(lds_waves);
    f4_t* s_red = reinterpret_cast<f4_t*>(lds_waves + 1024);   // [receiving wave][giving wave][TBN][64]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if constexpr (EPI == GemmEpilogue::LATENT_Q) {
        if ((int)blockIdx.x >= p.ride_from) {
            ride_along(p, 4, wave, lane);
            return;
        }
    }
    if constexpr (waves_carry_route(TBN, EPI, PL)) {
        if ((int)blockIdx.x >= p.ride_from) {
            if constexpr (EPI == GemmEpilogue::SWIGLU_A16) router_ride<4>(p, wave, lane, lds_waves);
            else route_sort<false, 256>(p.route.plan, nullptr, 0, reinterpret_cast<int*>(lds_waves));
            return;
        }
    }
    // every XCD a contiguous range of tiles, token tiles fastest: what runs together behind one L2 shares weights
    const int total = tiles_n * tiles_t;
    int id;
    {
        const int xcd = (int)blockIdx.x & 7, slot = (int)blockIdx.x >> 3, q = total >> 3, r = total & 7;
        id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + slot;
    }
    const int nb0 = id / tiles_t * FB, tb0 = id % tiles_t * TBN;
    const __half* W = p.W + (size_t)nb0 * p.nb_stride;
    const __half* A = p.A + (size_t)tb0 * p.Kb * PL * TILE_HALVES;
    unsigned of_w[FB], of_a[TBN];   // bytes to a block's first tile (blocks past the last: the last again, not stored)
#pragma unroll
    for (int f = 0; f < FB; f++) of_w[f] = (unsigned)min(f, p.NB - 1 - nb0) * (unsigned)(p.nb_stride * sizeof(__half));
#pragma unroll
    for (int j = 0; j < TBN; j++) of_a[j] = (unsigned)min(j, p.Tb - 1 - tb0) * (unsigned)(p.Kb * PL * 1024);

    const int mine = wave < p.Kb ? (p.Kb - wave + 3) >> 2 : 0;   // this wave's steps
    unsigned at_w = wave * 1024 + lane * 16, at_a = wave * (PL * 1024) + lane * 16;
    h8_t w[RING][FB], a[RING][NA];
    // A step past the last is requested through a descriptor of length zero: no traffic, and no branch in the loop.
    auto operand = [](const __half* base, bool live) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<__half*>(base), 0, live ? 0x7fffffff : 0, 0x00020000);
    };
    auto load = [](__amdgpu_buffer_rsrc_t from, unsigned lane_at, unsigned block_at) {
        return __builtin_bit_cast(h8_t, __builtin_amdgcn_raw_buffer_load_b128(from, lane_at, block_at, 0));
    };
    auto next_step = [&]() {
        at_w += 4096;
        at_a += 4096 * PL;
    };
    f4_t acc[FB][TBN];
#pragma unroll
    for (int f = 0; f < FB; f++)
#pragma unroll
        for (int j = 0; j < TBN; j++) acc[f][j] = f4_t{0.f, 0.f, 0.f, 0.f};
    // (in front of the first steps, which would be waited for with it; added up while they travel: q/k/v of Simivik at 1,029 tokens 23.5 -> 22.4 us)
    // Hyper-connection updates follow products of activations that nothing scales: those tiles keep no registers for it (six blocks 16 spilled
    // registers with them, 8 without).
    constexpr bool SCALED = hyper_streams(EPI) == 0;
    TileRinv<16 * TBN, 256> rinv;
    if (SCALED && p.e.ss_in != nullptr) rinv.request(p, tb0);
#pragma unroll
    for (int r = 0; r < RING; r++) {
        const auto rw = operand(W, r < mine), ra = operand(A, r < mine);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int f = 0; f < FB; f++) w[r][f] = load(rw, at_w, of_w[f]);
#pragma unroll
        for (int q = 0; q < NA; q++) a[r][q] = load(ra, at_a + (q % PL) * 1024, of_a[q / PL]);
        __builtin_amdgcn_sched_barrier(0);
        next_step();
    }
    if (SCALED && p.e.ss_in != nullptr) rinv.finish(p, s_rinv);

    // Step i out of registers r, each replaced by step i + RING's as soon as it has been multiplied.  The loop has one exit and
    // no condition around a request: where paths with and without requests meet, the compiler waits for all of them.
    int i = 0;
    auto step = [&](auto slot, auto reload) {
        constexpr int r = decltype(slot)::value;
        constexpr bool RELOAD = decltype(reload)::value;
        const auto rw = operand(W, i + r + RING < mine), ra = operand(A, i + r + RING < mine);
#pragma unroll
        for (int q = 0; q < NA; q++) {
#pragma unroll
            for (int f = 0; f < FB; f++) {
                acc[f][q / PL] = OP::mfma(w[r][f], a[r][q], acc[f][q / PL]);
                if (RELOAD && q == NA - 1) w[r][f] = load(rw, at_w, of_w[f]);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (RELOAD) a[r][q] = load(ra, at_a + (q % PL) * 1024, of_a[q / PL]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (RELOAD) next_step();
    };
    using yes = std::true_type;
    using no = std::false_type;
    for (; i + RING <= mine; i += RING) {
        step(std::integral_constant<int, 0>{}, yes{});
        step(std::integral_constant<int, 1>{}, yes{});
        if constexpr (RING > 2) step(std::integral_constant<int, 2>{}, yes{});
        if constexpr (RING > 3) step(std::integral_constant<int, 3>{}, yes{});
    }
    if (i < mine) step(std::integral_constant<int, 0>{}, no{});
    if constexpr (RING > 2)
        if (i + 1 < mine) step(std::integral_constant<int, 1>{}, no{});
    if constexpr (RING > 3)
        if (i + 2 < mine) step(std::integral_constant<int, 2>{}, no{});

    // what the residual epilogues add to travels while the sums meet (all of it: the steps' registers are free)
    PfResidual<2, TBN, EPI, TBN> residual;
    if constexpr (epi_is_residual(EPI)) residual.begin(p, nb0 + 2 * wave, tb0, lane);
    // the waves' sums meet: first the even row block of each wave's two, then the odd one
    f4_t sum[2][TBN];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        if (h) __syncthreads();   // the even blocks have been read
#pragma unroll
        for (int v = 0; v < 4; v++)
#pragma unroll
            for (int j = 0; j < TBN; j++) s_red[((v * 4 + wave) * TBN + j) * 64 + lane] = acc[2 * v + h][j];
        __syncthreads();          // (1/rms is visible too)
#pragma unroll
        for (int j = 0; j < TBN; j++) {
            f4_t z[4];
#pragma unroll
            for (int u = 0; u < 4; u++) z[u] = s_red[((wave * 4 + u) * TBN + j) * 64 + lane];
            sum[h][j] = (z[0] + z[1]) + (z[2] + z[3]);
        }
    }
    if constexpr (epi_is_residual(EPI)) residual.finish(p, sum, nb0 + 2 * wave, 0, tb0, s_rinv, lane, p.NB);
    else pf_epilogue<2, TBN, EPI, KVT, OP>(p, sum, nb0 + 2 * wave, 0, tb0, s_rinv, lane, p.NB);
}

template <int TBN, int EPI, typename KVT, typename OP>
bool launch_waves(GemmArgs a, int tiles_n, int tiles_t) {   // whether a.route rode
    constexpr int NEED = 1024 + 16 * TBN * 1024, LDS = EPI == GemmEpilogue::SWIGLU_A16 && waves_carry_route(TBN, EPI, OP::PLANES) ? std::max(NEED, ROUTER_RIDE_LDS) : NEED;
    static_assert(LDS <= 160 * 1024, "the waves' sums must fit the CU's LDS");
    if (hyper_streams(EPI) && a.e.ss_in) NVLLM_FATAL("hyper-connection updates take activations that are not scaled by token");
    static bool enabled = false;
    if (!enabled) {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_waves<TBN, EPI, KVT, OP>), hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
        enabled = true;
    }
    a.ride_from = tiles_n * tiles_t;
    const int route = waves_carry_route(TBN, EPI, OP::PLANES) ? route_groups(a, a.ride_from) : 0;
    static_assert((3 * 1024 + 1) * 4 <= NEED);   // (the sorting)
    NVLLM_LAUNCH((k_gemm_waves<TBN, EPI, KVT, OP>), dim3(a.ride_from + rider_groups(a, a.ride_from, 4) + route), dim3(256), route > 0 ? LDS : NEED, a, tiles_n, tiles_t);
    return route > 0;
}

// Seven blocks of two planes leave registers for two steps in flight, and lose: prompts of TinyLlama-1.1B, 1,547 tokens, w_down in such
// tiles 7,890 us a pass, in those of gemm_wide.h 7,790 (six blocks at 1,500 tokens 6,710 and 7,100).
constexpr int waves_tallest(int planes) { return planes == 1 ? 7 : 6; }
template <int EPI, typename KVT, typename OP>
bool launch_waves_height(const GemmArgs& a, int tbn) {
    const int tiles_n = cdiv(a.NB, WAVES_FB), tiles_t = cdiv(a.Tb, tbn);
    switch (tbn) {
        case 1: return launch_waves<1, EPI, KVT, OP>(a, tiles_n, tiles_t);
        case 2: return launch_waves<2, EPI, KVT, OP>(a, tiles_n, tiles_t);
        case 3: return launch_waves<3, EPI, KVT, OP>(a, tiles_n, tiles_t);
        case 4: return launch_waves<4, EPI, KVT, OP>(a, tiles_n, tiles_t);
        case 5: return launch_waves<5, EPI, KVT, OP>(a, tiles_n, tiles_t);
        case 6: return launch_waves<6, EPI, KVT, OP>(a, tiles_n, tiles_t);
        default:
            if constexpr (waves_tallest(OP::PLANES) == 7) return launch_waves<7, EPI, KVT, OP>(a, tiles_n, tiles_t);
            return false;
    }
}

// The lowest height whose tiles are one round of the chip; 0: none is.  (A second round costs as much as the first, a lower
// tile than needed only bytes.)
inline int waves_height(const GemmArgs& a, int tallest) {
    static const int env = getenv("NVLLM_GEMM_WAVES") ? atoi(getenv("NVLLM_GEMM_WAVES")) : -1;   // 0: never; token blocks: always that height
    if (env >= 0 || wide_env() > 0) return wide_env() > 0 ? 0 : std::min(env, tallest);
    const int tiles_n = cdiv(a.NB, WAVES_FB), room = rt().num_cus / tiles_n;   // token tiles that fit beside each other
    const int tbn = room ? cdiv(a.Tb, room) : tallest + 1;
    return tbn <= tallest ? tbn : 0;
}

}  // namespace

}  // namespace nvllm
