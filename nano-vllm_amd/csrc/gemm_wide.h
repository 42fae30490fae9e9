// gemm_wide.h -- projections of hundreds of tokens in tiles of 256 features: out[T, N] = act[T, K] x W[N, K]^T.
//
// What bounds a dense tile here is not the matrix cores but the bytes that feed them: about 45 bytes a cycle into a CU
// from L2, 128 out of its LDS.  A workgroup of four waves owns 256 features x 16 TBN tokens; wave w has features
// 64 w .. 64 w + 63 and ALL the tokens, so a K-step of 32 costs
//     (16 + PL TBN) KiB into the CU and 4 (4 + PL TBN) KiB out of LDS per 64 PL TBN matrix-core cycles
// (PL activation planes), e.g. fp16 hi + lo at 96 tokens 28 KiB and 64 KiB per 768 cycles, where the tiles of 128 x 96 in
// gemm_prefill_tile.h (2 x 2 waves) take 40 and 112 for the same products.  One wave per SIMD then has the register file to
// itself: accumulators for up to nine token blocks, and operands that are replaced as they are used, so that the LDS reads
// of step s + 1 and the copies of step s + RING - 1 are issued between the products of step s.  Copies go global -> LDS
// directly (one 1-KiB tile per wave instruction, both operands are stored in operand order) through a ring of RING stages
// with counted waits; one barrier a step publishes step s + 1 and frees the buffer of step s - 1, whose operands are in
// registers by then.  TinyLlama-1.1B's gate/up of 1,548 tokens: 175 us in the smaller tiles, 140 here (512 TFLOP/s of
// products, twice that in the matrix cores: hi + lo; large library products of this type reach 1,096).
//
// The epilogues are those of gemm_prefill_tile.h; the residual rows they add to are requested a token block ahead.
#pragma once

#include "gemm_prefill_tile.h"

namespace nvllm {

namespace {

template <int TBN, int PL>
struct WideGeom {
    static constexpr int FB = 16;                          // 16-row blocks of W per tile, four per wave
    static constexpr int TILES = FB + PL * TBN;            // 1-KiB tiles per stage
    static constexpr int CPW = (TILES + 3) / 4;            // copies per wave and stage (the last tile is copied by several waves when there are fewer)
    static constexpr int RING = TILES <= 24 ? 6 : TILES <= 30 ? 5 : 4;
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

// RESID_*, HYPER_*: the operands of token block j + 1 travel while block j is finished.
template <int TBN, int EPI>
__device__ __forceinline__ void wide_residual(const GemmArgs& p, const f4_t (&v)[4][TBN], int nb_first, int tb0, const float* s_rinv, int lane, int nb_lim) {
    const GemmEpilogue& ep = p.e;
    constexpr int HS = hyper_streams(EPI);
    const int n_of = nb_first * 16 + 4 * (lane >> 4);
    float4 xo[2][HS ? 1 : 4], gain[HS ? 1 : 4];
    HyperIn<HS ? HS : 1> hyper[2][HS ? 4 : 1];
    auto load = [&](int set, int j) {
        const int t = min((tb0 + j) * 16 + (lane & 15), p.T - 1);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int n = min(n_of + 16 * i, p.N - 4);
            if constexpr (HS > 0) hyper_load_4<HS>(hyper[set][i], ep, p.N, t, n);
            else xo[set][i] = *reinterpret_cast<const float4*>(ep.x + (size_t)t * p.N + n);
        }
    };
    if constexpr (HS == 0)
#pragma unroll
        for (int i = 0; i < 4; i++) gain[i] = *reinterpret_cast<const float4*>(ep.gain_next + min(n_of + 16 * i, p.N - 4));
    load(0, 0);
#pragma unroll
    for (int j = 0; j < TBN; j++) {
        if (j + 1 < TBN) load((j + 1) & 1, j + 1);
        const int tl = j * 16 + (lane & 15), t = tb0 * 16 + tl;
        const bool tok_live = t < p.T && tb0 + j < p.Tb;
        const float rinv = ep.ss_in ? s_rinv[tl] : 1.0f;
        float ssq[2] = {0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int n = n_of + 16 * i;
            const bool live = tok_live && nb_first + i < nb_lim;
            const float y[4] = {v[i][j][0] * rinv, v[i][j][1] * rinv, v[i][j][2] * rinv, v[i][j][3] * rinv};
            if (!live) continue;
            if constexpr (HS > 0) {
                hyper_update_4<HS>(hyper[j & 1][i], ep, p.N, t, n, y);
            } else if constexpr (EPI == GemmEpilogue::RESID_B16) {
                ssq[i >> 1] += resid_b16_4(ep, p.N, t, n, xo[j & 1][i], gain[i], y);
            } else {
                const float4 x = xo[j & 1][i], g = gain[i];
                // residual add as the reference's accum(): x = x + branch (layers.c:163-168)
                const float xn[4] = {__fadd_rn(x.x, y[0]), __fadd_rn(x.y, y[1]), __fadd_rn(x.z, y[2]), __fadd_rn(x.w, y[3])};
                *reinterpret_cast<float4*>(ep.x + (size_t)t * p.N + n) = make_float4(xn[0], xn[1], xn[2], xn[3]);
                const float z[4] = {xn[0] * g.x, xn[1] * g.y, xn[2] * g.z, xn[3] * g.w};
                store_a16_4(ep.a16_out, ep.Kb_out, t, n, z);
                ssq[i >> 1] += xn[0] * xn[0] + xn[1] * xn[1] + xn[2] * xn[2] + xn[3] * xn[3];
            }
        }
        if constexpr (epi_has_ss(EPI)) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                float sq = ssq[h];
                sq += __shfl_xor(sq, 16, 64);
                sq += __shfl_xor(sq, 32, 64);
                const int col = (nb_first + 2 * h) >> 1;
                if (lane < 16 && tok_live && col < (p.N + 31) >> 5) ep.ss_out[(size_t)t * ((p.N + 31) >> 5) + col] = sq;
            }
        }
    }
}

template <int TBN, int EPI, typename KVT, typename OP, bool EXP>
__global__ __launch_bounds__(256, 1) void k_gemm_wide(GemmArgs p, int tiles_n, int tiles_t) {
    constexpr int PL = OP::PLANES;
    using G = WideGeom<TBN, PL>;
    constexpr int RING = G::RING, CPW = G::CPW;
    if constexpr (EPI == GemmEpilogue::LATENT_Q) {
        if ((int)blockIdx.x >= p.ride_from) {
            latent_kv_ride(p.ride, ((int)blockIdx.x - p.ride_from) * 4 + (int)(threadIdx.x >> 6), threadIdx.x & 63);
            return;
        }
    }
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_wide[];
    float* s_rinv = reinterpret_cast<float*>(lds_wide);
    const h8_t* ring = reinterpret_cast<const h8_t*>(lds_wide + G::RINV_BYTES);

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // every XCD a contiguous range of tiles, token tiles fastest: what runs together behind one L2 shares weights
    const int total = tiles_n * tiles_t;
    int id;
    {
        const int xcd = (int)blockIdx.x & 7, slot = (int)blockIdx.x >> 3, q = total >> 3, r = total & 7;
        id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + slot;
    }
    const int nb0 = id / tiles_t * G::FB, tb0 = id % tiles_t * TBN;
    const __half* W = p.W;
    if constexpr (EXP) {
        const int e = __builtin_amdgcn_readfirstlane(p.block_expert[tb0]);
        if (e < 0) return;   // fewer rows than the launch has room for
        W += (size_t)e * p.expert_stride;
    }
    // wave w copies tiles w, w + 4, ...: weight blocks, then the planes of each token block (past the last: the last again, the
    // same bytes to the same place, so that no branch parts the loop)
    const __half* src[CPW];
    unsigned dst[CPW];
#pragma unroll
    for (int u = 0; u < CPW; u++) {
        const int q = min(wave + 4 * u, G::TILES - 1);
        dst[u] = (unsigned)(size_t)(lds_void*)lds_wide + G::RINV_BYTES + q * 1024;
        src[u] = q < G::FB ? W + (size_t)min(nb0 + q, p.NB - 1) * p.nb_stride
                           : p.A + ((size_t)min(tb0 + (q - G::FB) / PL, p.Tb - 1) * p.Kb * PL + (q - G::FB) % PL) * TILE_HALVES;
    }
    unsigned at_w = lane * 16, at_a = lane * 16;   // bytes from a source's start: its k-tile, this lane's piece
    auto copy = [&](int u, unsigned buf) {   // (whether a copy brings weights or activations depends on u alone: FB is a multiple of 4)
        wide_copy(src[u], 4 * u < G::FB ? at_w : at_a, dst[u], buf);
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
    // 1/rms of the tile's tokens from the producer's sums of squares, while the first stages travel: PARTS neighbouring
    // threads per token, every load of a thread requested at once (one after the other they cost 5 us)
    if (p.e.ss_in != nullptr) {
        constexpr int PARTS = TBN <= 4 ? 4 : TBN <= 8 ? 2 : 1;
        const int tl = (int)threadIdx.x / PARTS, part = (int)threadIdx.x % PARTS;
        const int t = min(tb0 * 16 + tl, p.T - 1), cols = p.e.ss_tiles;
        const float* sp = p.e.ss_in + (size_t)(p.e.ss_gather ? p.e.ss_gather[t] : t) * cols;
        float ss = 0.f;
        if ((cols & 3) == 0) {
            for (int j0 = 4 * part; j0 < cols; j0 += 64 * PARTS) {
                f4_t v[16];
#pragma unroll
                for (int j = 0; j < 16; j++) v[j] = *reinterpret_cast<const f4_t*>(sp + min(j0 + 4 * PARTS * j, cols - 4));
#pragma unroll
                for (int j = 0; j < 16; j++)
                    if (j0 + 4 * PARTS * j < cols) ss += (v[j][0] + v[j][1]) + (v[j][2] + v[j][3]);
            }
        } else {
            for (int j = part; j < cols; j += PARTS) ss += sp[j];
        }
#pragma unroll
        for (int o = 1; o < PARTS; o <<= 1) ss += __shfl_xor(ss, o, 64);
        if (part == 0 && tl < TBN * 16) s_rinv[tl] = __fdiv_rn(1.0f, sqrtf(__fadd_rn(__fdiv_rn(ss, (float)p.e.d_in), p.e.eps)));
    }

    f4_t acc[4][TBN];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < TBN; j++) acc[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};
    h8_t wa[4], wb[4], af[PL * TBN];   // weights of this stage and the next, in turn; activations: a block's are replaced as soon as it is done
    const h8_t* mine = ring + (size_t)wave * 4 * 64 + lane;
    const h8_t* acts = ring + (size_t)G::FB * 64 + lane;
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
        for (int j = 0; j < TBN; j++) {
#pragma unroll
            for (int m = 0; m < GROUP; m++) {
                const int i = m & 3, pl = m >> 2;
                acc[i][j] = OP::mfma(wf[i], af[PL * j + pl], acc[i][j]);
                if (READ && i == 3) af[PL * j + pl] = next_a[(PL * j + pl) * 64];
                if (READ && m == 1 && j < 4) wn[j] = next_w[j * 64];
                if (COPY && m == GROUP - 2 && j < CPW) copy(j, to);
                if (COPY && m == 0 && TBN + j < CPW) copy(TBN + j, to);
                if (COPY && m == 2 && PL == 2 && 2 * TBN + j < CPW) copy(2 * TBN + j, to);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        static_assert(CPW <= (PL == 2 ? 3 : 2) * TBN && TBN >= 4, "a place for every copy and every read");
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
    for (int f = 0; f < PL * TBN; f++) af[f] = acts[f * 64];
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

    const int nb_first = nb0 + wave * 4;
    if constexpr (EPI == GemmEpilogue::RESID_A16 || EPI == GemmEpilogue::RESID_B16 || hyper_streams(EPI) > 0)
        wide_residual<TBN, EPI>(p, acc, nb_first, tb0, s_rinv, lane, p.NB);
    else
        pf_epilogue<4, TBN, EPI, KVT, OP>(p, acc, nb_first, 0, tb0, s_rinv, lane, p.NB);
}

template <int TBN, int EPI, typename KVT, typename OP, bool EXP = false>
void launch_wide(const GemmArgs& a, int tiles_n, int tiles_t) {
    using G = WideGeom<TBN, OP::PLANES>;
    static bool enabled = false;
    if (!enabled) {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_wide<TBN, EPI, KVT, OP, EXP>), hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS));
        enabled = true;
    }
    const int riders = EPI == GemmEpilogue::LATENT_Q && a.ride.base ? cdiv(a.ride.T, 4) : 0;
    NVLLM_LAUNCH((k_gemm_wide<TBN, EPI, KVT, OP, EXP>), dim3(tiles_n * tiles_t + riders), dim3(256), G::LDS, a, tiles_n, tiles_t);
}

inline int wide_env() {   // NVLLM_GEMM_WIDE: 0 = never these tiles, a number of token blocks = always that height
    static const int v = getenv("NVLLM_GEMM_WIDE") ? atoi(getenv("NVLLM_GEMM_WIDE")) : -1;
    return v;
}
// Microseconds a launch takes in tiles of TBN token blocks: rounds of one workgroup per CU, each a start and an end beside its
// Kb steps.  Fitted to fp16 launches of 64 and 176 steps on a full chip (a round of 4, 6 and 9 blocks: 36, 45 and 60 us; 92,
// 120 and 140 us).
inline double wide_us(int tiles, int Kb, int TBN, int PL, int cus) {
    return (double)cdiv(tiles, cus) * (5.0 + 0.8 * TBN + Kb * (0.23 + 0.027 * PL * TBN));
}

}  // namespace

}  // namespace nvllm
