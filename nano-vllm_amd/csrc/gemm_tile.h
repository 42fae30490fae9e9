// gemm_tile.h -- one output tile of a decode-sized projection as a device function: what a
// workgroup of the projection kernel does (gemm.hip describes the decomposition and the
// epilogues).  Two callers:
//   k_gemm           one launch per projection; operands written by earlier launches (COH = false)
//   k_decode_chain   every projection and attention of a decode step in ONE launch; a tile's
//                    activations were written by other workgroups of the same launch (COH = true)
//
// COH = true changes how bytes that another workgroup of the SAME launch wrote or will read move:
// every such store is write-through (sc1) and every such load bypasses this CU's vector cache
// (sc1), so that the caller can hand tiles over with a drained counter add on the producer and a
// relaxed poll on the consumer, without cache write-backs or invalidates.  Weights, gains, RoPE
// angles and the integer arrays of the step are read-only during the launch and stay on plain loads.
#pragma once

#include <algorithm>

#include "gemm_common.h"

namespace nvllm {

// Weight tiles are read once per launch: non-temporal loads (a build knob for A/B runs)
#ifdef NVLLM_W_PLAIN
#define NVLLM_WLOAD(p) (*(p))
#else
#define NVLLM_WLOAD(p) __builtin_nontemporal_load(p)
#endif

constexpr int AUX_SC1 = 16;   // cache-policy bits of the raw buffer builtins on gfx950: bit 4 = sc1

typedef unsigned int u2_t __attribute__((ext_vector_type(2)));

// position of a tile in its projection's grid (what blockIdx / gridDim are to k_gemm)
struct TileIdx {
    int x, y, z;   // feature tile, K slice, token group
    int gx;        // feature tiles per token group (grid width, padding included)
};

// K-steps of weights and of activations in flight per wave.  Loads return in the order of their requests, so weights are in flight no
// further ahead than the activations asked for behind them, and a CU takes no more in for more requests: what is in flight beyond the trip's
// length queues.  Most rings are of one length; four steps of weights and two of activations hold fewer registers, which is faster where
// 64 features meet 32 tokens or the steps are few.  us a launch at the widths of TinyLlama and of the 1.2B designs, 64 rows unless said, with
// a wait for everything in flight in every step (weights 4, activations 2) | weights 4, activations 2 | 3 of both | 4 of both | others:
//   features x tokens                two planes                                   one plane
//   32 x 16  wo                      7.6 | 7.5 | 7.6 | - | 6: 7.7, 8: 7.9         7.1 | 7.4 | 7.2 | - | 6: 6.7, 8: 6.7
//            wo of stories42M, 32    5.2 | 4.9 | 5.2 | - | 6: 5.1, 8: 5.1
//   32 x 32  q/k/v                   10.3 | 9.6 | 9.8 | 9.8                       13.7 | 13.1 | 12.8 | 12.6
//   64 x 16  w_down, 9 rows          8.9 | 8.4 | 8.2 | 8.4                        experts' gate/up 43.3 | 40.8 | 40.6 | 39.4
//            classifier, 9 rows      44.2 | 44.8 | 43.0 | 44.5                     44.9 | 44.2 | 43.4 | 44.1
//            classifier, one row                                                  27.8 | 29.5 | 27.7 | 28.3 (experts' w_down 17.9 | 19.3 | 17.1 | 17.1)
//   64 x 32  w_down (RESID)          12.6 | 12.5 | 12.9 | 12.9                    11.7 | 11.5 | 12.2 | 12.0
//            w_down (HYPER)                                                       12.1 | 12.4 | 12.4 | 12.0
//            gate/up 32 rows, shared expert's w_down (F32)
//                                    15.7 | 14.5 | 14.9 | 14.7 | 2: 14.5          12.3 | 13.7 | 13.2 | 13.2 | 2: 11.9
//   96 x 32  gate/up                 17.2 | 16.8 | 16.9 | 16.3                    15.4 | 15.2 | 15.5 | 15.3
//   64 x 64  classifier              177 | 176 | 175 | spills | 2: 174            175 | 175 | 173 | - | 2: 173
//            gate/up                 9.7 | 10.1 | 9.9 | spills | 2: 9.3           14.4 | 12.9 | 12.7 | - | 2: 13.4
//            products by head (K 64)                                              4.8 | 5.1 | 5.4 | - | 2: 5.3
// (Two runs of one build differ by 0.1 to 0.3.  The products by head take 5.3 with the old wait too, behind the launch of 32 x 32 tiles that
// ends 0.5 sooner now.)
// Tiles of 64 x 64 whose epilogue adds to rows: a loop that waits for everything in flight in every step, and holds nothing over it for the
// epilogue (w_down of TinyLlama, 160 and 200 tokens 22.5 and 23.2 us against 23.2 and 24.0 without those waits, of Suselorn-1.2B, 101 tokens 14.7 against 15.1).
constexpr bool gemm_step_waits(int TB, int epi) { return TB == 4 && (epi == GemmEpilogue::RESID_A16 || hyper_streams(epi) > 0); }
constexpr int gemm_ring(int NBW, int TB, int planes, int epi, bool groups = false) {
    if (NBW == 2) return TB == 1 && planes == 1 ? 8 : 4;
    if (NBW == 4 && TB == 2) return epi == GemmEpilogue::F32 || epi == GemmEpilogue::SWIGLU_A16 ? 2 : 4;
    if (TB == 4) return gemm_step_waits(TB, epi) || groups ? 4 : planes == 2 ? 2 : 3;
    return NBW == 4 && TB == 1 && epi == GemmEpilogue::F32 ? 3 : 4;   // (a classifier of up to 16 rows: two workgroups share a CU)
}
constexpr int gemm_ring_act(int NBW, int TB, int planes, int epi, bool groups = false) {
    const int ring = gemm_ring(NBW, TB, planes, epi, groups);
    const bool narrow = NBW == 2 && TB == 1 && planes == 2, wide = NBW == 4 && TB == 2 && hyper_streams(epi) == 0, tall = TB == 4 && ring == 4;
    return narrow || wide || tall ? 2 : ring;
}

// bytes of dynamic LDS a tile needs: the waves' partial tiles, then four small arrays
template <int NBW, int TB, int NW>
constexpr int gemm_tile_lds() {
    return NW * NBW * TB * 64 * 16 + (TB * 16 + NW * 64 + 2 * TB * 16) * 4 + 16;
}

// Bytes of LDS a launch of F32 takes when its rows go to the host: with two workgroups per CU all tiles of a 32,000-word classifier
// are resident and done at once, and PCIe would idle until then; one per CU, and the first half's rows cross beside the second's
// products (64 rows of TinyLlama: the pass 6 us shorter than with a copy behind it, and 20 like this).  Up to 16 rows the weights take as long as PCIe: left alone.
constexpr int GEMM_LDS_ALONE = 84 * 1024;
template <int NBW, int TB, int NW>
inline int gemm_tile_lds(const GemmEpilogue& e) {
    constexpr int need = gemm_tile_lds<NBW, TB, NW>();
    return TB > 1 && e.out_host && need < GEMM_LDS_ALONE ? GEMM_LDS_ALONE : need;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t gemm_rsrc(const void* base, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

// 4 consecutive k of token t into hi/lo tiles with write-through stores (n % 4 == 0), 16 bytes per
// lane: the lane that holds k..k+3 and the lane 16 further on, which holds k+4..k+7 of the same
// token, are both active here; the first gets both hi halves and stores the hi plane's 16-byte
// chunk, the second both lo halves and stores the lo plane's (narrow write-through stores each cost
// a transaction of their own on the way to memory).  `rs` covers the whole a16 buffer.
__device__ __forceinline__ void store_a16_4_sc1(__amdgpu_buffer_rsrc_t rs, int Kb_out, int t, int n, const float* y, int lane) {
    alignas(8) __half hi[4], lo[4];
    split16_4(y, hi, lo);
    const u2_t H = *reinterpret_cast<const u2_t*>(hi), L = *reinterpret_cast<const u2_t*>(lo);
    const bool first = (lane & 16) == 0;          // k % 8 == 0
    const u2_t send = first ? L : H;
    u2_t recv;
    recv[0] = (unsigned)__shfl_xor((int)send[0], 16, 64);
    recv[1] = (unsigned)__shfl_xor((int)send[1], 16, 64);
    const u4_t out = first ? u4_t{H[0], H[1], recv[0], recv[1]} : u4_t{recv[0], recv[1], L[0], L[1]};
    const int k8 = n & ~7;
    const int tile = ((t >> 4) * Kb_out + (k8 >> 5)) * 2 + (first ? 0 : 1);
    const int off = ((t & 15) + 16 * ((k8 >> 3) & 3)) * 8;
    __builtin_amdgcn_raw_buffer_store_b128(out, rs, (tile * TILE_HALVES + off) * 2, 0, AUX_SC1);
}

template <typename KVT>
__device__ __forceinline__ void kv_put4_sc1(KVT* dst, const float* y);
template <>
__device__ __forceinline__ void kv_put4_sc1<float>(float* dst, const float* y) {
    alignas(8) float a[2] = {y[0], y[1]}, b[2] = {y[2], y[3]};
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(dst), *reinterpret_cast<unsigned long long*>(a),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(dst + 2), *reinterpret_cast<unsigned long long*>(b),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <>
__device__ __forceinline__ void kv_put4_sc1<__half>(__half* dst, const float* y) {
    alignas(8) __half h[4] = {kv_sat_half(y[0]), kv_sat_half(y[1]), kv_sat_half(y[2]), kv_sat_half(y[3])};
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(dst), *reinterpret_cast<unsigned long long*>(h),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename KVT>
__device__ __forceinline__ void kv_put4_strided_sc1(KVT* dst, const float* y);
template <>
__device__ __forceinline__ void kv_put4_strided_sc1<float>(float*, const float*) {}
template <>
__device__ __forceinline__ void kv_put4_strided_sc1<__half>(__half* dst, const float* y) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const __half h = kv_sat_half(y[e]);
        __hip_atomic_store(reinterpret_cast<unsigned short*>(dst + 4 * e), *reinterpret_cast<const unsigned short*>(&h),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// The first RW K-steps of a wave's weight stream: they depend on nothing the step computes, so a
// caller that knows its next tile may issue them long before that tile's activations exist.
// Must be followed by gemm_tile<..., PRE = true> with the same arguments.
// `tid` = threadIdx.x (a caller that runs many tiles in a loop passes it through an opaque copy, so that
// the compiler does not hoist every tile's per-lane index arithmetic out of that loop and keep it in registers).
// part / nparts: only the ring entries s with s * nparts / RW == part (a caller that spreads the
// requests over several places calls once per part); part < 0: all of them.
template <int NBW, int NW, int RW>
__device__ __forceinline__ void gemm_tile_prefetch(const GemmArgs& p, const TileIdx ix, h8_t (&w)[RW][NBW], const int tid, const bool on = true,
                                                   const int part = -1, const int nparts = 1) {
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb0 = ix.x * NBW;
    const int kb_begin = ix.y * p.kb_per_split;
    const int kb_end = min(p.Kb, kb_begin + p.kb_per_split);
    const int first = kb_begin + wave;
    // `on` = the workgroup has a tile at all; every ring entry is written either way (zeros where there
    // is nothing to load), so that no entry carries a value over from an earlier use of the registers
    const int nsteps = on && nb0 < p.NB && first < kb_end ? (kb_end - first + NW - 1) / NW : 0;
    const h8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < RW; s++) {
        if (part >= 0 && (s * nparts) / RW != part) continue;
        if (s < nsteps) {
            const int kb = first + NW * s;
#pragma unroll
            for (int i = 0; i < NBW; i++)
                w[s][i] = NVLLM_WLOAD(reinterpret_cast<const h8_t*>(p.W + (size_t)min(nb0 + i, p.NB - 1) * p.nb_stride) + lane +
                                      (size_t)kb * 64);
        } else {
#pragma unroll
            for (int i = 0; i < NBW; i++) w[s][i] = zero;
        }
    }
}

// One tile.  Returns true when this workgroup wrote the tile's results (false: grid padding, or a
// K slice that was not the last to arrive).  `slot_free(r)` is called exactly once for every r in
// [0, RW), as soon as the wave will not load ring entry r again for this tile -- inside the K loop,
// spread over its last RW steps: the place to start loads for later work, a few at a time.
// PRE: 0 = the tile requests its first RW K-steps of weights itself; 1 = the caller has (gemm_tile_prefetch);
// 2 = the caller says at run time (`prefetched`, uniform over the workgroup).
// OP: operand format (gemm_common.h); GRP: a block-diagonal product, whose tiles never cross a group; EXP: rows sorted by expert.
template <int NBW, int TB, int NW, int RW, int RA, int EPI, typename KVT, bool COH, int PRE, typename OP = OpF16x2, bool GRP = false, bool EXP = false, typename Hook>
__device__ __forceinline__ bool gemm_tile(const GemmArgs& p, const TileIdx ix, unsigned char* lds_dyn, h8_t (&w)[RW][NBW],
                                          Hook&& slot_free, const int tid, const bool prefetched = true) {
    static_assert(NBW % 2 == 0, "row blocks are reduced in pairs");
    static_assert(RW % RA == 0, "the activation ring must divide the weight ring");
    constexpr int ROUNDS = NBW / 2;    // LDS reduction rounds, two row blocks each
    constexpr int ITEMS = 2 * TB * 64; // float4 results per round
    constexpr int WITEMS = ROUNDS * ITEMS;                        // float4 results of the tile: item w = round * ITEMS + e
    constexpr int FPT = (WITEMS + NW * 64 - 1) / (NW * 64);     // items per thread: thread tid takes w = tid + s * NW*64
    constexpr int ITEMS_SHIFT = TB == 1 ? 7 : (TB == 2 ? 8 : 9);
    static_assert((1 << ITEMS_SHIFT) == ITEMS, "2, 4 or 8 row-block x token-block pairs of 64 lanes per round");
    constexpr int PARTS = (NW * 64) / (TB * 16);
    // the waves' partial tiles, all row blocks at once: red[wave][row block][token block][lane]
    typedef f4_t RedTile[NBW][TB][64];
    RedTile* red = reinterpret_cast<RedTile*>(lds_dyn);
    float* s_rinv = reinterpret_cast<float*>(lds_dyn + NW * NBW * TB * 64 * 16);   // [TB * 16]
    float (*s_part)[TB * 16 + 1] = reinterpret_cast<float (*)[TB * 16 + 1]>(s_rinv + TB * 16);   // [PARTS], rows of another bank each
    static_assert(PARTS <= 2 * TB * 16, "the rows' pads fit what lies behind");
    unsigned* s_ticket = reinterpret_cast<unsigned*>(s_rinv + TB * 16 + NW * 64 + 2 * TB * 16);

    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = GRP ? ix.x / p.group_tiles : 0;
    const int nb0 = GRP ? grp * p.group_nb + (ix.x - grp * p.group_tiles) * NBW : ix.x * NBW;
    const int nb_lim = GRP ? min(p.NB, (grp + 1) * p.group_nb) : p.NB;   // row blocks this tile may touch
    if (nb0 >= nb_lim) {   // grid padded for XCD alignment
#pragma unroll
        for (int r = 0; r < RW; r++) slot_free(r);
        return false;
    }
#ifdef NVLLM_STAMPS
    unsigned long long* const stamps_wg = p.stamps ? p.stamps + (size_t)((ix.z * p.ksplit + ix.y) * ix.gx + ix.x) * 8 : nullptr;
#endif
    NVLLM_TSTAMP(0, lane);
    const int kb_begin = ix.y * p.kb_per_split;
    const int kb_end = min(p.Kb, kb_begin + p.kb_per_split);
    const int tb0 = ix.z * TB;
    const __half* W = p.W;
    if constexpr (EXP) {
        const int e = __builtin_amdgcn_readfirstlane(p.block_expert[tb0]);
        if (e < 0) {   // fewer rows than the launch has room for
#pragma unroll
            for (int r = 0; r < RW; r++) slot_free(r);
            return false;
        }
        W += (size_t)e * p.expert_stride;
    }
    const int first = kb_begin + wave;
    const int nsteps = first < kb_end ? (kb_end - first + NW - 1) / NW : 0;
    const h8_t* wp[NBW];
#pragma unroll
    for (int i = 0; i < NBW; i++)
        wp[i] = reinterpret_cast<const h8_t*>(W + (size_t)min(nb0 + i, nb_lim - 1) * p.nb_stride) + lane;
    // activations: pointers (plain loads), or byte offsets into a buffer descriptor (sc1 loads)
    const h8_t* ap[TB];
    int aoff[TB];
    __amdgpu_buffer_rsrc_t rs_a = gemm_rsrc(p.A, (unsigned)p.Tb * (unsigned)p.Kb * 2048u);
#pragma unroll
    for (int j = 0; j < TB; j++) {
        ap[j] = reinterpret_cast<const h8_t*>(p.A + ((size_t)min(tb0 + j, p.Tb - 1) * (GRP ? p.act_Kb : p.Kb) + (GRP ? grp * p.Kb : 0)) * OP::PLANES * TILE_HALVES) + lane;
        if constexpr (EXP) {
            if (p.source) {   // every lane gathers its own row
                const int r = p.source[(tb0 + j) * 16 + (lane & 15)];
                ap[j] = reinterpret_cast<const h8_t*>(p.A + (size_t)(r >> 4) * p.Kb * TILE_HALVES) + (r & 15) + 16 * (lane >> 4);
            }
        }
        aoff[j] = min(tb0 + j, p.Tb - 1) * p.Kb * 2048 + lane * 16;
    }
    static_assert(!COH || (OP::PLANES == 2 && !GRP), "the one-launch step runs fp16 models");
    auto load_act = [&](int j, int kb, h8_t& hi, h8_t& lo) {
        if constexpr (OP::PLANES == 1) {
            hi = ap[j][(size_t)kb * 64];
        } else if constexpr (COH) {
            hi = __builtin_bit_cast(h8_t, __builtin_amdgcn_raw_buffer_load_b128(rs_a, aoff[j], kb * 2048, AUX_SC1));
            lo = __builtin_bit_cast(h8_t, __builtin_amdgcn_raw_buffer_load_b128(rs_a, aoff[j] + 1024, kb * 2048, AUX_SC1));
        } else {
            hi = ap[j][(size_t)kb * 128];
#ifdef NVLLM_ABLATE_LO   // diagnostic builds only: what the second activation plane costs (results are then fp16-activation results)
            lo = hi;
#else
            lo = ap[j][(size_t)kb * 128 + 64];
#endif
        }
    };

    f4_t acc[NBW][TB];
#pragma unroll
    for (int i = 0; i < NBW; i++)
#pragma unroll
        for (int j = 0; j < TB; j++) acc[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};

    h8_t ah[RA][TB], al[RA][TB];
    auto kb_of = [&](int s) { return first + NW * s; };
    auto load_w = [&](int r, int s) {
#pragma unroll
        for (int i = 0; i < NBW; i++) w[r][i] = NVLLM_WLOAD(wp[i] + (size_t)kb_of(s) * 64);
    };
    auto load_a = [&](int r, int s) {
#pragma unroll
        for (int j = 0; j < TB; j++) load_act(j, kb_of(s), ah[r][j], al[r][j]);
    };
    // requests stay in the order of their use: waits count what is younger
    auto load = [&](int r, int s) {   // step s into entry r of rings of the same length
        __builtin_amdgcn_sched_barrier(0);
        load_w(r, s);
        load_a(r % RA, s);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](int r) {
#pragma unroll
        for (int i = 0; i < NBW; i++)
#pragma unroll
            for (int j = 0; j < TB; j++) {
                acc[i][j] = OP::mfma(w[r][i], ah[r % RA][j], acc[i][j]);
#ifndef NVLLM_ABLATE_LO
                if constexpr (OP::PLANES == 2) acc[i][j] = OP::mfma(w[r][i], al[r % RA][j], acc[i][j]);
#endif
            }
    };

    const GemmEpilogue& ep = p.e;
    constexpr bool STEP_WAITS = COH || gemm_step_waits(TB, EPI);
    // 1/rms of this token group comes from the producer's per-tile sums of squares: every thread sums a slice of one token's tiles; the slices
    // meet in LDS before the epilogue.  Up to SS_HELD of them are requested behind the first steps and held in registers over the K loop.  (Summed in
    // front of it, each load waited for all before it: two to sixteen trips to memory before the first product.)  The one-launch step, whose
    // registers hold the next tile's weights, sums them beside the first steps.
    constexpr int SS_HELD = PARTS < 64 ? 64 / PARTS : 1;
    float ss_held[SS_HELD];
    const float* ss_row = nullptr;
    const int ss_tl = tid / PARTS, ss_part = tid % PARTS;   // (lanes side by side read one token's sums: a line, and not one line each)
    // What the epilogue needs beside the sums: requested behind the first steps and waited for behind the last.  With STEP_WAITS requested behind the
    // last: held over the loop they made the one-launch step spill (64 tokens: 230 registers -> 256 and 58 more in scratch)
    float4 pf_x[FPT], pf_g[FPT];
    int pf_pos = 0, pf_row = -1;
    f4_t pf_turn[FPT];
    __amdgpu_buffer_rsrc_t rs_x = gemm_rsrc(ep.x, (unsigned)p.T * (unsigned)p.N * 4u);
    auto request_positions = [&] {
        if (EPI == GemmEpilogue::ROPE_KV) {   // all items of a thread belong to one token (NW*64 is a multiple of TB*64)
            const int e = min(tid, WITEMS - 1) & (ITEMS - 1);
            const int t = min(tb0 * 16 + ((e >> 6) % TB) * 16 + (e & 15), p.T - 1);
            pf_pos = ep.pos[t];
            pf_row = ep.kv_row[t];
        }
    };
    auto request_operands = [&] {
#pragma unroll
        for (int s = 0; s < FPT; s++) {
            const int w_ = min(tid + s * NW * 64, WITEMS - 1);
            const int h = w_ >> ITEMS_SHIFT, e = w_ & (ITEMS - 1);
            const int l = e & 63, j = (e >> 6) % TB, i = (e >> 6) / TB;
            const int n0 = (nb0 + 2 * h + i) * 16 + 4 * (l >> 4);
            if (EPI == GemmEpilogue::RESID_A16 || EPI == GemmEpilogue::RESID_B16) {
                const int t = min(tb0 * 16 + j * 16 + (l & 15), p.T - 1), n = min(n0, p.N - 4);
                if constexpr (COH)
                    pf_x[s] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rs_x, (t * p.N + n) * 4, 0, AUX_SC1));
                else
                    pf_x[s] = *reinterpret_cast<const float4*>(ep.x + (size_t)t * p.N + n);
                pf_g[s] = *reinterpret_cast<const float4*>(ep.gain_next + n);
            }
            // (q and k begin at multiples of hd; values have an angle that nobody uses)
            if (EPI == GemmEpilogue::ROPE_KV) pf_turn[s] = *reinterpret_cast<const f4_t*>(ep.rope + (size_t)pf_pos * (ep.hd >> 1) + ((n0 % ep.hd) >> 1));
        }
    };
    if constexpr (!COH) request_positions();
    auto request_side = [&] {
        if (ep.ss_in != nullptr) {
            const int t = min(tb0 * 16 + ss_tl, p.T - 1);
            int src = t;
            if (ep.ss_gather) {
                src = ep.ss_gather[t];
                asm volatile("" ::"v"(src));
            }
            ss_row = ep.ss_in + (size_t)src * ep.ss_tiles;
            if constexpr (COH) {
                float ss = 0.f;
                for (int j = ss_part; j < ep.ss_tiles; j += PARTS)
                    ss += __builtin_bit_cast(float, __hip_atomic_load(reinterpret_cast<const unsigned*>(ss_row + j), __ATOMIC_RELAXED,
                                                                      __HIP_MEMORY_SCOPE_AGENT));
                s_part[ss_part][ss_tl] = ss;
            } else {
#pragma unroll
                for (int q = 0; q < SS_HELD; q++) ss_held[q] = ss_row[min(ss_part + q * PARTS, ep.ss_tiles - 1)];
            }
        }
        if constexpr (!STEP_WAITS) request_operands();
    };

    // Loads are issued only for steps that exist: a clamped re-load of the last tile would be real HBM traffic, since streamed
    // weights are loaded non-temporally and do not stay in L2.
    if constexpr (STEP_WAITS) {
        // (requests under conditions, each waited for with all before it: with the loop below the one-launch step needs 26 to 56 registers more)
        if (PRE == 0 || (PRE == 2 && !prefetched)) {
#pragma unroll
            for (int s = 0; s < RW; s++)
                if (s < nsteps) load_w(s, s);
        }
#pragma unroll
        for (int s = 0; s < RA; s++)
            if (s < nsteps) load_a(s, s);
        request_side();
        NVLLM_TSTAMP(1, lane);
        for (int s0 = 0; s0 < nsteps; s0 += RW) {
#pragma unroll
            for (int r = 0; r < RW; r++) {
                const int s = s0 + r;
                if (s < nsteps) {
                    multiply(r);
                    if (s == 0) NVLLM_TSTAMP(2, acc[NBW - 1][TB - 1][0]);
                    if (s + RW < nsteps) load_w(r, s + RW);
                    else slot_free(r);
                    if (s + RA < nsteps) load_a(r % RA, s + RA);
                }
            }
        }
#pragma unroll
        for (int r = 0; r < RW; r++)
            if (r >= nsteps) slot_free(r);   // entries a short K slice never used
    } else if (nsteps < RW) {
        static_assert(PRE == 0);
#pragma unroll
        for (int s = 0; s + 1 < RW; s++)
            if (s < nsteps) {
                load_w(s, s);
                if (s < RA) load_a(s, s);
            }
        request_side();
        NVLLM_TSTAMP(1, lane);
#pragma unroll
        for (int s = 0; s + 1 < RW; s++)
            if (s < nsteps) {
                multiply(s);
                if (s == 0) NVLLM_TSTAMP(2, acc[NBW - 1][TB - 1][0]);
                if (s + RA < nsteps) load_a(s % RA, s + RA);
                slot_free(s);
            }
#pragma unroll
        for (int r = 0; r < RW; r++)
            if (r >= nsteps) slot_free(r);
    } else {
        // The steady loop requests without a condition: where paths with and without requests meet, the compiler waits for all of them.
        if constexpr (RA == RW) {
#pragma unroll
            for (int r = 0; r < RW; r++) load(r, r);
        } else {
#pragma unroll
            for (int r = 0; r < RW; r++) load_w(r, r);
#pragma unroll
            for (int r = 0; r < RA; r++) load_a(r, r);
        }
        request_side();
        NVLLM_TSTAMP(1, lane);
        int i0 = 0;
        for (; i0 + 2 * RW <= nsteps; i0 += RW) {
#pragma unroll
            for (int r = 0; r < RW; r++) {
                multiply(r);
                if (i0 + r == 0) NVLLM_TSTAMP(2, acc[NBW - 1][TB - 1][0]);
                if constexpr (RA == RW) {
                    load(r, i0 + r + RW);
                } else {
                    load_w(r, i0 + r + RW);
                    load_a(r % RA, i0 + r + RA);
                }
            }
        }
#pragma unroll
        for (int r = 0; r < RW; r++) {
            multiply(r);
            if (i0 + r + RW < nsteps) load_w(r, i0 + r + RW);
            else slot_free(r);
            if (i0 + r + RA < nsteps) load_a(r % RA, i0 + r + RA);
        }
#pragma unroll
        for (int r = 0; r < RW; r++)
            if (i0 + RW + r < nsteps) {
                multiply(r);
                if (i0 + RW + r + RA < nsteps) load_a(r % RA, i0 + RW + r + RA);
                slot_free(r);
            }
    }
    NVLLM_TSTAMP(3, acc[NBW - 1][TB - 1][0]);
    if constexpr (COH) request_positions();
    if constexpr (STEP_WAITS) request_operands();
    if (!COH && ep.ss_in != nullptr) {
        float ss = 0.f;
#pragma unroll
        for (int q = 0; q < SS_HELD; q++)
            if (ss_part + q * PARTS < ep.ss_tiles) ss += ss_held[q];
#pragma unroll 4
        for (int j = ss_part + SS_HELD * PARTS; j < ep.ss_tiles; j += PARTS) ss += ss_row[j];
        s_part[ss_part][ss_tl] = ss;
    }
    // ---- 0. epilogue operands that do not depend on the sums and are too many to be held over the K loop: issue their loads now,
    // so that they travel while the K split is being closed (every workgroup does it;
    // only the one that ends up running the epilogue uses them).  Indices are clamped,
    // not predicated: unconditional loads.
    __amdgpu_buffer_rsrc_t rs_o = gemm_rsrc(ep.a16_out, (unsigned)p.Tb * (unsigned)ep.Kb_out * 2048u);
    __amdgpu_buffer_rsrc_t rs_q = gemm_rsrc(ep.q_out, (unsigned)p.T * (unsigned)ep.QD * 4u);
    constexpr int HS = hyper_streams(EPI);
    HyperIn<HS ? HS : 1> pf_hyper[HS ? FPT : 1];
    HyperMix<HS ? HS : 1> hyper_c;
    if constexpr (HS > 0) {
        hyper_c = hyper_mix<HS>(ep);
#pragma unroll
        for (int s = 0; s < FPT; s++) {
            const int w_ = min(tid + s * NW * 64, WITEMS - 1);
            const int h = w_ >> ITEMS_SHIFT, e = w_ & (ITEMS - 1);
            const int l = e & 63, j = (e >> 6) % TB, i = (e >> 6) / TB;
            hyper_load_4<HS>(pf_hyper[s], ep, p.N, min(tb0 * 16 + j * 16 + (l & 15), p.T - 1), min((nb0 + 2 * h + i) * 16 + 4 * (l >> 4), p.N - 4));
        }
    }
    // ---- 1. sum the waves' partial tiles through LDS: every wave stores all its tiles, ONE
    // barrier, then each thread collects its items w = (round h, e): the float4 for token t(e) and
    // features n(h, e) .. n+3, in wave order.  (The items of all rounds are dealt over all threads.)
    f4_t v[FPT];
#pragma unroll
    for (int i = 0; i < NBW; i++)
#pragma unroll
        for (int j = 0; j < TB; j++) red[wave][i][j][lane] = acc[i][j];
    __syncthreads();
    if (ep.ss_in != nullptr && tid < TB * 16) {
        // 1/rms per token from its slices' sums (s_part: visible since the barrier
        // above; s_rinv is read by the epilogue after at least one more barrier)
        float ss = 0.f;
#pragma unroll
        for (int q = 0; q < PARTS; q++) ss += s_part[q][tid];
        s_rinv[tid] = __fdiv_rn(1.0f, sqrtf(__fadd_rn(__fdiv_rn(ss, (float)ep.d_in), ep.eps)));
    }
#pragma unroll
    for (int s = 0; s < FPT; s++) {
        const int w_ = tid + s * NW * 64;
        f4_t sum = f4_t{0.f, 0.f, 0.f, 0.f};
        if (w_ < WITEMS) {
            const int h = w_ >> ITEMS_SHIFT, e = w_ & (ITEMS - 1);
            const int l = e & 63, j = (e >> 6) % TB, i = (e >> 6) / TB;
            sum = red[0][2 * h + i][j][l];
#pragma unroll
            for (int wv = 1; wv < NW; wv++) sum += red[wv][2 * h + i][j][l];
        }
        v[s] = sum;
    }
    __syncthreads();   // everybody has read the partial tiles (the epilogue reuses the array) and s_rinv is visible
    NVLLM_TSTAMP(4, v[FPT - 1][0]);
    // ---- 2. close the K split: write-through slab, ticket, last arriver reduces.
    const unsigned tile_id = ix.z * ix.gx + ix.x;
    if (p.ksplit > 1) {
        float* my = p.slab + ((size_t)tile_id * p.ksplit + ix.y) * (ROUNDS * ITEMS * 4);
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(my, 0, ROUNDS * ITEMS * 16, 0x00020000);
#pragma unroll
        for (int s = 0; s < FPT; s++) {
            const int w_ = tid + s * NW * 64;
            if (w_ < WITEMS)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4_t, v[s]), rs, w_ * 16, 0, /*sc1: write through*/ AUX_SC1);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // every storing wave drains its stores
        __syncthreads();
        if (tid == 0)
            *s_ticket = __hip_atomic_fetch_add(p.counters + tile_id, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*s_ticket != (unsigned)p.ksplit - 1) return false;     // not the last slice of this tile
        // The partials were stored write-through, every storing wave drained, and this workgroup's add came
        // last (its returned value says so, read behind the barrier above).  They may then be loaded past the
        // vector cache (sc1) with no invalidate: such a load misses that cache whoever shares the CU, and no
        // cache holds an older copy, because a line of the slab is stored once and read once in a launch, here,
        // and launches begin with clean caches.  Tiles and riders beside this one load no line of its partials.
        // Otherwise an agent acquire comes first.
        const bool past_l1 = p.close_sc1;
        if (!past_l1) {
            if (tid == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the invalidate has completed
            __syncthreads();
        }
        const float* base = p.slab + (size_t)tile_id * p.ksplit * (ROUNDS * ITEMS * 4);
        __amdgpu_buffer_rsrc_t rs_all = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0,
                                                                           p.ksplit * ROUNDS * ITEMS * 16, 0x00020000);
        // Every slab load of both rounds is issued before the first add: one round trip.
        // Slice indices past the end are clamped (a repeated load), not predicated, so the
        // loads stay unconditional; sums are taken in slice order.
#pragma unroll
        for (int s = 0; s < FPT; s++) v[s] = f4_t{0.f, 0.f, 0.f, 0.f};
        for (int s0 = 0; s0 < p.ksplit; s0 += 8) {
            f4_t part[FPT][8];
#pragma unroll
            for (int s = 0; s < FPT; s++) {
                const int w_ = min(tid + s * NW * 64, WITEMS - 1);
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    const int sl = min(s0 + u, p.ksplit - 1);
                    if (past_l1)
                        part[s][u] = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(rs_all, (sl * WITEMS + w_) * 16, 0, AUX_SC1));
                    else
                        part[s][u] = *reinterpret_cast<const f4_t*>(base + ((size_t)sl * WITEMS + w_) * 4);
                }
            }
#pragma unroll
            for (int s = 0; s < FPT; s++)
#pragma unroll
                for (int u = 0; u < 8; u++)
                    if (s0 + u < p.ksplit) v[s] += part[s][u];
        }
        // ready for the next launch (nobody else touches this tile's counter any more)
        if (tid == 0) __hip_atomic_store(p.counters + tile_id, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    NVLLM_TSTAMP(5, v[FPT - 1][0]);
    // ---- 3. epilogue on complete sums
    float ssq[FPT];
#pragma unroll
    for (int s = 0; s < FPT; s++) ssq[s] = 0.f;
    if (EPI == GemmEpilogue::SWIGLU_A16) {
        // gate (even row block, i = 0) and up (odd, i = 1) sit in different threads: swap through LDS so that
        // the i = 0 thread has both.  All rounds at once, each in its own part of the array (the partial tiles
        // in it have been consumed: a barrier back), so one barrier serves them all.
#pragma unroll
        for (int s = 0; s < FPT; s++) {
            const int w_ = tid + s * NW * 64;
            const int h = w_ >> ITEMS_SHIFT, e = w_ & (ITEMS - 1);
            if (w_ < WITEMS) red[0][2 * h + (e >> 6) / TB][(e >> 6) % TB][e & 63] = v[s];
        }
        __syncthreads();
    }
    {
#pragma unroll
        for (int s = 0; s < FPT; s++) {
            const int w_ = tid + s * NW * 64;
            if (w_ >= WITEMS) continue;
            const int h = w_ >> ITEMS_SHIFT, e = w_ & (ITEMS - 1);
            const int l = e & 63, j = (e >> 6) % TB, i = (e >> 6) / TB;
            const int tl = j * 16 + (l & 15);
            const int t = tb0 * 16 + tl;
            const int nb = nb0 + 2 * h + i;
            const int n = nb * 16 + 4 * (l >> 4);
            const bool live = t < p.T && tb0 + j < p.Tb && nb < nb_lim;
            const float rinv = ep.ss_in ? s_rinv[tl] : 1.0f;
            float y[4] = {v[s][0] * rinv, v[s][1] * rinv, v[s][2] * rinv, v[s][3] * rinv};
            if constexpr (HS > 0) {
                if (live) hyper_update_4<HS>(pf_hyper[s], hyper_c, ep, p.N, t, n, y);
            } else if constexpr (epi_is_point(EPI)) {
                if (live) ssq[s] += epi_point<EPI>(ep, p.N, t, n, y);
            } else if (EPI == GemmEpilogue::F32) {
                if constexpr (OP::PLANES == 1) {
                    if (ep.softcap > 0.f)
#pragma unroll
                        for (int r = 0; r < 4; r++) y[r] = ep.softcap * tanhf(y[r] / ep.softcap);
                }
                if (live) {
                    // logits rows go to the host from here: 64-byte pieces cross PCIe as fast as a copy's (64 rows of 32,000:
                    // 157 us, a copy kernel 151), beside the products instead of after them and after a launch's gap
                    for (float* rows = ep.out; rows; rows = rows == ep.out ? ep.out_host : nullptr) {
                        float* o = rows + (size_t)t * ep.ldo + n;
                        if (n + 3 < p.N && (ep.ldo & 3) == 0) {
                            *reinterpret_cast<float4*>(o) = make_float4(y[0], y[1], y[2], y[3]);
                        } else {
#pragma unroll
                            for (int r = 0; r < 4; r++)
                                if (n + r < p.N) o[r] = y[r];
                        }
                    }
                }
                if (ep.amax_pairs != nullptr) {
                    // this item's four outputs: first index of their maximum (a NaN never wins, -inf may)
                    float bv = -INFINITY, bi = -1.0f;
                    if (live) {
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            if (n + r < p.N && (y[r] > bv || (bi < 0.f && y[r] == bv))) {
                                bv = y[r];
                                bi = (float)(n + r);
                            }
                        // the reference's scan starts from logits[0], and nothing displaces a NaN there
                        // (sampler.c:86-97): +inf at index 0 wins every comparison downstream
                        if (n == 0 && y[0] != y[0]) {
                            bv = INFINITY;
                            bi = 0.f;
                        }
                    }
                    // (the partial tiles in `red` have been consumed: two barriers back)
                    float2* am = reinterpret_cast<float2*>(&red[0][0][0][0]);
                    am[((2 * h + i) * 4 + (l >> 4)) * (TB * 16) + tl] = make_float2(bv, bi);
                }
            } else if (EPI == GemmEpilogue::SWIGLU_A16) {
                if (i == 0 && live) {
                    const f4_t u = red[0][2 * h + 1][j][l];
                    float z[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        float gate = y[r], up = u[r] * rinv;
                        if constexpr (OP::PLANES == 1) {   // (the up row of a hidden unit is 16 rows further on)
                            if (ep.bias) {
                                gate += ep.bias[n + r];
                                up += ep.bias[n + 16 + r];
                            }
                            if (ep.row_weight) {
                                gate *= ep.row_weight[t];
                                up *= ep.row_weight[t];
                            }
                        }
                        z[r] = silu_mul(gate, up);
                    }
                    const int hid = (nb >> 1) * 16 + 4 * (l >> 4);
                    if constexpr (OP::PLANES == 1) store_b16_4(ep.a16_out, ep.Kb_out, t, hid, z);
                    else if constexpr (COH) store_a16_4_sc1(rs_o, ep.Kb_out, t, hid, z, l);
                    else store_a16_4(ep.a16_out, ep.Kb_out, t, hid, z);
                }
            } else if (EPI == GemmEpilogue::RESID_B16) {
                if (live) ssq[s] += resid_b16_4(ep, p.N, t, n, pf_x[s], pf_g[s], y);
            } else if (EPI == GemmEpilogue::RESID_A16) {
                if (live) {
                    float* xr = ep.x + (size_t)t * p.N + n;
                    const float4 xo = pf_x[s];
                    const float4 g = pf_g[s];
                    // residual add as the reference's accum(): x = x + branch (layers.c:163-168)
                    const float xn[4] = {__fadd_rn(xo.x, y[0]), __fadd_rn(xo.y, y[1]), __fadd_rn(xo.z, y[2]), __fadd_rn(xo.w, y[3])};
                    if constexpr (COH)
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4_t, make_float4(xn[0], xn[1], xn[2], xn[3])), rs_x,
                                                               (t * p.N + n) * 4, 0, AUX_SC1);
                    else
                        *reinterpret_cast<float4*>(xr) = make_float4(xn[0], xn[1], xn[2], xn[3]);
                    const float z[4] = {xn[0] * g.x, xn[1] * g.y, xn[2] * g.z, xn[3] * g.w};
                    if constexpr (COH) store_a16_4_sc1(rs_o, ep.Kb_out, t, n, z, l);
                    else store_a16_4(ep.a16_out, ep.Kb_out, t, n, z);
                    ssq[s] += xn[0] * xn[0] + xn[1] * xn[1] + xn[2] * xn[2] + xn[3] * xn[3];
                }
            } else {  // ROPE_KV
                if (live) {
                    if (n < ep.QD + ep.KD) {   // q or k: rotate the two pairs of this float4 (layers.c:118-141)
                        const float2 c0 = make_float2(pf_turn[s][0], pf_turn[s][1]), c1 = make_float2(pf_turn[s][2], pf_turn[s][3]);
                        const float a0 = y[0], b0 = y[1], a1 = y[2], b1 = y[3];
                        y[0] = __fsub_rn(__fmul_rn(a0, c0.x), __fmul_rn(b0, c0.y));
                        y[1] = __fadd_rn(__fmul_rn(a0, c0.y), __fmul_rn(b0, c0.x));
                        y[2] = __fsub_rn(__fmul_rn(a1, c1.x), __fmul_rn(b1, c1.y));
                        y[3] = __fadd_rn(__fmul_rn(a1, c1.y), __fmul_rn(b1, c1.x));
                    }
                    if (n < ep.QD) {
                        if constexpr (COH)
                            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4_t, make_float4(y[0], y[1], y[2], y[3])), rs_q,
                                                                   (t * ep.QD + n) * 4, 0, AUX_SC1);
                        else *reinterpret_cast<float4*>(ep.q_out + (size_t)t * ep.QD + n) = make_float4(y[0], y[1], y[2], y[3]);
                    } else if (pf_row >= 0) {
                        const long block = pf_row / ep.bs;
                        const int key = pf_row % ep.bs;
                        const bool is_k = n < ep.QD + ep.KD;
                        const int c = is_k ? n - ep.QD : n - ep.QD - ep.KD;
                        KVT* pool = reinterpret_cast<KVT*>(is_k ? ep.pool_k : ep.pool_v) + ep.layer_off;
                        if (sizeof(KVT) == 4) {   // the reference's rows (memory.c:37-43)
                            if constexpr (COH) kv_put4_sc1<KVT>(pool + (block * ep.bs + key) * ep.KD + c, y);
                            else kv_put4<KVT>(pool + (block * ep.bs + key) * ep.KD + c, y);
                        } else {                  // fp16 pages in matrix-core operand order
                            const int kvh = c / ep.hd, d = c % ep.hd;
                            KVT* page = pool + kv16_page(block, kvh, ep.KD / ep.hd, ep.hd);
                            if constexpr (COH) {
                                if (is_k) kv_put4_sc1<KVT>(page + kv16_k_off(key, d), y);
                                else kv_put4_strided_sc1<KVT>(page + kv16_v_off(key, d), y);
                            } else {
                                if (is_k) kv_put4<KVT>(page + kv16_k_off(key, d), y);
                                else kv_put4_strided<KVT>(page + kv16_v_off(key, d), y);
                            }
                        }
                    }
                }
            }
        }
    }
    if (EPI == GemmEpilogue::F32 && ep.amax_pairs != nullptr) {
        // per token, over the tile's features in ascending order: the first maximum
        __syncthreads();
        if (tid < TB * 16) {
            const float2* am = reinterpret_cast<const float2*>(&red[0][0][0][0]);
            float2 best = am[tid];
#pragma unroll
            for (int s = 1; s < NBW * 4; s++) {
                const float2 c = am[s * (TB * 16) + tid];
                if (c.y >= 0.f && (c.x > best.x || best.y < 0.f)) best = c;
            }
            const int t = tb0 * 16 + tid;
            if (t < p.T) ep.amax_pairs[(size_t)ix.x * ep.amax_ld + t] = best;
        }
    }
    if (epi_has_ss(EPI)) {
        // per-token sum of x^2 over each 32-feature group (= one round: two row blocks):
        // over the 4 lane groups (l>>4), then over the round's two row blocks (i)
        const int ss_cols = EPI == GemmEpilogue::LATENT_IN ? ep.latent_q >> 5 : (p.N + 31) >> 5;
        // all rounds' halves meet in the array of the partial tiles (consumed: a barrier back), [round][half][token]:
        // one barrier for all rounds
        float (*ss_lds)[2][TB * 16] = reinterpret_cast<float (*)[2][TB * 16]>(lds_dyn);
#pragma unroll
        for (int s = 0; s < FPT; s++) {
            float sq = ssq[s];
            sq += __shfl_xor(sq, 16, 64);
            sq += __shfl_xor(sq, 32, 64);
            const int w_ = tid + s * NW * 64;
            const int h = w_ >> ITEMS_SHIFT, e = w_ & (ITEMS - 1);
            if (w_ < WITEMS && (e & 63) < 16) ss_lds[h][(e >> 6) / TB][((e >> 6) % TB) * 16 + (e & 15)] = sq;
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < ROUNDS; h++) {
            if (tid < TB * 16) {
                const int t = tb0 * 16 + tid;
                const int col = ix.x * ROUNDS + h;
                if (t < p.T && col < ss_cols) {
                    const float sum = ss_lds[h][0][tid] + ss_lds[h][1][tid];
                    if constexpr (COH)
                        __hip_atomic_store(reinterpret_cast<unsigned*>(ep.ss_out + (size_t)t * ss_cols + col),
                                           __builtin_bit_cast(unsigned, sum), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    else
                        ep.ss_out[(size_t)t * ss_cols + col] = sum;
                }
            }
        }
    }
#ifdef NVLLM_STAMPS
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // stores issued so far have left the CU
#endif
    NVLLM_TSTAMP(6, ssq[0]);
    return true;
}

}  // namespace nvllm
