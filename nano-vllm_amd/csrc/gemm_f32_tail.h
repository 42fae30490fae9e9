// gemm_f32_tail.h -- what follows the sums of a projection whose activations are fp32 rows (gemm_f32.hip, gemm_thin.hip).
#pragma once

#include "gemm_common.h"
#include "gemm_f32.h"

namespace nvllm {

// The segment of a feature tile (those that a launch has not begin past every tile).
__device__ __forceinline__ int f32_segment(const F32Gemm& p, int tile) {
    int s = 0;
#pragma unroll
    for (int i = 1; i < F32_SEGMENTS; i++) s += tile >= p.seg[i].first;
    return s;
}

// The angles of features n .. n+3 of a head (n % 4 == 0) at position `pos`.
__device__ __forceinline__ bool f32_turns(const F32Segment& sg) { return sg.kind == F32Out::ROPE_Q || sg.kind == F32Out::ROPE_K; }
__device__ __forceinline__ f4_t f32_angles(const F32Gemm& p, int pos, int n) {
    return *reinterpret_cast<const f4_t*>(p.rope + (size_t)pos * (p.hd >> 1) + ((n % p.hd) >> 1));   // (hd is a multiple of 8)
}
__device__ __forceinline__ int f32_row(const F32Gemm& p, const F32Segment& sg, int t) {
    return sg.kind == F32Out::ROPE_K || sg.kind == F32Out::KV_V ? p.kv_row[t] : -1;
}
// What follows a token's complete sums of features n .. n+3 (n % 4 == 0).  `side`: what ADD adds to, or the angles of a quad that turns;
// `row`: its token's cache row.
template <bool PAIR>
__device__ __forceinline__ void f32_finish(const F32Gemm& p, const F32Segment& sg, int t, int n, f4_t y, const f4_t u, const f4_t side, int row) {
    if constexpr (PAIR) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int f = min(n + r, sg.N - 1);
            y[r] = silu_mul(sg.bias ? y[r] + sg.bias[f] : y[r], sg.bias2 ? u[r] + sg.bias2[f] : u[r]);
        }
    } else {
        switch (sg.kind) {
            case F32Out::ADD:
#pragma unroll
                for (int r = 0; r < 4; r++) y[r] = __fadd_rn(side[r], y[r]);
                break;
            case F32Out::SILU:
#pragma unroll
                for (int r = 0; r < 4; r++) y[r] = silu_mul(y[r], 1.f);
                break;
            case F32Out::RELU2:
#pragma unroll
                for (int r = 0; r < 4; r++) y[r] = fmaxf(y[r], 0.f) * fmaxf(y[r], 0.f);
                break;
            case F32Out::ROPE_Q:
            case F32Out::ROPE_K: {   // the two pairs of this quad turn (layers.c:118-141)
                const float2 c0 = make_float2(side[0], side[1]), c1 = make_float2(side[2], side[3]);
                y = f4_t{__fsub_rn(__fmul_rn(y[0], c0.x), __fmul_rn(y[1], c0.y)), __fadd_rn(__fmul_rn(y[0], c0.y), __fmul_rn(y[1], c0.x)),
                         __fsub_rn(__fmul_rn(y[2], c1.x), __fmul_rn(y[3], c1.y)), __fadd_rn(__fmul_rn(y[2], c1.y), __fmul_rn(y[3], c1.x))};
                break;
            }
            default: break;
        }
        if (sg.kind == F32Out::ROPE_K || sg.kind == F32Out::KV_V) {
            if (row < 0) return;
            const bool is_k = sg.kind == F32Out::ROPE_K;
            const float z[4] = {y[0], y[1], y[2], y[3]};
            if (p.kv_elem_bytes == 4) {   // the reference's rows (memory.c:37-43)
                kv_put4<float>(reinterpret_cast<float*>(is_k ? p.pool_k : p.pool_v) + p.layer_off + (size_t)row * p.KD + n, z);
            } else {                      // fp16 pages in matrix-core operand order
                __half* page = reinterpret_cast<__half*>(is_k ? p.pool_k : p.pool_v) + p.layer_off + kv16_page(row / p.bs, n / p.hd, p.KD / p.hd, p.hd);
                if (is_k) kv_put4<__half>(page + kv16_k_off(row % p.bs, n % p.hd), z);
                else kv_put4_strided<__half>(page + kv16_v_off(row % p.bs, n % p.hd), z);
            }
            return;
        }
    }
    for (float* rows = sg.out; rows; rows = rows == sg.out ? p.out_host : nullptr) {
        float* o = rows + (size_t)t * sg.ldo + n;
        if (sg.vec) {
            *reinterpret_cast<f4_t*>(o) = y;
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (n + r < sg.N) o[r] = y[r];
        }
    }
}
__device__ __forceinline__ f4_t f32_old(const F32Segment& sg, int t, int n) {   // t < T; features past the last are those of the last
    const float* o = sg.out + (size_t)t * sg.ldo;
    if (sg.vec) return *reinterpret_cast<const f4_t*>(o + min(n, sg.N - 4));
    f4_t v;
#pragma unroll
    for (int r = 0; r < 4; r++) v[r] = o[min(n + r, sg.N - 1)];
    return v;
}

// The first maximum of a block's 16 features per token, by the reference's scan (sampler.c:86-97): strict >, so a NaN never wins --
// except at index 0, which nothing displaces: +inf there wins every comparison downstream.  Lane (x, g): features n0 .. n0 + 3 of token x; the
// whole wave comes here.
__device__ __forceinline__ void f32_pairs(const F32Gemm& p, int N, int block, int n0, int t, bool writes, const f4_t& y) {
    float bv = -INFINITY, bi = -1.0f;
#pragma unroll
    for (int r = 0; r < 4; r++)
        if (n0 + r < N && (y[r] > bv || (bi < 0.f && y[r] == bv))) {
            bv = y[r];
            bi = (float)(n0 + r);
        }
    if (n0 == 0 && y[0] != y[0]) {
        bv = INFINITY;
        bi = 0.f;
    }
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {
        const float ov = __shfl_xor(bv, o, 64), oi = __shfl_xor(bi, o, 64);
        if (oi >= 0.f && (ov > bv || bi < 0.f || (ov == bv && oi < bi))) {
            bv = ov;
            bi = oi;
        }
    }
    if (writes) p.amax_pairs[(size_t)block * p.amax_ld + t] = make_float2(bv, bi);
}

}  // namespace nvllm
