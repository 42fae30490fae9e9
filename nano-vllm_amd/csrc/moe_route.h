// moe_route.h -- choosing experts and sorting a batch's (token, expert) pairs, on the device: launches of their own (moe.hip), or a
// workgroup beside a projection's tiles (gemm_b16.hip).
#pragma once

#include "attn_tile.h"
#include "moe.h"

namespace nvllm {

// Maximum over a wave, in every lane, on the vector unit alone (many waves of one CU would queue for the LDS crossbar):
// rotations within rows of 16 lanes, then the rows.
template <int N>
__device__ __forceinline__ float row_rotate(float x) {
    const int v = __builtin_bit_cast(int, x);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(v, v, 0x120 + N, 0xf, 0xf, false));
}
__device__ __forceinline__ float wave_max(float x) {
    x = fmaxf(x, row_rotate<8>(x));
    x = fmaxf(x, row_rotate<4>(x));
    x = fmaxf(x, row_rotate<2>(x));
    x = fmaxf(x, row_rotate<1>(x));
    return rows_max(x);
}

// One wave chooses for one token: `top` times the best of what comes after the previous choice in the order
// (score descending, index ascending).
__device__ __forceinline__ void route_token(const RoutePlan& r, const float* __restrict__ z, int t, int lane) {
    float last = INFINITY;
    int last_e = -1;
    for (int j = 0; j < r.top; j++) {
        float best = -INFINITY;
        int best_e = 0x7fffffff;
        for (int e = lane; e < r.E; e += 64) {
            const float v = z[e];
            const bool open = v < last || (v == last && e > last_e);
            if (open && v > best) {
                best = v;
                best_e = e;
            }
        }
        const float top = wave_max(best);
        int first = best == top ? best_e : 0x7fffffff;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) first = min(first, __shfl_xor(first, o, 64));
        best = top;
        best_e = first;
        if (best_e >= r.E) best_e = 0;   // (no number compares: NaN logits)
        last = best;
        last_e = best_e;
        if (lane == 0) {
            r.choice[(size_t)t * r.top + j] = best_e;
            r.score[(size_t)t * r.top + j] = 1.f / (1.f + expf(-best));
        }
    }
}
// The same for four tokens of up to 64 experts, a logit per lane (lanes past the last expert: -INFINITY).  put(token, place, expert, score) in lane 0.
template <class Put>
__device__ __forceinline__ void choose_four(float (&v)[4], int E, int top, int lane, Put&& put) {
    for (int j = 0; j < top; j++) {
        float best[4];
#pragma unroll
        for (int u = 0; u < 4; u++) best[u] = wave_max(v[u]);
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const unsigned long long at = __ballot(v[u] == best[u] && lane < E);
            const int e = at ? __ffsll(at) - 1 : 0;   // (no number compares: NaN logits)
            if (lane == e) v[u] = -INFINITY;
            if (lane == 0) put(u, j, e, 1.f / (1.f + expf(-best[u])));
        }
    }
}
// One workgroup: counts, segment starts, then every choice takes a row of its expert's segment (in any order: a row's
// result does not depend on its place).
// lds_r: counts [E], next free row [E], segment start [E + 1], CHOOSE: choices and scores [T * top].
template <bool CHOOSE, int NT>
__device__ __forceinline__ void route_sort(RoutePlan r, const float* __restrict__ z, int ldz, int* lds_r) {
    constexpr int WAVES = NT / 64;
    int* count = lds_r;
    int* cursor = count + r.E;
    int* start = cursor + r.E;
    const int tid = threadIdx.x, lane = tid & 63, pairs = r.T * r.top;
    int *choice = CHOOSE ? start + r.E + 1 : r.choice, *out_choice = r.choice;
    float* out_score = r.score;
    float* score = CHOOSE ? reinterpret_cast<float*>(choice + pairs) : r.score;
    for (int e = tid; e < r.E; e += NT) count[e] = 0;
    if (CHOOSE) {
        r.choice = choice;   // (route_token fills the LDS copies)
        r.score = score;
        if (r.E <= 64) {   // a logit per lane, four tokens at a time
            for (int t0 = tid >> 6; t0 < r.T; t0 += 4 * WAVES) {
                float v[4];
#pragma unroll
                for (int u = 0; u < 4; u++) v[u] = lane < r.E ? z[(size_t)min(t0 + WAVES * u, r.T - 1) * ldz + lane] : -INFINITY;
                choose_four(v, r.E, r.top, lane, [&](int u, int j, int e, float sc) {
                    const int t = t0 + WAVES * u;
                    if (t < r.T) {
                        choice[t * r.top + j] = e;
                        score[t * r.top + j] = sc;
                    }
                });
            }
        } else {
            for (int t = tid >> 6; t < r.T; t += WAVES) route_token(r, z + (size_t)t * ldz, t, lane);
        }
    }
    __syncthreads();
    for (int i = tid; i < pairs; i += NT) atomicAdd(count + choice[i], 1);
    __syncthreads();
    if (tid < 64) {   // the first wave sums the padded counts
        int base = 0;
        for (int e0 = 0; e0 < r.E; e0 += 64) {
            const int e = e0 + tid, n = e < r.E ? (count[e] + r.pad - 1) / r.pad * r.pad : 0;
            int sum = n;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int v = __shfl_up(sum, o, 64);
                if (tid >= o) sum += v;
            }
            if (e < r.E) start[e] = cursor[e] = base + sum - n;
            base += __shfl(sum, 63, 64);
        }
        if (tid == 0) start[r.E] = base;
    }
    __syncthreads();   // the last one: from here on everybody only writes results (a barrier would wait for the stores)
    const int used = start[r.E];
    for (int b = used / 16 + tid; b < r.capacity / 16; b += NT) r.block_expert[b] = -1;
    for (int i = used + tid; i < r.capacity; i += NT) {   // (a tile may look up rows behind its own: they name a token too)
        r.source[i] = 0;
        r.weight[i] = 0.f;
    }
    for (int e = tid >> 4; e < r.E; e += NT / 16) {   // 16 threads per expert: its blocks, and the padding of its segment
        const int lo = start[e], hi = start[e + 1], n = count[e];
        for (int b = lo / 16 + (tid & 15); b < hi / 16; b += 16) r.block_expert[b] = e;
        for (int i = lo + n + (tid & 15); i < hi; i += 16) {
            r.source[i] = 0;
            r.weight[i] = 0.f;
        }
    }
    for (int i = tid; i < pairs; i += NT) {
        const int row = atomicAdd(cursor + choice[i], 1);
        r.source[row] = i / r.top;
        r.weight[row] = score[i];
        r.row_of[i] = row;
        if (CHOOSE) {
            out_choice[i] = choice[i];
            out_score[i] = score[i];
        }
    }
}

// bytes of LDS of route_sort<true>
static inline size_t route_sort_lds(int T, int E, int top) { return ((size_t)3 * E + 1) * sizeof(int) + (size_t)T * top * 8; }
constexpr int ROUTE_ONE = 256;      // tokens up to which one workgroup chooses and sorts

// us that a workgroup takes to choose and sort: a step of a wave picks the best of what is left for four tokens (one, past 64 experts).
// 256 tokens, 4, 8 and 16 waves: 8 of 64 experts 114, 69, 54; 2 of 128 140, 66, 34; 8 of 512 952, 537, 316; 8 of 2,048 3,449, -, 1,150.
static inline double route_us(int T, int E, int top, int waves) {
    const double step = E > 64 ? 0.9 + 0.18 * E / 64 : waves <= 4 ? 0.9 : waves <= 8 ? 1.03 : 1.7;
    return 2.0 + step * top * (double)((E > 64 ? T + waves - 1 : (T + 4 * waves - 1) / 4) / waves);
}
// Whether that rides in a workgroup of `waves` waves beside tiles of `tiles_us`: where it then ends no later than a launch of its own would,
// which costs another microsecond and has 16 waves.  fp32 pairs of 2,816 features over 1,024 k, both ways (tiles alone): 80 tokens, 2 of 16 experts 28 and 36 us (28); 128, 2
// of 64 28 and 39 (29); 8 of 64, 96 tokens 40 and 53 (26), 192 86 and 80 (36); 2 of 128, 48 tokens 16 and 25 (16), 64 34 and 29, 256 140 and 82
// (44); 8 of 512, 256 tokens 952 and 365.  bf16, 1,024 features over 2,816 k: 2 of 16, 64 tokens 11 and 16 (10); 8 of 64, 128 36 and 39 (9); 2 of 65,
// 64 tokens 19 and 22 (10), 128 34 and 29; 8 of 512, 16 tokens 36 and 30 (8).
static inline bool route_rides(const RoutePlan& r, int waves, double tiles_us) {
    return r.T <= ROUTE_ONE && route_us(r.T, r.E, r.top, waves) <= tiles_us + 1.0 + route_us(r.T, r.E, r.top, 16);
}

}  // namespace nvllm
