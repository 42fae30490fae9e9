// moe.hip -- routing, sorting and summing for mixtures of experts (moe.h).
#include "moe.h"

#include <algorithm>

#include "gemm_common.h"
#include "moe_route.h"

namespace nvllm {

namespace {
constexpr int MAX_EXPERTS = 4096;
}

int route_pad(int T, int E, int top) {
    const long per = (long)T * top / E;   // rows an expert gets on average
    return per >= 96 ? 128 : per >= 40 ? 64 : per > 20 ? 32 : 16;
}
// Tiles of 256 features as tall as an expert's rows where they make one round of the chip, else 128 features by 16 to 128 rows.
// 16 experts of 2 x 1,408 x 2,048, two per token, 1,029 tokens: groups of 128 rows, which every other expert's overflow, took 74 us
// and 44 for the two products; of 160 56 and 41.
ExpertGroups expert_groups(int T, int E, int top, const B16Weight& up, const B16Weight& down) {
    const int wide = expert_rows_wide(T * top, E, up, down);
    return {wide ? wide : route_pad(T, E, top), wide != 0};
}
static int route_capacity(int T, int E, int top, int pad) {
    const long rows = (long)T * top, groups = std::min(rows, rows / pad + E);   // full groups, and one partly filled per expert
    return (int)(groups * pad);
}
size_t route_ints(int T, int E, int top, int pad) {
    const size_t cap = (size_t)route_capacity(T, E, top, pad);
    return cap / 16 + 2 * cap + 3 * (size_t)T * top + 64;
}
// (the sizes are checked here, for plans whose choices ride in a projection's launch too)
RoutePlan route_plan(int* mem, int T, int E, int top, int pad) {
    if (E < 1 || E > MAX_EXPERTS || top < 1 || top > E) NVLLM_FATAL("routing: %d of %d experts per token", top, E);
    RoutePlan r{};
    r.T = T; r.E = E; r.top = top; r.pad = pad;
    r.capacity = route_capacity(T, E, top, pad);
    r.block_expert = mem;
    r.source = r.block_expert + r.capacity / 16;
    r.weight = (float*)(r.source + r.capacity);
    r.row_of = (int*)(r.weight + r.capacity);
    r.choice = r.row_of + (size_t)T * top;
    r.score = (float*)(r.choice + (size_t)T * top);
    return r;
}

__global__ __launch_bounds__(256) void k_route(RoutePlan r, const float* __restrict__ z, int ldz) {
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t < r.T) route_token(r, z + (size_t)t * ldz, t, threadIdx.x & 63);
}

template <bool CHOOSE>
__global__ __launch_bounds__(1024) void k_route_sort(RoutePlan r, const float* __restrict__ z, int ldz) {
    extern __shared__ int lds_r[];
    route_sort<CHOOSE, 1024>(r, z, ldz, lds_r);
}

void launch_route(const RoutePlan& r, const float* z, int ldz, bool chosen) {
    if (r.T <= 0) return;
    const size_t lds = ((size_t)3 * r.E + 1) * sizeof(int);
    const size_t lds_one = route_sort_lds(r.T, r.E, r.top);
    if (!chosen && r.T <= ROUTE_ONE && lds_one <= 64 * 1024) {
        ProfScope ps(PC_ROUTE, choice_bytes(r), 0);
        NVLLM_LAUNCH((k_route_sort<true>), dim3(1), dim3(1024), lds_one, r, z, ldz);
        return;
    }
    if (!chosen) {
        ProfScope ps(PC_ROUTE, choice_bytes(r), 0);
        NVLLM_LAUNCH(k_route, dim3(cdiv(r.T, 4)), dim3(256), 0, r, z, ldz);
    }
    ProfScope ps(PC_ROUTE, sort_bytes(r), 0);
    NVLLM_LAUNCH((k_route_sort<false>), dim3(1), dim3(1024), lds, r, z, ldz);
}

// A workgroup per 16 rows, a wave per tile: lane (row, k group) reads 32 bytes of its row and writes its piece of the tile.
__global__ __launch_bounds__(256) void k_expert_rows(__half* __restrict__ dst, const float* __restrict__ x, const float* __restrict__ gain, RoutePlan r, int ld) {
    const int blk = blockIdx.x, lane = threadIdx.x & 63, Kb = ld >> 5;
    if (r.block_expert[blk] < 0) return;
    const float* row = x + (size_t)r.source[blk * 16 + (lane & 15)] * ld + 8 * (lane >> 4);
    for (int kb = (int)blockIdx.y * 4 + (threadIdx.x >> 6); kb < Kb; kb += 4 * gridDim.y) {
        const f4_t a = *reinterpret_cast<const f4_t*>(row + kb * 32), b = *reinterpret_cast<const f4_t*>(row + kb * 32 + 4);
        const f4_t ga = *reinterpret_cast<const f4_t*>(gain + kb * 32 + 8 * (lane >> 4)), gb = *reinterpret_cast<const f4_t*>(gain + kb * 32 + 8 * (lane >> 4) + 4);
        b8_t v;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            v[e] = (__bf16)(a[e] * ga[e]);
            v[4 + e] = (__bf16)(b[e] * gb[e]);
        }
        *reinterpret_cast<b8_t*>(dst + ((size_t)blk * Kb + kb) * TILE_HALVES + lane * 8) = v;
    }
}
void launch_expert_rows(__half* dst, const float* x, const float* gain, const RoutePlan& r, int ld) {
    if (r.T <= 0) return;
    if (ld % 32) NVLLM_FATAL("expert rows: a row of %d is not padded to 32", ld);
    ProfScope ps(PC_EXPERT_ROWS, (double)r.T * r.top * ld * 2.0 + (double)r.T * ld * 4.0, 0);
    NVLLM_LAUNCH(k_expert_rows, dim3(r.capacity / 16, std::min(4, cdiv(ld, 128))), dim3(256), 0, dst, x, gain, r, ld);   // (slices of K: 9.3 us with one at 1,029 tokens of 2,048, 8.0 with four)
}

// One workgroup per token.  VEC 4: eight neighbouring threads cover 32 features.  Everything but the experts' rows is requested before
// the look-up of the rows is answered, and the rows two at a time: 1,029 tokens of 2,048, two experts
// and a shared one 14.2 -> 12.8 us, 64 tokens 6.3 -> 5.0.
template <int VEC>
__global__ __launch_bounds__(256) void k_moe_combine(MoeCombine m, int top) {
    const int t = blockIdx.x, Kb = m.ld >> 5;
    struct alignas(4 * VEC) Vec { float v[VEC]; };
    const float z = m.shared ? m.z[(size_t)t * m.ldz + m.z_col] : 0.f;
    const int* row_of = m.row_of + (size_t)t * top;
    const int wide = VEC == 4 ? ((m.ld + 255) & ~255) : m.ld;   // (whole waves: the sums cross lanes)
    for (int n = threadIdx.x * VEC; n < wide; n += 256 * VEC) {
        float sq = 0.f;
        if (n < m.ld) {
            Vec* xp = reinterpret_cast<Vec*>(m.x + (size_t)t * m.ld + n);
            Vec xv = *xp, y, sh;
            f4_t g = {0.f, 0.f, 0.f, 0.f};
            if (m.shared) sh = *reinterpret_cast<const Vec*>(m.shared + (size_t)t * m.ld + n);
            if (VEC == 4 && m.out_b16) g = *reinterpret_cast<const f4_t*>(m.gain + n);
#pragma unroll
            for (int e = 0; e < VEC; e++) y.v[e] = 0.f;
            for (int j = 0; j < top; j += 2) {
                const Vec r0 = *reinterpret_cast<const Vec*>(m.rows + (size_t)row_of[j] * m.ld + n);
                const Vec r1 = *reinterpret_cast<const Vec*>(m.rows + (size_t)row_of[min(j + 1, top - 1)] * m.ld + n);
#pragma unroll
                for (int e = 0; e < VEC; e++) {
                    y.v[e] += r0.v[e];
                    if (j + 1 < top) y.v[e] += r1.v[e];
                }
            }
            if (m.shared) {
                const float gate = 1.f / (1.f + expf(-z));
#pragma unroll
                for (int e = 0; e < VEC; e++) y.v[e] = fmaf(gate, sh.v[e], y.v[e]);
            }
#pragma unroll
            for (int e = 0; e < VEC; e++) {
                xv.v[e] += y.v[e];
                sq += xv.v[e] * xv.v[e];
            }
            *xp = xv;
            if (VEC == 4 && m.out_b16) {
                const float w[4] = {xv.v[0] * g[0], xv.v[1 % VEC] * g[1], xv.v[2 % VEC] * g[2], xv.v[3 % VEC] * g[3]};
                store_b16_4(m.out_b16, Kb, t, n, w);
            }
        }
        if (VEC == 4 && m.ss) {
            sq += __shfl_xor(sq, 1, 64);
            sq += __shfl_xor(sq, 2, 64);
            sq += __shfl_xor(sq, 4, 64);
            if ((threadIdx.x & 7) == 0 && n < m.ld) m.ss[(size_t)t * Kb + (n >> 5)] = sq;
        }
    }
}
void launch_moe_combine(const MoeCombine& m, int T) {
    if (T <= 0) return;
    if (m.out_b16 && m.ld % 32) NVLLM_FATAL("sum of experts: a row of %d is not padded to 32", m.ld);
    ProfScope ps(PC_MOE_COMBINE, (double)T * m.ld * (4.0 * m.top + (m.shared ? 4.0 : 0.0) + 8.0 + (m.out_b16 ? 2.0 : 0.0)), 0);
    if (m.ld % 4 == 0) NVLLM_LAUNCH((k_moe_combine<4>), dim3(T), dim3(256), 0, m, m.top);
    else NVLLM_LAUNCH((k_moe_combine<1>), dim3(T), dim3(256), 0, m, m.top);
}

}  // namespace nvllm
