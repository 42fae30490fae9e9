// row_attention.hip -- attention of single tokens over fp32 rows where a key/value head serves one or two query heads.
//
// k_paged_attn multiplies 16 (token, head) columns at a time in v_mfma_f32_16x16x4_f32, of which such a token fills one or two: 1,024
// matrix-core cycles a page for what the vector unit does in 250, and a page's 16 keys are one dependent chain.  Here a workgroup has a
// (token, key/value head), LPK lanes a key, four dims each; its waves deal the keys among themselves 64 / LPK at a time and request
// AHEAD such groups together, so a context of a few hundred tokens is one trip to memory.  Every group of lanes keeps a maximum, sums
// and results of its own: nothing but scores crosses its lanes; groups and waves meet once at the end.
// stories42M, 32 rows of 220 cached positions: 11.2 -> 7.4 us a layer; stories15M, one row of 240: 8.6 -> 5.0 (rows_alone() has both sides).  Bound: the
// chain of run, table, rows and the merge, of about a microsecond a step.  fp32 throughout, fused multiply-adds, scale after the dot product, expf.
#include "attn_tile.h"

namespace nvllm {

namespace {

typedef const __attribute__((address_space(4))) int* const_int_p;   // read-only for the whole launch: scalar loads

constexpr int ROW_WAVES = 8;

template <int HD, int G>
__global__ __launch_bounds__(64 * ROW_WAVES) void k_row_attn(AttnKArgs a) {
    request_arguments<sizeof(AttnKArgs)>();
    constexpr int LPK = row_attn_lanes(HD), KEYS = 64 / LPK, AHEAD = 8;
    static_assert(KEYS * ROW_WAVES * AHEAD == row_attn_keys(HD));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = lane & (LPK - 1), kg = lane / LPK;   // this lane's four dims, its key of a group
    const bool live = 4 * x < HD;
    const int d = live ? 4 * x : 0;
    const int kvh = (int)(blockIdx.x % (unsigned)a.KVH);
    const const_int_p run = (const_int_p)(uintptr_t)(a.runs + blockIdx.x / (unsigned)a.KVH);
    const int t = run[0], last = run[2];
    const const_int_p table = (const_int_p)(uintptr_t)(a.tables + run[3]);
    const int sh = a.bs_shift, groups = last / KEYS + 1;   // groups of keys; the last may go past the token
    const float* pk = reinterpret_cast<const float*>(a.pool_k) + a.layer_off + (size_t)kvh * HD + d;
    const float* pv = reinterpret_cast<const float*>(a.pool_v) + a.layer_off + (size_t)kvh * HD + d;
    af4_t q[G], o[G];
    float m[G], l[G];
#pragma unroll
    for (int h = 0; h < G; h++) {
        q[h] = *reinterpret_cast<const af4_t*>(a.q + ((size_t)t * a.H + kvh * G + h) * HD + d);
        o[h] = af4_t{0.f, 0.f, 0.f, 0.f};
        m[h] = -INFINITY, l[h] = 0.f;
    }
    for (int g0 = wave; g0 < groups; g0 += ROW_WAVES * AHEAD) {
        af4_t k[AHEAD], v[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {   // (groups past the last: the last again, not counted)
            const int grp = min(g0 + ROW_WAVES * u, groups - 1), page = grp * KEYS >> 4;
            const long row0 = ((long)table[page >> sh] << (4 + sh)) + ((page & ((1 << sh) - 1)) << 4) + ((grp * KEYS) & 15);
            const int over = max(grp * KEYS + kg - last, 0);   // keys past the token: its own row again (written, finite)
            const long at = (row0 + kg - over) * a.rowstride;
            k[u] = *reinterpret_cast<const af4_t*>(pk + at);
            v[u] = *reinterpret_cast<const af4_t*>(pv + at);
        }
#pragma unroll
        for (int h = 0; h < G; h++) {
            if (!live) q[h] = af4_t{0.f, 0.f, 0.f, 0.f};
            float dot[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; u++) {
                dot[u] = q[h][0] * k[u][0];
#pragma unroll
                for (int e = 1; e < 4; e++) dot[u] = fmaf(q[h][e], k[u][e], dot[u]);
            }
            float s = eight_sums<LPK>(dot, x) * a.scale;   // of key number x & 7
            const int grp = g0 + ROW_WAVES * (x & 7);
            if (grp * KEYS + kg > last) s = -INFINITY;
            const float top = fmaxf(m[h], eight_max<LPK>(s)), base = fmaxf(top, -3.0e38f);   // (a group of lanes that has seen no key: exp(-inf - finite) = 0)
            const float alpha = expf(m[h] - base), p = expf(s - base);
            l[h] = fmaf(l[h], alpha, p);
            o[h] *= alpha;
            m[h] = top;
            add_eight<LPK>(o[h], p, v, lane);
        }
    }
#pragma unroll
    for (int h = 0; h < G; h++) {   // (lanes x and x + 8 hold the same)
        l[h] += lane_moved<0xB1>(l[h]);
        l[h] += lane_moved<0x4E>(l[h]);
        l[h] += LPK == 8 ? __shfl_xor(l[h], 4, 64) : lane_moved<0x124>(l[h]);
    }
    // the groups of lanes of all waves meet
    __shared__ float s_m[G][ROW_WAVES * KEYS], s_l[G][ROW_WAVES * KEYS];
    __shared__ af4_t s_o[G][ROW_WAVES * KEYS][LPK];
#pragma unroll
    for (int h = 0; h < G; h++) {
        if (x == 0) s_m[h][wave * KEYS + kg] = m[h], s_l[h][wave * KEYS + kg] = l[h];
        s_o[h][wave * KEYS + kg][x] = o[h];
    }
    __syncthreads();
    if (wave >= G) return;
    // wave h finishes head h: lane (kg, x) adds every KEYS-th part, then the groups of lanes meet
    const int h = wave;
    float M = -INFINITY;
#pragma unroll
    for (int i = 0; i < ROW_WAVES * KEYS; i++) M = fmaxf(M, s_m[h][i]);
    float L = 0.f;
    af4_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < ROW_WAVES; i++) {
        const float f = expf(s_m[h][i * KEYS + kg] - M);   // parts without keys carry -inf: weight 0
        L = fmaf(s_l[h][i * KEYS + kg], f, L);
        const af4_t part = s_o[h][i * KEYS + kg][x];
#pragma unroll
        for (int e = 0; e < 4; e++) sum[e] = fmaf(part[e], f, sum[e]);
    }
#pragma unroll
    for (int w = LPK; w < 64; w <<= 1) {
        L += __shfl_xor(L, w, 64);
#pragma unroll
        for (int e = 0; e < 4; e++) sum[e] += __shfl_xor(sum[e], w, 64);
    }
    if (kg != 0 || !live) return;
    sum *= 1.0f / L;
    const int head = kvh * G + h;
    if (a.out_f32) *reinterpret_cast<af4_t*>(a.out_f32 + ((size_t)t * a.H + head) * HD + d) = sum;
    if (a.out_a16) {
        const int kk = head * HD + d;
        alignas(8) __half hi[4], lo[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float xv = fminf(fmaxf(sum[e], -65504.f), 65504.f);
            hi[e] = __float2half_rn(xv);
            lo[e] = __float2half_rn(xv - __half2float(hi[e]));
        }
        const size_t tl = ((size_t)(t >> 4) * a.Kb_out + (kk >> 5)) * 2;
        const size_t off = (size_t)((t & 15) + 16 * ((kk >> 3) & 3)) * 8 + (kk & 7);
        *reinterpret_cast<uint2*>(a.out_a16 + tl * TILE_HALVES + off) = *reinterpret_cast<const uint2*>(hi);
        *reinterpret_cast<uint2*>(a.out_a16 + (tl + 1) * TILE_HALVES + off) = *reinterpret_cast<const uint2*>(lo);
    }
}

template <int HD>
void launch(const AttnKArgs& k) {
    const dim3 grid((unsigned)(k.n_runs * k.KVH)), block(64 * ROW_WAVES);
    if (k.group == 1) NVLLM_LAUNCH((k_row_attn<HD, 1>), grid, block, 0, k);
    else NVLLM_LAUNCH((k_row_attn<HD, 2>), grid, block, 0, k);
}

}  // namespace

void launch_row_attn(const AttnKArgs& k, int hd) {
    switch (hd) {
        case 16: launch<16>(k); break;
        case 32: launch<32>(k); break;
        case 48: launch<48>(k); break;
        case 64: launch<64>(k); break;
        case 80: launch<80>(k); break;
        case 96: launch<96>(k); break;
        case 128: launch<128>(k); break;
        default: NVLLM_FATAL("no row attention for heads of %d", hd);
    }
}

}  // namespace nvllm
