// prompt_attention.hip -- causal attention of prompt portions over fp16 pages, in the arithmetic of k_paged_attn16 (attention.hip):
// queries and weights of positions as fp16 hi + lo planes, 32-bit sums, scores' maxima and exponentials in the log2 domain.
//
// k_paged_attn16 meets 16 keys at a time with 16 (token, head) columns a wave: per page some 150 instructions for 16 products, in
// one dependent chain, and every page enters the CU once per 16 columns.  Here a workgroup has 64 columns (4 CT tokens x GT heads) and
// a wave 32 of them against half of each block of 64 keys, in v_mfma_f32_16x16x32_f16 (two 16-dim pieces of a page's keys, or
// two pages' values, are one operand as they lie).  Blocks travel to LDS by direct copies, RING - 1 ahead, once per workgroup.  A lane
// keeps its column's sums and results (values are the first operand), so in most blocks nothing crosses lanes; the two waves
// of a column group meet once at the end.  Three portions of 512 tokens behind 512, 32 heads on 4 of 64: 61.3 -> 28.1 us a layer, 9.7 GFLOP (twice that in
// the matrix cores for the planes).  Bound: issue of about 95 vector instructions, 16 of them exponentials, beside 32 products per 32 keys
// and 32 columns; the depth of the ring and a fourth workgroup a CU change nothing.  Of the way there: 37 as first written; references that
// rise at every new maximum, and maxima over all lanes for it, cost 5; walks of three workgroups of a CU that are all long or all short 4 (stage_step).
// Error against 64 bits (2-norm of the results, queries of size 1, 4 and 30; k_paged_attn16 in brackets, 1e-7): heads of 64 1.43, 3.48, 7.73 (1.47, 3.61,
// 8.01), of 32 1.35, 3.09, 6.29 (1.46, 3.58, 7.50), of 96 1.50, 3.43, 7.42 (1.56, 3.71, 8.07), of 128 1.39, 3.41, 7.56 (1.53, 3.93, 8.31); with both planes of a
// block's weights in one chain of sums 1.54 at 128 (which took 30.1 us for 16 heads where it now takes 31.6), with all products of a score in one chain
// too 1.60, 3.87, 8.70 at 64.
#include "prompt_attention.h"

#include "gemm_common.h"

namespace nvllm {

namespace {

typedef float pf4_t __attribute__((ext_vector_type(4)));
typedef float pf2_t __attribute__((ext_vector_type(2)));
typedef _Float16 ph8_t __attribute__((ext_vector_type(8)));
typedef _Float16 ph2_t __attribute__((ext_vector_type(2)));
typedef unsigned int pu2_t __attribute__((ext_vector_type(2)));
typedef unsigned int pu4_t __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) int* const_int_p;   // read-only for the whole launch: scalar loads

__device__ __forceinline__ float rows_sum(float x) {   // over lanes l, l^16, l^32, l^48
    x += __shfl_xor(x, 16, 64);
    return x + __shfl_xor(x, 32, 64);
}

__device__ __forceinline__ float max2(float a, float b) { return __builtin_elementwise_maximum(a, b); }   // (no quieting of operands: one instruction for three)
__device__ __forceinline__ float rows_max2(float x) {   // rows_max (attn_tile.h) the same way
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const float m = max2(__builtin_bit_cast(float, (unsigned)a[0]), __builtin_bit_cast(float, (unsigned)a[1]));
    const unsigned v = __builtin_bit_cast(unsigned, m);
    const auto b = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return max2(__builtin_bit_cast(float, (unsigned)b[0]), __builtin_bit_cast(float, (unsigned)b[1]));
}
// fp16(e - hi) of two values: the difference is exact, so it is rounded once.  `minus` is -1, hidden from the compiler, which would
// make a conversion and a subtraction of it where fma with conversions of either end is one instruction
__device__ __forceinline__ ph2_t rest_of(pf2_t e, ph2_t hi, float minus) {
    return ph2_t{(_Float16)fmaf((float)hi[0], minus, e[0]), (_Float16)fmaf((float)hi[1], minus, e[1])};
}

constexpr int KEYS = 64;   // of a block
constexpr float LAZY = 8.f;

template <int HD>
struct PromptWave {
    static constexpr int NC = HD / 16, PAGE = 64 * HD, BLOCK = 4 * PAGE;   // bytes: keys then values of 16 positions; of 64
    static constexpr int LDS_MERGE = 4 * (NC * 1024 + 128);
};

template <int HD, int RING>
__device__ __forceinline__ void prompt_item(const PromptAttnArgs& p, unsigned widx, unsigned char* lds) {
    using W = PromptWave<HD>;
    constexpr int NC = W::NC, COPIES = HD / 16;   // copies of a wave and block
    const AttnKArgs& a = p.k;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = lane & 15, g = lane >> 4;
    const int half = wave & 1, part = wave >> 1;   // columns 32 half .., keys 32 part .. of each block
    const unsigned NG = (unsigned)a.NG;
    const int hg = (int)(widx % NG), item = (int)(widx / NG);
    const const_int_p run = (const_int_p)(uintptr_t)(p.long_runs + item);
    const int t0 = run[0], ntok = run[1], last = run[2];
    const const_int_p table = (const_int_p)(uintptr_t)(a.tables + run[3]);
    const int h0 = hg * a.GT, kvh = (int)((unsigned)h0 / (unsigned)a.group);
    const int p0 = last - (ntok - 1), n_blocks = last / KEYS + 1, last_page = last >> 4;
    const __half* pk = reinterpret_cast<const __half*>(a.pool_k) + a.layer_off + lane * 8;
    const __half* pv = reinterpret_cast<const __half*>(a.pool_v) + a.layer_off + lane * 8;
    const unsigned lds0 = (unsigned)(size_t)(lds_void*)lds;
    // wave w brings page w of a block (past the last: the last again, masked)
    auto block_id = [&](int b) { return table[min(4 * b + wave, last_page)]; };
    auto issue = [&](int id, int buf) {
        const long off = kv16_page(id, kvh, a.KVH, HD);
        const unsigned dst = lds0 + (unsigned)(buf * W::BLOCK + wave * W::PAGE);
#pragma unroll
        for (int c = 0; c < HD / 32; c++) copy_tile_to_lds(pk + off + 512 * c, __builtin_amdgcn_readfirstlane(dst + 1024u * c));
#pragma unroll
        for (int c = 0; c < HD / 32; c++) copy_tile_to_lds(pv + off + 512 * c, __builtin_amdgcn_readfirstlane(dst + 32u * HD + 1024u * c));
    };
    // column x of group j: a token and a head; columns past the run's tokens repeat its last and are not stored
    const int ctok = x >> a.gt_shift, head = h0 + (x & (a.GT - 1)), CT = 16 >> a.gt_shift;
    int tok[2];
    ph8_t qh[2][HD / 32], ql[2][HD / 32];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        tok[j] = (2 * half + j) * CT + ctok;
        const float* qr = a.q + ((size_t)(t0 + min(tok[j], ntok - 1)) * a.H + head) * HD + 4 * g;
#pragma unroll
        for (int c = 0; c < HD / 32; c++)
#pragma unroll
            for (int i = 0; i < 2; i++) {   // dims 32 c + 16 i + 4 g .. + 3
                const float4 f = *reinterpret_cast<const float4*>(qr + 32 * c + 16 * i);
                const float fv[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float cl = fminf(fmaxf(fv[e], -65504.f), 65504.f);
                    const _Float16 hi = (_Float16)cl;
                    qh[j][c][4 * i + e] = hi;
                    ql[j][c][4 * i + e] = (_Float16)(cl - (float)hi);
                }
            }
    }
#pragma unroll
    for (int i = 0; i < RING - 1; i++)
        if (i < n_blocks) issue(block_id(i), i);
    int next_id = block_id(RING - 1), buf = 0;
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int c = 0; c < HD / 32; c++) asm volatile("" : "+v"(qh[j][c]), "+v"(ql[j][c]));   // here, not in the loop, whose only loads are the copies
    // results; those of the weights' lo plane apart where registers allow, else a block's of both planes added to the sums as one: either way one
    // rounding to the size of the sums per 32 keys
    constexpr int SUMS = HD < 128 ? 2 : 1;
    pf4_t acc[SUMS][2][NC];
#pragma unroll
    for (int k = 0; k < SUMS; k++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int n = 0; n < NC; n++) acc[k][j][n] = pf4_t{0.f, 0.f, 0.f, 0.f};
    float m[2] = {-INFINITY, -INFINITY}, nm[2] = {0.f, 0.f}, lsum[2] = {0.f, 0.f};   // reference (a maximum of products), minus that as an exponent, sum
    float limit[2] = {-INFINITY, -INFINITY};
    const float sl2 = a.scale * 1.44269504088896340736f;
    const int first_sees = p0 + 2 * half * CT;                                  // last position that the wave's first token sees
    const int wave_sees = 2 * half * CT < ntok ? min(first_sees + 2 * CT - 1, last) : -1;
    const int sees[2] = {p0 + tok[0], p0 + tok[1]};
    float minus = -1.f;
    asm("" : "+s"(minus));
    int v_at[NC];   // where a lane's piece of the values' tile n lies in a page (hidden: pieces of one page would be read together and moved apart)
#pragma unroll
    for (int n = 0; n < NC; n++) {
        v_at[n] = lane * 8 + 32 * HD + 512 * n;
        asm("" : "+v"(v_at[n]));
    }
    for (int b = 0; b < n_blocks; b++) {
        if (b + RING - 1 <= n_blocks) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RING - 2) * COPIES) : "memory");   // all later blocks are on their way
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();   // everybody's copies of block b; block b - 1 has been consumed
        asm volatile("" ::: "memory");
        const unsigned char* blk = lds + buf * W::BLOCK + 2 * part * W::PAGE;
        if (b + RING - 1 < n_blocks) {
            issue(next_id, buf == 0 ? RING - 1 : buf - 1);
            next_id = block_id(b + RING);
        }
        buf = buf + 1 == RING ? 0 : buf + 1;
        const int from = KEYS * b + 32 * part;
        if (from > wave_sees) continue;
        auto pair = [&](int at, int step) {   // 8 bytes there and `step` further on
            const pu2_t lo = *reinterpret_cast<const pu2_t*>(blk + at), hi = *reinterpret_cast<const pu2_t*>(blk + at + step);
            return __builtin_bit_cast(ph8_t, pu4_t{lo[0], lo[1], hi[0], hi[1]});
        };
        // scores: lane (column x) has keys from + 16 page + 4 g + r
        pf4_t s[2][2];   // [column group][page]
#pragma unroll
        for (int j = 0; j < 2; j++) s[j][0] = s[j][1] = pf4_t{0.f, 0.f, 0.f, 0.f};
        ph8_t k[HD / 32][2];
#pragma unroll
        for (int c = 0; c < HD / 32; c++)
#pragma unroll
            for (int page = 0; page < 2; page++) k[c][page] = pair(lane * 8 + page * W::PAGE + 1024 * c, 512);
        pf4_t s2[2][2];   // wide heads: a second chain
#pragma unroll
        for (int j = 0; j < 2; j++) s2[j][0] = s2[j][1] = pf4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int plane = 0; plane < 2; plane++)   // the small products first, so that they are not rounded to the size of the others
#pragma unroll
            for (int c = 0; c < HD / 32; c++)
#pragma unroll
                for (int page = 0; page < 2; page++)
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        pf4_t& sum = HD > 64 && (c & 1) ? s2[j][page] : s[j][page];
                        sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(k[c][page], plane ? qh[j][c] : ql[j][c], sum, 0, 0, 0);
                    }
        if constexpr (HD > 64)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int page = 0; page < 2; page++) s[j][page] += s2[j][page];
        if (from + 31 > first_sees) {   // some column does not see all of them
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int page = 0; page < 2; page++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (from + 16 * page + 4 * g + r > sees[j]) s[j][page][r] = -INFINITY;
        }
        float mx[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            mx[j] = max2(max2(s[j][0][0], s[j][0][1]), s[j][0][2]);
            mx[j] = max2(max2(mx[j], s[j][0][3]), s[j][1][0]);
            mx[j] = max2(max2(mx[j], s[j][1][1]), s[j][1][2]);
            mx[j] = max2(mx[j], s[j][1][3]);
        }
        // a column's reference rises when a product is more than 2^LAZY times as heavy as it: its weights then stay far inside fp16, and
        // after a portion's first blocks hardly any block does more than look (of its own lanes' products)
        if (__any(mx[0] > limit[0] || mx[1] > limit[1])) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const float mn = max2(m[j], rows_max2(mx[j]));
                if (mn != -INFINITY) {
                    const float alpha = __builtin_amdgcn_exp2f((m[j] - mn) * sl2);
                    lsum[j] *= alpha;
#pragma unroll
                    for (int k = 0; k < SUMS; k++)
#pragma unroll
                        for (int n = 0; n < NC; n++) acc[k][j][n] *= alpha;
                    m[j] = mn;
                    nm[j] = -mn * sl2;
                    limit[j] = mn + LAZY / sl2;
                }
            }
        }
        ph8_t ph[2], pl[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < 4; i++) {   // keys 4 g + 2 (i & 1), + 1 of page i >> 1
                pf2_t e;
#pragma unroll
                for (int r = 0; r < 2; r++) e[r] = __builtin_amdgcn_exp2f(fmaf(s[j][i >> 1][2 * (i & 1) + r], sl2, nm[j]));
                const ph2_t hi = __builtin_convertvector(e, ph2_t);
                const ph2_t lo = rest_of(e, hi, minus);
                sum += e[0] + e[1];
                ph[j][2 * i] = hi[0], ph[j][2 * i + 1] = hi[1];
                pl[j][2 * i] = lo[0], pl[j][2 * i + 1] = lo[1];
            }
            lsum[j] += sum;
        }
        // results, transposed: values x weights
#pragma unroll
        for (int n = 0; n < NC; n += 2) {
            ph8_t val[2];
#pragma unroll
            for (int i = 0; i < 2; i++) val[i] = pair(v_at[n + i], W::PAGE);
            if constexpr (SUMS == 2) {
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++) acc[0][j][n + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(val[i], ph[j], acc[0][j][n + i], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++) acc[1][j][n + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(val[i], pl[j], acc[1][j][n + i], 0, 0, 0);
            } else {
                pf4_t block[2][2];
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++) block[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(val[i], pl[j], pf4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++) block[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(val[i], ph[j], block[i][j], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++) acc[0][j][n + i] += block[i][j];
            }
        }
    }
    // the two waves of 32 columns: each leaves the other's 16 and finishes its own (group j = part)
#pragma unroll
    for (int j = 0; j < 2; j++) lsum[j] = rows_sum(lsum[j]);
    if constexpr (SUMS == 2)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int n = 0; n < NC; n++) acc[0][j][n] += acc[1][j][n];
    __syncthreads();
    auto area = [&](int w) { return lds + w * (NC * 1024 + 128); };
    {
        unsigned char* mine = area(wave);
        const bool second = part == 0;   // group that this wave leaves
#pragma unroll
        for (int n = 0; n < NC; n++) reinterpret_cast<pf4_t*>(mine)[n * 64 + lane] = second ? acc[0][1][n] : acc[0][0][n];
        if (g == 0) reinterpret_cast<pf2_t*>(mine + NC * 1024)[x] = second ? pf2_t{m[1], lsum[1]} : pf2_t{m[0], lsum[0]};
    }
    __syncthreads();
    const unsigned char* other = area(wave ^ 2);
    const pf2_t ml = reinterpret_cast<const pf2_t*>(other + NC * 1024)[x];
    const float my_m = part ? m[1] : m[0], my_l = part ? lsum[1] : lsum[0];
    const float M = fmaxf(my_m, ml[0]), f0 = __builtin_amdgcn_exp2f((my_m - M) * sl2), f1 = __builtin_amdgcn_exp2f((ml[0] - M) * sl2);
    const float inv = 1.0f / fmaf(my_l, f0, ml[1] * f1);
    const int token = part ? tok[1] : tok[0], t = t0 + token;
    const bool store = token < ntok;
    pf4_t o[NC];
#pragma unroll
    for (int n = 0; n < NC; n++) {
        const pf4_t mine = part ? acc[0][1][n] : acc[0][0][n], his = reinterpret_cast<const pf4_t*>(other)[n * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; e++) o[n][e] = fmaf(his[e], f1, mine[e] * f0) * inv;
        if (store && a.out_f32) *reinterpret_cast<pf4_t*>(a.out_f32 + ((size_t)t * a.H + head) * HD + 16 * n + 4 * g) = o[n];
    }
    if (!a.out_a16) return;
#pragma unroll
    for (int n = 0; n < NC; n += 2) {
        unsigned hi[2][2], lo[2][2];
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const pf2_t c = {fminf(fmaxf(o[n + i][2 * e], -65504.f), 65504.f), fminf(fmaxf(o[n + i][2 * e + 1], -65504.f), 65504.f)};
                const ph2_t h = __builtin_convertvector(c, ph2_t);
                hi[i][e] = __builtin_bit_cast(unsigned, h);
                lo[i][e] = __builtin_bit_cast(unsigned, rest_of(c, h, minus));
            }
        // rows of lanes (g) 2i and 2i + 1 hold neighbouring fours of dims of tiles n and n + 1: after the swap the even row has
        // eight of n, the odd row eight of n + 1
        pu4_t vh, vl;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const auto sh = __builtin_amdgcn_permlane16_swap(hi[0][e], hi[1][e], false, false);
            const auto sl = __builtin_amdgcn_permlane16_swap(lo[0][e], lo[1][e], false, false);
            vh[e] = sh[0], vh[2 + e] = sh[1];
            vl[e] = sl[0], vl[2 + e] = sl[1];
        }
        if (!store) continue;
        const int kk = head * HD + 16 * (n + (g & 1)) + 8 * (g >> 1);
        const size_t tl = ((size_t)(t >> 4) * a.Kb_out + (kk >> 5)) * 2;
        const size_t off = (size_t)((t & 15) + 16 * ((kk >> 3) & 3)) * 8;
        *reinterpret_cast<pu4_t*>(a.out_a16 + tl * TILE_HALVES + off) = vh;
        *reinterpret_cast<pu4_t*>(a.out_a16 + (tl + 1) * TILE_HALVES + off) = vl;
    }
}

// Portions' items first; then, in the same launch, what is left of the batch (single tokens, ends of portions) as k_paged_attn16 does it
template <int HD, int RING>
__global__ __launch_bounds__(256, HD <= 64 ? 3 : 2) void k_prompt_attn16(PromptAttnArgs p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_attn[];
    const unsigned n = (unsigned)p.n_long * (unsigned)p.k.NG;
    if (blockIdx.x < n) {
        prompt_item<HD, RING>(p, blockIdx.x, lds_attn);
        return;
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    Attn16Wave<HD, 2, 4, false> w;
    w.setup(p.k, blockIdx.x - n, wave, threadIdx.x & 63, 0);
    w.load_q();
    w.start();
    w.loop();
    w.deposit(lds_attn, wave);
    __syncthreads();
    w.merge(lds_attn, wave);
}

template <int HD, int RING>
void launch(const PromptAttnArgs& a) {
    constexpr int lds = RING * PromptWave<HD>::BLOCK;
    static_assert(lds >= attn16_lds<HD>() && lds >= PromptWave<HD>::LDS_MERGE && RING >= 2);
    NVLLM_LAUNCH((k_prompt_attn16<HD, RING>), dim3((unsigned)((a.n_long + a.k.n_runs) * a.k.NG)), dim3(256), lds, a);
}

}  // namespace

void launch_prompt_attn16(const PromptAttnArgs& a, int hd) {
    switch (hd) {
        case 32: launch<32, 3>(a); break;
        case 64: launch<64, 3>(a); break;
        case 96: launch<96, 2>(a); break;
        case 128: launch<128, 2>(a); break;
        default: NVLLM_FATAL("no prompt attention for heads of %d", hd);
    }
}

}  // namespace nvllm
