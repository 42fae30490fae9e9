// latent_prompt.hip -- latent attention of prompt portions (latent_prompt.h).
//
// A token that attends over latents as they lie multiplies rank + rot values per key and head and adds up rank of them; with
// keys W_uk c and values W_uv c formed first it is dim + rot and vdim (64 + 64 and 64 instead of 512 + 64 and 512), and
// the queries need no product with W_uk, the results none with W_uv.  Forming them costs rank * (dim + vdim) products per
// position and head, shared by all tokens of the portion: it pays from about seventy tokens on.
//
// k_latent_expand   a wave owns 32 features of [all heads' keys; all heads' values], whose weights (32 x rank) stay in its
//                   registers, and multiplies page after page: two pages of 16 positions travel to LDS by direct copies, one pair
//                   ahead, for the eight waves of the workgroup.  Keys are formed as W x latent (a lane holds four dims of a position),
//                   values as latent x W^T (four positions of a dim), which are the orders the attention's operands lie in.
// k_latent_prompt   64 tokens x one head; the four waves have 16 tokens each and walk the keys in blocks of 64 that
//                   travel to LDS one block ahead.  Scores, maxima and sums are fp32; the weights of two pages are the next
//                   product's operand as they lie in the score registers.
// Keys, values and weights of positions are fp16 (the caller sees to their range, LatentPrompt): attention over latents rounds nothing
// key by key, and with bf16 here the logits were further off in 64 bits than its (root of the mean square over eight and six seeds,
// prompts beside rows: Suselorn-1.2B 0.0104 and 0.0100, -0.4B 0.0064 and 0.0060; in fp16 0.0090 and 0.0056, at the same speed).
// Bounds: the expansion its 32 KiB per pair into and 4 KiB per wave out of a CU; attention the issue of about 110 vector
// instructions per 64 keys and 16 tokens beside 24 products.
#include "latent_prompt.h"

#include <algorithm>
#include <array>
#include <climits>

#include "latent_expand.h"

namespace nvllm {

namespace {

struct PromptArgs {
    const __half* base;
    const int *items, *pages;
    const __half *q_tiles, *q_rows, *kv;
    const float* sink;
    float scale;
    int H;
    int q_kb;                 // tiles of a token block of q_tiles
    int row, rank_ld;
    __half* out;
    int Kb_out;
};

// DC, RC: chunks of 32 dims of a head's key, unrotated and rotated; VT: tiles of 16 dims of its value
template <int DC, int RC, int VT, int RING>
__global__ __launch_bounds__(256, 2) void k_latent_prompt(PromptArgs a) {
    constexpr int TILES = 4 * DC + 4 * RC + 2 * VT;   // of a block of 64 keys: keys by page, rotated parts by page, values by pair
    constexpr int COPIES = DC + RC + VT / 2;          // of a wave
    extern __shared__ __attribute__((aligned(16))) __half lds_prompt[];   // [RING][TILES] tiles
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = lane & 15, g = lane >> 4;
    // heads fastest: a head's items meet behind one L2 wherever the number of heads is a multiple of the eight XCDs
    const int h = (int)(blockIdx.x % (unsigned)a.H), item = (int)(blockIdx.x / (unsigned)a.H);
    const const_int_p it = (const_int_p)(uintptr_t)(a.items + 4 * item), pages = (const_int_p)(uintptr_t)a.pages;
    const int t0 = it[0], ntok = it[1], p0 = it[2], pair0 = it[3];
    const int last = p0 + ntok - 1, n_blocks = (last >> 6) + 1, last_pair = last >> 5;
    const int tok = 16 * wave + x, t = t0 + min(tok, ntok - 1);
    const int sees = tok < ntok ? p0 + tok : -1;                                  // last position of this lane's column
    const int wave_sees = 16 * wave < ntok ? min(p0 + 16 * wave + 15, last) : -1;   // ... of the wave's last column
    constexpr size_t HEAD = (size_t)(2 * DC + VT) * TILE_HALVES;
    const unsigned lds0 = (unsigned)(size_t)(lds_void*)lds_prompt;
    // wave w brings page w of a block: its key tiles, its rotated part, and every second value tile of its pair
    auto pair_of = [&](int b) { return pair0 + min(2 * b + (wave >> 1), last_pair); };   // (past the last: the last again, masked)
    auto issue = [&](int page_id, int b, int buf) {
        const unsigned dst = lds0 + (unsigned)(buf * TILES) * 1024u;
        const __half* own = a.kv + ((size_t)pair_of(b) * a.H + h) * HEAD + lane * 8;
        const __half* rot = a.base + ((size_t)page_id * 16 * a.row + (size_t)a.rank_ld * 16) + lane * 8;
#pragma unroll
        for (int c = 0; c < DC; c++)
            copy_tile_to_lds(own + (size_t)((wave & 1) * DC + c) * TILE_HALVES, __builtin_amdgcn_readfirstlane(dst + (unsigned)(wave * DC + c) * 1024u));
#pragma unroll
        for (int c = 0; c < RC; c++)
            copy_tile_to_lds(rot + (size_t)c * TILE_HALVES, __builtin_amdgcn_readfirstlane(dst + (unsigned)(4 * DC + wave * RC + c) * 1024u));
#pragma unroll
        for (int n = 0; n < VT / 2; n++)
            copy_tile_to_lds(own + (size_t)(2 * DC + 2 * n + (wave & 1)) * TILE_HALVES,
                             __builtin_amdgcn_readfirstlane(dst + (unsigned)(4 * DC + 4 * RC + (wave >> 1) * VT + 2 * n + (wave & 1)) * 1024u));
    };
    auto page_of = [&](int b) { return pages[2 * pair_of(b) + (wave & 1)]; };
    // queries as the second operand: column x, dims 32 c + 8 g .. + 7
    b8_t q[DC + RC];   // (the first DC as fp16 bits)
#pragma unroll
    for (int c = 0; c < DC; c++)
        q[c] = *reinterpret_cast<const b8_t*>(a.q_tiles + ((size_t)(t >> 4) * a.q_kb + h * DC + c) * TILE_HALVES + ((t & 15) + 16 * g) * 8);
#pragma unroll
    for (int c = 0; c < RC; c++) q[DC + c] = *reinterpret_cast<const b8_t*>(a.q_rows + ((size_t)t * a.H + h) * a.row + a.rank_ld + 32 * c + 8 * g);
#pragma unroll
    for (int i = 0; i < RING - 1; i++)
        if (i < n_blocks) issue(page_of(i), i, i);
    int next_page = page_of(RING - 1), buf = 0;
#pragma unroll
    for (int c = 0; c < DC; c++) q[c] = __builtin_bit_cast(b8_t, __builtin_convertvector(__builtin_convertvector(q[c], f8_t), h8_t));
#pragma unroll
    for (int c = 0; c < DC + RC; c++) asm volatile("" : "+v"(q[c]));   // here, not in the loop, whose only loads are the copies
    f4_t acc[VT];
#pragma unroll
    for (int n = 0; n < VT; n++) acc[n] = f4_t{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, lsum = 0.f;
    const float sl2 = a.scale * 1.44269504088896340736f;   // scores in the log2 domain
    for (int b = 0; b < n_blocks; b++) {
        if (b + RING - 1 <= n_blocks) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RING - 2) * COPIES) : "memory");   // all later blocks are on their way
        else copies_landed();
        prompt_barrier();   // everybody's copies of block b; block b - 1 has been consumed
        const b8_t* blk = reinterpret_cast<const b8_t*>(lds_prompt) + (size_t)buf * TILES * 64 + lane;
        if (b + RING - 1 < n_blocks) {
            issue(next_page, b + RING - 1, buf == 0 ? RING - 1 : buf - 1);
            next_page = page_of(b + RING);
        }
        buf = buf + 1 == RING ? 0 : buf + 1;
        if (64 * b > wave_sees) continue;
        f4_t s[4];
#pragma unroll
        for (int page = 0; page < 4; page++) {
            s[page] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < DC; c++)
                s[page] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, blk[(page * DC + c) * 64]), __builtin_bit_cast(h8_t, q[c]), s[page], 0, 0, 0);
#pragma unroll
            for (int c = 0; c < RC; c++) s[page] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(blk[(4 * DC + page * RC + c) * 64], q[DC + c], s[page], 0, 0, 0);
        }
        // lane (column x): keys 64 b + 16 page + 4 g + r
        if (64 * b + 63 > p0 + 16 * wave || 16 * wave + 15 >= ntok) {   // some column does not see all of them
            const int from = 64 * b + 4 * g;
#pragma unroll
            for (int page = 0; page < 4; page++)
#pragma unroll
                for (int r = 0; r < 4; r++) s[page][r] = from + 16 * page + r <= sees ? s[page][r] * sl2 : -INFINITY;
        } else {
#pragma unroll
            for (int page = 0; page < 4; page++) s[page] *= sl2;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int page = 0; page < 4; page++) mx = fmaxf(mx, fmaxf(fmaxf(s[page][0], s[page][1]), fmaxf(s[page][2], s[page][3])));
        mx = rows_max(mx);
        if (__any(mx > m)) {   // some column's maximum rises
            const float mn = fmaxf(m, mx), alpha = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - mn);
            lsum *= alpha;
#pragma unroll
            for (int n = 0; n < VT; n++) acc[n] *= alpha;
            m = mn;
        }
        const float msafe = fmaxf(m, -1.0e30f);   // nothing visible: exp2(-inf - finite) = 0, no NaN
        h8_t p[2];
#pragma unroll
        for (int pair = 0; pair < 2; pair++) {
            f8_t e;
#pragma unroll
            for (int r = 0; r < 8; r++) {
                e[r] = __builtin_amdgcn_exp2f(s[2 * pair + (r >> 2)][r & 3] - msafe);
                lsum += e[r];
            }
            p[pair] = __builtin_convertvector(e, h8_t);
        }
#pragma unroll
        for (int pair = 0; pair < 2; pair++)
#pragma unroll
            for (int n = 0; n < VT; n++)
                acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, blk[(4 * DC + 4 * RC + pair * VT + n) * 64]), p[pair], acc[n], 0, 0, 0);
    }
    lsum += __shfl_xor(lsum, 16, 64);
    lsum += __shfl_xor(lsum, 32, 64);
    if (tok >= ntok) return;
    const float sk = a.sink[h] * 1.44269504088896340736f, top = fmaxf(m, sk);
    const float w = __builtin_amdgcn_exp2f(m - top), f = w / fmaf(lsum, w, __builtin_amdgcn_exp2f(sk - top));
#pragma unroll
    for (int n = 0; n < VT; n++) {
        const float o[4] = {acc[n][0] * f, acc[n][1] * f, acc[n][2] * f, acc[n][3] * f};
        store_b16_4(a.out, a.Kb_out, t, h * VT * 16 + 16 * n + 4 * g, o);
    }
}

template <int DC, int RC, int VT>
void launch_prompt(const PromptArgs& k, int workgroups) {
    constexpr int TILES = 4 * DC + 4 * RC + 2 * VT, RING = TILES <= 26 ? 3 : 2;   // (two workgroups a CU)
    constexpr int lds = RING * TILES * 1024;
    static bool enabled = false;
    if (lds > 64 * 1024 && !enabled) {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_latent_prompt<DC, RC, VT, RING>), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        enabled = true;
    }
    NVLLM_LAUNCH((k_latent_prompt<DC, RC, VT, RING>), dim3(workgroups), dim3(256), lds, k);
}
template <int KC>
__global__ __launch_bounds__(512, 2) void k_latent_expand(ExpandArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_expand[];
    latent_expand<KC>(a, (int)blockIdx.x, (int)blockIdx.y, lds_expand);
}
template <int KC>
void launch_expand(const ExpandArgs& e, dim3 grid) {
    const int lds = (int)expand_lds(e);
    static bool enabled = false;
    if (!enabled) {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_latent_expand<KC>), hipFuncAttributeMaxDynamicSharedMemorySize, 4 * KC * 1024));
        enabled = true;
    }
    NVLLM_LAUNCH((k_latent_expand<KC>), grid, dim3(512), lds, e);
}

}  // namespace

int latent_portion(const int* pos, const int* seq_ids, int T, int t) {
    int n = 1;
    while (t + n < T && seq_ids[t + n] == seq_ids[t] && pos[t + n] == pos[t + n - 1] + 1) n++;
    return n;
}

LatentPromptPlan latent_prompt_plan(const int* pos, const int* seq_ids, int T) {
    LatentPromptPlan p;
    int alone_last = -1;
    long n_pairs = 0;
    for (int t = 0, n; t < T; t += n) {
        n = latent_portion(pos, seq_ids, T, t);
        if (n == 1) {
            if (alone_last < 0) p.alone_from = t / 16;
            alone_last = t;
            continue;
        }
        const int pairs = pos[t + n - 1] / 32 + 1;
        n_pairs += pairs;
        p.most_pairs = std::max(p.most_pairs, pairs);
        p.n_items += cdiv(n, LATENT_PROMPT_TOKENS);
        p.tokens += n;
        p.pairs_qk += (long)n * pos[t] + (long)n * (n + 1) / 2;
    }
    if (alone_last >= 0) p.alone_to = alone_last / 16 + 1;
    p.n_pairs = (int)n_pairs;
    if (n_pairs > INT_MAX / 32) p.n_items = 0;   // (no pool is as large)
    return p;
}

std::vector<int> latent_prompt_ints(const LatentPromptPlan& plan, const int* pos, const int* seq_ids, int T, BlockTable** tables, int block_size) {
    std::vector<std::array<int, 4>> items;
    std::vector<int> pages, ints;
    const int per_block = block_size / LATENT_PAGE;
    pages.reserve(2 * (size_t)plan.n_pairs);
    for (int t = 0, n; t < T; t += n) {
        n = latent_portion(pos, seq_ids, T, t);
        if (n == 1) continue;
        const BlockTable* table = tables[seq_ids[t]];
        const int last = pos[t + n - 1], first_pair = (int)pages.size() / 2;
        for (int q = 0; q < 2 * (last / 32 + 1); q++) {
            const int page = std::min(q, last / LATENT_PAGE), block = std::min(page / per_block, table->num_blocks - 1);   // (a short table ends the pass later)
            pages.push_back(block < 0 ? 0 : table->block_indices[block] * per_block + page % per_block);
        }
        for (int i = 0; i < n; i += LATENT_PROMPT_TOKENS) items.push_back({t + i, std::min(LATENT_PROMPT_TOKENS, n - i), pos[t] + i, first_pair});
    }
    std::stable_sort(items.begin(), items.end(), [](const auto& a, const auto& b) { return a[2] + a[1] > b[2] + b[1]; });
    for (const auto& i : items) ints.insert(ints.end(), i.begin(), i.end());
    ints.insert(ints.end(), pages.begin(), pages.end());
    while (ints.size() % 4) ints.push_back(0);
    return ints;
}

bool latent_prompt_fits(int rank_ld, int rot_ld, int dim_ld, int vdim_ld) {
    auto one_of = [](int v, int a, int b, int c) { return v == a || v == b || v == c; };
    return rank_ld <= 512 && one_of(dim_ld, 32, 64, 128) && (rot_ld == 32 || rot_ld == 64) && one_of(vdim_ld, 32, 64, 128);
}

constexpr double EXPAND_BYTES = 512e6;   // of keys and values at most
bool latent_prompt_pays(const LatentPromptPlan& plan, int H, int rank_ld, int dim_ld, int vdim_ld) {
    static const int env = getenv("NVLLM_LATENT_EXPAND") ? atoi(getenv("NVLLM_LATENT_EXPAND")) : -1;   // 0: never, 1: wherever it can be done
    const double positions = 32.0 * plan.n_pairs;
    if (env == 0 || plan.n_items == 0 || positions * H * (dim_ld + vdim_ld) * 2.0 > EXPAND_BYTES) return false;
    if (env > 0) return true;
    // us a layer, fitted to portions of 17 to 256 tokens at 0, 512 and 1,700 cached positions, alone and beside five single tokens,
    // of 32 heads with 512 latent values and 16 with 256: two launches less, unless single tokens beside the portions want
    // theirs as before; the walk of 64 keys after 64 keys, which few items do not hide; forming keys and values; and the products
    // saved per pair of token and position.  96 tokens behind 512, 32 heads: 107 us a layer -> 91, beside five tokens 126 -> 118;
    // 64 behind 1,700 93 -> 92; 17 behind 1,700 83 -> 89, not taken.  Passes of few columns (less than a thousand) gain the launches alone.
    if ((long)plan.tokens * H < 1024) return false;
    const double forming = 0.35 * plan.most_pairs / 2 + positions * H * (dim_ld + vdim_ld) * rank_ld / 4e8;
    const double launches = plan.alone_to > plan.alone_from ? 0.0 : 8.0;
    const double saved = plan.pairs_qk * (double)H * (2 * rank_ld - dim_ld - vdim_ld) / 2e8;
    return forming < launches + saved;
}

__half* latent_prompt_scratch(const LatentPromptPlan& plan, int H, int dim_ld, int vdim_ld) {
    static const double most = getenv("NVLLM_LATENT_EXPAND_BYTES") ? atof(getenv("NVLLM_LATENT_EXPAND_BYTES")) : EXPAND_BYTES;
    const size_t bytes = (size_t)plan.n_pairs * H * 32 * (dim_ld + vdim_ld) * sizeof(__half);
    return (double)bytes <= most ? (__half*)ws_try(WS_EXPANDED, bytes) : nullptr;
}

ExpandArgs latent_expand_args(const LatentPrompt& a, const LatentPromptPlan& plan, int wgs) {
    const LatentPool& P = a.pool;
    ExpandArgs e{};
    e.base = (const __half*)P.base;
    e.pages = a.pages;
    e.n_pairs = plan.n_pairs;
    e.chunks = P.rank_ld / 32;
    e.row_tiles = P.row() / 32;
    e.H = a.H;
    e.dc = a.dim_ld / 32;
    e.vt = a.vdim_ld / 16;
    e.uk = a.uk;
    e.uv = a.uv;
    e.kv = a.kv;
    e.per = std::max(4, cdiv(plan.n_pairs, std::max(1, wgs / expand_cols(e))));
    return e;
}

void latent_expand_work(const LatentPrompt& a, const LatentPromptPlan& plan, double* bytes, double* flops) {
    const double positions = 32.0 * plan.n_pairs, width = (double)a.H * (a.dim_ld + a.vdim_ld), rank = a.pool.rank_ld;
    *bytes = width * rank * 2.0 + positions * rank * 2.0 + positions * width * 2.0;
    *flops = 2.0 * positions * width * rank;
}

void launch_latent_prompt(const LatentPrompt& a, const LatentPromptPlan& plan, bool formed) {
    if (plan.n_items <= 0) return;
    const LatentPool& P = a.pool;
    const double positions = 32.0 * plan.n_pairs, width = (double)a.H * (a.dim_ld + a.vdim_ld);
    if (!formed) {
        const ExpandArgs e = latent_expand_args(a, plan, rt().num_cus);
        double bytes, flops;
        latent_expand_work(a, plan, &bytes, &flops);
        ProfScope ps(PC_LATENT_EXPAND, bytes, flops);
        const dim3 grid(expand_cols(e), cdiv(plan.n_pairs, e.per));
        if (e.chunks <= 8) launch_expand<8>(e, grid);
        else launch_expand<16>(e, grid);
    }
    PromptArgs k{};
    k.base = (const __half*)P.base;
    k.items = a.items;
    k.pages = a.pages;
    k.q_tiles = a.q_tiles;
    k.q_rows = a.q_rows;
    k.kv = a.kv;
    k.sink = a.sink;
    k.scale = a.scale;
    k.H = a.H;
    k.q_kb = a.H * a.dim_ld / 32;
    k.row = P.row();
    k.rank_ld = P.rank_ld;
    k.out = a.out;
    k.Kb_out = a.H * a.vdim_ld / 32;
    ProfScope ps(PC_LATENT_ATTN, positions * (width + P.rot_ld) * 2.0 + (double)plan.tokens * a.H * (a.dim_ld + P.rot_ld + a.vdim_ld) * 2.0,
                 2.0 * (double)plan.pairs_qk * a.H * (a.dim_ld + P.rot_ld + a.vdim_ld));
    auto values = [&](auto dc, auto rc) {
        constexpr int DC = decltype(dc)::value, RC = decltype(rc)::value;
        if (a.vdim_ld == 32) launch_prompt<DC, RC, 2>(k, plan.n_items * a.H);
        else if (a.vdim_ld == 64) launch_prompt<DC, RC, 4>(k, plan.n_items * a.H);
        else launch_prompt<DC, RC, 8>(k, plan.n_items * a.H);
    };
    auto rotated = [&](auto dc) {
        if (P.rot_ld == 32) values(dc, std::integral_constant<int, 1>{});
        else values(dc, std::integral_constant<int, 2>{});
    };
    if (a.dim_ld == 32) rotated(std::integral_constant<int, 1>{});
    else if (a.dim_ld == 64) rotated(std::integral_constant<int, 2>{});
    else rotated(std::integral_constant<int, 4>{});
}

}  // namespace nvllm
