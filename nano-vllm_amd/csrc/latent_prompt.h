// latent_prompt.h -- latent attention of prompt portions with keys and values of each head expanded from the cached latents.
#pragma once

#include <vector>

#include "latent_attention.h"

namespace nvllm {

// A pass's portions of several tokens, on the host, in items of up to LATENT_PROMPT_TOKENS tokens.
constexpr int LATENT_PROMPT_TOKENS = 64;
struct LatentPromptPlan {
    int n_items = 0, n_pairs = 0;   // pairs: of pool pages with the positions up to a portion's last
    int most_pairs = 0;      // of one portion
    int tokens = 0;          // tokens of the portions
    long pairs_qk = 0;       // (token, position) pairs
    // the 16-token blocks that hold the tokens which are their sequence's only ones (none: from == to)
    int alone_from = 0, alone_to = 0;
};
int latent_portion(const int* pos, const int* seq_ids, int T, int t);   // tokens of the portion that begins with token t
LatentPromptPlan latent_prompt_plan(const int* pos, const int* seq_ids, int T);
// What the kernels read: [n_items][4] (first token, count, position of the first, first pair), those that see most first, then
// [n_pairs][2] page ids; a multiple of four.
std::vector<int> latent_prompt_ints(const LatentPromptPlan& plan, const int* pos, const int* seq_ids, int T, BlockTable** tables, int block_size);

// Keys, values and unrotated queries are held in fp16: the caller sees to it that they fit (latent_model.hip, fp16_holds).
struct LatentPrompt {
    LatentPool pool;
    const __half* q_tiles;   // unrotated queries, bf16 activation tiles of [T, H * dim_ld]
    const __half* q_rows;    // [T][H][pool.row()]: the rotated parts at pool.rank_ld
    const float* sink;
    float scale;
    int H, dim_ld, vdim_ld;
    const __half *uk, *uv;   // tiles of [H * dim_ld, rank_ld] and [H * vdim_ld, rank_ld]
    __half* kv;              // latent_prompt_scratch()
    __half* out;             // activation tiles of [T, H * vdim_ld]
    const int *items, *pages;   // device copies of the plan
};
struct ExpandArgs {
    const __half* base;   // the pool
    const int* pages;     // [n_pairs][2]
    int n_pairs, per;     // pairs, and pairs of a workgroup
    int chunks, row_tiles;   // tiles of a page: of its latent, in all
    int H, dc, vt;        // tiles of 32 dims of a head's key; of 16 dims of its value
    const __half *uk, *uv;
    __half* kv;           // [pair][head][2 dc key tiles by page, vt value tiles]
};
// split for `wgs` workgroups, four pairs each at least (a wave's weights are as many bytes as two pairs)
ExpandArgs latent_expand_args(const LatentPrompt& a, const LatentPromptPlan& plan, int wgs);
// ... and its work, for kernel timing
void latent_expand_work(const LatentPrompt& a, const LatentPromptPlan& plan, double* bytes, double* flops);
// Whether there are kernels for rows and heads of these widths.
bool latent_prompt_fits(int rank_ld, int rot_ld, int dim_ld, int vdim_ld);
// Whether this is the way to go for the pass's portions.
bool latent_prompt_pays(const LatentPromptPlan& plan, int H, int rank_ld, int dim_ld, int vdim_ld);
// Memory for the portions' keys and values; null: none (the portions attend over latents).
__half* latent_prompt_scratch(const LatentPromptPlan& plan, int H, int dim_ld, int vdim_ld);
// The same beside the attention of the tokens that come alone, if that leaves enough of the chip.
struct LatentExpandRider {
    const LatentPrompt* prompt;
    const LatentPromptPlan* plan;
    bool rode = false;
};
// formed: the keys and values are there (LatentAttn::expand rode)
void launch_latent_prompt(const LatentPrompt& a, const LatentPromptPlan& plan, bool formed);

}  // namespace nvllm
