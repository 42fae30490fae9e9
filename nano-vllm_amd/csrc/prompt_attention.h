// prompt_attention.h -- attention of prompt portions over fp16 pages (prompt_attention.hip).
#pragma once

#include "attn_tile.h"

namespace nvllm {

// `long_runs` int4 (first token, token count, last position, table offset), at most attn_long_runs().tokens tokens each, one launch with
// the items of k.runs (one key slice each).
struct PromptAttnArgs {
    AttnKArgs k;
    const int4* long_runs;
    int n_long;
};
void launch_prompt_attn16(const PromptAttnArgs& a, int hd);

}  // namespace nvllm
