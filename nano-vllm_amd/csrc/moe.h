// moe.h -- mixture of experts: a sigmoid router, the chosen experts' rows sorted by expert, and the sum of their results.
// The chosen weight scales an expert's INPUT; its score is not renormalised.
#pragma once

#include "nvllm_internal.h"

namespace nvllm {

// The rows of a batch sorted by expert, every expert's segment padded to `pad` rows.
struct RoutePlan {
    int T, E, top, pad;
    int capacity;          // rows, a multiple of pad: no batch of T tokens needs more
    int* block_expert;     // [capacity / 16]
    int* source;           // [capacity] row -> token (padding and unused rows: token 0)
    float* weight;         // [capacity] row -> its expert's score (padding: 0)
    int* row_of;           // [T][top] row of a token's j-th choice
    int* choice;           // [T][top] expert
    float* score;          // [T][top]
};
int route_pad(int T, int E, int top);   // group size that suits a batch in tiles of 128 features or less
// The group size that suits a batch's products with [up] and [down] stacked by expert (bf16); wide: expert_rows_wide()'s.
struct ExpertGroups {
    int pad;
    bool wide;
};
ExpertGroups expert_groups(int T, int E, int top, const B16Weight& up, const B16Weight& down);
size_t route_ints(int T, int E, int top, int pad);  // 4-byte words route_plan() lays out
RoutePlan route_plan(int* mem, int T, int E, int top, int pad);
// z: [T][ldz] router logits in columns 0 .. E-1; the `top` largest (the first of equals) are chosen
void launch_route(const RoutePlan& r, const float* z, int ldz, bool chosen = false);   // chosen: sorting is left

// bytes for kernel timing: of the choice, and of the sorting as a launch of its own
inline double choice_bytes(const RoutePlan& r) { return (double)r.T * (r.E * 4.0 + r.top * 20.0); }
inline double sort_bytes(const RoutePlan& r) { return (double)r.T * r.top * 28.0; }

// Work that needs a fraction of the chip, beside the shared expert's products on the CUs those leave idle: the router beside the first,
// the choice beside the second (launch_gemm_b16); with hundreds of tokens the choice with the router, the sorting alone beside the second.
struct MoeRider {
    const B16Weight* router = nullptr;   // SWIGLU_A16 launches: its activations are the launch's
    GemmEpilogue router_epi;             // F32
    RoutePlan plan{};                    // F32 launches
    const float* z = nullptr;
    int ldz = 0;
    bool chosen = false;                 // (set by the SWIGLU_A16 launch)
};

// the rows x * gain of a batch in the plan's order, as activation tiles (x [T][ld])
void launch_expert_rows(__half* dst, const float* x, const float* gain, const RoutePlan& r, int ld);

// x += sum of the chosen experts' rows + sigmoid(z_shared) * shared;  then what the next sublayer needs of x
struct MoeCombine {
    float* x;                  // [T][ld]
    const float* rows;         // expert results [row][ld], rows by row_of
    const int* row_of;
    int top;
    const float* shared;       // [T][ld] or null
    const float* z;            // its gate's logits: z[t * ldz + z_col]
    int ldz, z_col;
    const float* gain;         // next norm
    __half* out_b16;           // x * gain tiles, and ...
    float* ss;                 // ... sums of squares per 32 features (both null: fp32 path)
    int ld;
};
void launch_moe_combine(const MoeCombine& m, int T);

}  // namespace nvllm
