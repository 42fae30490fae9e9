// gemm_wide_f16.hip -- launches of the 256-feature tiles (gemm_wide.h) for fp16 models.
#include "gemm_wide.h"

namespace nvllm {

namespace {

template <int TBN, typename KVT>
void launch_kind(const GemmArgs& a, int tiles_n, int tiles_t) {
    switch (a.e.kind) {
        case GemmEpilogue::F32: launch_wide<TBN, GemmEpilogue::F32, float, OpF16x2>(a, tiles_n, tiles_t); break;
        case GemmEpilogue::SWIGLU_A16: launch_wide<TBN, GemmEpilogue::SWIGLU_A16, float, OpF16x2>(a, tiles_n, tiles_t); break;
        case GemmEpilogue::RESID_A16: launch_wide<TBN, GemmEpilogue::RESID_A16, float, OpF16x2>(a, tiles_n, tiles_t); break;
        default: launch_wide<TBN, GemmEpilogue::ROPE_KV, KVT, OpF16x2>(a, tiles_n, tiles_t); break;
    }
}

}  // namespace

bool launch_gemm_wide_f16(const GemmArgs& a) {
    // 8: more steps than the deepest ring.  Short K (a 512-wide model has 16 steps) is mostly start and end, which the smaller
    // tiles overlap with each other: gate/up of that model at 1,800 tokens 19.3 us there, 19.7 here, q/k/v 20.1 and 21.9.
    if (a.Kb < (wide_env() < 0 ? 32 : 8) || wide_env() == 0) return false;
    const int cus = rt().num_cus, tiles_n = cdiv(a.NB, 16);
    int best = 0;
    double cost = 0;
    for (int tbn : {4, 6, 9}) {
        const double c = wide_us(tiles_n * cdiv(a.Tb, tbn), a.Kb, tbn, 2, cus);
        if (wide_env() == tbn || ((!best || c < cost) && wide_env() < 0)) best = tbn, cost = c;
    }
    if (!best) return false;
    // One workgroup per CU has nothing to run beside it, so where the tiles leave a third of the CUs empty the smaller ones of
    // gemm_prefill.hip win.  TinyLlama-1.1B, those against these: gate/up at 256 tokens (176 tiles) 43 -> 35 us, at 520 (176)
    // 74 -> 60, at 1,200 (396 of 512) 136 -> 119, at 3,000 310 -> 265; q/k/v at 1,200 tokens (190 tiles) 47 -> 43, but at 640
    // (100) 34 -> 39; w_down at 2,048 (256) 114 -> 97, at 1,380 (176) 87 -> 86, at 1,000 (128) 73 -> 81.  Decode batches of
    // Llama-2-7B, against the eight-wave tiles: gate/up (172 tiles) at 112, 120 and 128 rows 67.1, 68.3, 68.8 -> 64.5, 66.4, 67.1,
    // the classifier (250) 79.4, 80.3, 83.7 -> 79.8, 81.1, 81.0.
    const int tiles_t = cdiv(a.Tb, best), tiles = tiles_n * tiles_t;
    if (wide_env() < 0 && 100 * tiles < 65 * cus * cdiv(tiles, cus)) return false;
    const bool kv16 = a.e.kind == GemmEpilogue::ROPE_KV && a.e.kv_elem_bytes == 2;
    if (best == 4) kv16 ? launch_kind<4, __half>(a, tiles_n, tiles_t) : launch_kind<4, float>(a, tiles_n, tiles_t);
    else if (best == 6) kv16 ? launch_kind<6, __half>(a, tiles_n, tiles_t) : launch_kind<6, float>(a, tiles_n, tiles_t);
    else kv16 ? launch_kind<9, __half>(a, tiles_n, tiles_t) : launch_kind<9, float>(a, tiles_n, tiles_t);
    return true;
}

}  // namespace nvllm
