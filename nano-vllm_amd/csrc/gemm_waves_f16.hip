// gemm_waves_f16.hip -- launches of gemm_waves.h for fp16 models.
#include "gemm_waves.h"

namespace nvllm {

bool launch_gemm_waves_f16(const GemmArgs& a) {
    const int tbn = waves_height(a, waves_tallest(2));
    if (!tbn) return false;
    // Two planes make the products as long as the copies: with a short K several smaller workgroups on a CU (gemm_prefill.hip),
    // which overlap each other's starts and ends, come as close.  us there and here: K = 5,632, 2,048 features at 256, 640, 1,029, 1,400
    // tokens (heights of 1, 3, 5, 6 blocks) 51.7 -> 28.1, 56 -> 39, 76 -> 52, 81 -> 64; K = 2,048 22.6 -> 11.3, 25.2 -> 18.1,
    // 31.7 -> 25.8, 34.6 -> 31.0; K = 512, 1,536 features at 256, 1,029, 1,400, 2,000 tokens (1, 4, 5, 6) 10.1 -> 6.1, 12.5 -> 12.1,
    // 15.4 -> 15.2, 16.8 -> 18.1.  Passes: prompts of TinyLlama-1.1B of 256, 640, 1,100 tokens 3,240 -> 2,350 us, 4,130 -> 3,640,
    // 6,360 -> 5,700; of stories42M 531 -> 376, 622 -> 502, 659 -> 593.
    static const bool forced = getenv("NVLLM_GEMM_WAVES") != nullptr;
    if (!forced && tbn == 6 && a.Kb < 64) return false;
    const bool kv16 = a.e.kind == GemmEpilogue::ROPE_KV && a.e.kv_elem_bytes == 2;
    switch (a.e.kind) {
        case GemmEpilogue::F32: launch_waves_height<GemmEpilogue::F32, float, OpF16x2>(a, tbn); break;
        case GemmEpilogue::SWIGLU_A16: launch_waves_height<GemmEpilogue::SWIGLU_A16, float, OpF16x2>(a, tbn); break;
        case GemmEpilogue::RESID_A16: launch_waves_height<GemmEpilogue::RESID_A16, float, OpF16x2>(a, tbn); break;
        default:
            if (kv16) launch_waves_height<GemmEpilogue::ROPE_KV, __half, OpF16x2>(a, tbn);
            else launch_waves_height<GemmEpilogue::ROPE_KV, float, OpF16x2>(a, tbn);
    }
    return true;
}

}  // namespace nvllm
