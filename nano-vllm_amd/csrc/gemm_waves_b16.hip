// gemm_waves_b16.hip -- launches of gemm_waves.h for bf16 models.
#include "gemm_waves.h"

namespace nvllm {

// Every launch that is one round takes them.  us, tiles of gemm_b16.hip and here, 2,048 features: K = 5,632 at 256, 512, 900, 1,029,
// 1,400, 1,600 tokens (heights of 1, 2, 4, 5, 6, 7 blocks) 39 -> 28, 40 -> 29, 42 -> 34, 48 -> 38, 53 -> 42, 54 -> 45; K = 2,048
// 16.6 -> 10.6, 17.4 -> 11.9, 19.3 -> 16.8, 22.2 -> 18.9, 23.8 -> 21.9, 25.0 -> 23.9; 1,024 features x 1,024 k at 512 and 2,000
// tokens (1 and 4) 11.1 -> 7.9, 13.7 -> 13.5; 5,632 x 2,048 at 400 (5) 27.8 -> 20.1; few tiles of a long K too: 256 and 512 features x 8,192 k at
// 256 tokens (32 and 64 tiles) 54.3 -> 25.8, 52.7 -> 24.9, 512 x 4,096 31.3 -> 14.5.
bool launch_gemm_waves_b16(const GemmArgs& a, bool* rode) {
    const int tbn = waves_height(a, waves_tallest(1));
    if (!tbn) return false;
    switch (a.e.kind) {
        case GemmEpilogue::F32: *rode = launch_waves_height<GemmEpilogue::F32, float, OpBf16>(a, tbn); break;
        case GemmEpilogue::SWIGLU_A16: *rode = launch_waves_height<GemmEpilogue::SWIGLU_A16, float, OpBf16>(a, tbn); break;
        case GemmEpilogue::TILE_B16: launch_waves_height<GemmEpilogue::TILE_B16, float, OpBf16>(a, tbn); break;
        case GemmEpilogue::ROWS_B16: launch_waves_height<GemmEpilogue::ROWS_B16, float, OpBf16>(a, tbn); break;
        case GemmEpilogue::LATENT_IN: launch_waves_height<GemmEpilogue::LATENT_IN, float, OpBf16>(a, tbn); break;
        case GemmEpilogue::LATENT_Q: launch_waves_height<GemmEpilogue::LATENT_Q, float, OpBf16>(a, tbn); break;
        case GemmEpilogue::HYPER_2: launch_waves_height<GemmEpilogue::HYPER_2, float, OpBf16>(a, tbn); break;
        case GemmEpilogue::HYPER_4: launch_waves_height<GemmEpilogue::HYPER_4, float, OpBf16>(a, tbn); break;
        case GemmEpilogue::RESID_B16: launch_waves_height<GemmEpilogue::RESID_B16, float, OpBf16>(a, tbn); break;
        default: return false;
    }
    return true;
}

}  // namespace nvllm
