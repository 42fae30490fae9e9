// gemm_wide_b16.hip -- launches of the 256-feature tiles (gemm_wide.h) for bf16 models: the wide projections whose epilogue
// only writes (gated pairs, tiles, rows).
#include "gemm_wide.h"

namespace nvllm {

namespace {

template <int EPI>
bool launch_wide_b16(const GemmArgs& a) {
    // 8: more steps than the deepest ring.  Below 32 steps a launch is mostly start and end, which the smaller tiles overlap.
    if (a.Kb < (wide_env() < 0 ? 32 : 8) || wide_env() == 0) return false;
    // With one plane of activations a step multiplies for as long as it copies, and the tiles of gemm_b16.hip, three to a CU,
    // come close.  So only launches that are one round here: the lowest height that fits them into the CUs, and 85 of 100 CUs
    // with a tile.  2,048 x 2,048 k, those against these: gated pairs of 5,632 at 400 tokens (220 tiles of 96) 35.9 -> 34.1 us,
    // at 700 (220 of 160) 50 -> 46; of 2,816 at 700 (242 of 64) 30.4 -> 29, at 1,029 (242 of 96) 38 -> 34, at 1,600 (220 of
    // 160) 55 -> 45.  154 tiles of 64 measured the same, two rounds (484 of 96) 66 -> 69; heights of 13 and 16 blocks, whose
    // sums do not fit 256 registers, 65 -> 69 where they make one round of two.
    const int cus = rt().num_cus, tiles_n = cdiv(a.NB, 16);
    int tbn = 4;
    while (tbn < 10 && tiles_n * cdiv(a.Tb, tbn) > cus) tbn += 2;
    if (wide_env() > 0) tbn = wide_env();
    const int tiles_t = cdiv(a.Tb, tbn), tiles = tiles_n * tiles_t;
    if (wide_env() < 0 && (tiles > cus || 100 * tiles < 85 * cus)) return false;
    if (tbn == 4) launch_wide<4, EPI, float, OpBf16>(a, tiles_n, tiles_t);
    else if (tbn == 6) launch_wide<6, EPI, float, OpBf16>(a, tiles_n, tiles_t);
    else if (tbn == 8) launch_wide<8, EPI, float, OpBf16>(a, tiles_n, tiles_t);
    else if (tbn == 10) launch_wide<10, EPI, float, OpBf16>(a, tiles_n, tiles_t);
    else return false;
    return true;
}

}  // namespace

bool launch_gemm_wide_b16(const GemmArgs& a) {
    switch (a.e.kind) {
        case GemmEpilogue::SWIGLU_A16: return launch_wide_b16<GemmEpilogue::SWIGLU_A16>(a);
        case GemmEpilogue::TILE_B16: return launch_wide_b16<GemmEpilogue::TILE_B16>(a);
        case GemmEpilogue::ROWS_B16: return launch_wide_b16<GemmEpilogue::ROWS_B16>(a);
        default: return false;
    }
}

}  // namespace nvllm
