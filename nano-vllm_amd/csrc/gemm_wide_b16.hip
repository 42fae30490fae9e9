// gemm_wide_b16.hip -- launches of the 256-feature tiles (gemm_wide.h) for bf16 models: the wide projections whose epilogue
// only writes (gated pairs, tiles, rows).
#include <algorithm>
#include <cmath>
#include <iterator>

#include "gemm_wide.h"

namespace nvllm {

namespace {

template <int EPI, bool EXP>
bool launch_wide_height(const GemmArgs& a, int tbn, int tiles_n, int tiles_t, bool* rode = nullptr) {
    bool ride;
    switch (tbn) {
        case 4: ride = launch_wide<4, EPI, float, OpBf16, 1, EXP>(a, tiles_n, tiles_t); break;
        case 5: ride = launch_wide<5, EPI, float, OpBf16, 1, EXP>(a, tiles_n, tiles_t); break;
        case 6: ride = launch_wide<6, EPI, float, OpBf16, 1, EXP>(a, tiles_n, tiles_t); break;
        case 8: ride = launch_wide<8, EPI, float, OpBf16, 2, EXP>(a, tiles_n, tiles_t); break;
        case 10: ride = launch_wide<10, EPI, float, OpBf16, 2, EXP>(a, tiles_n, tiles_t); break;
        case 12: ride = launch_wide<12, EPI, float, OpBf16, 2, EXP>(a, tiles_n, tiles_t); break;
        case 14: ride = launch_wide<14, EPI, float, OpBf16, 2, EXP>(a, tiles_n, tiles_t); break;
        case 16: ride = launch_wide<16, EPI, float, OpBf16, 2, EXP>(a, tiles_n, tiles_t); break;
        default: return false;
    }
    if (rode) *rode = ride;
    return true;
}
constexpr int WIDE_HEIGHTS[] = {4, 5, 6, 8, 10, 12, 14, 16};   // token blocks

// Height in token blocks of the tiles that a launch takes, 0: none of these.
// With one plane of activations a step multiplies for as long as it copies, and the tiles of gemm_b16.hip, three to a CU,
// come close.  So only launches that are one round here, at the lowest height that fits them into the CUs, and fill most of it: two
// rounds (484 tiles of 96) 66 -> 69 us.  2,048 k, those against these, layers' weights in turn: four blocks with a tile on 81 % of the CUs
// 27.1 -> 28.4 (4,864 features, 700 tokens), 27.1 -> 28.2 (3,328, 1,024), 28.2 -> 28.6 (6,656, 512), on 95 % 30.4 -> 29 (5,632, 700); five on
// 81 % 27.8 -> 24.7 (6,656, 640), on 96 % 36.3 -> 32.1 (4,864, 1,024); six on 81 % 38.4 -> 35.2 (13,312, 380).  Eight waves, two to a SIMD, from
// eight blocks on: one's requests go out behind the other's products; eight to sixteen on 81 % 33.9 -> 29.4, 45.4 -> 35.8, 48.2 -> 41.7,
// 51.9 -> 47.8 (6,656; 1,024, 1,280, 1,536, 1,792), 73.9 -> 53.4 (13,312, 1,024).
int wide_height(int NB, int Kb, int Tb) {
    // 8: more steps than the deepest ring.  Below 32 steps a launch is mostly start and end, which the smaller tiles overlap.
    if (Kb < (wide_env() < 0 ? 32 : 8) || wide_env() == 0) return 0;
    if (wide_env() > 0) return wide_env();
    const int cus = rt().num_cus, tiles_n = cdiv(NB, 16);
    for (int h : WIDE_HEIGHTS) {
        const int tiles = tiles_n * cdiv(Tb, h);
        if (tiles <= cus) return 100 * tiles < (h == 4 ? 85 : 80) * cus ? 0 : h;
    }
    return 0;
}
template <int EPI>
bool launch_wide_b16(const GemmArgs& a, bool* rode = nullptr) {
    const int tbn = wide_height(a.NB, a.Kb, a.Tb);
    return tbn && launch_wide_height<EPI, false>(a, tbn, cdiv(a.NB, 16), cdiv(a.Tb, tbn), rode);
}

}  // namespace

bool launch_gemm_wide_b16(const GemmArgs& a, bool* rode) {
    switch (a.e.kind) {
        case GemmEpilogue::SWIGLU_A16: return launch_wide_b16<GemmEpilogue::SWIGLU_A16>(a, rode);
        case GemmEpilogue::TILE_B16: return launch_wide_b16<GemmEpilogue::TILE_B16>(a);
        case GemmEpilogue::ROWS_B16: return launch_wide_b16<GemmEpilogue::ROWS_B16>(a);
        case GemmEpilogue::LATENT_Q: return launch_wide_b16<GemmEpilogue::LATENT_Q>(a);
        default: return false;
    }
}

// Rows sorted by expert: groups as tall as hold the rows an expert gets from a batch of that many, with the chance that one of
// sixteen gets more at a few in a hundred (a second group then); 0: not for these sizes.  One round of the chip, and one that pays
// beside groups of 64 rows (from 96 rows an expert on: 128) in 128-feature tiles.  Passes of four layers of sixteen experts, two a token,
// 330 to 1,600 tokens, those groups -> these, by the share of the CUs that have a tile of the first and of the second product: 62 and 44,
// 62 and 50, 62 and 62, 69 and 50, 94 and 50 % always faster (780 -> 735, 820 -> 776, 993 -> 888, 843 -> 788, 933 -> 891 us at 330 tokens; 1,122 -> 1,036 ..
// 1,370 -> 1,201 at 1,029); 56 and 50, 56 and 56 at 50 rows an expert 766 -> 793, 825 -> 855, at 64 829 -> 819, 962 -> 909; 50 and 44 at 64 rows
// 718 -> 754, at 100 852 -> 826, at 200 the same; eight experts of 41 and 41 at 82 rows 996 -> 1,032, at 128 1,148 -> 1,114.
int expert_rows_wide(int rows, int experts, const B16Weight& up, const B16Weight& down) {
    const double per = (double)rows / experts;
    auto height = [](int h) { return std::find(std::begin(WIDE_HEIGHTS), std::end(WIDE_HEIGHTS), h) != std::end(WIDE_HEIGHTS); };
    if (wide_env() > 0) return up.K >= 256 && down.K >= 256 && height(wide_env()) ? 16 * wide_env() : 0;
    const int cus = rt().num_cus, tiles_up = cdiv(up.N, 256) * experts, tiles_down = cdiv(down.N, 256) * experts;
    if (wide_env() == 0 || up.K < 1024 || down.K < 1024 || std::max(tiles_up, tiles_down) > cus || 100 * std::min(tiles_up, tiles_down) < 40 * cus) return 0;
    if (per < (100 * tiles_up >= 60 * cus ? 40 : 100 * tiles_up >= 55 * cus ? 60 : 96)) return 0;
    for (int h : WIDE_HEIGHTS)
        if (16 * h >= per + 2.5 * std::sqrt(per)) return 16 * h;
    return 0;
}
bool launch_experts_wide_b16(const GemmArgs& a, int pad) {
    const int tbn = pad / 16, tiles_n = cdiv(a.NB, 16), tiles_t = a.Tb / tbn;
    if (a.e.kind == GemmEpilogue::SWIGLU_A16) return launch_wide_height<GemmEpilogue::SWIGLU_A16, true>(a, tbn, tiles_n, tiles_t);
    return a.e.kind == GemmEpilogue::F32 && launch_wide_height<GemmEpilogue::F32, true>(a, tbn, tiles_n, tiles_t);
}

}  // namespace nvllm

// the rules above, for tests
extern "C" int nvllm_internal_wide_height(int N, int K, int T) {
    nvllm::ensure_init();
    return nvllm::wide_height(nvllm::cdiv(N, 16), nvllm::cdiv(K, 32), nvllm::cdiv(T, 16));
}
extern "C" int nvllm_internal_expert_rows_wide(int rows, int experts, int up_n, int up_k, int down_n, int down_k) {
    nvllm::ensure_init();
    nvllm::B16Weight up, down;
    up.N = up_n; up.K = up_k;
    down.N = down_n; down.K = down_k;
    return nvllm::expert_rows_wide(rows, experts, up, down);
}
