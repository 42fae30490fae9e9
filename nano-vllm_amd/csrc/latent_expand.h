// latent_expand.h -- keys and values of each head formed from cached latents, for prompt portions: a launch of its own (latent_prompt.hip), or
// beside the attention of the tokens that come alone (latent_attention.hip).
#pragma once

#include "attn_tile.h"
#include "gemm_common.h"
#include "latent_prompt.h"

namespace nvllm {

namespace {

typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
typedef float f8_t __attribute__((ext_vector_type(8)));
typedef const __attribute__((address_space(4))) int* const_int_p;   // read-only for the whole launch: scalar loads

__device__ __forceinline__ void prompt_barrier() {   // this wave's LDS accesses are done, then everybody meets
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void copies_landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Eight waves; KC: tiles of a latent that a wave has registers for.  lds_expand: [2][2][chunks] tiles
template <int KC>
__device__ __forceinline__ void latent_expand(const ExpandArgs& a, int col, int group, unsigned char* lds_expand) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = lane & 15, g = lane >> 4;
    const int nc = a.chunks;
    const int unit = col * 8 + wave, key_units = a.H * a.dc, units = key_units + a.H * (a.vt / 2);
    const bool is_key = unit < key_units, live = unit < units;
    const int mine = min(unit, units - 1), block = (is_key ? mine : mine - key_units) * 2;   // this wave's first row block of its matrix
    const int pair0 = group * a.per, pair1 = min(a.n_pairs, pair0 + a.per);
    const const_int_p pages = (const_int_p)(uintptr_t)a.pages;
    const unsigned lds0 = (unsigned)(size_t)(lds_void*)lds_expand;
    auto issue = [&](int pair, int buf) {   // waves 0-3 bring the first page's tiles, 4-7 the second's
        const int half = wave >> 2;
        const __half* src = a.base + (size_t)pages[2 * pair + half] * a.row_tiles * TILE_HALVES + lane * 8;
        for (int c = wave & 3; c < nc; c += 4)
            copy_tile_to_lds(src + (size_t)c * TILE_HALVES, __builtin_amdgcn_readfirstlane(lds0 + (unsigned)((buf * 2 + half) * nc + c) * 1024u));
    };
    issue(pair0, 0);
    h8_t w[2][KC];
    {
        const __half* W = (is_key ? a.uk : a.uv) + (size_t)block * nc * TILE_HALVES + lane * 8;
#pragma unroll
        for (int f = 0; f < 2; f++)
#pragma unroll
            for (int k = 0; k < KC; k++) w[f][k] = *reinterpret_cast<const h8_t*>(W + ((size_t)f * nc + min(k, nc - 1)) * TILE_HALVES);
    }
    const size_t head_halves = (size_t)(2 * a.dc + a.vt) * TILE_HALVES;
    for (int pair = pair0; pair < pair1; pair++) {
        const int buf = (pair - pair0) & 1;
        copies_landed();
        prompt_barrier();
        if (pair + 1 < pair1) issue(pair + 1, buf ^ 1);
        const h8_t* lat = reinterpret_cast<const h8_t*>(lds_expand) + (size_t)buf * 2 * nc * 64 + lane;
        f4_t acc[2][2] = {};   // [row block][page]
        if (is_key) {
#pragma unroll
            for (int k = 0; k < KC; k++)
                if (k < nc) {
#pragma unroll
                    for (int page = 0; page < 2; page++) {
                        const h8_t c = lat[(page * nc + k) * 64];
#pragma unroll
                        for (int f = 0; f < 2; f++) acc[f][page] = OpBf16::mfma(w[f][k], c, acc[f][page]);
                    }
                }
            if (!live) continue;
            const int head = mine / a.dc, c = mine - head * a.dc;
            __half* out = a.kv + ((size_t)pair * a.H + head) * head_halves;
#pragma unroll
            for (int f = 0; f < 2; f++)
#pragma unroll
                for (int page = 0; page < 2; page++)   // dims 16 f + 4 g .. + 3 of position x
                    *reinterpret_cast<h4_t*>(out + (size_t)(page * a.dc + c) * TILE_HALVES + (x + 16 * (2 * f + (g >> 1))) * 8 + 4 * (g & 1)) =
                        __builtin_convertvector(acc[f][page], h4_t);
        } else {
#pragma unroll
            for (int k = 0; k < KC; k++)
                if (k < nc) {
#pragma unroll
                    for (int page = 0; page < 2; page++) {
                        const h8_t c = lat[(page * nc + k) * 64];
#pragma unroll
                        for (int f = 0; f < 2; f++) acc[f][page] = OpBf16::mfma(c, w[f][k], acc[f][page]);
                    }
                }
            if (!live) continue;
            const int head = block / a.vt, n = block - head * a.vt;
            __half* out = a.kv + ((size_t)pair * a.H + head) * head_halves + (size_t)(2 * a.dc + n) * TILE_HALVES;
#pragma unroll
            for (int f = 0; f < 2; f++) {   // positions 4 g .. + 3 of both pages, dim 16 (n + f) + x
                alignas(16) h4_t both[2];
#pragma unroll
                for (int page = 0; page < 2; page++) both[page] = __builtin_convertvector(acc[f][page], h4_t);
                *reinterpret_cast<u4_t*>(out + (size_t)f * TILE_HALVES + lane * 8) = *reinterpret_cast<const u4_t*>(both);
            }
        }
    }
}

inline int expand_cols(const ExpandArgs& e) { return cdiv(e.H * (e.dc + e.vt / 2), 8); }   // workgroups side by side over the row blocks
inline size_t expand_lds(const ExpandArgs& e) { return (size_t)4 * e.chunks * 1024; }

}  // namespace

}  // namespace nvllm
