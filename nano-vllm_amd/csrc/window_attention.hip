// window_attention.hip -- attention with a sliding window and kept first tokens (window_attention.h).
//
// k_window_attn (bf16 pages).  Pages are stored in the operand order of the matrix cores, so a wave reads a key page
// (operand A of S^T = K Q^T) and a value page (operand A of O^T = V^T P^T) straight from memory into registers; a score
// tile's result registers are already in the k order of the second product, and a column (one query) stays on its lane
// through scores, weights, sums and results: no LDS and no barrier in the loop.  A step takes two pages (32 keys) while
// the next step's travel.
//   prompts        a wave owns C groups of 16 neighbouring tokens x up to four heads of a key/value group;
//   single tokens  the columns are the heads of a group; the waves of a workgroup (and, when there are few items,
//                  several workgroups) take every n-th pair of pages and their sums meet in LDS (and in a merge launch).
// The walk visits the pages of the kept first tokens and those the item's window touches; only pages at an edge are masked.
// A soft cap bounds every score, so with a cap of up to 32 the largest weight is known beforehand: weights are
// exp(score - cap), no running maximum and no rescaling (exp(-2 * 32) is far inside the range of fp32 and bf16).
// Scores, caps, maxima and sums are fp32.
//
// k_window_rows (fp32 rows of whole float4s), k_window_attn_any (what is left): one workgroup per (token, head).
#include "window_attention.h"

#include "attn_tile.h"
#include "gemm_common.h"
#include "model_dir.h"

namespace nvllm {

KvPages kv_pages(void* base, int elem_bytes, int block_size, int num_blocks, int G, int dim, int vdim) {
    KvPages p{base, nullptr, elem_bytes, block_size, G, dim, vdim, dim, vdim};
    if (elem_bytes == 2) {
        if (block_size % KV_PAGE) NVLLM_FATAL("bf16 key and value pages hold 16 positions: block size %d is not a multiple of 16", block_size);
        p.dim_ld = pad32(dim);
        p.vdim_ld = pad32(vdim);
    }
    if (base) p.values = (char*)base + (size_t)num_blocks * block_size * G * p.dim_ld * elem_bytes;
    return p;
}
size_t kv_pages_bytes(int elem_bytes, int block_size, int num_blocks, int G, int dim, int vdim) {
    const KvPages p = kv_pages(nullptr, elem_bytes, block_size, num_blocks, G, dim, vdim);
    return ((size_t)num_blocks * block_size * G * (p.dim_ld + p.vdim_ld) * elem_bytes + 255) & ~(size_t)255;
}

// accumulators of k_window_attn_any: a set per group of threads, or one row that is wider than the workgroup
__host__ __device__ inline int window_any_acc(int vdim_ld, int vec) { return vdim_ld > 256 * vec ? vdim_ld : 256 * vec; }
__device__ __forceinline__ float b16_f32(unsigned short v) { return __builtin_bit_cast(float, (unsigned)v << 16); }
__device__ __forceinline__ size_t key_off(long row, int g, int G, int d, int dim_ld) {
    return ((size_t)(row >> 4) * G + g) * (KV_PAGE * dim_ld) + (d >> 5) * 512 + ((row & 15) + 16 * ((d >> 3) & 3)) * 8 + (d & 7);
}
__device__ __forceinline__ size_t value_off(long row, int g, int G, int d, int vdim_ld) {
    return ((size_t)(row >> 4) * G + g) * (KV_PAGE * vdim_ld) + (d >> 4) * 256 + (((row & 15) >> 2) * 16 + (d & 15)) * 4 + (row & 3);
}

// ------------------------------------------------------------------ convolution, rotation, cache write
struct ConvKArgs {
    ConvRope c;
    KvPages pool;
    const int4* spans;
    const int* span_of;
    const int* kv_row;
    int channels, QD, KD;
    int items_q, items_k, items_v, items;   // work items of a query head, a key head, a value head; of a token
};

template <typename RT, int VEC>
struct alignas(sizeof(RT) * VEC) ConvVec {
    RT v[VEC];
};

// A thread owns VEC neighbouring channels of a token, together with their rotation partners when they turn.  The tokens
// that still see the state of earlier passes belong to the thread of the portion's first token, which then renews it.
template <typename RT, int VEC>
__global__ __launch_bounds__(256) void k_conv_rope(ConvKArgs a) {
    typedef ConvVec<RT, VEC> Vec;
    const int item = blockIdx.y * 256 + threadIdx.x;
    if (item >= a.items) return;
    const int t_mine = blockIdx.x, keep = a.c.n_taps - 1;
    const int4 span = a.spans[a.span_of[t_mine]];   // (first token, count, first position, sequence)
    const int off_mine = t_mine - span.x;
    if (off_mine > 0 && off_mine < keep) return;
    const int n_mine = off_mine == 0 ? min(span.y, max(keep, 1)) : 1;
    const RT* raw = reinterpret_cast<const RT*>(a.c.raw) + (size_t)span.x * a.c.raw_ld;
    RT* state = keep > 0 ? reinterpret_cast<RT*>(a.c.state) + (size_t)span.w * keep * a.channels : nullptr;

    // which head, which dims: part 0 query, 1 key, 2 value
    int part, head, at, i = item;
    if (i < a.c.H * a.items_q) {
        part = 0;
        head = i / a.items_q;
        at = i - head * a.items_q;
    } else if ((i -= a.c.H * a.items_q) < a.pool.G * a.items_k) {
        part = 1;
        head = i / a.items_k;
        at = i - head * a.items_k;
    } else {
        i -= a.pool.G * a.items_k;
        part = 2;
        head = i / a.items_v;
        at = i - head * a.items_v;
    }
    const int half = part == 2 ? 0 : a.c.rot >> 1, turning = half / VEC;
    const bool turns = at < turning;
    const int d0 = turns ? at * VEC : 2 * half + (at - turning) * VEC;
    const int dim = part == 2 ? a.pool.vdim : a.pool.dim;
    const bool live = d0 < dim;   // (past it: the padding of a query row)
    const int ch0 = (part == 0 ? 0 : part == 1 ? a.QD : a.QD + a.KD) + head * dim;

    // the projected value at place `off` of this portion (negative: from the state; before the sequence: zero)
    auto input = [&](int off, int ch) {
        Vec v;
        if (off >= 0) {
            v = *reinterpret_cast<const Vec*>(raw + (size_t)off * a.c.raw_ld + ch);
        } else if (span.z + off >= 0) {
            v = *reinterpret_cast<const Vec*>(state + (size_t)(keep + off) * a.channels + ch);
        } else {
#pragma unroll
            for (int e = 0; e < VEC; e++) v.v[e] = (RT)0.f;
        }
        return v;
    };
    auto conv = [&](int off, int ch, float* y) {
        if (!a.c.taps) {
            const Vec u = input(off, ch);
#pragma unroll
            for (int e = 0; e < VEC; e++) y[e] = (float)u.v[e];
            return;
        }
#pragma unroll
        for (int e = 0; e < VEC; e++) y[e] = 0.f;
        constexpr int U = VEC == 1 ? 4 : 1;   // taps requested together (one after the other a token of three taps took 12.8 us)
        for (int j0 = 0; j0 <= keep; j0 += U) {
            Vec u[U];
            float wf[U][VEC];
#pragma unroll
            for (int i = 0; i < U; i++) {
                const int j = min(j0 + i, keep);
                u[i] = input(off - keep + j, ch);
#pragma unroll
                for (int e = 0; e < VEC; e++) wf[i][e] = a.c.taps[(size_t)j * a.channels + ch + e];
            }
#pragma unroll
            for (int i = 0; i < U; i++)
                if (j0 + i <= keep)
#pragma unroll
                    for (int e = 0; e < VEC; e++) y[e] = fmaf(wf[i][e], (float)u[i].v[e], y[e]);
        }
    };
    auto store = [&](int t, int d, const float* y) {
        if (part == 0) {
            Vec v;
#pragma unroll
            for (int e = 0; e < VEC; e++) v.v[e] = (RT)y[e];
            *reinterpret_cast<Vec*>(reinterpret_cast<RT*>(a.c.q_out) + ((size_t)t * a.c.H + head) * a.pool.dim_ld + d) = v;
            return;
        }
        const int row = a.kv_row[t];
        if (row < 0) return;
        if (sizeof(RT) == 4) {
            float* p = part == 1 ? (float*)a.pool.keys : (float*)a.pool.values;
#pragma unroll
            for (int e = 0; e < VEC; e++) p[((size_t)row * a.pool.G + head) * dim + d + e] = y[e];
        } else if (part == 1) {   // VEC 8: one 16-byte piece of the page (d is a multiple of VEC)
            Vec v;
#pragma unroll
            for (int e = 0; e < VEC; e++) v.v[e] = (RT)y[e];
            *reinterpret_cast<Vec*>(reinterpret_cast<RT*>(a.pool.keys) + key_off(row, head, a.pool.G, d, a.pool.dim_ld)) = v;
        } else {
#pragma unroll
            for (int e = 0; e < VEC; e++) reinterpret_cast<RT*>(a.pool.values)[value_off(row, head, a.pool.G, d + e, a.pool.vdim_ld)] = (RT)y[e];
        }
    };

    for (int k = 0; k < n_mine; k++) {
        const int off = off_mine + k, t = span.x + off;
        float y[VEC], z[VEC];
        if (!live) {
#pragma unroll
            for (int e = 0; e < VEC; e++) y[e] = 0.f;
            store(t, d0, y);
            continue;
        }
        conv(off, ch0 + d0, y);
        if (turns) {
            conv(off, ch0 + d0 + half, z);
            const float2* cs = a.c.rope + (size_t)(span.z + off) * half + d0;
#pragma unroll
            for (int e = 0; e < VEC; e++) {
                const float2 r = cs[e];
                const float u = y[e], v = z[e];
                y[e] = u * r.x - v * r.y;
                z[e] = v * r.x + u * r.y;
            }
            store(t, d0 + half, z);
        }
        store(t, d0, y);
    }
    if (off_mine == 0 && keep > 0 && live) {   // ascending rows: a row's source lies at or behind it
        for (int r = 0; r < keep; r++) {
            const int off = span.y - keep + r;
            RT* dst = state + (size_t)r * a.channels + ch0 + d0;
            const Vec v = input(off, ch0 + d0);
            *reinterpret_cast<Vec*>(dst) = v;
            if (turns) {
                const Vec w = input(off, ch0 + d0 + half);
                *reinterpret_cast<Vec*>(dst + half) = w;
            }
        }
    }
}

// The same for fp32 rows and KEEP + 1 taps, a channel (and its rotation partner) per thread: all that a thread needs -- its inputs, for a portion's
// first token also those of the tokens that still see the state, and the ones that renew it; taps and angles -- is requested together, behind
// the look-up of the portion.  80 tokens of a prompt and rows, 1,536 channels, four taps: 10.1 us in k_conv_rope, which takes the first
// tokens and the rows of the state one after the other, 4.9 here.
template <int KEEP>
__global__ __launch_bounds__(256) void k_conv_rope_f32(ConvKArgs a) {
    request_arguments<sizeof(ConvKArgs)>();
    const int item = blockIdx.y * 256 + threadIdx.x, t_mine = blockIdx.x;
    if (item >= a.items) return;
    const int4 span = a.spans[a.span_of[t_mine]];   // (first token, count, first position, sequence)
    const int off_mine = t_mine - span.x;
    if (off_mine > 0 && off_mine < KEEP) return;    // (the first token's)
    const int n_mine = off_mine == 0 ? min(span.y, KEEP) : 1;
    int part, head, at, i = item;
    if (i < a.c.H * a.items_q) {
        part = 0;
        head = i / a.items_q;
        at = i - head * a.items_q;
    } else if ((i -= a.c.H * a.items_q) < a.pool.G * a.items_k) {
        part = 1;
        head = i / a.items_k;
        at = i - head * a.items_k;
    } else {
        i -= a.pool.G * a.items_k;
        part = 2;
        head = i / a.items_v;
        at = i - head * a.items_v;
    }
    const int half = part == 2 ? 0 : a.c.rot >> 1;
    const bool turns = at < half;
    const int d0 = turns ? at : 2 * half + (at - half), dim = part == 2 ? a.pool.vdim : a.pool.dim;
    const int ch = (part == 0 ? 0 : part == 1 ? a.QD : a.QD + a.KD) + head * dim + d0, partner = turns ? half : 0;
    const float* raw = reinterpret_cast<const float*>(a.c.raw) + (size_t)span.x * a.c.raw_ld + ch;
    float* state = reinterpret_cast<float*>(a.c.state) + (size_t)span.w * KEEP * a.channels + ch;
    constexpr int N = 2 * KEEP;   // inputs of tokens off_mine - KEEP .. (the last KEEP - 1 for a portion's first token only)
    float in[N], inz[N], tail[KEEP], tailz[KEEP], w[KEEP + 1], wz[KEEP + 1];
    float2 turn[KEEP];
    int rows[KEEP];
    // the projected value at place `off` of this portion: from the state where negative, zero before the sequence
    auto input = [&](int off, float& v, float& z) {
        const bool old = off < 0, none = old && span.z + off < 0;
        const float* src = old && !none ? state + (size_t)(KEEP + off) * a.channels : raw + (size_t)max(off, 0) * a.c.raw_ld;
        v = src[0];
        z = src[partner];
        if (none) v = z = 0.f;
    };
#pragma unroll
    for (int j = 0; j < N; j++)
        if (j <= KEEP || off_mine == 0) input(min(off_mine - KEEP + j, span.y - 1), in[j], inz[j]);
    if (off_mine == 0) {
#pragma unroll
        for (int r = 0; r < KEEP; r++) input(span.y - KEEP + r, tail[r], tailz[r]);
    }
#pragma unroll
    for (int j = 0; j <= KEEP; j++) {
        w[j] = a.c.taps[(size_t)j * a.channels + ch];
        wz[j] = a.c.taps[(size_t)j * a.channels + ch + partner];
    }
#pragma unroll
    for (int k = 0; k < KEEP; k++) {
        const int off = off_mine + min(k, n_mine - 1);
        turn[k] = turns ? a.c.rope[(size_t)(span.z + off) * half + d0] : make_float2(1.f, 0.f);
        rows[k] = a.kv_row[span.x + off];
    }
#pragma unroll
    for (int k = 0; k < KEEP; k++) {
        float y = 0.f, z = 0.f;
#pragma unroll
        for (int j = 0; j <= KEEP; j++) {
            y = fmaf(w[j], in[k + j], y);
            z = fmaf(wz[j], inz[k + j], z);
        }
        const float u = y, v = z;
        if (turns) {
            y = u * turn[k].x - v * turn[k].y;
            z = v * turn[k].x + u * turn[k].y;
        }
        float* dst = nullptr;
        if (k >= n_mine) dst = nullptr;
        else if (part == 0) dst = reinterpret_cast<float*>(a.c.q_out) + ((size_t)(t_mine + k) * a.c.H + head) * a.pool.dim_ld + d0;
        else if (rows[k] >= 0) dst = reinterpret_cast<float*>(part == 1 ? a.pool.keys : a.pool.values) + ((size_t)rows[k] * a.pool.G + head) * dim + d0;
        if (dst) {
            dst[0] = y;
            if (turns) dst[half] = z;
        }
    }
    if (off_mine == 0) {   // (everything of the old state that this thread needs has been read)
#pragma unroll
        for (int r = 0; r < KEEP; r++) {
            state[(size_t)r * a.channels] = tail[r];
            if (turns) state[(size_t)r * a.channels + half] = tailz[r];
        }
    }
}

// The same for bf16 rows of 16-byte pieces and KEEP + 1 taps: a thread walks TOK neighbouring tokens with the taps and the
// last KEEP inputs in registers (what the tokens need is requested up front), and on to the end of those that see the state
// of a portion that starts among them.
struct alignas(16) Piece {
    __bf16 v[8];
};
template <int KEEP, int TOK>
__global__ __launch_bounds__(256) void k_conv_rope_walk(ConvKArgs a, int T) {
    request_arguments<sizeof(ConvKArgs)>();
    const int item = blockIdx.y * 256 + threadIdx.x, t0 = blockIdx.x * TOK;
    if (item >= a.items) return;
    int part, head, at, i = item;
    if (i < a.c.H * a.items_q) {
        part = 0;
        head = i / a.items_q;
        at = i - head * a.items_q;
    } else if ((i -= a.c.H * a.items_q) < a.pool.G * a.items_k) {
        part = 1;
        head = i / a.items_k;
        at = i - head * a.items_k;
    } else {
        i -= a.pool.G * a.items_k;
        part = 2;
        head = i / a.items_v;
        at = i - head * a.items_v;
    }
    const int half = part == 2 ? 0 : a.c.rot >> 1, turning = half / 8;
    const bool turns = at < turning;
    const int d0 = turns ? at * 8 : 2 * half + (at - turning) * 8;
    const int dim = part == 2 ? a.pool.vdim : a.pool.dim;
    const bool live = d0 < dim;   // (past it: the padding of a query row)
    const int ch = (part == 0 ? 0 : part == 1 ? a.QD : a.QD + a.KD) + head * dim + (live ? d0 : 0), partner = turns ? half : 0;
    const __bf16* raw = reinterpret_cast<const __bf16*>(a.c.raw) + ch;
    int4 spans[TOK];   // (first token, count, first position, sequence)
    int rows[TOK];
    Piece in[TOK], inz[TOK];
#pragma unroll
    for (int u = 0; u < TOK; u++) {
        const int t = min(t0 + u, T - 1);
        spans[u] = a.spans[a.span_of[t]];
        rows[u] = a.kv_row[t];
        in[u] = *reinterpret_cast<const Piece*>(raw + (size_t)t * a.c.raw_ld);
        inz[u] = *reinterpret_cast<const Piece*>(raw + (size_t)t * a.c.raw_ld + partner);
    }
    float w[KEEP + 1][8], wz[KEEP + 1][8];
#pragma unroll
    for (int j = 0; j <= KEEP; j++)
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
            const f4_t one = {1.f, 1.f, 1.f, 1.f};
            const f4_t u = a.c.taps ? *reinterpret_cast<const f4_t*>(a.c.taps + (size_t)j * a.channels + ch + e) : one;
            const f4_t v = a.c.taps ? *reinterpret_cast<const f4_t*>(a.c.taps + (size_t)j * a.channels + ch + partner + e) : one;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                w[j][e + r] = u[r];
                wz[j][e + r] = v[r];
            }
        }
    Piece win[KEEP + 1], winz[KEEP + 1];   // inputs of tokens t - KEEP .. t
    int have = -1;                         // the token they are complete for, but for its own input
    // values of four tokens that are a quarter of a page: stored together, a dim's four keys lie side by side
    bool quarter = false;
    if (TOK % 4 == 0 && part == 2) {
        const int off = t0 - spans[0].x;
        quarter = t0 + TOK <= T && spans[TOK - 1].x == spans[0].x && (spans[0].z + off) % 4 == 0 && (off == 0 || off >= KEEP) && rows[0] >= 0 && rows[TOK - 1] >= 0;
    }
    Piece values[TOK];
    auto token = [&](const int t, const int4 span, const int row, const Piece own, const Piece ownz, Piece& value) __attribute__((always_inline)) {
        const int off = t - span.x;
        __bf16* state = reinterpret_cast<__bf16*>(a.c.state) + (size_t)span.w * KEEP * a.channels + ch;
        if (have != t || off == 0) {
#pragma unroll
            for (int j = 0; j < KEEP; j++) {
                const int o = off - KEEP + j;
                const Piece zero = {};
                win[j] = winz[j] = zero;
                if (span.z + o >= 0) {
                    const __bf16* src = o >= 0 ? raw + (size_t)(span.x + o) * a.c.raw_ld : state + (size_t)(KEEP + o) * a.channels;
                    win[j] = *reinterpret_cast<const Piece*>(src);
                    winz[j] = *reinterpret_cast<const Piece*>(src + partner);
                }
            }
        }
        win[KEEP] = own;
        winz[KEEP] = ownz;
        float y[8], z[8];
#pragma unroll
        for (int e = 0; e < 8; e++) y[e] = z[e] = 0.f;
#pragma unroll
        for (int j = 0; j <= KEEP; j++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                y[e] = fmaf(w[j][e], (float)win[j].v[e], y[e]);
                z[e] = fmaf(wz[j][e], (float)winz[j].v[e], z[e]);
            }
        if (turns) {
            const float4* cs = reinterpret_cast<const float4*>(a.c.rope + (size_t)(span.z + off) * half + d0);   // {cos, sin} x 2
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                const float4 r = cs[e >> 1];
                const float u0 = y[e], v0 = z[e], u1 = y[e + 1], v1 = z[e + 1];
                y[e] = u0 * r.x - v0 * r.y;
                z[e] = v0 * r.x + u0 * r.y;
                y[e + 1] = u1 * r.z - v1 * r.w;
                z[e + 1] = v1 * r.z + u1 * r.w;
            }
        }
        Piece py, pz;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            py.v[e] = (__bf16)(live ? y[e] : 0.f);
            pz.v[e] = (__bf16)z[e];
        }
        if (part == 0) {
            __bf16* q = reinterpret_cast<__bf16*>(a.c.q_out) + ((size_t)t * a.c.H + head) * a.pool.dim_ld + d0;
            *reinterpret_cast<Piece*>(q) = py;
            if (turns) *reinterpret_cast<Piece*>(q + half) = pz;
        } else if (row >= 0) {
            if (part == 1) {
                __bf16* k = reinterpret_cast<__bf16*>(a.pool.keys);
                *reinterpret_cast<Piece*>(k + key_off(row, head, a.pool.G, d0, a.pool.dim_ld)) = py;
                if (turns) *reinterpret_cast<Piece*>(k + key_off(row, head, a.pool.G, d0 + half, a.pool.dim_ld)) = pz;
            } else if (quarter) {
                value = py;
            } else {
                __bf16* v = reinterpret_cast<__bf16*>(a.pool.values) + value_off(row, head, a.pool.G, d0, a.pool.vdim_ld);
#pragma unroll
                for (int e = 0; e < 8; e++) v[4 * e] = py.v[e];   // (d0 is a multiple of 8: the dims stay in one tile)
            }
        }
#pragma unroll
        for (int j = 0; j < KEEP; j++) {
            win[j] = win[j + 1];
            winz[j] = winz[j + 1];
        }
        have = t + 1;
        if (KEEP > 0 && live && off == min(span.y, KEEP) - 1) {   // nobody needs the old state any more
#pragma unroll
            for (int j = 0; j < KEEP; j++) {
                Piece u = win[j], v = winz[j];
                if (span.y > KEEP) {
                    const __bf16* src = raw + (size_t)(span.x + span.y - KEEP + j) * a.c.raw_ld;
                    u = *reinterpret_cast<const Piece*>(src);
                    v = *reinterpret_cast<const Piece*>(src + partner);
                }
                *reinterpret_cast<Piece*>(state + (size_t)j * a.channels) = u;
                if (turns) *reinterpret_cast<Piece*>(state + (size_t)j * a.channels + half) = v;
            }
        }
    };
#pragma unroll
    for (int u = 0; u < TOK; u++) {
        const int t = t0 + u, off = t - spans[u].x;
        // (a token that sees the state of a portion that starts in front of these belongs to the thread of its first token)
        if (t < T && !(off > 0 && off < KEEP && spans[u].x < t0)) token(t, spans[u], rows[u], in[u], inz[u], values[u]);
    }
    if (quarter) {
#pragma unroll
        for (int u = 0; u + 3 < TOK; u += 4) {
            b4_t* v = reinterpret_cast<b4_t*>(reinterpret_cast<__bf16*>(a.pool.values) + value_off(rows[u], head, a.pool.G, d0, a.pool.vdim_ld));
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = b4_t{values[u].v[e], values[u + 1].v[e], values[u + 2].v[e], values[u + 3].v[e]};
        }
    }
    Piece unused;
    quarter = false;
    const int4 last = spans[TOK - 1];   // the portion the next tokens may belong to
    for (int t = t0 + TOK; t < last.x + min(last.y, KEEP) && last.x >= t0; t++)
        token(t, last, a.kv_row[t], *reinterpret_cast<const Piece*>(raw + (size_t)t * a.c.raw_ld), *reinterpret_cast<const Piece*>(raw + (size_t)t * a.c.raw_ld + partner), unused);
}

template <int KEEP>
static void launch_walk(const ConvKArgs& a, int T) {
    const dim3 threads(std::min(256, (a.items + 63) & ~63));
    const int y = cdiv(a.items, 256);
    if ((long)T * a.items >= 4L * 64 * 16 * rt().num_cus)   // (enough waves even so; fewer loads of the taps)
        NVLLM_LAUNCH((k_conv_rope_walk<KEEP, 4>), dim3(cdiv(T, 4), y), threads, 0, a, T);
    else if (T >= 256) NVLLM_LAUNCH((k_conv_rope_walk<KEEP, 2>), dim3(cdiv(T, 2), y), threads, 0, a, T);
    else NVLLM_LAUNCH((k_conv_rope_walk<KEEP, 1>), dim3(T, y), threads, 0, a, T);
}

void launch_conv_rope(const ConvRope& c, const KvPages& pool, const StepArrays& st) {
    if (st.T <= 0) return;
    if (!st.d_spans || !st.d_kv_row) NVLLM_FATAL("convolution over time: the batch was staged without its portions");
    if (c.rot % 2 || c.rot > pool.dim || c.n_taps < 1) NVLLM_FATAL("convolution over time: %d taps, %d of %d dimensions rotated", c.n_taps, c.rot, pool.dim);
    ConvKArgs a{};
    a.c = c;
    a.pool = pool;
    a.spans = (const int4*)st.d_spans;
    a.span_of = st.d_span_of;
    a.kv_row = st.d_kv_row;
    a.QD = c.H * pool.dim;
    a.KD = pool.G * pool.dim;
    a.channels = a.QD + a.KD + pool.G * pool.vdim;
    const int half = c.rot / 2;
    const bool wide = pool.elem_bytes == 2 && pool.dim % 8 == 0 && pool.vdim % 8 == 0 && half % 8 == 0 && c.raw_ld % 8 == 0;
    const int vec = wide ? 8 : 1;
    a.items_q = half / vec + (pool.dim_ld - c.rot) / vec;
    a.items_k = half / vec + (pool.dim - c.rot) / vec;
    a.items_v = pool.vdim / vec;
    a.items = c.H * a.items_q + pool.G * (a.items_k + a.items_v);
    const double elems = (double)st.T * a.channels * 2.0;
    ProfScope ps(PC_CONV_ROPE, elems * pool.elem_bytes + (double)a.channels * c.n_taps * 4.0, elems * c.n_taps);
    const dim3 grid(st.T, cdiv(a.items, 256));
    if (wide && c.n_taps <= 5 && (c.taps || c.n_taps == 1)) {
        switch (c.n_taps) {
            case 1: launch_walk<0>(a, st.T); break;
            case 2: launch_walk<1>(a, st.T); break;
            case 3: launch_walk<2>(a, st.T); break;
            case 4: launch_walk<3>(a, st.T); break;
            default: launch_walk<4>(a, st.T); break;
        }
        return;
    }
    if (pool.elem_bytes == 4 && c.taps && c.n_taps >= 2 && c.n_taps <= 5) {
        switch (c.n_taps) {
            case 2: NVLLM_LAUNCH(k_conv_rope_f32<1>, grid, dim3(256), 0, a); break;
            case 3: NVLLM_LAUNCH(k_conv_rope_f32<2>, grid, dim3(256), 0, a); break;
            case 4: NVLLM_LAUNCH(k_conv_rope_f32<3>, grid, dim3(256), 0, a); break;
            default: NVLLM_LAUNCH(k_conv_rope_f32<4>, grid, dim3(256), 0, a); break;
        }
        return;
    }
    if (pool.elem_bytes == 4) NVLLM_LAUNCH((k_conv_rope<float, 1>), grid, dim3(256), 0, a);
    else if (wide) NVLLM_LAUNCH((k_conv_rope<__bf16, 8>), grid, dim3(256), 0, a);
    else NVLLM_LAUNCH((k_conv_rope<__bf16, 1>), grid, dim3(256), 0, a);
}

// ------------------------------------------------------------------ attention, fp32 rows of whole float4s
// The scheme of row_attention.hip for a window and kept first tokens: a workgroup per (token, head), LPK lanes a key (four dims each, up to
// 4 LPK), the waves deal the keys among themselves 64 / LPK at a time and request AHEAD such groups together; every group of lanes keeps a
// maximum, a sum and results of its own, and they meet once at the end.  What bounds it is the chain position and sequence, table, block,
// rows, merge.  80 tokens x 16 heads of 64, up to 200 keys: 13.6 us in k_window_attn_any (keys' rows, scores, maxima and weights one after the other
// through LDS), 9.4 here (12.0 with the cap and the exponential formed by every lane of a key).
template <int LPK, int WAVES, bool CAP>
__global__ __launch_bounds__(64 * WAVES) void k_window_rows(KvPages pool, const float* __restrict__ q, float scale, float cap, int size, int keep,
                                                            const int* __restrict__ pos, const int* __restrict__ seq, const int* __restrict__ tbl_off,
                                                            const int* __restrict__ tables, int H, float* __restrict__ out, int shift) {   // shift: log2 of the block size, -1: it is no power of two
    typedef const __attribute__((address_space(4))) int* scalar_int_p;   // read-only for the whole launch
    constexpr int KEYS = 64 / LPK, AHEAD = 8;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), x = lane & (LPK - 1), kg = lane / LPK;
    const int t = blockIdx.x, h = blockIdx.y, g = h / (H / pool.G), dim = pool.dim, vdim = pool.vdim;
    const int p = ((scalar_int_p)(uintptr_t)pos)[t], first_block = ((scalar_int_p)(uintptr_t)tbl_off)[((scalar_int_p)(uintptr_t)seq)[t]];
    const int* table = tables + first_block;
    const int lo = max(0, p - size + 1), first = min(keep, lo), n_keys = first + p - lo + 1;
    const bool has = 4 * x < dim, has_v = 4 * x < vdim;
    const int d = has ? 4 * x : 0, dv = has_v ? 4 * x : 0;
    const f4_t zero = {0.f, 0.f, 0.f, 0.f};
    f4_t qv = *reinterpret_cast<const f4_t*>(q + ((size_t)t * H + h) * dim + d), o = zero;
    if (!has) qv = zero;
    float m = -INFINITY, l = 0.f;
    for (int k0 = wave * KEYS + kg; k0 - kg < n_keys; k0 += KEYS * WAVES * AHEAD) {   // (the condition is the wave's)
        int row[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {   // (past the last key: the last again, not counted)
            const int i = min(k0 + KEYS * WAVES * u, n_keys - 1), key = i < first ? i : lo + i - first;
            row[u] = shift >= 0 ? (table[key >> shift] << shift) + (key & ((1 << shift) - 1)) : table[key / pool.block_size] * pool.block_size + key % pool.block_size;
        }
        f4_t k[AHEAD], v[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
            const size_t at = (size_t)row[u] * pool.G + g;
            k[u] = *reinterpret_cast<const f4_t*>((const float*)pool.keys + at * dim + d);
            v[u] = *reinterpret_cast<const f4_t*>((const float*)pool.values + at * vdim + dv);
        }
        float dot[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
            dot[u] = qv[0] * k[u][0];
#pragma unroll
            for (int e = 1; e < 4; e++) dot[u] = fmaf(qv[e], k[u][e], dot[u]);
        }
        float s = eight_sums<LPK>(dot, x) * scale;   // of key number x & 7
        if constexpr (CAP) s = cap * tanhf(s / cap);
        if (k0 + KEYS * WAVES * (x & 7) >= n_keys) s = -INFINITY;
        const float top = fmaxf(m, eight_max<LPK>(s)), base = fmaxf(top, -3.0e38f);   // (a group of lanes that has seen no key: exp(-inf - finite) = 0)
        const float alpha = expf(m - base), w = expf(s - base);
        l = fmaf(l, alpha, w);
        o *= alpha;
        m = top;
        add_eight<LPK>(o, w, v, lane);
    }
    l += lane_moved<0xB1>(l);   // (lanes x and x + 8 hold the same)
    l += lane_moved<0x4E>(l);
    l += lane_moved<0x124>(l);
    __shared__ float s_m[WAVES * KEYS], s_l[WAVES * KEYS];
    __shared__ f4_t s_o[WAVES * KEYS][LPK];
    if (x == 0) s_m[wave * KEYS + kg] = m, s_l[wave * KEYS + kg] = l;
    s_o[wave * KEYS + kg][x] = o;
    __syncthreads();
    if (wave > 0) return;
    float M = -INFINITY, L = 0.f;
#pragma unroll
    for (int i = 0; i < WAVES * KEYS; i++) M = fmaxf(M, s_m[i]);
    f4_t sum = zero;
#pragma unroll
    for (int i = 0; i < WAVES; i++) {
        const float f = expf(s_m[i * KEYS + kg] - M);   // parts without keys carry -inf: weight 0
        L = fmaf(s_l[i * KEYS + kg], f, L);
        const f4_t part = s_o[i * KEYS + kg][x];
#pragma unroll
        for (int e = 0; e < 4; e++) sum[e] = fmaf(part[e], f, sum[e]);
    }
#pragma unroll
    for (int w = LPK; w < 64; w <<= 1) {
        L += __shfl_xor(L, w, 64);
#pragma unroll
        for (int e = 0; e < 4; e++) sum[e] += __shfl_xor(sum[e], w, 64);
    }
    if (kg == 0 && has_v) *reinterpret_cast<f4_t*>(out + ((size_t)t * H + h) * vdim + dv) = sum * (1.0f / L);
}
// false: not for these heads
static bool launch_window_rows(const WindowAttn& w, const StepArrays& st) {
    const KvPages& pool = w.pool;
    const int widest = std::max(pool.dim, pool.vdim);
    if (pool.elem_bytes != 4 || pool.dim % 4 || pool.vdim % 4 || widest > 128 || ((uintptr_t)w.q | (uintptr_t)w.out_f32) % 16) return false;   // (a caller's rows of 16-byte pieces)
    // us a layer, k_window_attn_any and these, 16 heads of 64 (128), a window of 512 and 16 kept: 1 row of 40 and 300 cached 5.2 and 4.6, 13.0 and 7.9 (5.9
    // and 4.7, 17.2 and 11.0), 32 rows of 600 26.3 and 18.4 (38.4 and 29.6), prompts of 100, 200, 400 9.7 and 8.6, 23.1 and 19.8, 50.5 and 44.3 (11.1 and
    // 11.2, 29.6 and 28.4, 66.6 and 70.4: wide heads of many tokens stay there)
    if (widest > 64 && (long)st.T * w.H > 16L * rt().num_cus) return false;
    const long keys = std::min((long)st.max_pos + 1, (long)w.size + w.keep_first);
    // eight waves where four would walk more than two trips and the workgroups are not many
    const bool many = widest <= 64 ? keys > 256 : keys > 128, eight = many && (long)st.T * w.H <= 4L * rt().num_cus;
    int shift = 0;
    while ((1 << shift) < pool.block_size) shift++;
    if ((1 << shift) != pool.block_size) shift = -1;
    auto go = [&](auto lpk, auto waves) {
        constexpr int LPK = decltype(lpk)::value, WAVES = decltype(waves)::value;
        const dim3 grid(st.T, w.H), block(64 * WAVES);
        if (w.cap > 0.f)
            NVLLM_LAUNCH((k_window_rows<LPK, WAVES, true>), grid, block, 0, pool, (const float*)w.q, w.scale, w.cap, w.size, w.keep_first, st.d_pos, st.d_seq, st.d_tbl_off,
                         st.d_tables, w.H, w.out_f32, shift);
        else
            NVLLM_LAUNCH((k_window_rows<LPK, WAVES, false>), grid, block, 0, pool, (const float*)w.q, w.scale, w.cap, w.size, w.keep_first, st.d_pos, st.d_seq, st.d_tbl_off,
                         st.d_tables, w.H, w.out_f32, shift);
    };
    using std::integral_constant;
    auto by_waves = [&](auto lpk) {
        if (eight) go(lpk, integral_constant<int, 8>{});
        else go(lpk, integral_constant<int, 4>{});
    };
    if (widest <= 64) by_waves(integral_constant<int, 16>{});
    else by_waves(integral_constant<int, 32>{});
    return true;
}

// ------------------------------------------------------------------ attention, any size
// A workgroup per (token, head), keys in blocks of 256.  What bounds it is the latency of a block's loads: a key per thread,
// read value by value, and a thread per output over all the block's keys were two chains of hundreds of loads (90 us for 80
// tokens x 16 heads of 64 and 200 keys, 13 so).  So sixteen lanes share a key's row, four keys a group at once, and the threads
// beyond an output row's take other keys (VEC = 4: fp32 rows of whole float4s).
template <bool B16, int VEC>
__global__ __launch_bounds__(256) void k_window_attn_any(KvPages pool, const void* q, float scale, float cap, int size, int keep, const int* __restrict__ pos,
                                                         const int* __restrict__ seq, const int* __restrict__ tbl_off, const int* __restrict__ tables, int H,
                                                         float* out_f32, __half* out_b16, int Kb_out) {
    typedef float vec_t __attribute__((ext_vector_type(VEC)));
    extern __shared__ __attribute__((aligned(16))) float lds_any[];   // query [dim_ld], accumulators [window_any_acc()], weights [256], reductions [8], rows [256]
    float* sq = lds_any;
    float* acc = sq + pool.dim_ld;
    const int acc_n = window_any_acc(pool.vdim_ld, VEC);
    float* sp = acc + acc_n;
    float* red = sp + 256;
    int* srow = reinterpret_cast<int*>(red + 8);
    const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = h / (H / pool.G);
    for (int d = tid; d < pool.dim; d += 256) {
        const size_t i = ((size_t)t * H + h) * pool.dim_ld + d;
        sq[d] = B16 ? b16_f32(reinterpret_cast<const unsigned short*>(q)[i]) : reinterpret_cast<const float*>(q)[i];
    }
    for (int d = tid; d < acc_n; d += 256) acc[d] = 0.f;
    auto load = [&](const void* base, bool values, int row, int d) {
        vec_t v;
        if constexpr (B16) v[0] = b16_f32(reinterpret_cast<const unsigned short*>(base)[values ? value_off(row, g, pool.G, d, pool.vdim_ld) : key_off(row, g, pool.G, d, pool.dim_ld)]);
        else v = *reinterpret_cast<const vec_t*>(reinterpret_cast<const float*>(base) + ((size_t)row * pool.G + g) * (values ? pool.vdim : pool.dim) + d);
        return v;
    };
    // columns: VEC neighbouring outputs; `groups` of threads share the keys of a block where a row has fewer columns than threads
    const int cols = pool.vdim / VEC, per = min(cols, 256), groups = 256 / per, grp = tid / per, col0 = tid - grp * per;
    const int sub = lane & 15, quarter = wave * 4 + (lane >> 4);
    const int p = pos[t], lo = max(0, p - size + 1), first = min(keep, lo), n_keys = first + p - lo + 1;
    const int* table = tables + tbl_off[seq[t]];
    float m = -INFINITY, l = 0.f;   // the same in every thread
    for (int k0 = 0; k0 < n_keys; k0 += 256) {
        const int k = k0 + tid, n = min(256, n_keys - k0);
        if (k < n_keys) {
            const int key = k < first ? k : lo + k - first;
            srow[tid] = table[key / pool.block_size] * pool.block_size + key % pool.block_size;
        }
        __syncthreads();   // (and the query, the first time)
        for (int b = 0; b < n; b += 64) {
            constexpr int U = 4;
            float dot[U];
            int row[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                dot[u] = 0.f;
                row[u] = srow[min(b + 16 * u + quarter, n - 1)];
            }
            for (int d = sub * VEC; d < pool.dim; d += 16 * VEC) {
                const vec_t qv = *reinterpret_cast<const vec_t*>(sq + d);
                vec_t kv[U];
#pragma unroll
                for (int u = 0; u < U; u++) kv[u] = load(pool.keys, false, row[u], d);
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int e = 0; e < VEC; e++) dot[u] = fmaf(qv[e], kv[u][e], dot[u]);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
#pragma unroll
                for (int o = 8; o > 0; o >>= 1) dot[u] += __shfl_xor(dot[u], o, 64);
                if (sub == u) sp[b + 16 * u + quarter] = dot[u];   // (past the n-th key: unused)
            }
        }
        __syncthreads();
        float s = -INFINITY;
        if (tid < n) {
            s = sp[tid] * scale;
            if (cap > 0.f) s = cap * tanhf(s / cap);
        }
        float mx = s;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
        if (lane == 0) red[wave] = mx;
        __syncthreads();
        const float mn = fmaxf(m, fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])));
        const float e = tid < n ? expf(s - mn) : 0.f;
        sp[tid] = e;
        float sum = e;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
        if (lane == 0) red[4 + wave] = sum;
        __syncthreads();
        const float alpha = m == -INFINITY ? 0.f : expf(m - mn);
        l = l * alpha + ((red[4] + red[5]) + (red[6] + red[7]));
        m = mn;
        if (grp < groups)
            for (int c = col0; c < cols; c += per) {   // (one round unless the values are very wide: then groups = 1)
                float* mine = acc + ((size_t)grp * per + c) * VEC;
                vec_t o;
#pragma unroll
                for (int i = 0; i < VEC; i++) o[i] = mine[i] * alpha;
                constexpr int U = 4;   // keys in flight
                for (int j = grp; j < n; j += U * groups) {
                    vec_t v[U];
                    float w[U];
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const int at = j + u * groups;
                        v[u] = load(pool.values, true, srow[min(at, n - 1)], c * VEC);
                        w[u] = at < n ? sp[at] : 0.f;
                    }
#pragma unroll
                    for (int u = 0; u < U; u++)
                        if (j + u * groups < n)
#pragma unroll
                            for (int i = 0; i < VEC; i++) o[i] = fmaf(w[u], v[u][i], o[i]);
                }
#pragma unroll
                for (int i = 0; i < VEC; i++) mine[i] = o[i];
            }
        __syncthreads();   // weights, rows and reductions are free again; the sums are there
    }
    for (int d = tid; d < pool.vdim_ld; d += 256) {
        float o = 0.f;
        if (d < pool.vdim) {
            for (int i = 0; i < groups; i++) o += acc[i * per * VEC + d];
            o /= l;
        }
        if (B16) {
            const int k = h * pool.vdim_ld + d;
            reinterpret_cast<__bf16*>(out_b16)[((size_t)(t >> 4) * Kb_out + (k >> 5)) * TILE_HALVES + (size_t)((t & 15) + 16 * ((k >> 3) & 3)) * 8 + (k & 7)] = (__bf16)o;
        } else {
            out_f32[((size_t)t * H + h) * pool.vdim + d] = o;
        }
    }
}
template <bool B16, int VEC>
static void launch_window_any(const WindowAttn& w, const StepArrays& st, int Kb_out) {
    const KvPages& pool = w.pool;
    const size_t lds = ((size_t)pool.dim_ld + window_any_acc(pool.vdim_ld, VEC) + 256 + 8 + 256) * 4;
    static bool enabled = false;
    if (lds > 64 * 1024 && !enabled) {   // (up to 4 KiB more than the sizes the caller allows)
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_window_attn_any<B16, VEC>), hipFuncAttributeMaxDynamicSharedMemorySize, 72 * 1024));
        enabled = true;
    }
    NVLLM_LAUNCH((k_window_attn_any<B16, VEC>), dim3(st.T, w.H), dim3(256), lds, pool, w.q, w.scale, w.cap, w.size, w.keep_first, st.d_pos, st.d_seq, st.d_tbl_off,
                 st.d_tables, w.H, w.out_f32, w.out_b16, Kb_out);
}

// ------------------------------------------------------------------ attention, bf16 pages
struct WindowKArgs {
    const __half* keys;
    const __half* values;
    const __half* q;
    const int* tables;
    const int4* runs;      // (first token, count, last position, table offset)
    int n_runs, n_sub;     // items of CT tokens per run
    int HW, NHG;           // heads per item (prompts: 1, 2 or 4; single tokens: 16); head groups of a key/value group
    int G, rep, H;
    int kc, vt;            // dim_ld / 32, vdim_ld / 16
    int size, keep;
    float scale, cap;
    int nsplit;
    int page_shift;        // log2(pages per block)
    __half* out;
    int Kb_out;
    float* part_acc;       // [run][head][slice][16 * vt]
    float* part_ml;        // [run][head][slice][2], log2 domain
};
typedef const __attribute__((address_space(4))) int* const_int_p;   // read-only for the whole launch: scalar loads
typedef unsigned int u2_t __attribute__((ext_vector_type(2)));
constexpr float LOG2E = 1.44269504088896340736f;
constexpr float CAP_FIXED = 32.f;   // caps up to here: the shift of the weights is the cap itself
constexpr int window_waves(int VT, bool single) { return !single || VT > 8 ? 4 : 8; }
static size_t window_lds(int VT, int waves) { return (size_t)waves * (VT * 1024 + 16 * 8); }

// KC key chunks of 32 dims, VT value tiles of 16 dims held; C column groups of 16 per wave; CAP: 0 no cap, 1 cap with the
// shift known beforehand, 2 cap with a running maximum; EXACT: the sizes are KC and VT.
template <int KC, int VT, int C, bool SINGLE, int CAP, bool EXACT>
__global__ __launch_bounds__(64 * window_waves(VT, SINGLE), 2) void k_window_attn(WindowKArgs a) {
    constexpr int WAVES = window_waves(VT, SINGLE);
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_win[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = lane & 15, g4 = lane >> 4;
    const int kc = EXACT ? KC : a.kc, vt = EXACT ? VT : a.vt;

    // ---- the item: neighbouring items share keys and values and sit behind one L2 (workgroups are dealt to 8 XCDs)
    int idx;
    {
        const int n = gridDim.x, xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, qd = n >> 3, r = n & 7;
        idx = (xcd < r ? xcd * (qd + 1) : r * (qd + 1) + (xcd - r) * qd) + slot;
    }
    int split = 0;
    if (SINGLE) {
        split = idx % a.nsplit;
        idx /= a.nsplit;
    } else {
        idx = idx * WAVES + wave;
    }
    const int hg = idx % a.NHG;
    idx /= a.NHG;
    const int sub = SINGLE ? 0 : idx % a.n_sub;
    if (!SINGLE) idx /= a.n_sub;
    const int run_id = idx % a.n_runs, grp = idx / a.n_runs;
    if (grp >= a.G) return;
    const int4 run = a.runs[run_id];
    const int CT = SINGLE ? 1 : 16 * C / a.HW;
    const int first = sub * CT;
    if (first >= run.y) return;
    const int ntok = __builtin_amdgcn_readfirstlane(min(CT, run.y - first));
    const int pos_lo = __builtin_amdgcn_readfirstlane(run.z - run.y + 1 + first), pos_hi = pos_lo + ntok - 1;
    const const_int_p table = (const_int_p)(uintptr_t)(a.tables + __builtin_amdgcn_readfirstlane(run.w));

    // this lane's column of group c: (token of the item, head of the group); position -1 where there is none
    auto column = [&](int c, int& tok, int& h) {
        const int hl = SINGLE ? x : c % a.HW;
        tok = SINGLE ? 0 : (c / a.HW) * 16 + x;
        h = hg * a.HW + hl;
        const bool valid = tok < ntok && h < a.rep;
        tok = valid ? tok : 0;
        h = valid ? grp * a.rep + h : -1;
    };
    int pos[C];
    b8_t qf[C][KC];
#pragma unroll
    for (int c = 0; c < C; c++) {
        int tok, h;
        column(c, tok, h);
        pos[c] = h >= 0 ? pos_lo + tok : -1;
        const b8_t* qr = reinterpret_cast<const b8_t*>(a.q + ((size_t)(run.x + first + tok) * a.H + max(h, 0)) * (kc * 32)) + g4;
#pragma unroll
        for (int k = 0; k < KC; k++) qf[c][k] = qr[(EXACT ? k : min(k, kc - 1)) * 4];
    }

    // ---- the pages: those of the kept first tokens, then those the window touches
    const int first_pg = max(0, pos_lo - a.size + 1) >> 4, last_pg = pos_hi >> 4;
    const int n_kept = min((a.keep + 15) >> 4, first_pg), n_pages = n_kept + last_pg - first_pg + 1;
    const int n_pairs = (n_pages + 1) >> 1;
    const int per = SINGLE ? (n_pairs + a.nsplit - 1) / a.nsplit : n_pairs;
    const int it0 = split * per + (SINGLE ? wave : 0), it1 = min(n_pairs, split * per + per);
    constexpr int STRIDE = SINGLE ? WAVES : 1;
    auto page_at = [&](int i) { return i < n_kept ? i : first_pg + i - n_kept; };   // position / 16

    // Pages in registers: of two steps (DEEP: a step's are requested before the step ahead of it is computed) or of one.
    constexpr bool DEEP = EXACT && 2 * (8 * KC + 4 * VT) + C * 4 * (KC + VT) <= 176;
    constexpr int SETS = DEEP ? 2 : 1;
    h8_t kf[SETS][2][KC];
    u2_t vf[SETS][2][VT];
    // The step that is requested next: entries of the block table (looked up a step earlier; used as late as possible, so that
    // nothing waits for the look-up) and the pages' places in their blocks.
    int entry[2], inside[2];
    auto look_up = [&](int it) {
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int pg = page_at(min(2 * it + p, n_pages - 1));
            entry[p] = table[pg >> a.page_shift];
            inside[p] = pg & ((1 << a.page_shift) - 1);
        }
    };
    auto page_id = [&](int p) { return (entry[p] << a.page_shift) + inside[p]; };
    auto load_keys = [&](int set) {
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const h8_t* src = reinterpret_cast<const h8_t*>(a.keys + ((size_t)page_id(p) * a.G + grp) * (KV_PAGE * 32 * kc)) + lane;
#pragma unroll
            for (int k = 0; k < KC; k++)
                if (EXACT || k < kc) kf[set][p][k] = src[k * 64];
        }
    };
    auto load_values = [&](int set) {
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const u2_t* src = reinterpret_cast<const u2_t*>(a.values + ((size_t)page_id(p) * a.G + grp) * (KV_PAGE * 16 * vt)) + lane;
#pragma unroll
            for (int v = 0; v < VT; v++)
                if (EXACT || v < vt) vf[set][p][v] = src[v * 64];
        }
    };

    float m[C], lsum[C];
    f4_t acc[VT][C];
#pragma unroll
    for (int c = 0; c < C; c++) {
        m[c] = -1e30f;   // (finite: no difference of infinities)
        lsum[c] = 0.f;
#pragma unroll
        for (int v = 0; v < VT; v++) acc[v][c] = f4_t{0.f, 0.f, 0.f, 0.f};
    }
    const float plain = a.scale * LOG2E;                                            // no cap: log2-domain scores
    const float grow = CAP ? 2.f * a.scale / a.cap * LOG2E : 0.f;                   // cap: tanh(s/cap) = 1 - 2 / (1 + 2^(grow s))
    const float top = a.cap * LOG2E;

    // set: where this step's pages are.  The next step's are requested whether or not there is one (the last pages again, then:
    // no memory traffic): where paths with and without requests meet, the compiler waits for every request in flight.
    auto step = [&](const int it, const int set) __attribute__((always_inline)) {
        if (DEEP && (!SINGLE || it + STRIDE < it1)) {   // (single tokens: few steps, so that the last one's would weigh)
            load_keys(set ^ 1);
            load_values(set ^ 1);
            look_up(it + 2 * STRIDE);
        }
        f4_t s[2][C];
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int c = 0; c < C; c++) s[p][c] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < KC; k++)
            if (EXACT || k < kc)
#pragma unroll
                for (int p = 0; p < 2; p++)
#pragma unroll
                    for (int c = 0; c < C; c++)
                        s[p][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8_t, kf[set][p][k]), qf[c][k], s[p][c], 0, 0, 0);
        if (!DEEP) load_keys(0);
        // ---- weights
        const int pg0 = page_at(2 * it), pg1 = 2 * it + 1 < n_pages ? page_at(2 * it + 1) : 1 << 26;   // (a page that is not there lies past every query)
        auto open = [&](int pg) { return pg * 16 + 15 <= pos_lo && (pg * 16 > pos_hi - a.size || pg * 16 + 15 < a.keep); };
        const bool masked = !(open(pg0) && open(pg1)) || (!SINGLE && ntok < CT);
        b8_t pw[C];
#pragma unroll
        for (int c = 0; c < C; c++) {
            float e[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float z = s[i >> 2][c][i & 3];
                if (CAP == 0) e[i] = z * plain;
                else {
                    const float r = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(z * grow));
                    e[i] = CAP == 1 ? -2.f * top * r : fmaf(-2.f * top, r, top);
                }
            }
            if (masked) {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const int key = (i < 4 ? pg0 : pg1) * 16 + 4 * g4 + (i & 3);
                    const bool seen = key <= pos[c] && (key > pos[c] - a.size || key < a.keep);
                    e[i] = seen ? e[i] : -INFINITY;
                }
            }
            if (CAP != 1) {
                float mx = e[0];
#pragma unroll
                for (int i = 1; i < 8; i++) mx = fmaxf(mx, e[i]);
                const float mn = fmaxf(m[c], rows_max(mx));
                if (__any(mn > m[c])) {
                    const float alpha = __builtin_amdgcn_exp2f(m[c] - mn);
                    lsum[c] *= alpha;
#pragma unroll
                    for (int v = 0; v < VT; v++)
                        if (EXACT || v < vt) acc[v][c] *= alpha;
                    m[c] = mn;
                }
#pragma unroll
                for (int i = 0; i < 8; i++) e[i] -= m[c];
            }
            float part = 0.f;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                e[i] = __builtin_amdgcn_exp2f(e[i]);
                part += e[i];
            }
            const f4_t lo = {e[0], e[1], e[2], e[3]}, hi = {e[4], e[5], e[6], e[7]};
            pw[c] = __builtin_shufflevector(__builtin_convertvector(lo, b4_t), __builtin_convertvector(hi, b4_t), 0, 1, 2, 3, 4, 5, 6, 7);
            lsum[c] += part;
        }
        // ---- values
#pragma unroll
        for (int v = 0; v < VT; v++)
            if (EXACT || v < vt) {
                const u4_t both = {vf[set][0][v][0], vf[set][0][v][1], vf[set][1][v][0], vf[set][1][v][1]};
#pragma unroll
                for (int c = 0; c < C; c++)
                    acc[v][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8_t, both), pw[c], acc[v][c], 0, 0, 0);
            }
        if (!DEEP) {
            load_values(0);
            look_up(it + 2 * STRIDE);
        }
    };
    if (it0 < it1) {
        look_up(it0);
        load_keys(0);
        load_values(0);
        look_up(it0 + STRIDE);
        if constexpr (DEEP) {
#pragma clang loop unroll(disable)
            for (int it = it0; it < it1; it += 2 * STRIDE) {
                step(it, 0);
                if (it + STRIDE < it1) step(it + STRIDE, 1);
            }
        } else {
#pragma clang loop unroll(disable)
            for (int it = it0; it < it1; it += STRIDE) step(it, 0);
        }
    }
#pragma unroll
    for (int c = 0; c < C; c++) {   // the four lane rows of a column hold different keys
        lsum[c] += __shfl_xor(lsum[c], 16, 64);
        lsum[c] += __shfl_xor(lsum[c], 32, 64);
    }
    if (!SINGLE) {
#pragma unroll
        for (int c = 0; c < C; c++) {
            int tok, h;
            column(c, tok, h);
            if (h < 0) continue;
            const float inv = 1.f / lsum[c];
#pragma unroll
            for (int v = 0; v < VT; v++)
                if (EXACT || v < vt) {
                    const float y[4] = {acc[v][c][0] * inv, acc[v][c][1] * inv, acc[v][c][2] * inv, acc[v][c][3] * inv};
                    store_b16_4(a.out, a.Kb_out, run.x + first + tok, h * vt * 16 + v * 16 + 4 * g4, y);
                }
        }
        return;
    }
    // ---- single tokens: the waves' sums meet
    f4_t* s_acc = reinterpret_cast<f4_t*>(lds_win);                                  // [wave][VT][64]
    float2* s_ml = reinterpret_cast<float2*>(lds_win + (size_t)WAVES * VT * 1024);   // [wave][16]
#pragma unroll
    for (int v = 0; v < VT; v++) s_acc[(wave * VT + v) * 64 + lane] = acc[v][0];
    if (g4 == 0) s_ml[wave * 16 + x] = make_float2(CAP == 1 ? 0.f : m[0], lsum[0]);
    __syncthreads();
    float mx = -1e30f, f[WAVES], l = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; w++) mx = fmaxf(mx, s_ml[w * 16 + x].x);
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
        f[w] = CAP == 1 ? 1.f : __builtin_amdgcn_exp2f(s_ml[w * 16 + x].x - mx);
        l = fmaf(f[w], s_ml[w * 16 + x].y, l);
    }
    const int hl = hg * a.HW + x, h = grp * a.rep + hl;   // (the column stays with the lane)
    if (hl >= a.rep || x >= a.HW) return;
    for (int v = wave; v < vt; v += WAVES) {
        f4_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < WAVES; w++) sum += f[w] * s_acc[(w * VT + v) * 64 + lane];
        if (a.nsplit == 1) {
            const float inv = 1.f / l;
            const float y[4] = {sum[0] * inv, sum[1] * inv, sum[2] * inv, sum[3] * inv};
            store_b16_4(a.out, a.Kb_out, run.x, h * vt * 16 + v * 16 + 4 * g4, y);
        } else {
            const size_t slice = ((size_t)run_id * a.H + h) * a.nsplit + split;
            *reinterpret_cast<f4_t*>(a.part_acc + slice * (16 * vt) + v * 16 + 4 * g4) = sum;
            if (v == 0 && g4 == 0) *reinterpret_cast<float2*>(a.part_ml + 2 * slice) = make_float2(mx, l);
        }
    }
}

__global__ __launch_bounds__(64) void k_window_merge(WindowKArgs a) {
    const int run_id = blockIdx.x, h = blockIdx.y, row = 16 * a.vt, t = a.runs[run_id].x;
    const size_t slice = ((size_t)run_id * a.H + h) * a.nsplit;
    float mx = -1e30f, l = 0.f;
    for (int s = 0; s < a.nsplit; s++) mx = fmaxf(mx, a.part_ml[2 * (slice + s)]);
    for (int s = 0; s < a.nsplit; s++) l += __builtin_amdgcn_exp2f(a.part_ml[2 * (slice + s)] - mx) * a.part_ml[2 * (slice + s) + 1];
    for (int d = 4 * threadIdx.x; d < row; d += 256) {
        f4_t sum = {0.f, 0.f, 0.f, 0.f};
        for (int s = 0; s < a.nsplit; s++)
            sum += __builtin_amdgcn_exp2f(a.part_ml[2 * (slice + s)] - mx) * *reinterpret_cast<const f4_t*>(a.part_acc + (slice + s) * row + d);
        const float y[4] = {sum[0] / l, sum[1] / l, sum[2] / l, sum[3] / l};
        store_b16_4(a.out, a.Kb_out, t, h * row + d, y);
    }
}

template <int KC, int VT, int C, bool SINGLE, int CAP, bool EXACT>
static void launch_win(const WindowKArgs& a, int grid) {
    constexpr int WAVES = window_waves(VT, SINGLE);
    const size_t shmem = SINGLE ? window_lds(VT, WAVES) : 0;
    static bool enabled = false;
    if (shmem > 64 * 1024 && !enabled) {
        HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_window_attn<KC, VT, C, SINGLE, CAP, EXACT>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem));
        enabled = true;
    }
    NVLLM_LAUNCH((k_window_attn<KC, VT, C, SINGLE, CAP, EXACT>), dim3(grid), dim3(64 * WAVES), shmem, a);
}
template <int KC, int VT, int C, bool SINGLE, int CAP>
static void launch_win_exact(const WindowKArgs& a, int grid) {
    if (a.kc == KC && a.vt == VT) launch_win<KC, VT, C, SINGLE, CAP, true>(a, grid);
    else launch_win<KC, VT, C, SINGLE, CAP, false>(a, grid);
}
template <int KC, int VT, int C, bool SINGLE>
static void launch_win_cap(const WindowKArgs& a, int grid) {
    if (a.cap <= 0.f) launch_win_exact<KC, VT, C, SINGLE, 0>(a, grid);
    else if (a.cap <= CAP_FIXED) launch_win_exact<KC, VT, C, SINGLE, 1>(a, grid);
    else launch_win_exact<KC, VT, C, SINGLE, 2>(a, grid);
}

// Keys up to which a token's window stays whole: the merge of slices is a launch of its own.  Passes of twelve layers, 1, 6, 16 and 30
// rows, sliced -> whole: heads of 64 values at 1,500 keys 562 -> 526, 586 -> 544, 609 -> 580, 646 -> 626 us; of 128 at 900 565 -> 543, 587 -> 562,
// 636 -> 633, 669 -> 651, at 1,200 564 -> 555, 585 -> 576, 644 -> 683, 689 -> 689; of 256 at 520 574 -> 554, 595 -> 571, 623 -> 603, 639 -> 640, at 700
// 576 -> 573, 590 -> 594, 631 -> 630, 660 -> 692; of 192, in the form for other widths, at 300 601 -> 590, 618 -> 613, 637 -> 643, 647 -> 654, at 400
// 599 -> 634, 604 -> 645, 649 -> 686, 675 -> 736 (160: at 400 the same; 224: as 192).
static int window_whole(int cls, bool exact) { return cls == 0 ? 1536 : cls == 1 ? 960 : exact ? 576 : 320; }
void launch_window_attention(const WindowAttn& w, const StepArrays& st) {
    if (st.n_runs <= 0) return;
    const KvPages& pool = w.pool;
    if (w.H % pool.G) NVLLM_FATAL("%d query heads do not divide over %d key/value heads", w.H, pool.G);
    if (w.size < 1 || w.keep_first < 0) NVLLM_FATAL("a window of %d tokens with %d kept", w.size, w.keep_first);
    const int kc = pool.dim_ld / 32, vt = pool.vdim_ld / 16, rep = w.H / pool.G;
    const int ppb = pool.block_size / KV_PAGE;
    const int Kb_out = w.H * pool.vdim_ld / 32;
    if (pool.elem_bytes == 4 || kc > 8 || vt > 16 || (ppb & (ppb - 1))) {
        const size_t lds = ((size_t)pool.dim_ld + pool.vdim_ld + 256 + 8 + 256) * 4;
        if (lds > 64 * 1024) NVLLM_FATAL("attention heads of %d and %d values are too wide", pool.dim, pool.vdim);
        ProfScope ps(PC_WINDOW_ATTN, 0, 0);
        if (launch_window_rows(w, st)) return;
        if (pool.elem_bytes != 4) launch_window_any<true, 1>(w, st, Kb_out);
        else if (pool.dim % 4 || pool.vdim % 4) launch_window_any<false, 1>(w, st, Kb_out);
        else launch_window_any<false, 4>(w, st, Kb_out);
        return;
    }
    WindowKArgs a{};
    a.keys = (const __half*)pool.keys;
    a.values = (const __half*)pool.values;
    a.q = (const __half*)w.q;
    a.tables = st.d_tables;
    a.G = pool.G; a.rep = rep; a.H = w.H; a.kc = kc; a.vt = vt; a.size = w.size; a.keep = w.keep_first; a.scale = w.scale; a.cap = w.cap;
    a.page_shift = __builtin_ctz(ppb);
    a.out = w.out_b16;
    a.Kb_out = Kb_out;
    a.nsplit = 1;
    const int cls = kc <= 2 && vt <= 4 ? 0 : kc <= 4 && vt <= 8 ? 1 : 2;
    const long seen_cap = (long)w.size + w.keep_first;   // keys a token sees at most
    const double kv_bytes = (double)pool.G * (pool.dim_ld + pool.vdim_ld) * 2.0, io_bytes = (double)w.H * (pool.dim_ld + pool.vdim_ld) * 2.0;
    const double pair_flops = 2.0 * w.H * (pool.dim_ld + pool.vdim_ld);
    if (st.n_multi > 0) {
        a.runs = (const int4*)st.d_runs;
        a.n_runs = st.n_multi;
        // wide items share more of a page's load, narrow ones are more waves: the widest that still gives every SIMD one
        int C = cls == 0 ? 4 : cls == 1 ? 2 : 1, waves = 0;
        for (;; C /= 2) {
            a.HW = rep >= C ? C : rep >= 2 && C >= 2 ? 2 : 1;
            a.NHG = cdiv(rep, a.HW);
            a.n_sub = cdiv(std::min(st.max_run, WINDOW_RUN), 16 * C / a.HW);
            waves = a.G * a.n_runs * a.n_sub * a.NHG;
            if (C == 1 || waves >= 4 * rt().num_cus) break;
        }
        const int grid = cdiv(waves, 4);
        const double rows = (double)st.multi_rows(seen_cap), pairs = (double)st.multi_pairs(seen_cap);
        ProfScope ps(PC_WINDOW_ATTN, rows * kv_bytes + (double)(st.T - (st.n_runs - st.n_multi)) * io_bytes, pairs * pair_flops);
        if (cls == 0 && C == 4) launch_win_cap<2, 4, 4, false>(a, grid);
        else if (cls == 0 && C == 2) launch_win_cap<2, 4, 2, false>(a, grid);
        else if (cls == 0) launch_win_cap<2, 4, 1, false>(a, grid);
        else if (cls == 1 && C == 2) launch_win_cap<4, 8, 2, false>(a, grid);
        else if (cls == 1) launch_win_cap<4, 8, 1, false>(a, grid);
        else launch_win_cap<8, 16, 1, false>(a, grid);
    }
    const int n_single = st.n_runs - st.n_multi;
    if (n_single > 0) {
        a.runs = (const int4*)st.d_runs + st.n_multi;
        a.n_runs = n_single;
        a.n_sub = 1;
        a.HW = 16;
        a.NHG = cdiv(rep, 16);
        const int items = n_single * a.G * a.NHG, waves = window_waves(cls == 0 ? 4 : cls == 1 ? 8 : 16, true);
        const long longest = std::min<long>(st.max_pos + 1, seen_cap + 32);
        // slices until every CU has a workgroup, each wave of a slice with at least one pair of pages
        const int whole = window_whole(cls, kc == 8 && vt == 16);
        a.nsplit = longest <= whole ? 1 : (int)std::max<long>(1, std::min<long>(rt().num_cus / items, longest / 32 / waves));
        if (a.nsplit > 1) {
            const size_t slices = (size_t)n_single * w.H * a.nsplit;
            a.part_acc = (float*)ws_get(WS_ATT_PART, slices * (16 * vt + 2) * sizeof(float));
            a.part_ml = a.part_acc + slices * 16 * vt;
        }
        {
            const double rows = (double)st.single_rows(seen_cap);
            ProfScope ps(PC_WINDOW_ATTN_TOK, rows * kv_bytes + (double)n_single * io_bytes, rows * pair_flops);
            const int grid = items * a.nsplit;
            if (cls == 0) launch_win_cap<2, 4, 1, true>(a, grid);
            else if (cls == 1) launch_win_cap<4, 8, 1, true>(a, grid);
            else launch_win_cap<8, 16, 1, true>(a, grid);
        }
        if (a.nsplit > 1) {
            ProfScope ps(PC_ATTN_COMBINE, (double)n_single * w.H * (a.nsplit + 0.5) * vt * 64.0, 0);
            NVLLM_LAUNCH(k_window_merge, dim3(n_single, w.H), dim3(64), 0, a);
        }
    }
}

}  // namespace nvllm
