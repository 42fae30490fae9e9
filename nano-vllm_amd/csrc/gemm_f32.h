// gemm_f32.h -- projections whose activations are fp32 rows: of fp32 weights (row-major, as the files hold them), and of
// fp16 weights in tile order for a few tokens.
#pragma once

#include "moe.h"

namespace nvllm {

// What happens to a segment's complete sums y[t][n].
enum class F32Out {
    STORE,    // out[t][n] = y
    ADD,      // out[t][n] += y (residual)
    SILU,     // y * sigmoid(y)
    RELU2,    // max(y, 0)^2
    ROPE_Q,   // rotated -> out
    ROPE_K,   // rotated -> key rows of the block pool
    KV_V      // -> value rows of the block pool
};
struct F32Segment {
    const float* W;      // [N][K]; fp16 weights: tiles, ...
    const float* W2;     // second matrix of a gated pair: out = silu(y + bias) * (y2 + bias2) (null: none)
    const float *bias, *bias2;   // of a pair, per feature (null: none)
    long nb_stride;      // ... halves between their 16-row blocks
    int N;
    F32Out kind;
    float* out;          // [T][ldo]
    int ldo;
    int first;           // first feature tile of the launch (set by the launcher)
    bool vec;            // 16-byte stores (set by the launcher)
};
constexpr int F32_SEGMENTS = 4;
struct F32Gemm {
    const float* in;               // [rows][K]
    const int* in_rows = nullptr;  // row of `in` that token t reads (null: t)
    const float* gain = nullptr;   // RMS norm of the input: in * gain / rms(in)
    float eps = 0.f;
    int K, T;
    int n_segs = 0;
    F32Segment seg[F32_SEGMENTS];
    // rows sorted by expert, 16 of one expert at a time (moe.h): expert of a 16-row block (-1: none), floats between the
    // experts' matrices, and what a row's results are scaled by (null: nothing)
    const int* block_expert = nullptr;
    long expert_stride = 0;
    const float* row_weight = nullptr;
    int live, touched = 1;   // for the figures of a profile: rows that are some token's, matrices they can be of
    // one STORE segment: its rows also go to this page-locked host array, laid out like its `out` (null: no)
    float* out_host = nullptr;
    // one STORE segment: (maximum, its first index) of each 16 outputs of a token -> [block][amax_ld] ...
    float2* amax_pairs = nullptr;
    int amax_ld = 0;
    // ... and with them (launch_gemm_f32): every token's first index of its maximum, merged by a launch of its own; to a page-locked host array too
    int* amax_out = nullptr;
    int* amax_out_host = nullptr;
    // a mixture's choices and their sorting in one more workgroup, of pairs behind a norm (route.T 0: none)
    RoutePlan route{};
    const float* z = nullptr;   // router logits [T][ldz]
    int ldz = 0;
    int route_from;             // that workgroup (grid x, set by the launcher)
    // ROPE_*, KV_V
    const int* pos = nullptr;
    const int* kv_row = nullptr;
    const float2* rope = nullptr;
    void* pool_k = nullptr;
    void* pool_v = nullptr;
    int hd = 0, KD = 0, kv_elem_bytes = 4, bs = 16;
    long layer_off = 0;

    F32Gemm(const float* in_, int T_, int K_) : in(in_), K(K_), T(T_), live(T_) {}
    F32Gemm& norm(const float* g, float e) {
        gain = g;
        eps = e;
        return *this;
    }
    F32Gemm& add(const float* W, int N, float* out, F32Out kind = F32Out::STORE) {
        seg[n_segs++] = F32Segment{W, nullptr, nullptr, nullptr, 0, N, kind, out, N, 0, false};
        return *this;
    }
    F32Gemm& add16(const __half* tiles, long nb_stride, int N, float* out, F32Out kind = F32Out::STORE, const __half* tiles2 = nullptr) {
        seg[n_segs++] = F32Segment{(const float*)tiles, (const float*)tiles2, nullptr, nullptr, nb_stride, N, kind, out, N, 0, false};
        return *this;
    }
    F32Gemm& add_pair(const float* gate, const float* up, int N, float* out, const float* bias_gate = nullptr, const float* bias_up = nullptr) {
        seg[n_segs++] = F32Segment{gate, up, bias_gate, bias_up, 0, N, F32Out::STORE, out, N, 0, false};
        return *this;
    }
    F32Gemm& choose(const RoutePlan& r, const float* logits, int ld) {
        route = r;
        z = logits;
        ldz = ld;
        return *this;
    }
    F32Gemm& experts(const RoutePlan& r, long stride, const float* weight) {
        block_expert = r.block_expert;
        expert_stride = stride;
        row_weight = weight;
        live = r.T * r.top;
        touched = r.E < live ? r.E : live;
        return *this;
    }
};
// One launch for all segments: all of them gated pairs, or none.  Whether g.route rode.
bool launch_gemm_f32(const F32Gemm& g, int prof_cls);

// The same for fp16 weights in tile order (add16) and up to THIN_TOKENS tokens; K % 32 == 0.  Activations enter the matrix
// cores as fp16 hi + lo, as in gemm.hip.
constexpr int THIN_TOKENS = 6;   // (at most 16: one block of tokens)
void launch_gemm_thin(const F32Gemm& g, int prof_cls);

}  // namespace nvllm
