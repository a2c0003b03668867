// One decode step of a model as a single call: the launches of lyra/model.py:734-793 in decode mode (one token per sequence),
// issued from native code in the order in which the Python driver issues them, on the same kernels with the same arguments.
// Host code only.  What it saves is the host's work between launches: 8-12 us each from Python - reading tensors, allocating
// results, marshalling 25 arguments - against 2.5 us here, with 119-131 launches per step of lyra-small.
#include <algorithm>

#include "lyra_device.h"

namespace lyra {
namespace {

// Results of a layer live in one of two halves of the caller's scratch memory; the next layer writes the other one.
struct Carve {
    char* base = nullptr;
    size_t used = 0;
    template <typename T = void>
    T* take(size_t bytes) {
        char* p = base ? base + used : nullptr;
        used += (bytes + 255) / 256 * 256;
        return (T*)p;
    }
};

// The residual stream between layers: complete rows (x), token ids not gathered yet, the slices of a projection that still
// have to be added to x, or the expert outputs that still have to be combined with it.
struct Stream {
    enum Kind { kTokens, kRows, kSlices, kExperts } kind = kTokens;
    const void* x = nullptr;
    const float* slices = nullptr;
    int splits = 0;
    const float* bias = nullptr;
    float scale = 1.f;
    const void* rows = nullptr;
    const float* scores = nullptr;
    const int32_t* dest = nullptr;
};

struct Step {
    const lyra_step_t& s;
    bool dry;  // sizes only: nothing is launched
    Carve mem;
    const int32_t* one;
    lyra_stream_t st;

    size_t f32(size_t n) const { return n * sizeof(float); }
    size_t bf16(size_t rows, size_t cols) const { return rows * cols * 2; }
    size_t tiled(size_t cols) const { return ((size_t)s.B + 15) / 16 * 16 * cols * 2; }

    // RMS norm of the stream (completing it on the way) with an optional narrow projection; x becomes the completed rows
    int norm(Stream& t, const float* scale, void* h, const float* proj, const float* bias, void* y, int n, int mode) {
        const size_t xbytes = bf16(s.B, s.C);
        int rc = LYRA_OK;
        if (t.kind == Stream::kRows) {
            if (!dry) rc = lyra_rmsnorm_proj(t.x, scale, h, proj, bias, y, s.B, s.C, n, mode, s.eps, st);
            return rc;
        }
        void* x = mem.take(xbytes);
        if (!dry) {
            if (t.kind == Stream::kTokens)
                rc = lyra_rmsnorm_proj_embed(s.table, s.tokens, s.table_rows, x, scale, h, proj, bias, y, s.B, s.C, n, mode, s.eps, st);
            else if (t.kind == Stream::kSlices)
                rc = lyra_rmsnorm_proj_sum_bias(nullptr, t.slices, t.splits, t.bias, t.x, t.scale, x, scale, h, proj, bias, y, s.B, s.C, n,
                                                mode, s.eps, st);
            else
                rc = lyra_rmsnorm_proj_combine(t.rows, t.scores, t.dest, s.k_routed + s.n_shared, t.x, t.scale, x, scale, h, proj, bias,
                                               y, s.B, s.C, n, mode, s.eps, st);
        }
        t.kind = Stream::kRows;
        t.x = x;
        return rc;
    }

    // lhs @ w as K slices (splits > 0), rows: lhs holds B rows of K
    int partials(const void* lhs, bool lhs_tiled, const lyra_matrix_t& w, int K, int N, int splits, float* out) {
        if (dry) return LYRA_OK;
        return lyra_decode_gemm_partials(lhs, w.data, w.scale, w.bk, w.bn, one, out, f32((size_t)splits * s.B * N), s.B, K, N,
                                         w.dtype | (lhs_tiled ? LYRA_LHS_TILED16 : 0), st);
    }

    int attention(const lyra_layer_t& l, Stream& t) {
        const int W = (s.N + 2 * s.K) * s.H, heads = s.N * s.H;
        const int splits = lyra_decode_gemm_splits(s.B, s.C, W, l.qkv.scale ? l.qkv.bk : 0);
        void* h = mem.take(tiled(s.C));
        void* gate = l.gate_t ? mem.take(bf16(s.B, s.N)) : nullptr;
        int rc = norm(t, l.attn_norm, h, l.gate_t, nullptr, gate, l.gate_t ? s.N : 0, 1 | 4);
        if (rc != LYRA_OK) return rc;
        float* part = splits > 0 ? mem.take<float>(f32((size_t)splits * s.B * W)) : nullptr;
        void* qkv = splits > 0 ? nullptr : mem.take(bf16(s.B, W));
        void* out = mem.take(bf16(s.B, heads));
        rc = splits > 0 ? partials(h, true, l.qkv, s.C, W, splits, part)
                        : gemm(h, true, l.qkv, s.C, W, l.qkv_bias, l.qkv_bias ? 2 : 0, nullptr, 1.f, qkv);
        if (rc != LYRA_OK) return rc;
        if (!dry)
            rc = lyra_decode_attention_qkv_bias(qkv, part, splits, splits > 0 ? l.qkv_bias : nullptr, l.qnorm, l.knorm, s.cos_t, s.sin_t,
                                                s.rope_rows, s.eps, l.k, l.v, l.ks, l.vs, l.sinks, s.position, 0, gate, out,
                                                s.attn_ws, s.attn_ws_bytes, s.B, s.N, s.K, l.S, s.H, s.sm_scale, l.sliding_window,
                                                s.kv_dtype, LYRA_DTYPE_BF16, st);
        if (rc != LYRA_OK) return rc;
        return leave(t, out, false, l.out, heads, l.out_bias, s.residual_scale, t.x);
    }

    // one-group product summed by the launch itself; post: bits of lyra_decode_gemm_ex's post_scale
    int gemm(const void* lhs, bool lhs_tiled, const lyra_matrix_t& w, int K, int N, const float* bias, int post, const void* residual,
             float scale, void* out) {
        if (dry) return LYRA_OK;
        return lyra_decode_gemm_ex(lhs, nullptr, w.data, w.scale, w.bk, w.bn, one, bias, residual, scale, post, out, s.gemm_ws,
                                   s.gemm_ws_bytes, s.B, 1, K, N, w.dtype | (lhs_tiled ? LYRA_LHS_TILED16 : 0), LYRA_DTYPE_BF16, 0, s.beta,
                                   s.limit, st);
    }

    // the projection that ends a block, left to whoever reads the stream next where it runs split over K
    int leave(Stream& t, const void* lhs, bool lhs_tiled, const lyra_matrix_t& w, int K, const float* bias, float scale, const void* x) {
        const int splits = lyra_decode_gemm_splits(s.B, K, s.C, w.scale ? w.bk : 0);
        if (splits > 0) {
            float* part = mem.take<float>(f32((size_t)splits * s.B * s.C));
            t = Stream{};
            t.kind = Stream::kSlices;
            t.x = x; t.slices = part; t.splits = splits; t.bias = bias; t.scale = scale;
            return partials(lhs, lhs_tiled, w, K, s.C, splits, part);
        }
        void* out = mem.take(bf16(s.B, s.C));
        t = Stream{};
        t.kind = Stream::kRows;
        t.x = out;
        return gemm(lhs, lhs_tiled, w, K, s.C, bias, 1 | (bias ? 2 : 0), x, scale, out);
    }

    int dense(const lyra_layer_t& l, Stream& t) {
        const int Hd = s.dense_hidden;
        void* h = mem.take(tiled(s.C));
        void* act = mem.take(tiled(Hd));
        int rc = norm(t, l.mlp_norm, h, nullptr, nullptr, nullptr, 0, 2 | 4);
        const int bk_down = l.down.scale ? l.down.bk : 0;
        const int up = lyra_rows_proj_swiglu_exists(s.B, Hd, s.C, bk_down) ? lyra_decode_gemm_splits(s.B, s.C, 2 * Hd, l.up.scale ? l.up.bk : 0) : 0;
        if (rc == LYRA_OK && up > 0) {  // a few rows: SwiGLU inside the down projection's launch
            const int down = lyra_decode_gemm_splits(s.B, Hd, s.C, bk_down);
            float* part = mem.take<float>(f32((size_t)up * s.B * 2 * Hd));
            float* dpart = mem.take<float>(f32((size_t)down * s.B * s.C));
            rc = partials(h, true, l.up, s.C, 2 * Hd, up, part);
            if (rc == LYRA_OK && !dry)
                rc = lyra_rows_proj_swiglu(part, up, l.up_bias, s.beta, s.limit, l.down.data, l.down.scale, l.down.bk, l.down.bn, dpart,
                                           f32((size_t)down * s.B * s.C), s.B, Hd, s.C, l.down.dtype, st);
            const void* x = t.x;
            t = Stream{};
            t.kind = Stream::kSlices;
            t.x = x; t.slices = dpart; t.splits = down; t.bias = l.down_bias; t.scale = s.dense_residual_scale;
            return rc;
        }
        if (rc == LYRA_OK && !dry)
            rc = lyra_decode_gemm_ex(h, nullptr, l.up.data, l.up.scale, l.up.bk, l.up.bn, one, l.up_bias, nullptr, 1.f, 0, act, s.gemm_ws,
                                     s.gemm_ws_bytes, s.B, 1, s.C, 2 * Hd, l.up.dtype | LYRA_LHS_TILED16 | LYRA_OUT_TILED16,
                                     LYRA_DTYPE_BF16, 1, s.beta, s.limit, st);
        if (rc != LYRA_OK) return rc;
        return leave(t, act, true, l.down, Hd, l.down_bias, s.dense_residual_scale, t.x);
    }

    int experts(const lyra_layer_t& l, Stream& t) {
        const int topk = s.k_routed + s.n_shared, E = s.n_routed + s.n_shared, M = s.B * topk, Hd = s.expert_hidden;
        void* h = mem.take(tiled(s.C));
        float* logits = mem.take<float>(f32((size_t)s.B * s.n_routed));
        int rc = norm(t, l.mlp_norm, h, l.router_t, l.router_bias, logits, s.n_routed, 2 | 4);
        if (rc != LYRA_OK) return rc;
        float* scores = mem.take<float>(f32(M));
        int32_t* groups = mem.take<int32_t>(f32(E));
        int32_t* row_map = mem.take<int32_t>(f32(M));
        int32_t* dest = mem.take<int32_t>(f32(M));
        void* act = mem.take(((size_t)M + 15) / 16 * 16 * Hd * 2);
        void* rows = mem.take(bf16(M, s.C));
        if (!dry) {
            rc = lyra_moe_route(logits, scores, groups, row_map, dest, s.B, s.n_routed, s.n_shared, s.k_routed, st);
            if (rc != LYRA_OK) return rc;
            rc = lyra_decode_gemm_ex(h, row_map, l.up.data, l.up.scale, l.up.bk, l.up.bn, groups, l.up_bias, nullptr, 1.f, 0, act, s.gemm_ws,
                                     s.gemm_ws_bytes, M, E, s.C, 2 * Hd, l.up.dtype | LYRA_LHS_TILED16 | LYRA_OUT_TILED16, LYRA_DTYPE_BF16,
                                     1, s.beta, s.limit, st);
            if (rc != LYRA_OK) return rc;
            rc = lyra_decode_gemm_ex(act, nullptr, l.down.data, l.down.scale, l.down.bk, l.down.bn, groups, l.down_bias, nullptr, 1.f, 0,
                                     rows, s.gemm_ws, s.gemm_ws_bytes, M, E, Hd, s.C, l.down.dtype | LYRA_LHS_TILED16, LYRA_DTYPE_BF16, 0,
                                     s.beta, s.limit, st);
            if (rc != LYRA_OK) return rc;
        }
        const void* x = t.x;
        t = Stream{};
        t.kind = Stream::kExperts;
        t.x = x; t.scale = s.residual_scale; t.rows = rows; t.scores = scores; t.dest = dest;
        return LYRA_OK;
    }

    // every layer and the final norm; `half`: bytes of one half of the scratch memory (dry: the most a layer needs, returned)
    int run(size_t& half) {
        Stream t;
        size_t most = 0;
        for (int i = 0; i <= s.n_layers; ++i) {
            mem.used = 0;
            mem.base = dry ? nullptr : (char*)s.scratch + (i & 1) * half;
            int rc;
            if (i < s.n_layers) {
                const lyra_layer_t& l = s.layers[i];
                rc = attention(l, t);
                if (rc == LYRA_OK) rc = l.router_t ? experts(l, t) : dense(l, t);
            } else {
                rc = norm(t, s.final_norm, s.out, nullptr, nullptr, nullptr, 0, 2);
            }
            if (rc != LYRA_OK) return rc;
            most = std::max(most, mem.used);
        }
        if (dry) half = most;
        return LYRA_OK;
    }
};

int check(const lyra_step_t* s) {
    if (!s || !s->layers || s->n_layers <= 0 || s->B <= 0 || s->C <= 0 || s->N <= 0 || s->K <= 0 || s->H <= 0 || s->N % s->K) return LYRA_E_BADARG;
    if (s->C % 32 || (s->N * s->H) % 32 || s->B > LYRA_MAX_ROW_COUNT) return LYRA_E_UNSUPPORTED;
    for (int i = 0; i < s->n_layers; ++i) {
        const lyra_layer_t& l = s->layers[i];
        if (!l.attn_norm || !l.qkv.data || !l.out.data || !l.sinks || !l.k || !l.v || !l.mlp_norm || !l.up.data || !l.down.data) return LYRA_E_BADARG;
        const int hidden = l.router_t ? s->expert_hidden : s->dense_hidden;
        if (hidden <= 0 || hidden % 32) return LYRA_E_UNSUPPORTED;
        if (l.router_t && (s->n_routed <= 0 || s->k_routed <= 0 || s->n_shared < 0 || s->n_routed + s->n_shared < 2 || s->k_routed + s->n_shared > 16))
            return LYRA_E_UNSUPPORTED;
    }
    return LYRA_OK;
}

}  // namespace
}  // namespace lyra

extern "C" size_t lyra_decode_step_scratch(const lyra_step_t* step) {
    if (lyra::check(step) != LYRA_OK) return 0;
    lyra::Step run{*step, true, {}, nullptr, nullptr};
    size_t half = 0;
    return run.run(half) == LYRA_OK ? 2 * half : 0;
}

extern "C" int lyra_decode_step(const lyra_step_t* step, lyra_stream_t stream) {
    const int rc = lyra::check(step);
    if (rc != LYRA_OK) return rc;
    if (!step->table || !step->tokens || !step->cos_t || !step->sin_t || !step->position || !step->final_norm || !step->out || !step->scratch)
        return LYRA_E_BADARG;
    // all of the scratch memory is there before anything is launched (the pass that counts it takes a microsecond)
    lyra::Step count{*step, true, {}, nullptr, nullptr};
    size_t half = 0;
    const int fits = count.run(half);
    if (fits != LYRA_OK) return fits;
    if ((uintptr_t)step->scratch % 256 || step->scratch_bytes / 2 < half) return LYRA_E_WORKSPACE;
    const int32_t* counts = (const int32_t*)lyra_row_counts();
    if (!counts) return LYRA_E_LAUNCH;
    lyra::Step run{*step, false, {}, counts + step->B, stream};
    return run.run(half);
}
