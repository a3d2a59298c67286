// The layers of a Llama-shaped prefill on one GPU, issued from one call (host code: every launch is one of the
// library's own entry points).  A layer is eight to twelve launches; from Python each costs about 10 us of the host's
// time, which at short prompts is more than it runs for: 5 to 100 tokens through 22 layers of hidden size 2048 all took
// 2.5 ms, for 1.9 ms of kernels at 37.
//
// The launches are those of the layer taken op by op, with one exception: where the O or the down projection is cut into
// k-slices, the launch that adds them also does the addition and the norm behind the projection (gemm_prefill_run with a
// PostNorm), one launch and one pass over the rows less.  Same results bit for bit.  Whole prompts through 22 layers of hidden
// size 2048 (us, op by op from Python -> here): 37 tokens 2480 -> 1587, of which the projections' short form is about 250;
// four prompts of 509 through 16 layers of hidden size 4096 do not change: there the kernels outlast the host.
#include "common.h"

namespace mv {
enum { kLn1, kWqkv, kBqkv, kWo, kLn2, kWgu, kWd, kKcache, kVcache, kTensors };
}  // namespace mv

extern "C" size_t mv_llama_prefill_workspace_bytes(int tokens, int hidden, int inter, int hq, int hkv, int d) {
    if (tokens <= 0 || hidden <= 0 || inter <= 0 || hq <= 0 || hkv <= 0 || d <= 0) return 0;
    const int shapes[4][2] = {{(hq + 2 * hkv) * d, hidden}, {hidden, hq * d}, {2 * inter, hidden}, {hidden, inter}};
    size_t need = 0;
    for (int i = 0; i < 4; ++i) {
        const size_t b = mv_gemm_prefill_workspace_bytes(tokens, shapes[i][0], shapes[i][1]);
        if (b > need) need = b;
    }
    return need;
}

extern "C" int mv_llama_prefill_layers(const void* const* tensors, const float* eps, int n_layers, int rows, int seq,
                                       int hidden, int inter, int hq, int hkv, int d, const void* rot_cos,
                                       const void* rot_sin, int rot_max_pos, const int32_t* cache_seqlens,
                                       const int32_t* block_table, int bt_stride, int page, int num_pages, void* h,
                                       void* normed, void* qkv, void* attn, void* proj, void* resid, void* act,
                                       float scale, void* workspace, size_t workspace_bytes, mv_stream_t stream) {
    using namespace mv;
    if (!tensors || !eps || n_layers < 0 || rows <= 0 || seq <= 0 || (int64_t)rows * seq > 0x7fffffff) return MV_ERR_INVALID_ARG;
    if (!h || !normed || !qkv || !attn || !proj || !resid || !act) return MV_ERR_INVALID_ARG;
    if (hidden <= 0 || inter <= 0 || hq <= 0 || hkv <= 0 || d <= 0) return MV_ERR_INVALID_ARG;
    if (hidden % 64 || inter % 64 || (hq * d) % 64 || ((hq + 2 * hkv) * d) % 16) return MV_ERR_UNSUPPORTED;
    for (const void* p : {(const void*)h, (const void*)normed, (const void*)qkv, (const void*)attn, (const void*)proj,
                          (const void*)resid, (const void*)act})
        if (!aligned16(p)) return MV_ERR_INVALID_ARG;
    for (int i = 0; i < n_layers * kTensors; ++i)
        if (i % kTensors != kBqkv && (!tensors[i] || !aligned16(tensors[i]))) return MV_ERR_INVALID_ARG;
    if (workspace_bytes < mv_llama_prefill_workspace_bytes(rows * seq, hidden, inter, hq, hkv, d) ||
        (workspace_bytes && (!workspace || !aligned16(workspace))))
        return MV_ERR_INVALID_ARG;
    const int T = rows * seq, nq = hq * d, nqkv = (hq + 2 * hkv) * d;
    int rc = MV_OK;
    auto project = [&](const void* x, int k, const void* w, const void* bias, const void* residual, void* y, int ncols, int n,
                       int flags, PostNorm* norm) {
        return gemm_prefill_run(x, k, w, bias, residual, residual ? n : 0, y, ncols, T, n, k, flags, workspace, workspace_bytes,
                                norm, stream);
    };
    bool normed_done = false;
    for (int li = 0; li < n_layers && rc == MV_OK; ++li) {
        const void* const* t = tensors + (int64_t)li * kTensors;
        if (!normed_done) rc = mv_rmsnorm(h, t[kLn1], normed, T, hidden, hidden, hidden, eps[2 * li], stream);
        if (rc == MV_OK) rc = project(normed, hidden, t[kWqkv], t[kBqkv], nullptr, qkv, nqkv, nqkv, 0, nullptr);
        if (rc == MV_OK)
            rc = mv_rope_attn_prefill(qkv, nqkv, rot_cos, rot_sin, rot_max_pos, cache_seqlens, block_table, bt_stride,
                                      (void*)t[kKcache], (void*)t[kVcache], attn, nq, rows, seq, hq, hkv, d, page, num_pages, scale,
                                      stream);
        if (rc != MV_OK) break;
        // resid = attention's projection + h with its norm (over the unrounded sum, as mv_rmsnorm_residual takes it)
        PostNorm ln2 = {h, resid, t[kLn2], eps[2 * li + 1], normed, hidden, 0, (float*)proj, false};
        rc = project(attn, nq, t[kWo], nullptr, nullptr, proj, hidden, hidden, 0, &ln2);
        if (rc == MV_OK && !ln2.done)
            rc = mv_rmsnorm_residual(proj, h, t[kLn2], normed, resid, T, hidden, hidden, hidden, hidden, hidden, eps[2 * li + 1],
                                     stream);
        if (rc == MV_OK) rc = project(normed, hidden, t[kWgu], nullptr, nullptr, act, inter, 2 * inter, MV_GEMM_SWIGLU, nullptr);
        // h = the MLP's projection + resid, with the next layer's first norm (of the rounded sum, as mv_rmsnorm reads it)
        PostNorm ln1 = {resid, h, nullptr, 0.f, normed, hidden, 1, (float*)proj, false};
        if (li + 1 < n_layers) {
            ln1.ln_w = t[kTensors + kLn1];
            ln1.eps = eps[2 * li + 2];
        }
        if (rc == MV_OK)
            rc = project(act, inter, t[kWd], nullptr, resid, h, hidden, hidden, 0, ln1.ln_w ? &ln1 : nullptr);
        normed_done = ln1.done;
    }
    return rc;
}
