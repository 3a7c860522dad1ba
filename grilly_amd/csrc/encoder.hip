// One post-LN BERT encoder layer as a fixed sequence of launches on the context stream:
//   QKV GEMM (packed weight) -> flash attention on the packed buffer -> out-proj GEMM
//   -> LayerNorm(residual) -> FFN1 GEMM + GELU epilogue -> FFN2 GEMM -> LayerNorm(residual)
// Activations stay in HBM between kernels; nothing returns to the host.
// Recipe: utils/vulkan_sentence_transformer.py:972-1035 (post-LN order, eps passed by the
// caller, tanh GELU, key-padding mask as additive -1e9 bias, heads = plain reshape of the
// last dimension :985-995).
#include "common.hpp"
#include <cmath>
#include <cstring>

extern "C" int64_t grl_bert_layer_workspace(int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int64_t d_ff) {
    if (!grl_valid_dtype(dtype) || B < 0 || S < 0 || H <= 0 || D <= 0 || d_ff <= 0) return -1;
    const int64_t M = B * S, d = H * D;
    // qkv (M,3d) | attn (M,d) | proj (M,d) | ff (M,d_ff); each region padded to 256 B
    auto pad = [](int64_t v) { return (v + 255) / 256 * 256; };
    const int64_t es = (int64_t)grl_dtype_size(dtype);
    return pad(M * 3 * d * es) + 2 * pad(M * d * es) + pad(M * d_ff * es);
}

// attention on the packed (M, 3d) projection, of a rectangular batch (rg null) or a ragged one
static int layer_attention(grl_ctx* c, int dtype, int64_t B, int64_t S, int64_t H, int64_t D, const char* qkv, const float* mask, char* attn,
                           const grl_ragged* rg) {
    const int64_t d = H * D, es = (int64_t)grl_dtype_size(dtype);
    const float scale = 1.0f / sqrtf((float)D);
    if (rg) return grl_fa2_fwd_ragged(c, dtype, rg, H, D, qkv, qkv + d * es, qkv + 2 * d * es, attn, 3 * d, 3 * d, 3 * d, d, scale, 0,
                                      GRL_ROPE_NONE, 10000.f, 1.f);
    return grl_fa2_fwd_strided(c, dtype, B, S, H, D, qkv, qkv + d * es, qkv + 2 * d * es, mask, attn, 3 * d, 3 * d, 3 * d, d, scale, 0,
                               GRL_ROPE_NONE, 10000.f, 1.f);
}

static int bert_layer(grl_ctx* c, int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int64_t d_ff,
                      const grl_bert_layer* w, const float* mask, float eps, void* x, void* workspace, const grl_ragged* rg) {
    GRL_REQUIRE(c && w && x && workspace, GRL_ERR_ARG, "grl_bert_layer_fwd: null argument");
    GRL_REQUIRE(grl_valid_dtype(dtype), GRL_ERR_ARG, "grl_bert_layer_fwd: bad dtype %d", dtype);
    GRL_REQUIRE(B >= 0 && S >= 0 && H > 0 && d_ff > 0, GRL_ERR_SHAPE, "grl_bert_layer_fwd: bad shape");
    GRL_REQUIRE(D >= 1 && D <= 1024, GRL_ERR_SHAPE, "grl_bert_layer_fwd: head_dim must be between 1 and 1024 (got %lld)", (long long)D);
    GRL_REQUIRE(w->w_qkv && w->w_o && w->w_ff1 && w->w_ff2 && w->ln1_g && w->ln1_b && w->ln2_g && w->ln2_b,
                GRL_ERR_ARG, "grl_bert_layer_fwd: null weight");
    const int64_t M = rg ? rg->rows : B * S, d = H * D, es = (int64_t)grl_dtype_size(dtype);
    if (M == 0) return GRL_OK;
    auto pad = [](int64_t v) { return (v + 255) / 256 * 256; };
    char* qkv = (char*)workspace;
    char* attn = qkv + pad(M * 3 * d * es);
    char* proj = attn + pad(M * d * es);
    char* ff = proj + pad(M * d * es);
    int rc;
    grl_lap_mark(c);
    if ((rc = grl_gemm_nt(c, dtype, dtype, M, 3 * d, d, x, w->w_qkv, w->b_qkv, qkv, GRL_EPI_NONE))) return rc;
    grl_lap_mark(c);
    if ((rc = layer_attention(c, dtype, B, S, H, D, qkv, mask, attn, rg))) return rc;
    grl_lap_mark(c);
    if ((rc = grl_gemm_nt(c, dtype, dtype, M, d, d, attn, w->w_o, w->b_o, proj, GRL_EPI_NONE))) return rc;
    grl_lap_mark(c);
    if ((rc = grl_layernorm(c, dtype, M, d, x, proj, w->ln1_g, w->ln1_b, eps, x))) return rc;
    grl_lap_mark(c);
    if ((rc = grl_gemm_nt(c, dtype, dtype, M, d_ff, d, x, w->w_ff1, w->b_ff1, ff, GRL_EPI_GELU))) return rc;
    grl_lap_mark(c);
    if ((rc = grl_gemm_nt(c, dtype, dtype, M, d, d_ff, ff, w->w_ff2, w->b_ff2, proj, GRL_EPI_NONE))) return rc;
    grl_lap_mark(c);
    if ((rc = grl_layernorm(c, dtype, M, d, x, proj, w->ln2_g, w->ln2_b, eps, x))) return rc;
    grl_lap_mark(c);
    return GRL_OK;
}

extern "C" int grl_bert_layer_fwd(grl_ctx* c, int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int64_t d_ff,
                                  const grl_bert_layer* w, const float* mask, float eps, void* x, void* workspace) {
    return bert_layer(c, dtype, B, S, H, D, d_ff, w, mask, eps, x, workspace, nullptr);
}
extern "C" int grl_bert_layer_fwd_ragged(grl_ctx* c, int dtype, const grl_ragged* rg, int64_t H, int64_t D, int64_t d_ff,
                                         const grl_bert_layer* w, float eps, void* x, void* workspace) {
    int rc = grl_check_ragged("grl_bert_layer_fwd_ragged", rg);
    return rc ? rc : bert_layer(c, dtype, rg->sequences, rg->longest, H, D, d_ff, w, nullptr, eps, x, workspace, rg);
}

// ---- the same layer without a LayerNorm pass: the residual stream is kept as raw rows + row statistics ----------
extern "C" int64_t grl_bert_layer_fused_workspace(int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int64_t d_ff) {
    if (!grl_valid_dtype(dtype) || B < 0 || S < 0 || H <= 0 || D <= 0 || d_ff <= 0) return -1;
    const int64_t M = B * S, d = H * D;
    auto pad = [](int64_t v) { return (v + 255) / 256 * 256; };
    const int64_t es = (int64_t)grl_dtype_size(dtype);
    // qkv (M,3d) | attn (M,d) | ff (M,d_ff) | statistics of the middle residual (M,2) | row-statistics partials
    return pad(M * 3 * d * es) + pad(M * d * es) + pad(M * d_ff * es) + pad(M * 8) + pad(grl_gemm_nt_resln_workspace(M, d));
}

// `layers` layers, the first of which finds the statistics of r in stats.  Between them, and inside each, the statistics stay the partials
// that the residual products leave; with `last_merged` those of the final r are merged into stats (workspace: as of one layer then;
// else grl_bert_layers_fused_workspace, as the partials that a layer starts from live beside those of its middle).
static int bert_layers_fused(grl_ctx* c, int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int64_t d_ff,
                             const grl_bert_layer_fused* w, int64_t layers, bool last_merged, const float* mask, float eps, void* r, float* stats,
                             void* workspace, const grl_ragged* rg) {
    GRL_REQUIRE(c && w && r && stats && workspace && layers >= 0, GRL_ERR_ARG, "grl_bert_layer_fwd_fused: null argument");
    GRL_REQUIRE(grl_valid_dtype(dtype), GRL_ERR_ARG, "grl_bert_layer_fwd_fused: bad dtype %d", dtype);
    GRL_REQUIRE(B >= 0 && S >= 0 && H > 0 && d_ff > 0, GRL_ERR_SHAPE, "grl_bert_layer_fwd_fused: bad shape");
    GRL_REQUIRE(D >= 1 && D <= 1024, GRL_ERR_SHAPE, "grl_bert_layer_fwd_fused: head_dim must be between 1 and 1024 (got %lld)", (long long)D);
    for (int64_t l = 0; l < layers; ++l)
        GRL_REQUIRE(w[l].ws_qkv && w[l].c_qkv && w[l].bf_qkv && w[l].in_g && w[l].in_b && w[l].w_o && w[l].ln1_g && w[l].ln1_b && w[l].ws_ff1 && w[l].c_ff1 &&
                    w[l].bf_ff1 && w[l].w_ff2, GRL_ERR_ARG, "grl_bert_layer_fwd_fused: null weight");
    const int64_t M = rg ? rg->rows : B * S, d = H * D, es = (int64_t)grl_dtype_size(dtype), slab = 128 / es;
    GRL_REQUIRE(d % slab == 0 && d_ff % slab == 0, GRL_ERR_SHAPE,
                "grl_bert_layer_fwd_fused: d_model (%lld) and d_ff (%lld) must be multiples of %lld; use grl_bert_layer_fwd",
                (long long)d, (long long)d_ff, (long long)slab);
    if (M == 0) return GRL_OK;
    auto pad = [](int64_t v) { return (v + 255) / 256 * 256; };
    char* qkv = (char*)workspace;
    char* attn = qkv + pad(M * 3 * d * es);
    char* ff = attn + pad(M * d * es);
    float* stats1 = (float*)(ff + pad(M * d_ff * es));
    char* part = (char*)stats1 + pad(M * 8);
    char* part_next = part + pad(grl_gemm_nt_resln_workspace(M, d));
    grl_row_stats in = {stats, nullptr, 0, eps}, mid{};
    for (int64_t l = 0; l < layers; ++l, ++w) {
        int rc;
        grl_lap_mark(c);
        if ((rc = grl_ln_gemm_nt_from(c, dtype, M, 3 * d, d, r, w->ws_qkv, w->c_qkv, w->bf_qkv, in, stats, qkv, GRL_EPI_NONE))) return rc;
        grl_lap_mark(c);
        if ((rc = layer_attention(c, dtype, B, S, H, D, qkv, mask, attn, rg))) return rc;
        grl_lap_mark(c);
        if ((rc = grl_gemm_nt_resln_parts(c, dtype, M, d, d, attn, w->w_o, w->b_o, r, in, w->in_g, w->in_b, r, eps, stats1, part, &mid))) return rc;
        grl_lap_mark(c);
        if ((rc = grl_ln_gemm_nt_from(c, dtype, M, d_ff, d, r, w->ws_ff1, w->c_ff1, w->bf_ff1, mid, stats1, ff, GRL_EPI_GELU))) return rc;
        grl_lap_mark(c);
        // (the partials that the layer started from have been read by now)
        if (last_merged && l == layers - 1) {
            if (mid.nparts) {      // the one partials' buffer of a single layer is read and written by this product: other rows, other tiles
                if ((rc = grl_merge_row_stats(c, mid.parts, stats1, M, d, mid.nparts, eps))) return rc;
                mid = {stats1, nullptr, 0, eps};
            }
            rc = grl_gemm_nt_resln(c, dtype, M, d, d_ff, ff, w->w_ff2, w->b_ff2, r, mid.stats, w->ln1_g, w->ln1_b, r, eps, stats, part);
        } else rc = grl_gemm_nt_resln_parts(c, dtype, M, d, d_ff, ff, w->w_ff2, w->b_ff2, r, mid, w->ln1_g, w->ln1_b, r, eps, stats, part_next, &in);
        if (rc) return rc;
        grl_lap_mark(c);
    }
    return GRL_OK;
}

extern "C" int grl_bert_layer_fwd_fused(grl_ctx* c, int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int64_t d_ff,
                                        const grl_bert_layer_fused* w, const float* mask, float eps, void* r, float* stats,
                                        void* workspace) {
    return bert_layers_fused(c, dtype, B, S, H, D, d_ff, w, 1, true, mask, eps, r, stats, workspace, nullptr);
}
extern "C" int grl_bert_layer_fwd_fused_ragged(grl_ctx* c, int dtype, const grl_ragged* rg, int64_t H, int64_t D, int64_t d_ff,
                                               const grl_bert_layer_fused* w, float eps, void* r, float* stats, void* workspace) {
    int rc = grl_check_ragged("grl_bert_layer_fwd_fused_ragged", rg);
    return rc ? rc : bert_layers_fused(c, dtype, rg->sequences, rg->longest, H, D, d_ff, w, 1, true, nullptr, eps, r, stats, workspace, rg);
}

extern "C" int64_t grl_bert_layers_fused_workspace(int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int64_t d_ff) {
    const int64_t one = grl_bert_layer_fused_workspace(dtype, B, S, H, D, d_ff);
    return one < 0 ? one : one + (grl_gemm_nt_resln_workspace(B * S, H * D) + 255) / 256 * 256;
}
extern "C" int grl_bert_layers_fwd_fused(grl_ctx* c, int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int64_t d_ff,
                                         const grl_bert_layer_fused* w, int64_t layers, const float* mask, float eps, void* r, float* stats,
                                         void* workspace) {
    return bert_layers_fused(c, dtype, B, S, H, D, d_ff, w, layers, false, mask, eps, r, stats, workspace, nullptr);
}
extern "C" int grl_bert_layers_fwd_fused_ragged(grl_ctx* c, int dtype, const grl_ragged* rg, int64_t H, int64_t D, int64_t d_ff,
                                                const grl_bert_layer_fused* w, int64_t layers, float eps, void* r, float* stats, void* workspace) {
    int rc = grl_check_ragged("grl_bert_layers_fwd_fused_ragged", rg);
    return rc ? rc : bert_layers_fused(c, dtype, rg->sequences, rg->longest, H, D, d_ff, w, layers, false, nullptr, eps, r, stats, workspace, rg);
}

// ---- projection and attention with rotary positions ---------------------------------------------------------------
extern "C" int grl_rotary_attention(grl_ctx* c, int dtype, int64_t B, int64_t S, const grl_ragged* rg, int64_t H, int64_t D, const void* x,
                                    const void* w_qkv, const float* b_qkv, const float* mask, void* qkv, void* out, float rope_base, float rope_scaling) {
    GRL_REQUIRE(c && x && w_qkv && qkv && out, GRL_ERR_ARG, "grl_rotary_attention: null argument");
    GRL_REQUIRE(grl_valid_dtype(dtype), GRL_ERR_ARG, "grl_rotary_attention: bad dtype %d", dtype);
    GRL_REQUIRE(B >= 0 && S >= 0 && H > 0 && D >= 2 && D <= 128 && D % 2 == 0, GRL_ERR_SHAPE, "grl_rotary_attention: bad shape");
    GRL_REQUIRE(rope_base > 0.f && rope_scaling != 0.f, GRL_ERR_ARG, "grl_rotary_attention: bad rope base/scaling");
    if (rg) {
        const int rc = grl_check_ragged("grl_rotary_attention", rg);
        if (rc) return rc;
    }
    const int64_t M = rg ? rg->rows : B * S, longest = rg ? rg->longest : S, d = H * D, es = (int64_t)grl_dtype_size(dtype);
    if (M == 0) return GRL_OK;
    char* q = (char*)qkv;
    int rope = GRL_ROPE_HALF, rc;
    if (D == 64 && M < (1LL << 31) && 3 * d < (1LL << 31)) {
        bool taken = false;
        if ((rc = grl_gemm_nt_rope(c, dtype, M, 3 * d, d, x, w_qkv, b_qkv, qkv, 2 * d, rg ? rg->positions : nullptr, longest, rope_base, rope_scaling, &taken)))
            return rc;
        if (taken) rope = GRL_ROPE_NONE;
    }
    if (rope == GRL_ROPE_HALF && (rc = grl_gemm_nt(c, dtype, dtype, M, 3 * d, d, x, w_qkv, b_qkv, qkv, GRL_EPI_NONE))) return rc;
    const float scale = (float)(1.0 / sqrt((double)D));
    if (rg) return grl_fa2_fwd_ragged(c, dtype, rg, H, D, q, q + d * es, q + 2 * d * es, out, 3 * d, 3 * d, 3 * d, d, scale, 0, rope, rope_base, rope_scaling);
    return grl_fa2_fwd_strided(c, dtype, B, S, H, D, q, q + d * es, q + 2 * d * es, mask, out, 3 * d, 3 * d, 3 * d, d, scale, 0, rope, rope_base, rope_scaling);
}

// ---- the two products around the LayerNorm of a gated MLP ---------------------------------------------------------
extern "C" int grl_resln_ln_glu(grl_ctx* c, int dtype, int64_t M, int64_t d, int64_t K, int64_t d_ff, const void* A, const void* W, const float* bias,
                                const void* R, const float* r_stats, const float* r_gamma, const float* r_beta, void* C, const void* Wg_scaled,
                                const void* Wu_scaled, const float* colsum_gate, const float* colsum_up, const float* bias_gate_folded,
                                const float* bias_up_folded, float eps, float* stats, void* workspace, void* out, int activation) {
    grl_row_stats rows{};
    const int rc = grl_gemm_nt_resln_parts(c, dtype, M, d, K, A, W, bias, R, grl_row_stats{r_stats, nullptr, 0, 0.f}, r_gamma, r_beta, C, eps, stats, workspace, &rows);
    if (rc || M == 0 || d == 0) return rc;
    return grl_ln_glu_nt_from(c, dtype, M, d_ff, d, C, Wg_scaled, Wu_scaled, colsum_gate, colsum_up, bias_gate_folded, bias_up_folded, rows, stats, out, activation);
}

// ---- the same for few rows: five launches, no statistics pass, no partials to merge -------------------------------
// The products that read LayerNorm(r) take its row statistics from their own operand and leave them for the residual epilogue
// that needs them next, so between layers only the raw rows travel.  One 128-token sentence through twelve layers 768 wide in
// bf16: 521 us with seven launches a layer (two of them LayerNorm passes of 5 us over 128 rows), 443 us with these five.  Hidden
// states are 1 to 4 % nearer to their float64 values: a sublayer's output is rounded once, behind the residual, not before and after.
static int bert_layer_rows(grl_ctx* c, int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int64_t d_ff, const grl_bert_layer_fused* w,
                           const float* mask, float in_eps, float eps, void* r, void* workspace, const grl_ragged* rg) {
    GRL_REQUIRE(c && w && r && workspace, GRL_ERR_ARG, "grl_bert_layer_fwd_rows: null argument");
    GRL_REQUIRE(grl_valid_dtype(dtype), GRL_ERR_ARG, "grl_bert_layer_fwd_rows: bad dtype %d", dtype);
    GRL_REQUIRE(B >= 0 && S >= 0 && H > 0 && d_ff > 0, GRL_ERR_SHAPE, "grl_bert_layer_fwd_rows: bad shape");
    GRL_REQUIRE(D >= 1 && D <= 1024, GRL_ERR_SHAPE, "grl_bert_layer_fwd_rows: head_dim must be between 1 and 1024 (got %lld)", (long long)D);
    GRL_REQUIRE(w->ws_qkv && w->c_qkv && w->bf_qkv && w->in_g && w->in_b && w->w_o && w->ln1_g && w->ln1_b && w->ws_ff1 && w->c_ff1 &&
                w->bf_ff1 && w->w_ff2, GRL_ERR_ARG, "grl_bert_layer_fwd_rows: null weight");
    const int64_t M = rg ? rg->rows : B * S, d = H * D, es = (int64_t)grl_dtype_size(dtype), slab = 128 / es;
    GRL_REQUIRE(d % slab == 0 && d_ff % slab == 0, GRL_ERR_SHAPE,
                "grl_bert_layer_fwd_rows: d_model (%lld) and d_ff (%lld) must be multiples of %lld; use grl_bert_layer_fwd",
                (long long)d, (long long)d_ff, (long long)slab);
    if (M == 0) return GRL_OK;
    auto pad = [](int64_t v) { return (v + 255) / 256 * 256; };
    char* qkv = (char*)workspace;                  // the layout of the folded layer's workspace
    char* attn = qkv + pad(M * 3 * d * es);
    char* ff = attn + pad(M * d * es);
    float* stats = (float*)(ff + pad(M * d_ff * es));
    int rc;
    grl_lap_mark(c);
    if ((rc = grl_ln_gemm_nt_rows(c, dtype, M, 3 * d, d, r, w->ws_qkv, w->c_qkv, w->bf_qkv, in_eps, stats, qkv, GRL_EPI_NONE))) return rc;
    grl_lap_mark(c);
    if ((rc = layer_attention(c, dtype, B, S, H, D, qkv, mask, attn, rg))) return rc;
    grl_lap_mark(c);
    if ((rc = grl_gemm_nt_lnres(c, dtype, M, d, d, attn, w->w_o, w->b_o, r, stats, w->in_g, w->in_b, r))) return rc;
    grl_lap_mark(c);
    if ((rc = grl_ln_gemm_nt_rows(c, dtype, M, d_ff, d, r, w->ws_ff1, w->c_ff1, w->bf_ff1, eps, stats, ff, GRL_EPI_GELU))) return rc;
    grl_lap_mark(c);
    if ((rc = grl_gemm_nt_lnres(c, dtype, M, d, d_ff, ff, w->w_ff2, w->b_ff2, r, stats, w->ln1_g, w->ln1_b, r))) return rc;
    grl_lap_mark(c);
    return GRL_OK;
}

extern "C" int grl_bert_layer_fwd_rows(grl_ctx* c, int dtype, int64_t B, int64_t S, int64_t H, int64_t D, int64_t d_ff,
                                       const grl_bert_layer_fused* w, const float* mask, float in_eps, float eps, void* r, void* workspace) {
    return bert_layer_rows(c, dtype, B, S, H, D, d_ff, w, mask, in_eps, eps, r, workspace, nullptr);
}
extern "C" int grl_bert_layer_fwd_rows_ragged(grl_ctx* c, int dtype, const grl_ragged* rg, int64_t H, int64_t D, int64_t d_ff,
                                              const grl_bert_layer_fused* w, float in_eps, float eps, void* r, void* workspace) {
    int rc = grl_check_ragged("grl_bert_layer_fwd_rows_ragged", rg);
    return rc ? rc : bert_layer_rows(c, dtype, rg->sequences, rg->longest, H, D, d_ff, w, nullptr, in_eps, eps, r, workspace, rg);
}

// ---- a padded batch without its padding: host side --------------------------------------------------------------
int grl_check_ragged(const char* who, const grl_ragged* rg) {
    GRL_REQUIRE(rg && rg->offsets && rg->positions, GRL_ERR_ARG, "%s: null ragged batch", who);
    GRL_REQUIRE(rg->sequences >= 0 && rg->rows >= 0 && rg->longest >= 0 && rg->longest <= rg->rows && rg->rows < (1LL << 31), GRL_ERR_SHAPE,
                "%s: bad ragged batch (sequences=%lld rows=%lld longest=%lld)", who, (long long)rg->sequences, (long long)rg->rows, (long long)rg->longest);
    return GRL_OK;
}

template <typename M>
static int pack_batch(int64_t B, int64_t S, int64_t vocab, const int64_t* ids, const M* mask, int32_t* all_ids, float* all_mask, int32_t* out,
                      int64_t* rows, int64_t* longest) {
    int32_t* offsets = out;
    int32_t* positions = out + (B + 1);
    int32_t* kept = positions + B * S;
    int64_t n = 0, most = 0;
    bool prefix = true;
    const int32_t top = (int32_t)vocab;
    bool bad_id = false, bad_mask = false;
    for (int64_t b = 0; b < B; ++b) {
        const int64_t first = n;
        const int64_t* row = ids + b * S;
        offsets[b] = (int32_t)n;
        for (int64_t s = 0; s < S; ++s) {
            const int32_t id = (int32_t)row[s];
            bad_id |= (uint32_t)id >= (uint32_t)top;
            bool keep = true;
            if (mask) {
                const M m = mask[b * S + s];
                keep = m != (M)0;
                bad_mask |= keep && m != (M)1;
                if (all_mask) all_mask[b * S + s] = (float)m;
            }
            if (all_ids) all_ids[b * S + s] = id;
            prefix &= !keep || n - first == s;
            positions[n] = (int32_t)s;           // overwritten by the next token when this one is not kept
            kept[n] = id;
            n += keep;
        }
        if (n - first > most) most = n - first;
    }
    offsets[B] = (int32_t)n;
    if (n < B * S) memmove(positions + n, kept, (size_t)n * sizeof(int32_t));
    *rows = n; *longest = most;
    if (bad_id) return GRL_PACK_BAD_ID;
    if (bad_mask) return GRL_PACK_OTHER_MASK;
    return prefix ? GRL_PACK_PREFIX : GRL_PACK_SCATTERED;
}

extern "C" int grl_pack_inputs(int64_t B, int64_t S, int64_t vocab, const int64_t* ids, const void* mask, int mask_kind,
                               int32_t* all_ids, float* all_mask, int32_t* out, int64_t* rows, int64_t* longest) {
    GRL_REQUIRE(B >= 0 && S >= 0 && B * S < (1LL << 31) && vocab > 0 && vocab < (1LL << 31), GRL_ERR_SHAPE, "grl_pack_batch: bad shape");
    GRL_REQUIRE(out && rows && longest && (B * S == 0 || ids), GRL_ERR_ARG, "grl_pack_batch: null argument");
    switch (mask ? mask_kind : 0) {
        case 0: return pack_batch<int64_t>(B, S, vocab, ids, nullptr, all_ids, nullptr, out, rows, longest);
        case 1: return pack_batch<int64_t>(B, S, vocab, ids, (const int64_t*)mask, all_ids, all_mask, out, rows, longest);
        case 2: return pack_batch<float>(B, S, vocab, ids, (const float*)mask, all_ids, all_mask, out, rows, longest);
        default: break;
    }
    grl_set_error("grl_pack_batch: mask_kind must be 0 (none), 1 (int64) or 2 (float32)");
    return GRL_ERR_ARG;
}

extern "C" int grl_pack_batch(int64_t B, int64_t S, int64_t vocab, const int64_t* ids, const void* mask, int mask_kind,
                              int32_t* out, int64_t* rows, int64_t* longest) {
    return grl_pack_inputs(B, S, vocab, ids, mask, mask_kind, nullptr, nullptr, out, rows, longest);
}
