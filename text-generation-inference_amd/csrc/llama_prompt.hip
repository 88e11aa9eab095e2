// The layers of a dense Llama model on the rows of prompts, launched from here: the launches that the model's own forward makes one by one,
// with the same arguments and the same results, without its way back to Python between them.  A layer of a short prompt is seven launches of 4 to
// 17 us, each of which took 9 us of host time to prepare; here it is 2 - 3 us.  47 tokens through 22 layers of 2048: 1820 -> 1540 us.
#include "common.h"

#define TRY(call)                          \
    do {                                   \
        const int rc_ = (call);            \
        if (rc_ != TGIS_OK) return rc_;    \
    } while (0)

// Up to 64 rows in bf16: the launches of dense_rows.hip, six or seven a layer.  A prefill of 47 tokens through 22 layers of 2048, us, the launches below / these:
// 1519 / 1305 (a layer 54.5 / 43.6: qkv 11.0 / 7.1, o and the norm 10.2 / 7.0, gate | up 16.0 / 12.8, down and the norm 13.0 / 11.9).
static int rows16_prompt(const TgisLlamaLayer* layers, int n_layers, TgisLlamaPrompt* p, void* stream) {
    TGIS_CHECK_ARG(p->x && p->hw && p->sums && p->last && p->qkv && p->att && p->act && p->res[0] && p->slabs && p->dtype == TGIS_BF16,
                   "tgis_llama_prompt: null buffer, or rows that are not bf16");
    const int64_t T = p->T, HD = (int64_t)p->H * p->D, QKV = HD + 2 * (int64_t)p->Hkv * p->D;
    TRY(tgis_dense_rows16_embed(nullptr, p->x, layers[0].input_norm, p->h, p->hw, p->sums, T, p->hidden, 0, stream));
    for (int i = 0; i < n_layers; ++i) {
        const TgisLlamaLayer& l = layers[i];
        TRY(tgis_dense_rows16_norm_rope(p->hw, p->sums, p->eps, l.qkv_rope, l.qkv_bias, p->positions, p->slots, p->cos, p->sin, p->qkv, QKV, l.k_pool,
                                        l.v_pool, T, p->hidden, p->H, p->Hkv, p->D, stream));
        TRY(tgis_attn_paged_fragments(p->qkv, QKV, l.k_pool, l.v_pool, p->block_tables, p->max_pages, p->ctx_lens, p->cu_seqlens, p->att, p->B, p->H,
                                      p->Hkv, p->D, p->max_q_len, p->max_ctx, p->scale, p->dtype, stream));
        TRY(tgis_dense_rows16_residual(p->att, l.o, l.post_norm, p->h, p->hw, p->sums, p->slabs, p->slabs_bytes, T, HD, p->hidden, stream));
        TRY(tgis_dense_rows16_norm_silu(p->hw, p->sums, p->eps, l.gate_up, p->act, T, p->hidden, 2 * p->inner, stream));
        if (i + 1 < n_layers)
            TRY(tgis_dense_rows16_residual(p->act, l.down, layers[i + 1].input_norm, p->h, p->hw, p->sums, p->slabs, p->slabs_bytes, T, p->inner, p->hidden,
                                           stream));
        else
            TRY(tgis_dense_rows16_leave(p->act, l.down, p->h, p->res[0], p->last, p->slabs, p->slabs_bytes, T, p->inner, p->hidden, stream));
    }
    p->num_slabs = 1;
    p->slab_ld = p->hidden;
    return TGIS_OK;
}

extern "C" int tgis_llama_prompt(const TgisLlamaLayer* layers, int n_layers, TgisLlamaPrompt* p, void* stream) {
    TGIS_CHECK_ARG(layers && n_layers >= 1 && p && p->T >= 1, "tgis_llama_prompt: bad arguments");
    if (p->h) return rows16_prompt(layers, n_layers, p, stream);
    TGIS_CHECK_ARG(p->x && p->y && p->qkv && p->att && p->act && p->res[0] && p->res[1] && p->workspace && p->workspace_bytes >= 4096,
                   "tgis_llama_prompt: null buffer");
    const bool tall = p->T >= TGIS_DENSE_TALL_MIN_M;
    TGIS_CHECK_ARG(p->slabs || (tall && p->out), "tgis_llama_prompt: no room for the products behind the residual stream");
    const int64_t T = p->T, HD = (int64_t)p->H * p->D, QKV = HD + 2 * (int64_t)p->Hkv * p->D;
    uint8_t* ws = (uint8_t*)p->workspace;
    int S = 0;        // the last product lies in `slabs` as S partial sums (0: in x0)
    int64_t ld = 0;
    const void* x0 = p->x;
    const void* res = nullptr;
    int next = 0;
    auto norm = [&](const void* w, float eps) -> int {
        void* to = p->res[next];
        if (S > 0)
            TRY(tgis_rmsnorm_residual_partial(p->slabs, S, ld, nullptr, res, w, p->y, p->hidden, to, T, p->hidden, eps, p->dtype, stream));
        else
            TRY(tgis_rmsnorm_residual(x0, res, w, p->y, p->hidden, res ? to : nullptr, T, p->hidden, eps, p->dtype, stream));
        if (S > 0 || res) {
            res = to;
            next ^= 1;
        } else {
            res = x0;
        }
        return TGIS_OK;
    };
    // which of the two kernels leaves a product in parts, and whether qkv is left so
    const bool left = p->slabs != nullptr;
    auto tall_parts = [&](int64_t K, int64_t N) { return tall && left && tgis_dense_tall_partial_bytes(T, K, N) >= 0; };
    const bool qkv_tall = tall_parts(p->hidden, QKV), o_tall = tall_parts(HD, p->hidden), down_tall = tall_parts(p->inner, p->hidden);
    const bool qkv_whole = tall && (!left || (p->fresh && tgis_dense_tall_bytes(T, p->hidden, QKV, 0) >= 0));
    const bool q_later = tgis_attn_rotates_q(p->H, p->Hkv, p->D, p->max_q_len);  // the attention rotates q as it reads it
    auto parts = [&](bool by_tall, const void* in, const void* image, int64_t K, int64_t N, int* slabs, int64_t* row) -> int {
        if (by_tall) return tgis_dense_tall_partial(in, K, image, T, K, N, p->dtype, p->slabs, p->slabs_bytes, slabs, row, stream);
        return tgis_dense_gemm_partial(in, K, image, T, K, N, p->dtype, 0, p->slabs, p->slabs_bytes, slabs, row, stream);
    };
    auto product = [&](bool by_tall, const void* in, const void* image, int64_t K) -> int {  // [T, hidden], summed by the norm behind it
        if (!left) {
            x0 = p->out;
            return tgis_dense_tall(in, K, image, nullptr, p->out, p->hidden, T, K, p->hidden, p->dtype, 0, 0, 0.f, 0.f, ws + 4096,
                                   p->workspace_bytes - 4096, stream);
        }
        return parts(by_tall, in, image, K, p->hidden, &S, &ld);
    };
    for (int i = 0; i < n_layers; ++i) {
        const TgisLlamaLayer& l = layers[i];
        TRY(norm(l.input_norm, p->eps));
        if (!tall) {
            TRY(tgis_dense_gemm_rope(p->y, p->hidden, l.qkv_rope, l.qkv_bias, p->positions, p->slots, p->cos, p->sin, p->qkv, QKV, l.k_pool, l.v_pool,
                                     T, p->hidden, QKV, p->H, p->Hkv, p->D, p->dtype, stream));
        } else if (!qkv_whole) {
            int qkv_slabs = 0;
            int64_t row = 0;
            TRY(parts(qkv_tall, p->y, l.qkv, p->hidden, QKV, &qkv_slabs, &row));
            TRY(tgis_rope_kv_write_partial(p->slabs, qkv_slabs, row, l.qkv_bias, p->qkv, QKV, p->cos, p->sin, p->positions, p->slots, l.k_pool, l.v_pool, T,
                                           p->H, p->Hkv, p->D, p->D, p->dtype, stream));
        } else {
            TRY(tgis_dense_tall(p->y, p->hidden, l.qkv, l.qkv_bias, p->qkv, QKV, T, p->hidden, QKV, p->dtype, 0, 0, 0.f, 0.f, ws + 4096,
                                p->workspace_bytes - 4096, stream));
            if (p->fresh && q_later)
                TRY(tgis_rope_k_write_prefill(p->qkv, QKV, p->cos, p->sin, p->positions, p->cu_seqlens, p->block_tables, p->max_pages, l.k_pool,
                                              l.v_pool, p->B, T, p->max_q_len, p->H, p->Hkv, p->D, p->D, p->dtype, stream));
            else if (p->fresh)
                TRY(tgis_rope_kv_write_prefill(p->qkv, QKV, p->cos, p->sin, p->positions, p->cu_seqlens, p->block_tables, p->max_pages, l.k_pool,
                                               l.v_pool, p->B, T, p->max_q_len, p->H, p->Hkv, p->D, p->D, p->dtype, stream));
            else
                TRY(tgis_rope_kv_write(p->qkv, QKV, p->cos, p->sin, p->positions, p->slots, l.k_pool, l.v_pool, T, p->H, p->Hkv, p->D, p->D,
                                       p->dtype, stream));
        }
        if (qkv_whole && p->fresh && q_later)
            TRY(tgis_attn_paged_rope(p->qkv, QKV, p->cos, p->sin, p->positions, l.k_pool, l.v_pool, p->block_tables, p->max_pages, p->ctx_lens, p->cu_seqlens,
                                     p->att, p->B, p->H, p->Hkv, p->D, p->max_q_len, p->max_ctx, p->scale, p->dtype, stream));
        else
            TRY(tgis_attn_paged(p->qkv, QKV, l.k_pool, l.v_pool, p->block_tables, p->max_pages, p->ctx_lens, p->cu_seqlens, p->att, HD, p->B, p->H,
                                p->Hkv, p->D, p->max_q_len, p->max_ctx, p->scale, p->dtype, 1, nullptr, 0, stream));
        TRY(product(o_tall, p->att, l.o, HD));
        TRY(norm(l.post_norm, p->eps));
        if (tall)
            TRY(tgis_dense_tall(p->y, p->hidden, l.gate_up, nullptr, p->act, p->inner, T, p->hidden, 2 * p->inner, p->dtype, 0, 2, 0.f, 0.f, ws + 4096,
                                p->workspace_bytes - 4096, stream));
        else
            TRY(tgis_dense_gemm(p->y, p->hidden, l.gate_up, nullptr, p->act, p->inner, T, p->hidden, 2 * p->inner, p->dtype, 0, 2, ws,
                                p->workspace_bytes, stream));
        TRY(product(down_tall, p->act, l.down, p->inner));
    }
    p->num_slabs = S;
    p->slab_ld = ld;
    return TGIS_OK;
}
