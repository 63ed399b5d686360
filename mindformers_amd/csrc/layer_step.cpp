// One decode step of a weight-only layer from one call: the launches of QuantDecodeLayer.forward in its order.
//
// A step is seven to nine launches of about 3 us of host time each; reaching every one of them through its own wrapper (checks,
// an allocation, a call with 12 to 20 arguments) took another 40 us a layer, which is what a step of few sequences waits for: two layers of
// 512 x 1376 at 4 sequences, through the serving runner, 178 to 187 us, 119 with this call (80 on the device then, 64 now).  Every entry point
// called here checks its own arguments.
#include "../../include/mf_decode.h"

void mf_set_error(const char* fmt, ...);

namespace {
size_t aligned(size_t bytes) { return (bytes + 255) & ~(size_t)255; }
struct Scratch {
    size_t n1, qkv, attn, h, n2, act, end;
    Scratch(int64_t rows, int64_t hidden, int64_t nq, int64_t nkv, int64_t ffn) {
        n1 = 0;
        qkv = n1 + aligned(2 * rows * hidden);
        attn = qkv + aligned(2 * rows * (nq + 2 * nkv));
        h = attn + aligned(2 * rows * nq);
        n2 = h + aligned(2 * rows * hidden);
        act = n2 + aligned(2 * rows * hidden);
        end = act + aligned(2 * rows * ffn);
    }
};
}  // namespace

extern "C" size_t mf_decode_layer_args_bytes(void) { return sizeof(mf_decode_layer_args); }

extern "C" size_t mf_decode_layer_scratch_bytes(int rows, int hidden, int n_heads, int n_kv_heads, int head_dim, int ffn) {
    if (rows <= 0 || hidden <= 0 || n_heads <= 0 || n_kv_heads <= 0 || head_dim <= 0 || ffn <= 0) return 0;
    return Scratch(rows, hidden, (int64_t)n_heads * head_dim, (int64_t)n_kv_heads * head_dim, ffn).end;
}

extern "C" size_t mf_decode_layer_workspace_bytes(int rows, int hidden, int n_heads, int n_kv_heads, int head_dim, int ffn) {
    const int nq = n_heads * head_dim, nqkv = nq + 2 * n_kv_heads * head_dim;
    size_t need = mf_w8a16_workspace_bytes(rows, nqkv, hidden);
    const int shapes[3][2] = {{hidden, nq}, {2 * ffn, hidden}, {hidden, ffn}};
    for (const auto& s : shapes) {
        const size_t b = mf_w8a16_workspace_bytes(rows, s[0], s[1]);
        need = b > need ? b : need;
    }
    return need;
}

extern "C" int mf_decode_layer_step(const mf_decode_layer_args* a) {
    if (!a || !a->scratch || !a->out) {
        mf_set_error("decode_layer_step: null argument");
        return 1;
    }
    const int rows = (int)a->rows, hidden = (int)a->hidden, nh = (int)a->n_heads, nkv = (int)a->n_kv_heads, d = (int)a->head_dim;
    const int ffn = (int)a->ffn, dtype = (int)a->dtype;
    const Scratch at(rows, hidden, (int64_t)nh * d, (int64_t)nkv * d, ffn);
    if (rows <= 0 || (size_t)a->scratch_bytes < at.end) {
        mf_set_error("decode_layer_step: scratch of %zu bytes needed, %lld given", at.end, (long long)a->scratch_bytes);
        return 1;
    }
    char* s = (char*)a->scratch;
    void *n1 = s + at.n1, *qkv = s + at.qkv, *attn = s + at.attn, *h = s + at.h, *n2 = s + at.n2, *act = s + at.act;
    void *ws = a->workspace, *st = a->stream;
    const size_t wsb = (size_t)a->workspace_bytes;
    int rc;
    const void* in = a->normed;
    if (!in) {
        in = n1;
        if ((rc = mf_rmsnorm(n1, nullptr, a->x, nullptr, a->attn_gamma, (float)a->eps, rows, hidden, dtype,
                             (int)a->attn_gamma_dtype, st)))
            return rc;
    }
    if ((rc = mf_w8a16_qkv_rope_and_cache(qkv, in, a->qkv_w, a->qkv_scale, a->qkv_bias, a->cos, a->sin, a->key_cache,
                                          a->value_cache, a->slot_mapping, rows, nh, nkv, d, a->num_blocks * a->block_size, hidden,
                                          dtype, (int)a->table_dtype, ws, wsb, st)))
        return rc;
    if ((rc = mf_paged_attention_decode(attn, qkv, a->key_cache, a->value_cache, a->block_tables, a->context_lens, rows, nh, nkv, d,
                                        (int)a->block_size, (int)a->max_blocks, (int)a->num_blocks, (float)a->scale,
                                        (int64_t)(nh + 2 * nkv) * d, dtype, a->attn_workspace, (size_t)a->attn_workspace_bytes,
                                        st)))
        return rc;
    if ((rc = mf_w8a16_gemm_add_rmsnorm(n2, h, attn, a->wo_w, a->wo_scale, nullptr, a->x, a->ffn_gamma, (float)a->eps, rows, hidden,
                                        nh * d, dtype, (int)a->ffn_gamma_dtype, ws, wsb, st)))
        return rc;
    if ((rc = mf_w8a16_gemm_silu_mul(act, n2, a->fc1_w, a->fc1_scale, nullptr, rows, 2 * ffn, hidden, dtype, ws, wsb, st))) return rc;
    if (a->next_gamma)
        return mf_w8a16_gemm_add_rmsnorm(a->norm_out, a->out, act, a->fc2_w, a->fc2_scale, nullptr, h, a->next_gamma,
                                         (float)a->next_eps, rows, hidden, ffn, dtype, (int)a->next_gamma_dtype, ws, wsb, st);
    return mf_w8a16_gemm(a->out, act, a->fc2_w, a->fc2_scale, nullptr, h, rows, hidden, ffn, dtype, ws, wsb, st);
}
