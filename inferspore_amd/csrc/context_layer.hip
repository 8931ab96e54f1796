// isp_context_layer_rows_f16: a whole context-decoder layer of packed fp16 rows in one call (isp_context_layer_f16: up to 64 of them);
// isp_context_layer_rows_f32: of fp32 rows.
// Seven to ten launches (two more where rows are wider than 8192 columns).  A product whose k is split over workgroups leaves fp32 partial sums, and the step that follows adds them where it
// would have read the product -- QKV bias + RoPE + KV append, residual + RMSNorm (twice), SwiGLU; a gate / up product that is not
// split computes SwiGLU itself.  As separate calls a layer
// takes up to 14 launches (four products, their four additions, six steps) and host time in Python for each.  us per two layers, step by
// step and in one call: 16 sequences at 256-1023 keys, 4096 wide, 268, 260; one prompt of 37 tokens 240, 230; 664 tokens, 1024 wide (the
// steps' products by the library), 223, 130.
// The steps and their order are those of the reference's kernel comments (see inferspore_amd/context_layer.py).
#include <math.h>

#include "linear_rows.h"

namespace isp {

struct LayerPlans {
    ProductPlan qkv, o, gate_up, down;
    size_t bytes;  // of the largest product (or its partial sums), or the attention's: they are used one after the other
};

static LayerPlans layer_plans(int batch, int tokens, int hidden, int head_num, int kv_head_num, int head_size, int max_q_len,
                              int max_k_len, int inter) {
    const int width = (head_num + 2 * kv_head_num) * head_size, ctx = head_num * head_size;
    const int splits = tokens > 65535 ? 1 : kTiledMaxSplits;  // the kernels that add them up have a grid row per token
    LayerPlans p;
    p.qkv = product_plan(tokens, width, hidden, splits);
    p.o = product_plan(tokens, hidden, ctx, splits);
    p.gate_up = product_plan(tokens, 2 * inter, hidden, splits, true);
    p.down = product_plan(tokens, hidden, inter, splits);
    p.bytes = attention_workspace(batch, head_num, kv_head_num, head_size, max_q_len, max_k_len);
    const size_t sizes[] = {p.qkv.bytes(tokens, width), p.o.splits() == 1 ? 0 : p.o.bytes(tokens, hidden),
                            p.gate_up.tiled && p.gate_up.splits() == 1 ? 0 : p.gate_up.bytes(tokens, 2 * inter),
                            p.down.splits() == 1 ? 0 : p.down.bytes(tokens, hidden)};
    for (size_t s : sizes) p.bytes = s > p.bytes ? s : p.bytes;
    return p;
}

// ISP_OK where the layer runs here.  `vector`: elements of 16 bytes, of which rows are whole numbers.
static int layer_shape(int layer, int batch, int tokens, int hidden, int head_num, int kv_head_num, int head_size, int max_q_len,
                       int max_k_len, int max_seq_len, int inter, int rotary_dim, int vector = 8) {
    if (layer < 0 || batch <= 0 || tokens <= 0 || hidden <= 0 || head_num <= 0 || kv_head_num <= 0 || head_size <= 0 ||
        max_q_len <= 0 || max_k_len <= 0 || max_seq_len <= 0 || inter <= 0 || rotary_dim < 0 || head_num % kv_head_num != 0 ||
        rotary_dim % 2 != 0 || rotary_dim > head_size)
        return ISP_ERR_BAD_SHAPE;
    const long long widest = ((long long)head_num + 2ll * kv_head_num) * head_size;
    const int most = tokens <= kSkinnyMaxRows && vector == 8 ? kSkinnyMaxExtent : kTiledMaxExtent;
    if ((head_size != 64 && head_size != 96 && head_size != 128) || hidden % vector != 0 || inter % vector != 0 || batch > 65535 ||
        max_q_len > 65535 * 16 || (long long)batch * max_q_len > 0x7fffffffll || hidden > most || inter > most || widest > most)
        return ISP_ERR_UNSUPPORTED;
    // the steps between the products index vectors of 16 bytes in 32 bits
    if ((long long)tokens * (widest > 2ll * inter ? widest : 2ll * inter) > 0xffffffffll) return ISP_ERR_UNSUPPORTED;
    // the fp32 products are calls of their own: none may refuse once another has run
    if (vector == 4 && (2ll * inter > kTiledMaxExtent || (long long)tokens * hidden >= kTiledMaxValues)) return ISP_ERR_UNSUPPORTED;
    return ISP_OK;
}

// What isp_context_layer_f16 is for: a few rows, of products whose weights these kernels read faster than the library does (above 16 rows 32768
// columns: 48 rows of 6144, inter 24576, take 295 us a layer here and 278 with the library's).
static int few_rows_shape(int tokens, int hidden, int head_num, int kv_head_num, int head_size, int inter) {
    if (tokens > kSkinnyMaxRows || hidden > kNormSumsMaxHidden) return ISP_ERR_UNSUPPORTED;
    if (tokens > 16 && (2ll * inter > 32768 || ((long long)head_num + 2ll * kv_head_num) * head_size > 32768)) return ISP_ERR_UNSUPPORTED;
    return ISP_OK;
}

// residual + RMSNorm of a product: its partial sums, or what it has stored in `out`.  Rows of more than kNormSumsMaxHidden columns are wider
// than the workgroup that adds and normalises one: their sums are added first, as behind a product of its own.
static int layer_norm(const ProductPlan& plan, const float* sums, void* residual, void* out, const void* gamma, float eps, int tokens,
                      int hidden, hipStream_t stream) {
    const bool wide = hidden > kNormSumsMaxHidden;
    if (wide && plan.splits() > 1) {
        launch_add_splits(sums, plan.splits(), static_cast<__half*>(out), tokens, hidden, stream);
        const int status = note_launch(hipGetLastError());
        if (status != ISP_OK) return status;
    }
    if (wide || plan.splits() == 1)
        return isp_fused_add_bias_residual_rmsnorm_f16(residual, out, nullptr, gamma, eps, tokens, hidden, 0, stream);
    launch_norm_sums(sums, plan.splits(), static_cast<__half*>(residual), static_cast<__half*>(out), static_cast<const __half*>(gamma), eps,
                     tokens, hidden, stream);
    return note_launch(hipGetLastError());
}

static int context_layer(const void* normed, void* residual, void* out, const void* qkv_weight, const void* qkv_bias,
                         const void* o_weight, const void* gate_up_weight, const void* down_weight, const void* ffn_norm,
                         const void* next_norm, void* q, void* k_cache, void* v_cache, void* context, void* act,
                         const int32_t* padding_offset, const int32_t* history_length, const int32_t* input_length,
                         const int32_t* context_length, void* workspace, int layer, int batch, int tokens, int hidden, int head_num,
                         int kv_head_num, int head_size, int max_q_len, int max_k_len, int max_seq_len, int inter, int rotary_dim,
                         float rotary_base, float eps, hipStream_t stream) {
    const void* needed[] = {normed, residual, out, qkv_weight, o_weight, gate_up_weight, down_weight, ffn_norm, next_norm,
                            q, k_cache, v_cache, context, act, padding_offset, history_length, input_length, context_length, workspace};
    for (const void* p : needed) ISP_REQUIRE_PTR(p);
    const void* vectors[] = {normed, residual, out, qkv_weight, qkv_bias, o_weight, gate_up_weight, down_weight, ffn_norm,
                             next_norm, q, k_cache, v_cache, context, act, workspace};
    for (const void* p : vectors)
        if (!aligned16(p)) return ISP_ERR_UNSUPPORTED;
    const auto half_in = [](const void* p) { return static_cast<const __half*>(p); };
    const auto half_out = [](void* p) { return static_cast<__half*>(p); };
    const LayerPlans plan = layer_plans(batch, tokens, hidden, head_num, kv_head_num, head_size, max_q_len, max_k_len, inter);
    float* sums = static_cast<float*>(workspace);
    __half* product = half_out(workspace);
    const int width = (head_num + 2 * kv_head_num) * head_size, ctx = head_num * head_size;

    launch_product(plan.qkv, half_in(normed), half_in(qkv_weight), product, sums, tokens, width, hidden, stream);
    int status = note_launch(hipGetLastError());
    if (status != ISP_OK) return status;
    if (plan.qkv.splits() == 1) {
        status = isp_qkv_bias_rope_transpose_append_f16(q, nullptr, nullptr, k_cache, v_cache, layer, max_seq_len, product, qkv_bias,
                                                        padding_offset, history_length, input_length, batch, max_q_len, tokens,
                                                        head_num, kv_head_num, head_size, rotary_dim, rotary_base, stream);
    } else {
        const size_t slice = (size_t)layer * batch * kv_head_num * max_seq_len * head_size;
        launch_qkv_sums(sums, plan.qkv.splits(), half_in(qkv_bias), half_out(q), half_out(k_cache) + slice, half_out(v_cache) + slice,
                        padding_offset, history_length, input_length, batch, max_q_len, tokens, head_num, kv_head_num, head_size,
                        max_seq_len, rotary_dim, rotary_base, stream);
        status = note_launch(hipGetLastError());
    }
    if (status != ISP_OK) return status;
    status = context_attention(static_cast<const _Float16*>(q), static_cast<const _Float16*>(k_cache),
                               static_cast<const _Float16*>(v_cache), static_cast<_Float16*>(context), history_length,
                               input_length, context_length, layer, batch, head_num, kv_head_num, head_size, max_q_len, max_k_len,
                               max_seq_len, tokens, (float)(1.0 / sqrt((double)head_size)), sums, stream);
    if (status != ISP_OK) return status;
    launch_product(plan.o, half_in(context), half_in(o_weight), half_out(out), sums, tokens, hidden, ctx, stream);
    status = note_launch(hipGetLastError());
    if (status != ISP_OK) return status;
    status = layer_norm(plan.o, sums, residual, out, ffn_norm, eps, tokens, hidden, stream);
    if (status != ISP_OK) return status;
    if (plan.gate_up.splits() > 1) {
        launch_product(plan.gate_up, half_in(out), half_in(gate_up_weight), nullptr, sums, tokens, 2 * inter, hidden, stream);
        launch_swiglu_sums(sums, plan.gate_up.splits(), half_out(act), tokens, inter, stream);
        status = note_launch(hipGetLastError());
    } else if (plan.gate_up.tiled) {  // both products of a column meet in one wavefront: neither is stored
        launch_tiled_swiglu(plan.gate_up.tile, half_in(out), half_in(gate_up_weight), half_out(act), tokens, inter, hidden, stream);
        status = note_launch(hipGetLastError());
    } else {
        launch_product(plan.gate_up, half_in(out), half_in(gate_up_weight), product, sums, tokens, 2 * inter, hidden, stream);
        status = isp_swiglu_f16(workspace, act, tokens, inter, stream);
    }
    if (status != ISP_OK) return status;
    launch_product(plan.down, half_in(act), half_in(down_weight), half_out(out), sums, tokens, hidden, inter, stream);
    status = note_launch(hipGetLastError());
    if (status != ISP_OK) return status;
    return layer_norm(plan.down, sums, residual, out, next_norm, eps, tokens, hidden, stream);
}

// The same steps in fp32, on a workspace that holds the wider of the two products stored on the way and, behind it, partial sums.
// Residual + RMSNorm adds the splits of its product (rows of up to one vector per lane), the gate / up product computes SwiGLU where that
// takes no longer than a split product, the addition and the kernel of its own (2.5 us and 4.5 TB/s).  Eight to eleven launches.
// 4 prompts of up to 100 tokens, 2048 wide, us per two layers, with separate additions and SwiGLU and so: 592, 580.
struct LayerSpaceF32 {
    size_t product, bytes;
};
static LayerSpaceF32 layer_space_f32(int tokens, int hidden, int head_num, int kv_head_num, int head_size, int inter) {
    const int width = (head_num + 2 * kv_head_num) * head_size, ctx = head_num * head_size, widest = width > 2 * inter ? width : 2 * inter;
    const int extents[][2] = {{width, hidden}, {hidden, ctx}, {2 * inter, hidden}, {hidden, inter}};
    size_t sums = 0;
    for (const auto& e : extents) {
        const size_t need = isp_linear_rows_f32_workspace(tokens, e[0], e[1]);
        sums = need > sums ? need : sums;
    }
    const size_t product = (size_t)tokens * (size_t)widest * sizeof(float);  // rows of whole 16 bytes
    return {product, product + sums};
}

static int context_layer_f32(const void* normed, void* residual, void* out, const void* qkv_weight, const void* qkv_bias,
                             const void* o_weight, const void* gate_up_weight, const void* down_weight, const void* ffn_norm,
                             const void* next_norm, void* q, void* k_cache, void* v_cache, void* context, void* act,
                             const int32_t* padding_offset, const int32_t* history_length, const int32_t* input_length,
                             const int32_t* context_length, void* workspace, int layer, int batch, int tokens, int hidden, int head_num,
                             int kv_head_num, int head_size, int max_q_len, int max_k_len, int max_seq_len, int inter, int rotary_dim,
                             float rotary_base, float eps, hipStream_t stream) {
    const void* needed[] = {normed, residual, out, qkv_weight, o_weight, gate_up_weight, down_weight, ffn_norm, next_norm,
                            q, k_cache, v_cache, context, act, padding_offset, history_length, input_length, context_length, workspace};
    for (const void* p : needed) ISP_REQUIRE_PTR(p);
    const void* vectors[] = {normed, residual, out, qkv_weight, qkv_bias, o_weight, gate_up_weight, down_weight, ffn_norm,
                             next_norm, q, k_cache, v_cache, context, act, workspace};
    for (const void* p : vectors)
        if (!aligned16(p)) return ISP_ERR_UNSUPPORTED;
    const int width = (head_num + 2 * kv_head_num) * head_size, ctx = head_num * head_size;
    void* product = workspace;
    void* sums = static_cast<char*>(workspace) + layer_space_f32(tokens, hidden, head_num, kv_head_num, head_size, inter).product;

    int status = isp_linear_rows_f32(normed, qkv_weight, product, sums, tokens, width, hidden, stream);
    if (status != ISP_OK) return status;
    status = isp_qkv_bias_rope_transpose_append_f32(q, nullptr, nullptr, k_cache, v_cache, layer, max_seq_len, product, qkv_bias,
                                                    padding_offset, history_length, input_length, batch, max_q_len, tokens, head_num,
                                                    kv_head_num, head_size, rotary_dim, rotary_base, stream);
    if (status != ISP_OK) return status;
    status = isp_context_attention_f32(q, k_cache, v_cache, context, history_length, input_length, context_length, layer, batch,
                                       head_num, kv_head_num, head_size, max_q_len, max_k_len, max_seq_len, tokens,
                                       (float)(1.0 / sqrt((double)head_size)), stream);
    if (status != ISP_OK) return status;
    // the kernel that adds splits has a vector per lane; its bits are the norm's own where that has, too
    int per_lane = 0;
    const bool norm_adds = isp_norm_launch_config(4, tokens, hidden, 1, nullptr, &per_lane, nullptr, nullptr) == ISP_OK && per_lane == 1;
    const auto normed_product = [&](const void* in, const void* weight, const void* gamma, int k) {
        const TiledPlan plan = tiled_plan_f32(tokens, hidden, k, kTiledMaxSplits, nullptr);
        if (plan.splits == 1 || !norm_adds) {
            const int made = isp_linear_rows_f32(in, weight, out, sums, tokens, hidden, k, stream);
            return made != ISP_OK ? made : isp_fused_add_bias_residual_rmsnorm_f32(residual, out, nullptr, gamma, eps, tokens, hidden, 0, stream);
        }
        float* partial = static_cast<float*>(sums);
        launch_tiled_f32(plan, static_cast<const float*>(in), static_cast<const float*>(weight), partial, tokens, hidden, k, stream);
        launch_norm_sums(partial, plan.splits, static_cast<float*>(residual), static_cast<float*>(out), static_cast<const float*>(gamma), eps,
                         tokens, hidden, stream);
        return note_launch(hipGetLastError());
    };
    status = normed_product(context, o_weight, ffn_norm, ctx);
    if (status != ISP_OK) return status;
    double fused_us, split_us;
    const TiledPlan fused = tiled_plan_f32(tokens, 2 * inter, hidden, 1, &fused_us);
    tiled_plan_f32(tokens, 2 * inter, hidden, kTiledMaxSplits, &split_us);
    if (fused_us <= split_us + 2.5 + 12.0 * tokens * inter / 4.5 * 1e-6) {
        launch_tiled_swiglu_f32(fused, static_cast<const float*>(out), static_cast<const float*>(gate_up_weight), static_cast<float*>(act),
                                tokens, inter, hidden, stream);
        status = note_launch(hipGetLastError());
    } else {
        status = isp_linear_rows_f32(out, gate_up_weight, product, sums, tokens, 2 * inter, hidden, stream);
        if (status != ISP_OK) return status;
        status = isp_swiglu_f32(product, act, tokens, inter, stream);
    }
    if (status != ISP_OK) return status;
    return normed_product(act, down_weight, next_norm, inter);
}

}  // namespace isp

extern "C" {

size_t isp_context_layer_rows_f16_workspace(int batch, int token_num, int hidden, int head_num, int kv_head_num, int head_size,
                                            int max_q_len, int max_k_len, int max_seq_len, int inter) {
    if (isp::layer_shape(0, batch, token_num, hidden, head_num, kv_head_num, head_size, max_q_len, max_k_len, max_seq_len, inter,
                         0) != ISP_OK)
        return 0;
    return isp::layer_plans(batch, token_num, hidden, head_num, kv_head_num, head_size, max_q_len, max_k_len, inter).bytes;
}

int isp_context_layer_rows_f16(const void* normed, void* residual, void* out, const void* qkv_weight, const void* qkv_bias,
                               const void* o_weight, const void* gate_up_weight, const void* down_weight, const void* ffn_norm,
                               const void* next_norm, void* q, void* k_cache, void* v_cache, void* context, void* act,
                               const int32_t* padding_offset, const int32_t* history_length, const int32_t* input_length,
                               const int32_t* context_length, void* workspace, int layer, int batch, int token_num, int hidden,
                               int head_num, int kv_head_num, int head_size, int max_q_len, int max_k_len, int max_seq_len, int inter,
                               int rotary_dim, float rotary_base, float eps, isp_stream_t stream) {
    const int shape = isp::layer_shape(layer, batch, token_num, hidden, head_num, kv_head_num, head_size, max_q_len, max_k_len,
                                       max_seq_len, inter, rotary_dim);
    if (shape != ISP_OK) return shape;
    return isp::context_layer(normed, residual, out, qkv_weight, qkv_bias, o_weight, gate_up_weight, down_weight, ffn_norm, next_norm, q,
                              k_cache, v_cache, context, act, padding_offset, history_length, input_length, context_length, workspace,
                              layer, batch, token_num, hidden, head_num, kv_head_num, head_size, max_q_len, max_k_len, max_seq_len,
                              inter, rotary_dim, rotary_base, eps, static_cast<hipStream_t>(stream));
}

size_t isp_context_layer_f16_workspace(int batch, int token_num, int hidden, int head_num, int kv_head_num, int head_size,
                                       int max_q_len, int max_k_len, int max_seq_len, int inter) {
    if (isp::few_rows_shape(token_num, hidden, head_num, kv_head_num, head_size, inter) != ISP_OK) return 0;
    return isp_context_layer_rows_f16_workspace(batch, token_num, hidden, head_num, kv_head_num, head_size, max_q_len, max_k_len,
                                                max_seq_len, inter);
}

int isp_context_layer_f16(const void* normed, void* residual, void* out, const void* qkv_weight, const void* qkv_bias,
                          const void* o_weight, const void* gate_up_weight, const void* down_weight, const void* ffn_norm,
                          const void* next_norm, void* q, void* k_cache, void* v_cache, void* context, void* act,
                          const int32_t* padding_offset, const int32_t* history_length, const int32_t* input_length,
                          const int32_t* context_length, void* workspace, int layer, int batch, int token_num, int hidden,
                          int head_num, int kv_head_num, int head_size, int max_q_len, int max_k_len, int max_seq_len, int inter,
                          int rotary_dim, float rotary_base, float eps, isp_stream_t stream) {
    const int shape = isp::layer_shape(layer, batch, token_num, hidden, head_num, kv_head_num, head_size, max_q_len, max_k_len,
                                       max_seq_len, inter, rotary_dim);
    if (shape != ISP_OK) return shape;
    const int few = isp::few_rows_shape(token_num, hidden, head_num, kv_head_num, head_size, inter);
    if (few != ISP_OK) return few;
    return isp_context_layer_rows_f16(normed, residual, out, qkv_weight, qkv_bias, o_weight, gate_up_weight, down_weight, ffn_norm,
                                      next_norm, q, k_cache, v_cache, context, act, padding_offset, history_length, input_length,
                                      context_length, workspace, layer, batch, token_num, hidden, head_num, kv_head_num, head_size,
                                      max_q_len, max_k_len, max_seq_len, inter, rotary_dim, rotary_base, eps, stream);
}

size_t isp_context_layer_rows_f32_workspace(int batch, int token_num, int hidden, int head_num, int kv_head_num, int head_size,
                                            int max_q_len, int max_k_len, int max_seq_len, int inter) {
    if (isp::layer_shape(0, batch, token_num, hidden, head_num, kv_head_num, head_size, max_q_len, max_k_len, max_seq_len, inter, 0,
                         4) != ISP_OK)
        return 0;
    return isp::layer_space_f32(token_num, hidden, head_num, kv_head_num, head_size, inter).bytes;
}

int isp_context_layer_rows_f32(const void* normed, void* residual, void* out, const void* qkv_weight, const void* qkv_bias,
                               const void* o_weight, const void* gate_up_weight, const void* down_weight, const void* ffn_norm,
                               const void* next_norm, void* q, void* k_cache, void* v_cache, void* context, void* act,
                               const int32_t* padding_offset, const int32_t* history_length, const int32_t* input_length,
                               const int32_t* context_length, void* workspace, int layer, int batch, int token_num, int hidden,
                               int head_num, int kv_head_num, int head_size, int max_q_len, int max_k_len, int max_seq_len, int inter,
                               int rotary_dim, float rotary_base, float eps, isp_stream_t stream) {
    const int shape = isp::layer_shape(layer, batch, token_num, hidden, head_num, kv_head_num, head_size, max_q_len, max_k_len,
                                       max_seq_len, inter, rotary_dim, 4);
    if (shape != ISP_OK) return shape;
    return isp::context_layer_f32(normed, residual, out, qkv_weight, qkv_bias, o_weight, gate_up_weight, down_weight, ffn_norm,
                                  next_norm, q, k_cache, v_cache, context, act, padding_offset, history_length, input_length,
                                  context_length, workspace, layer, batch, token_num, hidden, head_num, kv_head_num, head_size,
                                  max_q_len, max_k_len, max_seq_len, inter, rotary_dim, rotary_base, eps,
                                  static_cast<hipStream_t>(stream));
}

}  // extern "C"
