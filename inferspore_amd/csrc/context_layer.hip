// isp_context_layer_f16: a whole context-decoder layer for up to 64 packed fp16 rows (a decode step, a short prompt) in one call.
// Nine or ten launches: each of the four products leaves fp32 partial sums, and the step that follows adds them where it
// would have read the product -- QKV bias + RoPE + KV append, residual + RMSNorm (twice), SwiGLU.  As separate calls a layer
// takes 14 launches (four products, their four additions, six steps) and, from Python, about 13 us of host time each, more than a
// small layer's kernels take: 16 sequences at 256-1023 keys 271 against 262 us for two layers, one prompt of 37 tokens 256
// against 246.
// The steps and their order are those of the reference's kernel comments (see inferspore_amd/context_layer.py).
#include <math.h>

#include "linear_rows.h"

namespace isp {

struct LayerPlans {
    SkinnyPlan qkv, o, gate_up, down;
    size_t floats;  // of the largest product's partial sums, or the attention's: they are used one after the other
};

static LayerPlans layer_plans(int batch, int tokens, int hidden, int head_num, int kv_head_num, int head_size, int max_q_len,
                              int max_k_len, int inter) {
    const int width = (head_num + 2 * kv_head_num) * head_size, ctx = head_num * head_size;
    LayerPlans p;
    p.qkv = skinny_plan(tokens, width, hidden);
    p.o = skinny_plan(tokens, hidden, ctx);
    p.gate_up = skinny_plan(tokens, 2 * inter, hidden);
    p.down = skinny_plan(tokens, hidden, inter);
    p.floats = attention_workspace(batch, head_num, kv_head_num, head_size, max_q_len, max_k_len) / sizeof(float);
    const size_t sizes[] = {p.qkv.partial_floats(tokens, width), p.o.partial_floats(tokens, hidden),
                            p.gate_up.partial_floats(tokens, 2 * inter), p.down.partial_floats(tokens, hidden)};
    for (size_t s : sizes) p.floats = s > p.floats ? s : p.floats;
    return p;
}

// ISP_OK where the layer runs here.
static int layer_shape(int layer, int batch, int tokens, int hidden, int head_num, int kv_head_num, int head_size, int max_q_len,
                       int max_k_len, int max_seq_len, int inter, int rotary_dim) {
    if (layer < 0 || batch <= 0 || tokens <= 0 || hidden <= 0 || head_num <= 0 || kv_head_num <= 0 || head_size <= 0 ||
        max_q_len <= 0 || max_k_len <= 0 || max_seq_len <= 0 || inter <= 0 || rotary_dim < 0 || head_num % kv_head_num != 0 ||
        rotary_dim % 2 != 0 || rotary_dim > head_size)
        return ISP_ERR_BAD_SHAPE;
    if (tokens > kSkinnyMaxRows || (head_size != 64 && head_size != 96 && head_size != 128) || hidden % 8 != 0 || hidden > kNormSumsMaxHidden ||
        inter % 8 != 0 || batch > 65535 || max_q_len > 65535 * 16 || (long long)batch * max_q_len > 0x7fffffffll ||
        ((long long)head_num + 2ll * kv_head_num) * head_size > (1 << 24) || inter > (1 << 24))
        return ISP_ERR_UNSUPPORTED;
    // wide products of many rows are the library's (5120 x 40928, 64 rows: 85 us there, 124 here); below the line a whole layer is
    // ahead of its steps, with the library's products or with these (4096 wide, 64 rows, 2 x inter 20480 ... 32768: 159 ... 172 us
    // against 163 ... 174, 166 ... 188 with the library for gate / up and 244 ... 293 with it for all four)
    if (tokens > 16 && (2 * inter > 32768 || (head_num + 2 * kv_head_num) * head_size > 32768)) return ISP_ERR_UNSUPPORTED;
    return ISP_OK;
}

}  // namespace isp

extern "C" {

size_t isp_context_layer_f16_workspace(int batch, int token_num, int hidden, int head_num, int kv_head_num, int head_size,
                                       int max_q_len, int max_k_len, int max_seq_len, int inter) {
    if (isp::layer_shape(0, batch, token_num, hidden, head_num, kv_head_num, head_size, max_q_len, max_k_len, max_seq_len, inter,
                         0) != ISP_OK)
        return 0;
    return isp::layer_plans(batch, token_num, hidden, head_num, kv_head_num, head_size, max_q_len, max_k_len, inter).floats *
           sizeof(float);
}

int isp_context_layer_f16(const void* normed, void* residual, void* out, const void* qkv_weight, const void* qkv_bias,
                          const void* o_weight, const void* gate_up_weight, const void* down_weight, const void* ffn_norm,
                          const void* next_norm, void* q, void* k_cache, void* v_cache, void* context, void* act,
                          const int32_t* padding_offset, const int32_t* history_length, const int32_t* input_length,
                          const int32_t* context_length, void* workspace, int layer, int batch, int token_num, int hidden,
                          int head_num, int kv_head_num, int head_size, int max_q_len, int max_k_len, int max_seq_len, int inter,
                          int rotary_dim, float rotary_base, float eps, isp_stream_t stream_) {
    using namespace isp;
    const int shape = layer_shape(layer, batch, token_num, hidden, head_num, kv_head_num, head_size, max_q_len, max_k_len,
                                  max_seq_len, inter, rotary_dim);
    if (shape != ISP_OK) return shape;
    const void* needed[] = {normed, residual, out, qkv_weight, o_weight, gate_up_weight, down_weight, ffn_norm, next_norm,
                            q, k_cache, v_cache, context, act, padding_offset, history_length, input_length, context_length, workspace};
    for (const void* p : needed) ISP_REQUIRE_PTR(p);
    const void* vectors[] = {normed, residual, out, qkv_weight, qkv_bias, o_weight, gate_up_weight, down_weight, ffn_norm,
                             next_norm, q, k_cache, v_cache, context, act, workspace};
    for (const void* p : vectors)
        if (!aligned16(p)) return ISP_ERR_UNSUPPORTED;
    const hipStream_t stream = static_cast<hipStream_t>(stream_);
    const auto half_in = [](const void* p) { return static_cast<const __half*>(p); };
    const auto half_out = [](void* p) { return static_cast<__half*>(p); };
    const LayerPlans plan = layer_plans(batch, token_num, hidden, head_num, kv_head_num, head_size, max_q_len, max_k_len, inter);
    float* sums = static_cast<float*>(workspace);
    const int width = (head_num + 2 * kv_head_num) * head_size, ctx = head_num * head_size;
    const size_t slice = (size_t)layer * batch * kv_head_num * max_seq_len * head_size;

    launch_skinny(plan.qkv, half_in(normed), half_in(qkv_weight), nullptr, sums, token_num, width, hidden, stream);
    launch_qkv_sums(sums, plan.qkv.splits, half_in(qkv_bias), half_out(q), half_out(k_cache) + slice, half_out(v_cache) + slice,
                    padding_offset, history_length, input_length, batch, max_q_len, token_num, head_num, kv_head_num, head_size,
                    max_seq_len, rotary_dim, rotary_base, stream);
    int status = note_launch(hipGetLastError());
    if (status != ISP_OK) return status;
    status = context_attention(static_cast<const _Float16*>(q), static_cast<const _Float16*>(k_cache),
                               static_cast<const _Float16*>(v_cache), static_cast<_Float16*>(context), history_length,
                               input_length, context_length, layer, batch, head_num, kv_head_num, head_size, max_q_len, max_k_len,
                               max_seq_len, token_num, (float)(1.0 / sqrt((double)head_size)), sums, stream);
    if (status != ISP_OK) return status;
    launch_skinny(plan.o, half_in(context), half_in(o_weight), nullptr, sums, token_num, hidden, ctx, stream);
    launch_norm_sums(sums, plan.o.splits, half_out(residual), half_out(out), half_in(ffn_norm), eps, token_num, hidden, stream);
    if (plan.gate_up.splits == 1) {  // nothing to add: the product itself, in half the bytes
        launch_skinny(plan.gate_up, half_in(out), half_in(gate_up_weight), half_out(workspace), nullptr, token_num, 2 * inter,
                      hidden, stream);
        status = isp_swiglu_f16(workspace, act, token_num, inter, stream_);
        if (status != ISP_OK) return status;
    } else {
        launch_skinny(plan.gate_up, half_in(out), half_in(gate_up_weight), nullptr, sums, token_num, 2 * inter, hidden, stream);
        launch_swiglu_sums(sums, plan.gate_up.splits, half_out(act), token_num, inter, stream);
    }
    launch_skinny(plan.down, half_in(act), half_in(down_weight), nullptr, sums, token_num, hidden, inter, stream);
    launch_norm_sums(sums, plan.down.splits, half_out(residual), half_out(out), half_in(next_norm), eps, token_num, hidden, stream);
    return note_launch(hipGetLastError());
}

}  // extern "C"
