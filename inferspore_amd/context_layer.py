"""Caller-side glue: one LLaMA context-decoder (prefill) layer built from this library's kernels.

The reference ships the kernels but not the layer code that calls them (its `src/layers` and
`Llama<T>` class are absent); this module is the call sequence its kernel comments and weight layout
imply (fused QKV weight `[H, 3H]`, fused gate/up weight `[H, 2I]`, reference
src/weights/llama/layer_weights.cc:19-62), so that the kernels can be exercised and timed in the
order a model runs them:

    normed, residual                       (packed [tokens, H]; `normed` = RMSNorm(residual) by attn_norm)
    qkv      = normed @ Wqkv                                 product
    q, cache += k, v = add_fused_qkv_bias_transpose_rope_and_append(qkv)    * this library
    packed   = context_attention(q, cache)                   * this library (heads of 64, 96 or 128 elements; others, and
                                                               a state with a mask of its own: repeat_kv_cache, torch's
                                                               attention, transpose_out_remove_padding)
    attn_out = packed @ Wo                                   product
    residual, normed2 = fused_add_bias_residual_rmsnorm(residual, attn_out, ffn_norm)      * this library
    act      = SwiGLU(normed2 @ Wgate_up)                    product + * this library
    ffn_out  = act @ Wdown                                   product
    residual, normed_next = fused_add_bias_residual_rmsnorm(residual, ffn_out, next attn_norm)   * this library

A layer of float16 or float32 rows is one call of the C ABI (isp_context_layer_rows_f16, _f32), products included.  Where a layer runs
step by step (a mask of its own, unaligned buffers, gradients, a dispatch mode, few rows with the widest products), products of up to 64
float16 rows go to ops.linear and the others to torch's library calls (hipBLASLt GEMMs); everything marked * goes through the C ABI.  All
work is issued on torch's current stream.
"""
import math

import torch

from . import capi, ops

_PADDED = frozenset(("mask", "k_all", "v_all"))


class LayerWeights:
    """Weights of one layer in the reference's fused layout."""

    def __init__(self, hidden, inter, dtype, device="cuda", generator=None, qkv_bias=False):
        def w(*shape, scale):
            return (scale * torch.randn(shape, device=device, generator=generator)).to(dtype)

        self.qkv = w(hidden, 3 * hidden, scale=hidden ** -0.5)
        self.qkv_bias = w(3 * hidden, scale=0.02) if qkv_bias else None
        self.o = w(hidden, hidden, scale=hidden ** -0.5)
        self.gate_up = w(hidden, 2 * inter, scale=hidden ** -0.5)   # columns [0, I) gate, [I, 2I) up
        self.down = w(inter, hidden, scale=inter ** -0.5)
        self.attn_norm = (0.5 + torch.rand(hidden, device=device, generator=generator)).to(dtype)
        self.ffn_norm = (0.5 + torch.rand(hidden, device=device, generator=generator)).to(dtype)


def _padded_is_faster(dtype, batch, max_q_len, max_k_len, head_num, kv_head_num, head_size):
    """Thousands of contexts of a few keys.  The attention alone: a workgroup of the fused kernels costs 5 to 10 ns of the chip even then,
    one per key head (up to 16 queries per group) or per query head; torch's kernel works in tiles of 16 keys and takes 2.5 to 9 ns per head.
    float16, 128 elements, us fused and padded: 1000 prompts of 7 / 12 / 16 tokens, 32 heads over 8 313 and 172 / 331 and 240 / 340
    and 296, of 24 363 and 673; 4000 decode rows of 8 keys, 8 heads 193 and 123, 8 over 2 below it.  Beyond ten thousand
    sequences the lengths that every workgroup adds up count as well: 16000 decode rows of 8 keys, 8 heads 959 and 470; in float32
    60000 of 1 / 8 / 12 keys 5359 and 3141 / 5585 and 4017 / level.  Heads of 96 in float16 lie in between (4000 rows of 2 keys
    132 and 117, 16000 of 12 876 and 808).  Fewer workgroups are over before torch's launches are: 1000 rows of 4 keys, 8 heads of
    64, 30 and 41.
    Whole layers, which in the padded form have the library's products as well: decode rows keep that gain (4000 rows of 8 keys, 1024
    wide, 342 in one call and 284 padded; 16000 x 4096 9470 and 7680; 30000 in float32 7810 and 7650); prompts do not (1000 of 7 / 12 / 16
    tokens, 4096 wide, 2342 and 2644 / 3703 and 4426 / 4835 and 5197): for them the line is still the attention's."""
    if max_k_len > 16 or batch * head_num * head_size < 1000000:
        return False
    tiled = head_num // max(kv_head_num, 1) * max_q_len > 16
    if not tiled and head_num != kv_head_num:
        return False
    if dtype == torch.float32:
        return max_k_len <= batch // 7000
    if head_size == 96:
        return batch >= 4000 and max_k_len <= min(12, batch // 2000)
    return tiled or batch >= 16000 or max_k_len <= 8


class BatchState:
    """Padding bookkeeping of one ragged prefill batch plus the buffers a layer needs."""

    def __init__(self, lengths, max_q_len, head_num, kv_head_num, head_size, inter, max_seq_len, layers, dtype,
                 history=None):
        dev = "cuda"
        self.batch = len(lengths)
        self.max_q_len, self.max_seq_len = max_q_len, max_seq_len
        self.head_num, self.kv_head_num, self.head_size = head_num, kv_head_num, head_size
        self.lengths = torch.as_tensor(lengths, dtype=torch.int32).to(dev)
        self.history = (torch.zeros(self.batch, dtype=torch.int32, device=dev) if history is None
                        else torch.as_tensor(history, dtype=torch.int32).to(dev))
        self.context = self.lengths + self.history
        self.tokens = int(sum(lengths))
        self.max_k_len = int(max(int(l) + int(h) for l, h in zip(lengths, self.history.tolist())))
        self.padding_offset = torch.zeros((self.batch, max_q_len), dtype=torch.int32, device=dev)
        self.cum_seqlens = torch.zeros(self.batch + 1, dtype=torch.int32, device=dev)
        ops.cal_padding_offset(self.padding_offset, self.cum_seqlens, self.lengths)
        z = lambda *s: torch.zeros(s, dtype=dtype, device=dev)
        self.q = z(self.batch, head_num, max_q_len, head_size)
        self.k_cache = z(layers, self.batch, kv_head_num, max_seq_len, head_size)
        self.v_cache = z(layers, self.batch, kv_head_num, max_seq_len, head_size)
        self.packed_ctx = z(self.tokens, head_num, head_size)
        self.act = z(self.tokens, inter)

        self._attended = None   # the layer whose attention ran last without the buffers below
        if (not ops.context_attention_supports(dtype, head_size) or
                (self.tokens > 64 and _padded_is_faster(dtype, self.batch, max_q_len, self.max_k_len, head_num, kv_head_num,
                                                        head_size))):
            self._padded_buffers()

    def _padded_buffers(self):
        """What the padded form of the attention (repeat, mask, transpose) works on; what a program has set itself stays."""
        shape = (self.batch, self.head_num, self.max_k_len, self.head_size)
        missing = [name for name in ("k_all", "v_all") if name not in self.__dict__]
        for name in missing:
            self.__dict__[name] = torch.zeros(shape, dtype=self.q.dtype, device=self.q.device)
        attended = self.__dict__.get("_attended")   # missing in a state saved before layers left a note
        if missing and attended is not None:
            ops.repeat_kv_cache(self.k_cache, self.v_cache, self.context, attended, self.k_all, self.v_all)
        if "mask" not in self.__dict__:
            self.mask = self._build_mask()

    def __getattr__(self, name):
        # The fused attention needs none of them: they are built when a program first asks, k_all and v_all with the broadcast of
        # the layer that ran last.  From then on (or from when a program sets one) the layers take the padded form, so that an
        # edited mask counts and k_all, v_all hold what a layer attended to.
        if name not in _PADDED or "act" not in self.__dict__:
            raise AttributeError(name)
        self._padded_buffers()
        return self.__dict__[name]

    def _build_mask(self):
        """Additive attention mask [batch, 1, max_q_len, max_k_len]: query s of sequence b sees keys
        0 .. history[b] + s, and only when s is a valid position."""
        dev = self.q.device
        s = torch.arange(self.max_q_len, device=dev)[None, :, None]
        kpos = torch.arange(self.max_k_len, device=dev)[None, None, :]
        hist = self.history[:, None, None]
        visible = (kpos <= hist + s) & (s < self.lengths[:, None, None])
        mask = torch.zeros((self.batch, 1, self.max_q_len, self.max_k_len), dtype=self.q.dtype, device=dev)
        mask.masked_fill_(~visible[:, None], float("-inf"))
        # fully padded query rows would be all -inf: let them see key 0 (their output is discarded)
        mask[:, :, :, 0].masked_fill_(~(s[:, :, 0] < self.lengths[:, None])[:, None], 0.0)
        return mask


def _padded_asked(st):
    """Whether a program has set or asked for the padded form's mask or buffers.  Its own state object has the mask that the padded
    form needs, or was made for the fused one."""
    if not isinstance(st, BatchState):
        return hasattr(st, "mask")
    return not _PADDED.isdisjoint(st.__dict__) or hasattr(type(st), "mask")


def _fused_attention(st):
    """Whether a layer's attention is the fused kernel's: not where that does not take the state's buffers (an unaligned view in a
    program's own cache, say), nor where a program has asked for the padded form."""
    return not _padded_asked(st) and ops.context_attention_takes(st.q, st.k_cache, st.v_cache, st.packed_ctx)


def _layer_in_one_call(normed, residual, w, st, layer_id, gamma, rotary_dim, rotary_base, eps):
    """The whole layer as one call of the C ABI, or None where it is not the plain case of float16 or float32 rows: everything
    that the steps below accept or refuse otherwise stays with them."""
    if normed.dtype not in (torch.float16, torch.float32) or _padded_asked(st):
        return None
    out = capi.calls().context_layer(
        normed, residual, w.qkv, w.qkv_bias, w.o, w.gate_up, w.down, w.ffn_norm, gamma, st.q, st.k_cache, st.v_cache, st.packed_ctx,
        st.act, st.padding_offset, st.history, st.lengths, st.context, int(layer_id), int(st.tokens), int(st.head_num),
        int(st.kv_head_num), int(st.head_size), int(st.max_k_len), int(rotary_dim), float(rotary_base), float(eps))
    if type(out) is int:
        capi.check(out, "isp_context_layer")
    if out is not None and isinstance(st, BatchState):
        st._attended = int(layer_id)
    return out


def _linear(x, w):
    return ops.linear(x, w) if ops.linear_supports(x, w) else x @ w


def context_decoder_layer(normed, residual, w, state, layer_id, next_norm_gamma, rotary_dim=128,
                          rotary_base=10000.0, eps=1e-5):
    """Runs one prefill layer.  `normed` and `residual` are packed [tokens, H]; `residual` is updated in
    place; returns the next layer's normalised input (a new tensor)."""
    st = state
    out = _layer_in_one_call(normed, residual, w, st, layer_id, next_norm_gamma, rotary_dim, rotary_base, eps)
    if out is not None:
        return out
    qkv = _linear(normed, w.qkv)                                                 # [tokens, 3H]
    qkv = qkv.view(st.tokens, st.head_num + 2 * st.kv_head_num, st.head_size)
    # bias + RoPE + re-pad of q, with k and v written straight into the cache (one launch, no padded k / v)
    ops.add_fused_qkv_bias_transpose_rope_and_append(st.q, None, None, st.k_cache, st.v_cache, layer_id, qkv,
                                                     w.qkv_bias, st.padding_offset, st.history, st.lengths,
                                                     rotary_dim, rotary_base)
    if _fused_attention(st):
        ops._expect(st.context.shape[0] == st.q.shape[0], "batch extents differ")
        ops.context_attention(st.q, st.k_cache, st.v_cache, layer_id, st.history, st.lengths, st.context, st.max_k_len,
                              st.packed_ctx)
        if isinstance(st, BatchState):
            st._attended = int(layer_id)
    else:
        ops.repeat_kv_cache(st.k_cache, st.v_cache, st.context, layer_id, st.k_all, st.v_all)
        ctx = torch.nn.functional.scaled_dot_product_attention(st.q, st.k_all, st.v_all, attn_mask=st.mask,
                                                               scale=1.0 / math.sqrt(st.head_size))
        ops.transpose_out_remove_padding(ctx.contiguous(), st.padding_offset, st.packed_ctx)
    attn_out = _linear(st.packed_ctx.view(st.tokens, -1), w.o)
    ops.fused_add_bias_residual_rmsnorm(residual, attn_out, None, w.ffn_norm, eps)   # attn_out := normed
    gate_up = _linear(attn_out, w.gate_up).view(st.tokens, 2, -1)
    ops.act(gate_up, st.act)
    ffn_out = _linear(st.act, w.down)
    ops.fused_add_bias_residual_rmsnorm(residual, ffn_out, None, next_norm_gamma, eps)
    return ffn_out
