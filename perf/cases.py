"""The work a user of this framework has it do, as cases that a timing program can prepare and run.

Two kinds of program call the framework, and the cases are passes of these two:

  "model"    a LLaMA stack built from `inferspore_amd.context_layer`: token ids -> embedding -> RMSNorm -> every
             layer by `context_decoder_layer` -> the final-normed hidden state, with keys and values left in the cache.
             The same call is a first prompt (no history), a later turn (history and new tokens) and a decode step
             (history and one new token per sequence).
  "kernels"  a program that has its own GEMMs and attention and calls `inferspore_amd.ops` for everything around
             them: the calls that one layer of a prompt batch ("prefill") or of a decode step ("decode") makes, on
             buffers that stand for what its GEMMs wrote.

A case is a dict of plain numbers:
  dtype          "f16" or "f32"
  batch, max_q   sequences and the longest query; the lengths are ragged (see `lengths`) unless max_q is 1
  history        longest history in the cache (0: first prompt); ragged when there is one
  max_seq        positions a cache row holds
  heads, kv_heads, head_size, inter, vocab, bias, layers   the model's dimensions (kernels: layers of the cache)
  step           kernels only: "prefill" or "decode"
  fused          kernels, prefill only: the QKV step with the KV append in one call, or the separate calls of the
                 reference's interface (QKV step, concat, repeat)
"""
import random

import torch

from inferspore_amd import ops
from inferspore_amd.context_layer import BatchState, LayerWeights, context_decoder_layer

EPS = 1e-5
ROTARY_BASE = 10000.0
DTYPES = {"f16": torch.float16, "f32": torch.float32}


def _model(name, **kw):
    case = dict(name=name, kind="model", dtype="f16", batch=1, max_q=1, history=0, max_seq=1024, heads=32, kv_heads=32,
                head_size=128, inter=11008, vocab=32000, bias=False, layers=2)
    case.update(kw)
    return case


def _kernels(name, **kw):
    case = dict(name=name, kind="kernels", step="prefill", fused=True, dtype="f16", batch=8, max_q=512, history=0,
                max_seq=1024, heads=32, kv_heads=32, head_size=128, inter=11008, vocab=32000, bias=False, layers=1)
    case.update(kw)
    return case


def listed():
    return [
        # A batch of ragged prompts on the 32 x 128-head, 4096-wide model: what a serving process does for new requests.
        _model("prompt_batch", batch=8, max_q=512),
        # One short question to an idle server: the time to the first token.
        _model("prompt_one_short", batch=1, max_q=37, max_seq=256),
        # Documents: long prompts, where attention's quadratic part shows.
        _model("prompt_long", batch=4, max_q=2048, max_seq=2048),
        # A later turn of conversations: some new tokens on top of a history in the cache.
        _model("second_turn", batch=8, max_q=96, history=512),
        # One decode step of a running batch with long contexts.
        _model("decode_batch", batch=16, history=1023),
        # One decode step of a larger batch on a model with grouped key / value heads.
        _model("decode_grouped", batch=64, history=500, max_seq=512, heads=32, kv_heads=8, inter=14336),
        # A small model (64-element heads, 1024 wide): prompts of a few hundred tokens.
        _model("small_model_prompt", batch=5, max_q=200, max_seq=512, heads=16, kv_heads=16, head_size=64, inter=2816),
        # fp32, as a numerics check of a model is run: small batch, short prompts.
        _model("prompt_f32", dtype="f32", batch=4, max_q=100, max_seq=256, heads=16, kv_heads=16, inter=5632, vocab=8192),
        # The calls around a caller's own GEMMs in a decode step of 16 sequences: a few rows, latency and launches.
        _kernels("kernels_decode", step="decode", batch=16, max_q=1, history=1023),
        # The same calls of a prompt batch, with biases: the sizes the benchmark is quoted on.
        _kernels("kernels_prompt_bias", bias=True),
        # A large prompt batch on grouped heads.
        _kernels("kernels_prompt_large", batch=16, max_q=1024, kv_heads=8, inter=14336),
        # The reference's separate calls in fp32 on a wider model with an odd number of tokens and sequences.
        _kernels("kernels_separate_f32", dtype="f32", fused=False, batch=5, max_q=301, max_seq=512, heads=40, kv_heads=8,
                 inter=13824, vocab=8192),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _cost(case):
    w = work(case)
    return w["bytes"] / 5e12 + w["flops"] / (1e15 if case["dtype"] == "f16" else 1e14)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _kernels("") if rng.random() < 0.4 else _model("")
        del case["name"]
        case["dtype"] = "f32" if rng.random() < 0.2 else "f16"
        case["head_size"] = rng.choice((128, 128, 128, 64, 96))
        case["heads"] = rng.choice((8, 12, 16, 24, 32, 40))
        case["kv_heads"] = case["heads"] // rng.choice((1, 1, 2, 4))
        # feed-forward widths lie between two and four times the hidden width, in multiples of 16
        hidden = case["heads"] * case["head_size"]
        case["inter"] = int(hidden * rng.uniform(2.0, 4.0)) // 16 * 16
        case["vocab"] = rng.choice((8192, 32000))
        case["bias"] = rng.random() < 0.25
        if rng.random() < 0.35:   # a decode step
            case["batch"] = _log_int(rng, 1, 128)
            case["max_q"], case["history"] = 1, _log_int(rng, 8, 2000)
            if case["kind"] == "kernels":
                case["step"] = "decode"
        else:
            case["batch"] = _log_int(rng, 1, 24)
            # A layer's outputs are comparable over the extents for which torch's scaled_dot_product_attention, a plain
            # way to write its attention, repeats itself bit for bit on an MI355X.  It does for 128-element heads up
            # to contexts of 1024 and for smaller heads up to about 230 queries; beyond, single 16-query stripes differ
            # from one call to the next by up to the result's own size, in 5 to 100 % of calls (320 random extents,
            # 24 calls each; the listed extents repeat themselves over 60 calls).
            longest = 2048 if case["kind"] == "kernels" else 1000 if case["head_size"] == 128 else 200
            case["max_q"] = _log_int(rng, 7, longest)
            case["history"] = _log_int(rng, 16, 1024) if rng.random() < 0.3 else 0
            if case["kind"] == "kernels":
                case["fused"] = rng.random() < 0.7
            else:
                case["history"] = min(case["history"], 1024 - case["max_q"])
        case["max_seq"] = -(-(case["max_q"] + case["history"]) // 64) * 64
        if _cost(case) <= most:
            return case


def lengths(case):
    """(query lengths, history lengths) of the batch: the longest first, the others from a quarter of it upwards."""
    r = random.Random(case["batch"] * 1000003 + case["max_q"] * 1009 + case["history"])
    some = lambda most: [most if b == 0 else r.randint((most + 3) // 4, most) for b in range(case["batch"])]  # noqa: E731
    return some(case["max_q"]), some(case["history"])


def _randn(g, dtype, *shape, scale=1.0):
    return torch.empty(shape, device="cuda", dtype=dtype).normal_(0.0, scale, generator=g)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    q_len, hist = lengths(case)
    tokens, hidden = sum(q_len), case["heads"] * case["head_size"]
    s = {"case": case, "q_len": q_len, "rotary_dim": case["head_size"]}
    s["table"] = _randn(g, dtype, case["vocab"], hidden, scale=0.02)
    s["ids"] = torch.randint(0, case["vocab"], (tokens,), device="cuda", dtype=torch.int32, generator=g)
    s["residual"] = torch.empty((tokens, hidden), device="cuda", dtype=dtype)
    return _prepare_model(s, case, g, dtype, hist) if case["kind"] == "model" else _prepare_kernels(s, case, g, dtype, hist)


def _prepare_model(s, case, g, dtype, hist):
    heads, kv, hs = case["heads"], case["kv_heads"], case["head_size"]
    hidden = heads * hs
    s["weights"] = []
    for _ in range(case["layers"]):
        w = LayerWeights(hidden, case["inter"], dtype, generator=g, qkv_bias=case["bias"])
        if kv != heads:   # grouped heads: a narrower fused projection
            w.qkv = w.qkv[:, :(heads + 2 * kv) * hs].contiguous()
            w.qkv_bias = None if w.qkv_bias is None else w.qkv_bias[:(heads + 2 * kv) * hs].contiguous()
        s["weights"].append(w)
    s["final_norm"] = (0.5 + torch.rand(hidden, device="cuda", generator=g)).to(dtype)
    st = BatchState(s["q_len"], case["max_q"], heads, kv, hs, case["inter"], case["max_seq"], case["layers"], dtype, history=hist)
    if case["history"]:
        for cache in (st.k_cache, st.v_cache):
            cache.normal_(generator=g)
    s["state"] = st
    return s


def _prepare_kernels(s, case, g, dtype, hist):
    batch, max_q, heads, kv, hs, inter = (case[k] for k in ("batch", "max_q", "heads", "kv_heads", "head_size", "inter"))
    tokens, hidden, all_heads = s["ids"].numel(), heads * hs, heads + 2 * kv
    zeros = lambda *shape: torch.zeros(shape, device="cuda", dtype=dtype)   # noqa: E731
    ints = lambda v: torch.tensor(v, device="cuda", dtype=torch.int32)      # noqa: E731
    s["lens"], s["hist"] = ints(s["q_len"]), ints(hist)
    s["context"] = s["lens"] + s["hist"]
    s["gamma"] = (0.5 + torch.rand(hidden, device="cuda", generator=g)).to(dtype)
    s["o_bias"] = _randn(g, dtype, hidden, scale=0.02) if case["bias"] else None
    s["attn_out"] = _randn(g, dtype, tokens, hidden)
    s["qkv"] = _randn(g, dtype, tokens, all_heads, hs)
    s["gate_up"] = _randn(g, dtype, tokens, 2, inter)
    s["act"] = zeros(tokens, inter)
    cache = (case["layers"], batch, kv, case["max_seq"], hs)
    s["k_cache"], s["v_cache"] = zeros(*cache), zeros(*cache)
    if case["step"] == "decode":
        return s
    s["qkv_bias"] = _randn(g, dtype, all_heads * hs, scale=0.02) if case["bias"] else None
    s["padding_offset"] = torch.zeros((batch, max_q), device="cuda", dtype=torch.int32)
    s["cum"] = torch.zeros(batch + 1, device="cuda", dtype=torch.int32)
    s["q"] = zeros(batch, heads, max_q, hs)
    s["ctx"] = _randn(g, dtype, batch, heads, max_q, hs)
    s["packed"] = zeros(tokens, heads, hs)
    if not case["fused"]:
        s["k"], s["v"] = zeros(batch, kv, max_q, hs), zeros(batch, kv, max_q, hs)
        longest = max(a + b for a, b in zip(s["q_len"], hist))
        s["k_all"], s["v_all"] = zeros(batch, heads, longest, hs), zeros(batch, heads, longest, hs)
    return s


def run(s):
    if s["case"]["kind"] == "model":
        return _run_model(s)
    return _run_decode_kernels(s) if s["case"]["step"] == "decode" else _run_prefill_kernels(s)


def _run_model(s):
    residual, weights, st = s["residual"], s["weights"], s["state"]
    ops.input_embedding(s["ids"], residual, s["table"])
    hidden = residual.clone()
    ops.rmsnorm(hidden, weights[0].attn_norm, EPS)
    for layer, w in enumerate(weights):
        following = weights[layer + 1].attn_norm if layer + 1 < len(weights) else s["final_norm"]
        hidden = context_decoder_layer(hidden, residual, w, st, layer, following, rotary_dim=s["rotary_dim"],
                                       rotary_base=ROTARY_BASE, eps=EPS)
    return {"hidden": hidden, "residual": residual, "k_cache": st.k_cache, "v_cache": st.v_cache}


def _run_prefill_kernels(s):
    ops.cal_padding_offset(s["padding_offset"], s["cum"], s["lens"])
    ops.input_embedding(s["ids"], s["residual"], s["table"])
    out = {name: s[name] for name in ("padding_offset", "residual", "attn_out", "q", "k_cache", "v_cache", "packed", "act")}
    if s["case"]["fused"]:
        ops.add_fused_qkv_bias_transpose_rope_and_append(s["q"], None, None, s["k_cache"], s["v_cache"], 0, s["qkv"],
                                                         s["qkv_bias"], s["padding_offset"], s["hist"], s["lens"],
                                                         s["rotary_dim"], ROTARY_BASE)
    else:
        ops.add_fused_qkv_bias_transpose_and_rope(s["q"], s["k"], s["v"], s["qkv"], s["qkv_bias"], s["padding_offset"],
                                                  s["hist"], s["lens"], s["rotary_dim"], ROTARY_BASE)
        ops.concat_kv_cache(s["k"], s["v"], 0, s["lens"], s["hist"], s["k_cache"], s["v_cache"])
        ops.repeat_kv_cache(s["k_cache"], s["v_cache"], s["context"], 0, s["k_all"], s["v_all"])
        out.update(k=s["k"], v=s["v"], k_all=s["k_all"], v_all=s["v_all"])
    ops.transpose_out_remove_padding(s["ctx"], s["padding_offset"], s["packed"])
    ops.fused_add_bias_residual_rmsnorm(s["residual"], s["attn_out"], s["o_bias"], s["gamma"], EPS)
    ops.act(s["gate_up"], s["act"])
    return out


def _run_decode_kernels(s):
    ops.input_embedding(s["ids"], s["residual"], s["table"])
    ops.rope_decode_and_append(s["qkv"], None, s["k_cache"], s["v_cache"], 0, s["hist"], 0, s["case"]["heads"],
                               s["rotary_dim"], ROTARY_BASE)
    ops.fused_add_bias_residual_rmsnorm(s["residual"], s["attn_out"], s["o_bias"], s["gamma"], EPS)
    ops.act(s["gate_up"], s["act"])
    return {name: s[name] for name in ("residual", "qkv", "k_cache", "v_cache", "attn_out", "act")}


def work(case):
    q_len, hist = lengths(case)
    tokens, es = sum(q_len), 2 if case["dtype"] == "f16" else 4
    heads, kv, hs, inter, layers = (case[k] for k in ("heads", "kv_heads", "head_size", "inter", "layers"))
    hidden, qkv_cols = heads * hs, (heads + 2 * kv) * hs
    if case["kind"] == "model":
        matrix = hidden * qkv_cols + hidden * hidden + 3 * hidden * inter
        cache_rows = tokens + sum(hist)            # new rows written, history rows read
        pairs = sum(n * h + n * (n + 1) // 2 for n, h in zip(q_len, hist))
        return {"bytes": es * (layers * (matrix + 2 * cache_rows * kv * hs) + 3 * tokens * hidden),
                "flops": layers * (2.0 * tokens * matrix + 4.0 * pairs * heads * hs)}
    rows = 4 * hidden + 3 * inter                  # table row, residual, the norm's input and output; gate, up, product
    if case["step"] == "decode":
        rows += 2 * qkv_cols + 2 * kv * hs         # packed row in and out, the cache rows
        return {"bytes": es * tokens * rows, "flops": 12.0 * tokens * (hidden + inter)}
    rows += 2 * qkv_cols + 2 * hidden              # packed row in, q and the cache rows out; attention output in and out
    extra = 0
    if not case["fused"]:                          # the padded k and v, and the history and the broadcast over all heads
        extra = 2 * tokens * kv * hs + 2 * sum(hist) * kv * hs + 2 * (tokens + sum(hist)) * hidden
    return {"bytes": es * (tokens * rows + extra), "flops": 12.0 * tokens * (hidden + inter)}


# What two right implementations differ by, times four:
#   model, f16    two layers in f16 against the same in f32: rel 0.0014, max 0.012; against itself with the hidden and
#                 feed-forward columns permuted, i.e. every sum in another order: rel 0.001, max 0.009
#   model, f32    with the columns permuted: rel 5.6e-6, max 3.9e-5
#   kernels, f16  one rounding: rel 2.1e-4, max 4.9e-4 (two implementations may round to different neighbours)
#   kernels, f32  against float64: the norm and SwiGLU rel 6e-8, max 3e-7; the rotation, whose angle of up to a thousand
#                 radians is formed in f32, rel 3.5e-6, max 1.9e-4 (and so in the f32 model's cache: its max)
TOLERANCES = {("model", "f16"): {"rel": 5e-3, "max": 5e-2}, ("model", "f32"): {"rel": 2.5e-5, "max": 8e-4},
              ("kernels", "f16"): {"rel": 8e-4, "max": 2e-3}, ("kernels", "f32"): {"rel": 1.4e-5, "max": 8e-4}}


def tolerance(case):
    return TOLERANCES[case["kind"], case["dtype"]]
