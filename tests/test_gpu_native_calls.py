"""The native module takes the wrappers' calls on plain operands and leaves everything else to the general path: both give the same bits,
and what one refuses so does the other."""
import pytest
import torch

pytestmark = pytest.mark.gpu


class Sub(torch.Tensor):
    pass


def _calls(isp, dtype):
    """name -> (arguments of plain tensors, positions of the results among them); the wrapper's own order."""
    g = torch.Generator(device="cuda").manual_seed(7)
    r = lambda *s: torch.randn(s, device="cuda", generator=g).to(dtype)   # noqa: E731
    i = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")       # noqa: E731
    batch, heads, kv, seq, hs, tokens, max_seq = 3, 4, 2, 5, 24, 9, 11
    lens, hist = i([5, 1, 3]), i([2, 0, 4])
    offset = torch.zeros(batch, seq, dtype=torch.int32, device="cuda")
    isp.cal_padding_offset(offset, torch.zeros(batch + 1, dtype=torch.int32, device="cuda"), lens)
    cache = lambda: r(2, batch, kv, max_seq, hs)   # noqa: E731
    return {
        "input_embedding": ([i([3, 0, 7]), r(3, 33), r(8, 33)], [1]),
        "cal_padding_offset": ([torch.zeros_like(offset), i([0] * (batch + 1)), lens], [0, 1]),
        "rmsnorm": ([r(tokens, 40), r(40), 1e-5], [0]),
        "fused_add_bias_residual_rmsnorm": ([r(tokens, 40), r(tokens, 40), r(40), r(40), 1e-5], [0, 1]),
        "add_fused_qkv_bias_transpose_and_rope": ([r(batch, heads, seq, hs), r(batch, kv, seq, hs), r(batch, kv, seq, hs),
                                                   r(tokens, heads + 2 * kv, hs), r((heads + 2 * kv) * hs), offset, hist, lens, 16, 10000.0],
                                                  [0, 1, 2]),
        "add_fused_qkv_bias_transpose_rope_and_append": ([r(batch, heads, seq, hs), None, None, cache(), cache(), 1,
                                                          r(tokens, heads + 2 * kv, hs), None, offset, hist, lens, 24, 500], [0, 3, 4]),
        "act": ([r(tokens, 2, 20), r(tokens, 20)], [1]),
        "rope_decode_and_append": ([r(batch, heads + 2 * kv, hs), r((heads + 2 * kv) * hs), cache(), cache(), 0, hist, 0, heads, 24, 10000.0],
                                   [0, 2, 3]),
        "transpose_out_remove_padding": ([r(batch, heads, seq, hs), offset, r(tokens, heads, hs)], [2]),
        "concat_kv_cache": ([r(batch, kv, seq, hs), r(batch, kv, seq, hs), 1, lens, hist, cache(), cache()], [5, 6]),
        "repeat_kv_cache": ([cache(), cache(), lens + hist, 1, r(batch, heads, 9, hs), r(batch, heads, 9, hs)], [4, 5]),
    }


NATIVE = {"add_fused_qkv_bias_transpose_and_rope": "qkv_bias_rope_transpose",
          "add_fused_qkv_bias_transpose_rope_and_append": "qkv_bias_rope_transpose_append", "rope_decode_and_append": "rope_decode_append"}
DEFAULTS = {"input_embedding": [True], "fused_add_bias_residual_rmsnorm": [0], "add_fused_qkv_bias_transpose_and_rope": [2048, False]}
NAMES = ["input_embedding", "cal_padding_offset", "rmsnorm", "fused_add_bias_residual_rmsnorm", "add_fused_qkv_bias_transpose_and_rope",
         "add_fused_qkv_bias_transpose_rope_and_append", "act", "rope_decode_and_append", "transpose_out_remove_padding",
         "concat_kv_cache", "repeat_kv_cache"]


def _copy(args):
    return [a.clone() if isinstance(a, torch.Tensor) else a for a in args]


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("name", NAMES)
def test_native_equals_general(isp, name, dtype, monkeypatch):
    from inferspore_amd import capi, ops
    args, results = _calls(isp, dtype)[name]
    native, general, subclass = _copy(args), _copy(args), _copy(args)
    fn = getattr(capi.calls(), NATIVE.get(name, name))
    assert fn(*native, *DEFAULTS.get(name, [])) == capi.OK, "plain operands must be taken"
    monkeypatch.setattr(ops.capi, "calls", capi._NoCalls)
    getattr(ops, name)(*general)
    monkeypatch.undo()
    # a tensor class of the program's own is left to the general path
    at = next(i for i, a in enumerate(subclass) if isinstance(a, torch.Tensor))
    subclass[at] = subclass[at].as_subclass(Sub)
    assert fn(*subclass, *DEFAULTS.get(name, [])) is None
    getattr(ops, name)(*subclass)
    for i in results:
        assert torch.equal(native[i], general[i]) and torch.equal(subclass[i].as_subclass(torch.Tensor), general[i]), (name, i)


@pytest.mark.parametrize("name", NAMES)
def test_native_leaves_what_is_not_plain(isp, name):
    """Each tensor in turn on the CPU, of another type, not contiguous, missing or one element short in its last extent; one argument less."""
    from inferspore_amd import capi
    args, _ = _calls(isp, torch.float16)[name]
    fn, rest = getattr(capi.calls(), NATIVE.get(name, name)), DEFAULTS.get(name, [])
    optional = {"fused_add_bias_residual_rmsnorm": (0, 2), "add_fused_qkv_bias_transpose_and_rope": (4, 7),
                "add_fused_qkv_bias_transpose_rope_and_append": (7,), "rope_decode_and_append": (1,)}.get(name, ())
    for at, a in enumerate(args):
        if not isinstance(a, torch.Tensor):
            continue
        wide = torch.zeros(tuple(a.shape[:-1]) + (2 * a.shape[-1],), dtype=a.dtype, device="cuda")
        bad = [a.cpu(), a.double() if a.is_floating_point() else a.long(), wide[..., ::2]] + ([] if at in optional else [None])
        bad.append(a[..., :-1].contiguous())
        for b in bad:
            mixed = _copy(args)
            mixed[at] = b
            if b is not None and b.dtype == a.dtype and b.is_cuda and b.shape != a.shape and a.dtype == torch.int32 and \
                    a.dim() == 2 and b.numel() >= 9:
                continue   # a padding offset that still holds every token is taken
            assert fn(*mixed, *rest) is None, (name, at, None if b is None else (b.dtype, b.shape))
    assert fn(*args[:-1], *rest) is None


def test_layer_takes_numbers_as_the_steps_do(isp):
    """Integral and boolean numbers of other classes, weights as parameters outside autograd, and what leaves the one call."""
    import numpy as np
    from inferspore_amd import context_layer as cl
    half = torch.float16
    w = cl.LayerWeights(128, 256, half)
    w.qkv = torch.nn.Parameter(w.qkv, requires_grad=False)
    gamma = torch.ones(128, dtype=half, device="cuda")
    x = torch.randn(20, 128, device="cuda").to(half)
    outs = []
    for layer, rot, base in ((0, 64, 10000.0), (np.int64(0), np.int32(64), 10000)):
        st = cl.BatchState([12, 8], 12, 2, 2, 64, 256, 32, 1, half)
        outs.append(cl._layer_in_one_call(x, x.clone(), w, st, layer, gamma, rot, base, 1e-5))
    assert outs[0] is not None and torch.equal(*outs)
    st = cl.BatchState([12, 8], 12, 2, 2, 64, 256, 32, 1, half)
    call = lambda a=x, b=None, weights=w, rot=64: cl._layer_in_one_call(a, x.clone() if b is None else b, weights, st, 0, gamma, rot, 10000.0, 1e-5)  # noqa: E731
    assert call() is not None
    same = x.clone()
    assert call(a=same, b=same) is None and call(rot=63) is None and call(a=x[:, ::1].t().contiguous().t()) is None
    assert call(a=x.as_subclass(Sub)) is None and call(a=x.bfloat16()) is None
    w.down = torch.nn.Parameter(w.down.clone())
    assert call() is None
    with torch.no_grad():
        assert call() is not None
        with torch.autocast("cuda", torch.float16):
            assert call() is None


@pytest.mark.parametrize("rows,dtype", [(100, torch.float16), (3, torch.float32)])
def test_a_dispatch_mode_sees_the_products(isp, rows, dtype):
    """torch's own counter of operations counts a layer's four products, whose library calls it sees in the steps."""
    from torch.utils.flop_counter import FlopCounterMode

    from inferspore_amd import context_layer as cl
    hidden, inter = 128, 320
    w = cl.LayerWeights(hidden, inter, dtype)
    st = cl.BatchState([rows], rows, 2, 2, 64, inter, rows, 1, dtype)
    x = torch.randn(rows, hidden, device="cuda").to(dtype)
    with FlopCounterMode(display=False) as counter:
        got = cl.context_decoder_layer(x, x.clone(), w, st, 0, w.attn_norm, rotary_dim=64)
    assert counter.get_total_flops() == 2 * rows * (hidden * 3 * hidden + hidden * hidden + 3 * hidden * inter)
    want = cl.context_decoder_layer(x, x.clone(), w, st, 0, w.attn_norm, rotary_dim=64)
    # the library's sums and these: in float16 the four products are rounded to 2^-11 on either side
    assert (got.float() - want.float()).abs().max() <= 2.0 ** -8 * want.float().abs().max()
