"""A layer of a few rows in one call against the same layer step by step through ops (ops.linear and the kernels of the
separate entry points): the same operations in the same order on the same partial sums, so everything must be EQUAL --
attention included, which both reach by the same kernels.  The extents are where the kernels of the one call can go wrong: rows
that do not fill a wavefront, rotation of part of a head, a bias, grouped heads, padded sequences, an empty one, several
splits, the widest rows, caches that end before the last token."""
import pytest
import torch

pytestmark = pytest.mark.gpu

#        lens              history          heads kv hs   inter  max_q max_seq rot  bias   hidden
CASES = [([1], [0], 2, 2, 64, 264, 1, 8, 64, False, 128),
         ([5, 3], [0, 0], 2, 1, 128, 520, 5, 16, 128, True, 256),
         ([1] * 16, list(range(0, 160, 10)), 8, 2, 128, 1040, 1, 256, 96, False, 1024),
         ([7, 0, 20], [3, 9, 0], 4, 4, 64, 1000, 24, 32, 64, True, 264),
         ([1, 4], [50, 0], 6, 3, 96, 392, 4, 64, 96, True, 576),
         ([64], [0], 12, 3, 128, 88, 64, 64, 128, False, 1536),
         ([1, 1, 1], [30, 31, 40], 16, 16, 64, 2816, 1, 32, 0, True, 1024),   # the last two sequences' rows are past the cache
         ([2, 2], [100, 7], 64, 8, 128, 4096, 2, 128, 128, False, 8192),
         # rows wider than the kernel that adds splits and normalises takes: the splits are added by themselves
         ([1], [9], 2, 2, 64, 264, 1, 16, 64, False, 8320),
         ([1] * 16, list(range(16)), 2, 1, 128, 1040, 1, 32, 128, True, 10240),
         ([9, 8], [0, 5], 2, 2, 128, 1040, 9, 32, 128, False, 8320)]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_one_call_equals_the_steps(isp, case, monkeypatch):
    from inferspore_amd import context_layer as cl
    lens, hist, heads, kv, hs, inter, max_q, max_seq, rot, bias, hidden = CASES[case]
    print("[case] layer in one call %s" % (CASES[case],), flush=True)
    g = torch.Generator(device="cuda").manual_seed(case)
    half = torch.float16
    rnd = lambda *s, scale=1.0: (scale * torch.randn(s, device="cuda", generator=g)).to(half)   # noqa: E731
    w = cl.LayerWeights(hidden, inter, half, generator=g)
    width = (heads + 2 * kv) * hs
    w.qkv, w.o = rnd(hidden, width, scale=hidden ** -0.5), rnd(heads * hs, hidden, scale=hidden ** -0.5)
    w.qkv_bias = rnd(width, scale=0.1) if bias else None
    gamma = rnd(hidden)
    normed, residual = rnd(sum(lens), hidden), rnd(sum(lens), hidden)
    cache = rnd(2, len(lens), kv, max_seq, hs)
    got = []
    for one in (True, False):
        st = cl.BatchState(lens, max_q, heads, kv, hs, inter, max_seq, 2, half, history=hist)
        st.k_cache.copy_(cache)
        st.v_cache.copy_(-cache)
        r = residual.clone()
        if one:
            out = cl._layer_in_one_call(normed, r, w, st, 1, gamma, rot, 10000.0, 1e-5)
            assert out is not None
        else:
            monkeypatch.setattr(cl, "_layer_in_one_call", lambda *a: None)
            out = cl.context_decoder_layer(normed, r, w, st, 1, gamma, rotary_dim=rot)
        got.append((out, r, st.q, st.k_cache, st.v_cache, st.packed_ctx, st.act))
    for name, a, b in zip(("out", "residual", "q", "k_cache", "v_cache", "context", "act"), *got):
        assert torch.isfinite(a).all(), name
        assert torch.equal(a, b), name


def test_what_is_not_plain_goes_step_by_step(isp):
    from inferspore_amd import context_layer as cl
    w = cl.LayerWeights(256, 512, torch.float16)
    st = cl.BatchState([3], 3, 2, 2, 128, 512, 8, 1, torch.float16)
    x = torch.randn(3, 256, device="cuda").half()
    call = lambda n, w=w: cl._layer_in_one_call(n, x.clone(), w, st, 0, w.attn_norm, 128, 1e4, 1e-5)   # noqa: E731
    assert call(x) is not None
    assert call(x.float()) is None and call(x[:2]) is None and call(x.t().contiguous().t()) is None
    w.down = w.down.t().contiguous().t()
    assert call(x) is None
    out = cl.context_decoder_layer(x, x.clone(), w, st, 0, w.attn_norm)
    w.down = w.down.contiguous()
    assert (out.float() - call(x).float()).abs().max() <= 2.0 ** -9 * out.float().abs().max()


def test_a_few_tokens_among_thousands_of_empty_sequences(isp):
    """More than 65535 query rows: the layer still runs in one call."""
    from inferspore_amd import context_layer as cl
    w = cl.LayerWeights(64, 64, torch.float16)
    st = cl.BatchState([5] + [0] * 4198 + [2], 16, 1, 1, 64, 64, 16, 1, torch.float16)
    x = torch.randn(7, 64, device="cuda").half()
    out = cl._layer_in_one_call(x, x.clone(), w, st, 0, w.attn_norm, 64, 1e4, 1e-5)
    assert out is not None and torch.isfinite(out).all()
    assert torch.equal(st.packed_ctx[[0, 5], 0], st.v_cache[0, [0, 4199], 0, 0])   # a first token attends to itself


@pytest.mark.parametrize("rows,hidden,inter,kv,one", [(16, 64, 16392, 1, True), (17, 64, 16392, 1, False), (64, 64, 16384, 1, True),
                                                      (33, 64, 64, 171, False), (64, 64, 64, 170, True), (65, 64, 16392, 1, True),
                                                      (128, 8200, 24416, 1, False), (129, 8200, 24416, 1, True),
                                                      (65, 8192, 24416, 1, True), (65, 8200, 24376, 1, True), (128, 8200, 39640, 1, True),
                                                      (192, 9224, 21688, 1, False), (193, 9224, 21688, 1, True)])
def test_layers_that_are_faster_step_by_step(isp, rows, hidden, inter, kv, one):
    """Few rows with wide products keep the library's product for them."""
    from inferspore_amd import context_layer as cl
    print("[case] route of %s" % ((rows, hidden, inter, kv),), flush=True)
    zeros = lambda *s: torch.zeros(s, dtype=torch.float16, device="cuda")   # noqa: E731
    w = cl.LayerWeights.__new__(cl.LayerWeights)
    w.qkv, w.qkv_bias, w.o, w.gate_up = zeros(hidden, 3 * kv * 64), None, zeros(kv * 64, hidden), zeros(hidden, 2 * inter)
    w.down, w.ffn_norm, w.attn_norm = zeros(inter, hidden), zeros(hidden), zeros(hidden)
    st = cl.BatchState([1] * rows, 1, kv, kv, 64, inter, 1, 1, torch.float16)
    x = zeros(rows, hidden)
    assert (cl._layer_in_one_call(x, x.clone(), w, st, 0, w.attn_norm, 64, 1e4, 1e-5) is not None) == one
