"""Products in float32 (isp_linear_rows_f32) against a float64 product: every tile that the plan knows, whole and with its k split over
workgroups, at extents where a tile, its last step of k, its columns or the last split end early; and whole float32 layers in one call
against their steps.

Bound: a sum of k products, each rounded at most once with its addition, has an error of at most k 2^-24 of the sum of the terms'
magnitudes; adding up to sixteen splits rounds fifteen times more."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

#         m     n     k   rows cols  split
SHAPES = [(1, 4, 4, 32, 64, False), (1, 1392, 144, 32, 64, False), (1, 180, 1112, 32, 64, True), (141, 3444, 72, 32, 128, False),
          (1, 2696, 504, 32, 128, True), (400, 3608, 4, 64, 128, False), (2100, 80, 1784, 64, 128, True), (132, 104, 16, 96, 64, False),
          (844, 8, 944, 96, 64, True), (714, 5544, 4, 160, 64, False), (271, 1824, 1008, 160, 64, True)]


def _product(isp, x, w):
    from inferspore_amd import capi
    lib, (m, k), n = capi.lib(), x.shape, w.shape[1]
    guard = 4096
    buf = torch.full((m * n + 2 * guard,), 7.0, device="cuda")
    out = buf[guard:guard + m * n]
    need = lib.isp_linear_rows_f32_workspace(m, n, k)
    work = torch.empty(need, dtype=torch.uint8, device="cuda") if need else None
    capi.check(lib.isp_linear_rows_f32(isp._p(x), isp._p(w), out.data_ptr(), isp._p(work), m, n, k, isp._stream()), "linear_rows_f32")
    assert (buf[:guard] == 7).all() and (buf[guard + m * n:] == 7).all(), "written outside the result"
    return out.view(m, n)


@pytest.mark.parametrize("m,n,k,rows,cols,split", SHAPES)
def test_tiles_match_float64(isp, m, n, k, rows, cols, split):
    from inferspore_amd import capi
    print("[case] linear_rows_f32 %d %d %d" % (m, n, k), flush=True)
    a, b, s = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert capi.lib().isp_linear_rows_f32_plan(m, n, k, ctypes.byref(a), ctypes.byref(b), ctypes.byref(s)) == 0
    assert (a.value, b.value, s.value > 1) == (rows, cols, split), "the shape no longer meets the tile that it is here for"
    g = torch.Generator(device="cuda").manual_seed(m * 7919 + n + k)
    x = torch.randn(m, k, generator=g, device="cuda")
    w = torch.randn(k, n, generator=g, device="cuda")
    expect = x.double() @ w.double()
    size = x.double().abs() @ w.double().abs()
    assert ((_product(isp, x, w).double() - expect).abs() <= (k + 15) * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("m,n,k", [(1, 68, 36), (132, 104, 20), (714, 5544, 4), (271, 1824, 1004)])
def test_infinite_neighbours_do_not_leak(isp, m, n, k):
    """What a tile loads from past the last row, column or k is never mixed in."""
    x = torch.ones(m, k, device="cuda")
    w = torch.ones(k, n, device="cuda")
    w[k - 1, n - 3] = float("inf")
    x[m - 1, k - 2] = float("inf")
    expect = torch.full((m, n), float(k), device="cuda")
    expect[m - 1] = float("inf")
    expect[:, n - 3] = float("inf")
    assert torch.equal(_product(isp, x, w), expect)


def test_what_the_products_refuse(isp):
    from inferspore_amd import capi
    lib = capi.lib()
    p = torch.zeros(64, device="cuda").data_ptr()
    call = lambda m, n, k, a=p: lib.isp_linear_rows_f32(a, p, p, p, m, n, k, isp._stream())   # noqa: E731
    for m, n, k in ((100, 6, 8), (100, 8, 6), (100, 8, 0), (100, 2 ** 22 + 4, 8), (100, 8, 2 ** 22 + 4)):
        assert call(m, n, k) == capi.ERR_UNSUPPORTED
        assert lib.isp_linear_rows_f32_workspace(m, n, k) == 0
    assert call(100, 8, 8, p + 4) == capi.ERR_UNSUPPORTED and call(0, 8, 8) == 0


#        lens               history        heads kv hs   inter  max_q max_seq rot  bias   hidden
LAYERS = [([1], [0], 2, 2, 64, 12, 1, 16, 64, False, 36),
          ([100, 0, 31], [3, 9, 0], 4, 2, 128, 1000, 100, 128, 96, True, 520),
          ([300, 299], [50, 0], 6, 3, 96, 1540, 300, 384, 96, True, 572),
          ([1] * 70, [7] * 70, 16, 2, 128, 4112, 1, 16, 128, False, 2048),
          # the gate / up product with SwiGLU inside, on each of the tiles; a last one with rows too wide for the norm to add splits
          ([1], [0], 1, 1, 64, 4, 1, 16, 64, False, 44), ([30, 3], [0, 0], 1, 1, 64, 4124, 30, 32, 64, False, 36),
          ([100, 63], [0, 0], 1, 1, 64, 4132, 100, 128, 64, False, 36), ([65], [0], 1, 1, 64, 2732, 65, 128, 64, False, 36),
          ([300, 60], [0, 0], 1, 1, 64, 2716, 300, 320, 64, False, 68), ([5, 4], [0, 3], 33, 3, 128, 200, 5, 16, 128, False, 4224)]


@pytest.mark.parametrize("case", range(len(LAYERS)))
def test_one_call_equals_the_steps(isp, case, monkeypatch):
    """The same products step by step: the same kernels in the same order, so everything is EQUAL."""
    from inferspore_amd import context_layer as cl
    lens, hist, heads, kv, hs, inter, max_q, max_seq, rot, bias, hidden = LAYERS[case]
    print("[case] float32 layer in one call %s" % (LAYERS[case],), flush=True)
    g = torch.Generator(device="cuda").manual_seed(case)
    rnd = lambda *s, scale=1.0: scale * torch.randn(s, device="cuda", generator=g)   # noqa: E731
    w = cl.LayerWeights(hidden, inter, torch.float32, generator=g)
    width = (heads + 2 * kv) * hs
    w.qkv, w.o = rnd(hidden, width, scale=hidden ** -0.5), rnd(heads * hs, hidden, scale=hidden ** -0.5)
    w.qkv_bias = rnd(width, scale=0.1) if bias else None
    gamma = rnd(hidden)
    normed, residual = rnd(sum(lens), hidden), rnd(sum(lens), hidden)
    cache = rnd(2, len(lens), kv, max_seq, hs)
    got = []
    for one in (True, False):
        st = cl.BatchState(lens, max_q, heads, kv, hs, inter, max_seq, 2, torch.float32, history=hist)
        st.k_cache.copy_(cache)
        st.v_cache.copy_(-cache)
        r = residual.clone()
        if one:
            out = cl._layer_in_one_call(normed, r, w, st, 1, gamma, rot, 10000.0, 1e-5)
            assert out is not None
        else:
            monkeypatch.setattr(cl, "_layer_in_one_call", lambda *a: None)
            monkeypatch.setattr(cl, "_linear", lambda x, y: _product(isp, x, y))
            out = cl.context_decoder_layer(normed, r, w, st, 1, gamma, rotary_dim=rot)
        got.append((out, r, st.q, st.k_cache, st.v_cache, st.packed_ctx, st.act))
    for name, a, b in zip(("out", "residual", "q", "k_cache", "v_cache", "context", "act"), *got):
        assert torch.isfinite(a).all(), name
        assert torch.equal(a, b), name
