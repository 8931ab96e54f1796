"""Products of more than 16 rows (isp_linear_rows_f16) against a float64 product: every tile that the plan knows, whole and with its k
split over workgroups, at extents where a tile, its last step of k, its columns or the last split end early; and whole layers of
prompts in one call against their steps.

Bound: the products are exact in float32 and the sum of k terms has a relative error of at most k 2^-24 of the sum of their
magnitudes; the result is rounded once, 2^-11, or to a subnormal, 2^-25."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

#         m     n     k   rows cols  split
SHAPES = [(17, 16, 8, 32, 128, False), (18, 16, 208, 32, 128, True), (31, 12296, 72, 32, 128, False),
          (65, 248, 96, 64, 64, False), (68, 240, 216, 64, 64, True), (260, 5520, 1112, 64, 128, False),
          (65, 1632, 4488, 64, 128, True), (129, 5984, 224, 128, 64, False), (132, 1832, 1976, 128, 64, True),
          (386, 4752, 584, 128, 128, False), (130, 3624, 3272, 128, 128, True), (644, 6040, 72, 128, 192, False),
          (393, 5384, 7112, 128, 192, True), (1330, 5528, 208, 128, 256, False), (137, 5472, 5232, 128, 256, True),
          (3369, 3488, 72, 192, 256, False), (517, 6768, 3656, 192, 256, True), (3846, 1056, 464, 256, 128, False),
          (403, 2720, 4784, 256, 128, True), (2752, 4464, 72, 256, 256, False), (904, 4360, 3992, 256, 256, True)]


def _product(isp, x, w):
    from inferspore_amd import capi
    lib, (m, k), n = capi.lib(), x.shape, w.shape[1]
    guard = 4096
    buf = torch.full((m * n + 2 * guard,), 7.0, dtype=torch.float16, device="cuda")
    out = buf[guard:guard + m * n]
    need = lib.isp_linear_rows_f16_workspace(m, n, k)
    work = torch.empty(need, dtype=torch.uint8, device="cuda") if need else None
    capi.check(lib.isp_linear_rows_f16(isp._p(x), isp._p(w), out.data_ptr(), isp._p(work), m, n, k, isp._stream()), "linear_rows")
    assert (buf[:guard] == 7).all() and (buf[guard + m * n:] == 7).all(), "written outside the result"
    return out.view(m, n)


# 17 to 48 rows by the kernel for few rows (tile 0 x 0): two and three tiles of 16 rows, whole and split, with a last step of 8, 16 or 24
# rows of the weight and a strip that ends early
SHAPES += [(25, 30056, 744, 0, 0, False), (17, 2456, 9064, 0, 0, True), (17, 14568, 1520, 0, 0, True), (41, 32560, 1904, 0, 0, False),
           (33, 16344, 4280, 0, 0, True)]


@pytest.mark.parametrize("m,n,k,rows,cols,split", SHAPES)
def test_tiles_match_float64(isp, m, n, k, rows, cols, split):
    from inferspore_amd import capi
    print("[case] linear_rows %d %d %d" % (m, n, k), flush=True)
    a, b, s = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert capi.lib().isp_linear_rows_f16_plan(m, n, k, ctypes.byref(a), ctypes.byref(b), ctypes.byref(s)) == 0
    assert (a.value, b.value, s.value > 1) == (rows, cols, split), "the shape no longer meets the tile that it is here for"
    g = torch.Generator(device="cuda").manual_seed(m * 7919 + n + k)
    x = torch.randn(m, k, generator=g, device="cuda").half()
    w = torch.randn(k, n, generator=g, device="cuda").half()
    expect = x.double() @ w.double()
    size = x.double().abs() @ w.double().abs()
    got = _product(isp, x, w).double()
    assert ((got - expect).abs() <= 2.0 ** -11 * expect.abs() + 2.0 ** -25 + k * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("m,n,k", [(18, 136, 216), (70, 264, 72), (300, 520, 8), (2752, 4464, 72), (25, 30056, 744),
                                   (41, 32560, 1904)])
def test_infinite_neighbours_do_not_leak(isp, m, n, k):
    """What a tile loads from past the last row, column or k is never mixed in."""
    x = torch.ones(m, k, dtype=torch.float16, device="cuda")
    w = torch.ones(k, n, dtype=torch.float16, device="cuda")
    w[k - 1, n - 3] = float("inf")
    x[m - 1, k - 2] = float("inf")
    expect = torch.full((m, n), float(k), device="cuda")
    expect[m - 1] = float("inf")
    expect[:, n - 3] = float("inf")
    assert torch.equal(_product(isp, x, w).float(), expect)


def test_what_the_products_refuse(isp):
    from inferspore_amd import capi
    lib = capi.lib()
    p = torch.zeros(64, dtype=torch.float16, device="cuda").data_ptr()
    call = lambda m, n, k, a=p: lib.isp_linear_rows_f16(a, p, p, p, m, n, k, isp._stream())   # noqa: E731
    for m, n, k in ((100, 12, 8), (100, 8, 12), (100, 8, 0), (100, 2 ** 22 + 8, 8), (100, 8, 2 ** 22 + 8)):
        assert call(m, n, k) == capi.ERR_UNSUPPORTED
        assert lib.isp_linear_rows_f16_workspace(m, n, k) == 0
    assert call(100, 8, 8, p + 2) == capi.ERR_UNSUPPORTED and call(0, 8, 8) == 0
    assert lib.isp_linear_f16(p, p, p, p, 65, 8, 8, isp._stream()) == capi.ERR_UNSUPPORTED


#        lens               history        heads kv hs   inter  max_q max_seq rot  bias   hidden
LAYERS = [([40, 37], [0, 0], 2, 2, 64, 264, 40, 64, 64, False, 128),
          ([100, 0, 31], [3, 9, 0], 4, 2, 128, 1000, 100, 128, 96, True, 520),
          ([70] * 8, list(range(0, 80, 10)), 8, 2, 128, 2816, 70, 256, 128, False, 1024),
          ([300, 299], [50, 0], 6, 3, 96, 1544, 300, 384, 96, True, 576),
          ([300, 299], [0, 3], 20, 5, 128, 6912, 300, 320, 128, False, 2560),
          ([80], [0], 65, 65, 128, 96, 80, 128, 128, False, 8320),       # rows wider than the kernel that adds splits and normalises takes
          ([1] * 130, [7] * 130, 16, 2, 128, 4112, 1, 16, 128, False, 2048)]


def _rows(m, inter, hidden):
    return ([1] * m, [3] * m, 1, 1, 64, inter, 1, 8, 64, False, hidden)


# SwiGLU inside the gate / up product, on each of the tiles
INSIDE = {(32, 128): (17, 16, 32), (64, 64): (70, 16, 32), (64, 128): (130, 8680, 32), (128, 64): (787, 624, 224),
          (128, 128): (874, 1168, 616), (128, 192): (66, 16400, 40), (128, 256): (274, 8856, 144), (192, 256): (523, 9928, 48),
          (256, 128): (1542, 1296, 240), (256, 256): (390, 14224, 40)}
LAYERS += [_rows(*extents) for extents in INSIDE.values()]
# gate / up products that take another kernel by themselves than with SwiGLU to follow or inside: the one for few rows, of four tiles of
# 16 rows, and a tile
LAYERS += [_rows(57, 16384, 4096), _rows(31, 14728, 736)]


def _plan(name, *extents):
    from inferspore_amd import capi
    a, b, s = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert getattr(capi.lib(), name)(*extents, ctypes.byref(a), ctypes.byref(b), ctypes.byref(s)) == 0
    return a.value, b.value, s.value


@pytest.mark.parametrize("tile", INSIDE)
def test_layers_meet_every_tile(isp, tile):
    assert _plan("isp_gate_up_rows_f16_plan", *INSIDE[tile]) == tile + (1,), "the layer no longer meets the tile that it is here for"


@pytest.mark.parametrize("case", range(len(LAYERS)))
def test_one_call_equals_the_steps(isp, case, monkeypatch):
    """The same products step by step: the same sums in the same order, so everything is EQUAL, SwiGLU inside the product included.
    Tiles add k in one order, whatever their size; only where the gate / up product takes the kernel for few rows here and not there
    are the orders others, each value rounded once or twice."""
    from inferspore_amd import context_layer as cl
    lens, hist, heads, kv, hs, inter, max_q, max_seq, rot, bias, hidden = LAYERS[case]
    print("[case] prompt layer in one call %s" % (LAYERS[case],), flush=True)
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
            monkeypatch.setattr(cl, "_linear", lambda x, y: _product(isp, x, y))
            out = cl.context_decoder_layer(normed, r, w, st, 1, gamma, rotary_dim=rot)
        got.append((out, r, st.q, st.k_cache, st.v_cache, st.packed_ctx, st.act))
    here, there = (_plan("isp_gate_up_rows_f16_plan", sum(lens), inter, hidden), _plan("isp_linear_rows_f16_plan", sum(lens), 2 * inter, hidden))
    same_order = here[2] == there[2] and (here[0] == 0) == (there[0] == 0)
    assert same_order or LAYERS[case] in LAYERS[-2:]
    for name, a, b in zip(("out", "residual", "q", "k_cache", "v_cache", "context", "act"), *got):
        assert torch.isfinite(a).all(), name
        if same_order:
            assert torch.equal(a, b), name
        else:
            assert (a.float() - b.float()).abs().max() <= 2.0 ** -9 * b.float().abs().max(), name
