"""What a program does to a BatchState is what its layers see: an edited or replaced mask counts, and k_all / v_all hold the
broadcast of the layer that ran last, whichever form of the attention the layer would take by itself.

Bound of the attention: as in test_gpu_context_attention (float16 2e-3, float32 2e-5 of the largest output)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

HEADS, KV, HS, INTER, HIDDEN = 4, 2, 64, 128, 256
LENS = {"few": [7, 4], "many": [50, 33]}   # up to 64 rows: a layer of float16 rows is one call


def layers(edit, dtype, rows, count=1):
    from inferspore_amd import context_layer as cl
    lens = LENS[rows]
    g = torch.Generator(device="cuda").manual_seed(4)
    st = cl.BatchState(lens, max(lens), HEADS, KV, HS, INTER, 64, 2, dtype)
    x = torch.randn(sum(lens), HIDDEN, device="cuda", generator=g).to(dtype)
    edit(st)
    for layer in range(count):
        w = cl.LayerWeights(HIDDEN, INTER, dtype, generator=g)
        w.qkv = w.qkv[:, :(HEADS + 2 * KV) * HS].contiguous()
        cl.context_decoder_layer(x, x.clone(), w, st, layer, w.attn_norm, rotary_dim=HS)
    return st, lens


def attention64(st, lens, hidden_key):
    """Packed attention of layer 0 from the state's queries and caches; queries past 0 do not see `hidden_key` (None: see all)."""
    rows = []
    for b, n in enumerate(lens):
        k, v = (c[0, b, :, :n].double().repeat_interleave(HEADS // KV, 0) for c in (st.k_cache, st.v_cache))
        s = (st.q[b, :, :n].double()[:, :, None] * k[:, None]).sum(-1) * HS ** -0.5
        i = torch.arange(n, device="cuda")
        s.masked_fill_(i[None] > i[:, None], float("-inf"))
        if hidden_key is not None:
            s[:, 1:, hidden_key] = float("-inf")
        rows.append((torch.softmax(s, -1)[..., None] * v[:, None]).sum(2).transpose(0, 1))
    return torch.cat(rows)


@pytest.mark.parametrize("rows", ["few", "many"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("how", ["edited", "replaced"])
def test_the_states_mask_counts(isp, dtype, rows, how):
    def edit(st):
        mask = st.mask if how == "edited" else st._build_mask()
        mask[:, :, 1:, 0] = float("-inf")
        for b, n in enumerate(LENS[rows]):
            mask[b, :, n:, 0] = 0.0   # padded queries see something; their output is dropped
        if how == "replaced":
            st.mask = mask

    st, lens = layers(edit, dtype, rows)
    expect = attention64(st, lens, 0)
    bound = (2e-3 if dtype == torch.float16 else 2e-5) * expect.abs().max()
    assert (st.packed_ctx.double() - expect).abs().max() <= bound
    assert (attention64(st, lens, None) - expect).abs().max() > 10 * bound   # the mask makes a difference


@pytest.mark.parametrize("rows", ["few", "many"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("asked", ["before", "after"])
def test_k_all_holds_what_the_last_layer_attended_to(isp, dtype, rows, asked):
    st, lens = layers(lambda st: st.k_all if asked == "before" else None, dtype, rows, count=2)
    for got, cache in ((st.k_all, st.k_cache), (st.v_all, st.v_cache)):
        for b, n in enumerate(lens):
            assert torch.equal(got[b, :, :n], cache[1, b, :, :n].repeat_interleave(HEADS // KV, 0))
            assert not got[b, :, n:].any()
    assert (st.packed_ctx.double() - attention_of_layer_1(st, lens)).abs().max() <= 2e-3 * st.packed_ctx.abs().max()


def attention_of_layer_1(st, lens):
    from types import SimpleNamespace
    return attention64(SimpleNamespace(q=st.q, k_cache=st.k_cache[1:], v_cache=st.v_cache[1:]), lens, None)


def test_a_state_that_keeps_its_own_buffers_is_not_rebuilt(isp):
    """A copy keeps what was set, and an attribute that never existed is still an error."""
    import copy
    from inferspore_amd import context_layer as cl
    st = cl.BatchState([3], 3, HEADS, KV, HS, INTER, 8, 1, torch.float16)
    own = torch.full((1, 1, 3, 3), -1.0, dtype=torch.float16, device="cuda")
    st.mask = own
    assert st.k_all.shape == (1, HEADS, 3, HS) and st.mask is own and copy.copy(st).mask is own
    with pytest.raises(AttributeError):
        st.masks


def shifted(t):
    """The same extents one element past an aligned address."""
    flat = torch.zeros(t.numel() + 8, dtype=t.dtype, device="cuda")
    return flat[1:1 + t.numel()].view(t.shape)


@pytest.mark.parametrize("rows", ["few", "many"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("name", ["q", "k_cache", "v_cache", "packed_ctx", "packed_ctx in q"])
def test_a_programs_own_unaligned_buffers(isp, dtype, rows, name):
    def edit(st):
        if name == "packed_ctx in q":
            st.packed_ctx = st.q.view(-1)[:st.packed_ctx.numel()].view(st.packed_ctx.shape)
        else:
            setattr(st, name, shifted(getattr(st, name)))

    st, lens = layers(edit, dtype, rows)
    if name == "packed_ctx in q":   # the queries are gone: against the run with buffers of their own
        expect = layers(lambda st: st.mask, dtype, rows)[0].packed_ctx.double()
    else:
        expect = attention64(st, lens, None)
    assert (st.packed_ctx.double() - expect).abs().max() <= (2e-3 if dtype == torch.float16 else 2e-5) * expect.abs().max()


def test_more_sequences_than_a_grid_holds(isp):
    """65536 sequences of one token: the padded form, as ever."""
    from inferspore_amd import context_layer as cl
    n = 65536
    st = cl.BatchState([1] * n, 1, 1, 1, 64, 16, 1, 1, torch.float16)
    w = cl.LayerWeights(64, 16, torch.float16)
    x = torch.randn(n, 64, device="cuda").half()
    cl.context_decoder_layer(x, x.clone(), w, st, 0, w.attn_norm, rotary_dim=64)
    assert torch.equal(st.packed_ctx[:, 0], st.v_cache[0, :, 0, 0])   # one key: its value


@pytest.mark.parametrize("rows", ["few", "many"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_context_lengths_of_another_batch_are_refused(isp, dtype, rows):
    def edit(st):
        st.context = torch.cat([st.context, st.context])

    with pytest.raises(RuntimeError, match="batch extents"):
        layers(edit, dtype, rows)


@pytest.mark.parametrize("dtype,hs,lens,heads,kv", [(torch.float16, 64, [7, 3] * 1000, 8, 2), (torch.float16, 128, [1] * 4000, 2, 2),
                                                    (torch.float16, 96, [2, 1] * 2700, 2, 2), (torch.float32, 64, [1, 2] * 8000, 1, 1)])
def test_thousands_of_tiny_contexts_take_the_padded_form(isp, dtype, hs, lens, heads, kv):
    from inferspore_amd import context_layer as cl
    hidden = 64
    g = torch.Generator(device="cuda").manual_seed(2)
    st = cl.BatchState(lens, max(lens), heads, kv, hs, 32, max(lens), 1, dtype)
    assert "k_all" in st.__dict__
    w = cl.LayerWeights(hidden, 32, dtype, generator=g)
    width = (heads + 2 * kv) * hs
    w.qkv = (torch.randn(hidden, width, device="cuda", generator=g) * hidden ** -0.5).to(dtype)
    w.o = (torch.randn(heads * hs, hidden, device="cuda", generator=g) * hidden ** -0.5).to(dtype)
    x = torch.randn(sum(lens), hidden, device="cuda", generator=g).to(dtype)
    cl.context_decoder_layer(x, x.clone(), w, st, 0, w.attn_norm, rotary_dim=hs)
    padded = st.packed_ctx.clone()
    isp.context_attention(st.q, st.k_cache, st.v_cache, 0, st.history, st.lengths, st.context, st.max_k_len, st.packed_ctx)
    assert (padded.float() - st.packed_ctx.float()).abs().max() <= (4e-3 if dtype == torch.float16 else 4e-5) * padded.abs().max()


@pytest.mark.parametrize("lens,history", [([7] * 200, 0), ([24] * 1000, 0), ([1] * 4000, 31)])
def test_other_batches_build_no_padded_buffers(isp, lens, history):
    from inferspore_amd import context_layer as cl
    st = cl.BatchState(lens, max(lens), 8, 2, 64, 32, max(lens) + history, 1, torch.float16, history=[history] * len(lens))
    assert "k_all" not in st.__dict__ and "mask" not in st.__dict__


@pytest.mark.parametrize("rows", ["few", "many"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_a_programs_own_state_object(isp, dtype, rows):
    """An object with the attributes that the steps of a layer read, and no others."""
    from types import SimpleNamespace
    from inferspore_amd import context_layer as cl
    lens = LENS[rows]
    st = cl.BatchState(lens, max(lens), HEADS, KV, HS, INTER, 64, 1, dtype)
    names = ("tokens", "head_num", "kv_head_num", "head_size", "q", "k_cache", "v_cache", "padding_offset", "history", "lengths",
             "context", "packed_ctx", "act", "k_all", "v_all", "mask")
    own = SimpleNamespace(**{n: getattr(st, n) for n in names})
    g = torch.Generator(device="cuda").manual_seed(9)
    w = cl.LayerWeights(HIDDEN, INTER, dtype, generator=g)
    w.qkv = w.qkv[:, :(HEADS + 2 * KV) * HS].contiguous()
    x = torch.randn(sum(lens), HIDDEN, device="cuda", generator=g).to(dtype)
    out = cl.context_decoder_layer(x, x.clone(), w, own, 0, w.attn_norm, rotary_dim=HS)
    expect = attention64(own, lens, None)
    assert torch.isfinite(out).all()
    assert (own.packed_ctx.double() - expect).abs().max() <= (2e-3 if dtype == torch.float16 else 2e-5) * expect.abs().max()


def test_a_state_saved_before(isp):
    """A copy without what a layer notes in it still builds its buffers."""
    import copy
    from inferspore_amd import context_layer as cl
    st = copy.copy(cl.BatchState([3, 2], 3, HEADS, KV, HS, INTER, 8, 1, torch.float16))
    del st.__dict__["_attended"]
    assert st.mask.shape == (2, 1, 3, 3) and not st.k_all.any()
