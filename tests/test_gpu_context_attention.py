"""ops.context_attention against a float64 attention on the CPU, at the extents where its kernels can go wrong: queries
and keys that end inside, at and just past a tile, a single query over long and short histories, grouped heads, an
empty sequence, padded extents larger than the longest query.  Rows that must not be read hold NaN.

Bound in float16: the probabilities are rounded to fp16 before the second product (relative 2^-11 each, averaging out over the
keys) and the result once more; 2e-3 of the largest output is several times that.
In float32: a score of size S has an error of about S 2^-23 (S up to 100 here: sums of 128 products of 2 x 2 standard deviations,
times log2 e / sqrt(128)), which is the relative error of its probability: 100 x 2^-23 = 1.2e-5, and 2e-5 is the bound."""
import pytest
import torch

pytestmark = pytest.mark.gpu

#        lens                 history              heads kv  max_q max_seq
CASES = [([5], [0], 2, 2, 5, 8),
         ([16, 5, 11], [0, 9, 30], 4, 2, 16, 48),
         ([200, 133], [0, 70], 2, 2, 210, 300),
         ([129], [0], 8, 1, 130, 130),
         ([64, 64], [0, 64], 2, 1, 64, 128),
         ([40, 0, 17], [0, 5, 9], 2, 2, 40, 64),
         ([1, 1, 1], [1000, 63, 64], 4, 2, 1, 1100),
         ([1, 1, 1, 1], [0, 31, 32, 33], 8, 2, 1, 64),
         ([1, 1], [255, 700], 32, 1, 1, 1024),
         ([1] * 9, [3, 700, 128, 127, 129, 511, 512, 513, 0], 16, 16, 1, 768),
         ([2, 1, 3], [100, 257, 64], 6, 2, 3, 300),
         ([1, 0, 1], [300, 200, 700], 8, 2, 1, 1024),   # an empty sequence among split keys (fp16)
         ([0, 1, 0], [3, 20, 0], 4, 4, 2, 32),          # and among whole ones
         ([1] * 50 + [0] + [1] * 250, [b % 37 for b in range(301)], 4, 4, 1, 40),   # more sequences than a workgroup has threads,
         ([20, 3, 0, 17] * 75, [b % 5 for b in range(300)], 2, 1, 20, 25),          # which add up the lengths before a sequence's
         ([129, 64], [0, 64], 32, 4, 130, 200),         # from here on more than 256 tiles of 16 queries: fp16 heads of 96 take
         ([31, 0, 17], [97, 5, 9], 64, 8, 33, 130),     # the tiled kernel
         ([33, 32], [31, 96], 64, 64, 33, 128)]


def reference(q, k, v, lens, hist, out):
    heads, hs, group = q.shape[1], q.shape[3], q.shape[1] // k.shape[1]
    t = 0
    for b, (n, h) in enumerate(zip(lens, hist)):
        kk = k[b, :, :h + n].double().repeat_interleave(group, 0)
        vv = v[b, :, :h + n].double().repeat_interleave(group, 0)
        s = (q[b, :, :n].double()[:, :, None, :] * kk[:, None]).sum(-1) * hs ** -0.5
        s.masked_fill_(torch.arange(h + n)[None, None] > h + torch.arange(n)[None, :, None], float("-inf"))
        out[t:t + n] = (torch.softmax(s, -1)[..., None] * vv[:, None]).sum(2).transpose(0, 1)
        t += n
    return out


@pytest.mark.parametrize("dtype,hs", [(torch.float16, 128), (torch.float16, 96), (torch.float16, 64), (torch.float32, 128), (torch.float32, 96),
                                      (torch.float32, 64)])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_attention_matches_float64(isp, dtype, hs, case):
    lens, hist, heads, kv, max_q, max_seq = CASES[case]
    print("[case] attention %s %s hs %d" % (CASES[case], dtype, hs), flush=True)
    g = torch.Generator().manual_seed(case)
    batch, tokens = len(lens), sum(lens)
    nan = float("nan")
    q = torch.full((batch, heads, max_q, hs), nan, dtype=dtype)
    k, v = (torch.full((2, batch, kv, max_seq, hs), nan, dtype=dtype) for _ in range(2))
    for b in range(batch):
        q[b, :, :lens[b]] = 2 * torch.randn(heads, lens[b], hs, generator=g)
        n = lens[b] + hist[b]
        k[1, b, :, :n] = 2 * torch.randn(kv, n, hs, generator=g)
        v[1, b, :, :n] = torch.randn(kv, n, hs, generator=g)
    expect = reference(q, k[1], v[1], lens, hist, torch.zeros(tokens, heads, hs, dtype=torch.float64))
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")   # noqa: E731
    out = torch.full((tokens, heads, hs), nan, dtype=dtype, device="cuda")
    context = [a + b for a, b in zip(lens, hist)]
    isp.context_attention(q.cuda(), k.cuda(), v.cuda(), 1, ints(hist), ints(lens), ints(context), max(context), out)
    got = out.cpu().double()
    assert torch.isfinite(got).all()
    assert (got - expect).abs().max() <= (2e-3 if dtype == torch.float16 else 2e-5) * expect.abs().max()


@pytest.mark.parametrize("dtype,hs", [(torch.float16, 128), (torch.float16, 96), (torch.float16, 64), (torch.float32, 128),
                                      (torch.float32, 96), (torch.float32, 64)])
@pytest.mark.parametrize("even", [False, True])   # equal probabilities: powers of two before the division
@pytest.mark.parametrize("lens,hist,heads", [([1, 1, 1], [40, 100, 2], 4), ([20, 5], [0, 13], 4), ([121, 40], [0, 13], 32)])
def test_an_infinite_value_reaches_only_its_own_sum(isp, dtype, hs, lens, hist, heads, even):
    """An infinite element of a sequence's last visible value row, where no block of keys ends: the queries that see it get
    infinity in that element (not NaN: the rest of the block counts as nothing), and no other element is touched."""
    print("[case] infinite value %s hs %d %s" % (dtype, hs, lens), flush=True)
    g = torch.Generator().manual_seed(hs)
    batch, max_seq = len(lens), 128
    q = (0 if even else 1) * torch.randn(batch, heads, max(lens), hs, generator=g).to(dtype)
    k, v = (torch.randn(1, batch, 2, max_seq, hs, generator=g).to(dtype) for _ in range(2))
    context = [a + b for a, b in zip(lens, hist)]
    expect = reference(q, k[0], v[0], lens, hist, torch.zeros(sum(lens), heads, hs, dtype=torch.float64))
    for b in range(batch):
        v[0, b, :, context[b] - 1, 5] = float("inf")
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")   # noqa: E731
    out = torch.zeros(sum(lens), heads, hs, dtype=dtype, device="cuda")
    isp.context_attention(q.cuda(), k.cuda(), v.cuda(), 0, ints(hist), ints(lens), ints(context), max(context), out)
    got = out.cpu().double()
    last = torch.tensor(lens).cumsum(0) - 1
    assert (got[last, :, 5] == float("inf")).all()
    others = torch.arange(hs) != 5
    assert (got - expect)[:, :, others].abs().max() <= (2e-3 if dtype == torch.float16 else 2e-5) * expect.abs().max()


@pytest.mark.parametrize("dtype,hs", [(torch.float16, 128), (torch.float16, 96), (torch.float16, 64), (torch.float32, 128),
                                      (torch.float32, 96), (torch.float32, 64)])
@pytest.mark.parametrize("lens,heads", [([1, 1, 1], 2), ([1] * 90, 8), ([20, 33, 40], 2), ([130, 33, 40], 64)])
def test_a_context_of_no_keys_gives_zeros(isp, dtype, hs, lens, heads):
    """context_length 0 for one sequence (inconsistent lengths): nothing to attend to, zeros -- with split keys, whole ones and
    in the prompt kernels; its neighbours are untouched."""
    print("[case] no keys %s hs %d %s" % (dtype, hs, lens[:3]), flush=True)
    g = torch.Generator().manual_seed(hs)
    batch, max_seq = len(lens), 600 if max(lens) == 1 else max(lens)
    hist = [max_seq - n for n in lens]
    q = torch.randn(batch, heads, max(lens), hs, generator=g).to(dtype)
    k, v = (torch.randn(1, batch, heads, max_seq, hs, generator=g).to(dtype) for _ in range(2))
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")   # noqa: E731
    out = torch.full((sum(lens), heads, hs), float("nan"), dtype=dtype, device="cuda")
    context = [max_seq, 0] + [max_seq] * (batch - 2)
    isp.context_attention(q.cuda(), k.cuda(), v.cuda(), 0, ints(hist), ints(lens), ints(context), max_seq, out)
    first = lens[0]
    assert not out[first:first + lens[1]].any()
    rest = [0, batch - 1]
    expect = reference(q[rest], k[0][rest], v[0][rest], [lens[b] for b in rest], [hist[b] for b in rest],
                       torch.zeros(lens[0] + lens[-1], heads, hs, dtype=torch.float64))
    got = torch.cat([out[:first], out[-lens[-1]:]]).cpu().double()
    assert (got - expect).abs().max() <= (2e-3 if dtype == torch.float16 else 2e-5) * expect.abs().max()


@pytest.mark.parametrize("hs", [128, 64])
def test_more_short_prompts_than_a_grid_row(isp, hs):
    """4200 sequences of up to 16 tokens: more than 65535 query rows, and few enough queries per group for the decode kernel."""
    g = torch.Generator().manual_seed(1)
    lens = [[16, 1, 5, 0][b % 4] for b in range(4200)]
    q = torch.randn(len(lens), 1, 16, hs, generator=g).half()
    k, v = (torch.randn(1, len(lens), 1, 16, hs, generator=g).half() for _ in range(2))
    ints = torch.tensor(lens, dtype=torch.int32, device="cuda")
    out = torch.zeros(sum(lens), 1, hs, dtype=torch.float16, device="cuda")
    isp.context_attention(q.cuda(), k.cuda(), v.cuda(), 0, torch.zeros_like(ints), ints, ints, 16, out)
    some = [b for b in range(len(lens)) if b % 4 != 3][-300:]
    first = torch.tensor([0] + lens).cumsum(0)
    expect = reference(q[some], k[0][some], v[0][some], [lens[b] for b in some], [0] * len(some),
                       torch.zeros(sum(lens[b] for b in some), 1, hs, dtype=torch.float64))
    got = torch.cat([out[first[b]:first[b + 1]] for b in some]).cpu().double()
    assert (got - expect).abs().max() <= 2e-3 * expect.abs().max()


@pytest.mark.parametrize("lens,hist,heads,kv,max_seq", [([300, 77], [0, 0], 16, 2, 320), ([65, 130], [900, 30], 32, 8, 1000),
                                                          ([24], [3000], 2, 2, 3100)])
def test_float16_heads_of_96_keep_their_probabilities(isp, lens, hist, heads, kv, max_seq):
    """The probabilities of 96-element heads are not rounded to fp16 (two halves, 21 bits): the error is the result's own rounding, 2^-11,
    and 2e-5 of the largest output for the scores, as in float32."""
    g = torch.Generator().manual_seed(7)
    batch, context = len(lens), [a + b for a, b in zip(lens, hist)]
    q = 2 * torch.randn(batch, heads, max(lens), 96, generator=g).half()
    k, v = (torch.randn(1, batch, kv, max_seq, 96, generator=g).half() for _ in range(2))
    expect = reference(q, k[0], v[0], lens, hist, torch.zeros(sum(lens), heads, 96, dtype=torch.float64))
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")   # noqa: E731
    out = torch.zeros(sum(lens), heads, 96, dtype=torch.float16, device="cuda")
    isp.context_attention(q.cuda(), k.cuda(), v.cuda(), 0, ints(hist), ints(lens), ints(context), max(context), out)
    assert ((out.cpu().double() - expect).abs() <= 2.0 ** -11 * expect.abs() + 2e-5 * expect.abs().max()).all()
