"""ops.linear against a float64 product at the extents where its kernel can go wrong: every number of 16-row tiles and rows
that do not fill one, column strips that end early, a last step of 8, 16 or 24 rows of the weight, fewer steps than
wavefronts, one and many splits.

Bound: the products are exact in float32 and the sum of k terms has a relative error of at most k 2^-24 of the sum of their
magnitudes (about 1.1 sqrt(k) standard deviations' worth here: far below the rounding); the result is rounded once, 2^-11."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 8, 8), (1, 128, 32), (2, 136, 40), (15, 120, 136), (16, 4096, 4096), (17, 1024, 2816), (31, 264, 1000),
          (33, 3072, 1024), (48, 640, 4112), (49, 520, 88), (64, 256, 14336), (64, 32768, 64), (16, 33000, 64), (5, 12288, 1536)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_linear_matches_float64(isp, m, n, k):
    print("[case] linear %d %d %d" % (m, n, k), flush=True)
    g = torch.Generator().manual_seed(m * 7919 + n + k)
    x = torch.randn(m, k, generator=g).half()
    w = torch.randn(k, n, generator=g).half()
    expect = x.double() @ w.double()
    size = x.double().abs() @ w.double().abs()
    assert isp.linear_supports(x.cuda(), w.cuda())
    got = isp.linear(x.cuda(), w.cuda()).cpu().double()
    assert torch.isfinite(got).all()
    assert ((got - expect).abs() <= 2.0 ** -11 * expect.abs() + k * 2.0 ** -24 * size).all()


def test_infinite_neighbours_do_not_leak(isp):
    """Rows of the activation and columns of the weight past the requested extents are never mixed in: an infinite value
    reaches only the outputs that contain it."""
    x = torch.ones(3, 40, dtype=torch.float16, device="cuda")
    w = torch.ones(40, 24, dtype=torch.float16, device="cuda")
    w[39, 5] = float("inf")
    x[1, 0] = float("inf")
    got = isp.linear(x, w).cpu()
    expect = torch.full((3, 24), 40.0)
    expect[1] = float("inf")
    expect[:, 5] = float("inf")
    assert torch.equal(got.float(), expect)


def test_other_products_stay_with_torch(isp):
    x = torch.ones(3, 40, dtype=torch.float16, device="cuda")
    w = torch.ones(40, 24, dtype=torch.float16, device="cuda")
    assert not isp.linear_supports(x.expand(65, 3, 40)[:, 0], w)          # too many rows
    assert not isp.linear_supports(x, torch.ones(24, 40, dtype=torch.float16, device="cuda").t())
    assert not isp.linear_supports(x.float(), w.float())
    assert not isp.linear_supports(x[:, :36].contiguous(), w[:36])        # k not a multiple of 8
    assert not isp.linear_supports(x, w.clone().requires_grad_())
