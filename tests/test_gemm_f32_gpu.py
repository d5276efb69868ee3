"""The float32 product of many rows (operands split into three bfloat16 parts) against float64: every tile shape at the edges
of its tiles, slices of K, and values at the ends of float32's range."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

TILES = [-1, 0, 1, 2, 3]


def ops():
    from litellmengine_amd.csrc.ops import default_ops

    return default_ops()


def operands(M, N, K, seed=0):
    g = torch.Generator(device="cuda").manual_seed(1000 * seed + M + 7 * N + 13 * K)
    x = torch.randn(M, K, generator=g, device="cuda") * torch.exp2(torch.randint(-8, 9, (M, 1), generator=g, device="cuda").float())
    return x, torch.randn(N, K, generator=g, device="cuda") * 0.02


def exponent(w):
    return math.frexp(float(w.abs().max()))[1] - 1


def check(got, x, w):
    """Every element within what K float32 additions may lose of the sum of its products' sizes; all together within 6 x 2^-24 of
    those (with random signs a sum stays sqrt(K) below its products' sizes, and so do its roundings; without the third parts
    of the operands it would be 2^-18 sqrt(1 / K) or more off at these K)."""
    want = x.double() @ w.double().T
    size = x.double().abs() @ w.double().abs().T
    K = x.shape[1]
    off = (got.double() - want).abs()
    assert bool((off <= 2.0 ** -24 * (K + 16) * size).all())
    assert float(off.norm() / size.norm()) <= 2.0 ** -24 * 6 / math.sqrt(K) * max(1.0, K / 64)


@pytest.mark.parametrize("tiles", TILES)
@pytest.mark.parametrize("M,N,K", [(1, 1, 4), (65, 64, 32), (64, 129, 36), (257, 127, 100), (128, 256, 28), (300, 2049, 64), (66, 131, 4)])
def test_tiles_at_their_edges(tiles, M, N, K):
    x, w = operands(M, N, K)
    check(ops().linear_f32_tiles(x, w, tiles=tiles)[0], x, w)


@pytest.mark.parametrize("slices,K", [(2, 128), (3, 260), (8, 96), (5, 1028)])
def test_slices_add_up(slices, K):
    """(8 slices of three steps: the last ones are empty)"""
    x, w = operands(70, 192, K, seed=1)
    parts = ops().linear_f32_tiles(x, w, slices=slices)
    assert parts.shape == (slices, 70, 192) and bool(torch.isfinite(parts).all())
    check(parts.double().sum(0), x, w)


def test_the_product_takes_slices_where_its_reader_adds_them_up():
    from litellmengine_amd.parts import PartialSums

    o = ops()
    x, w = operands(100, 1024, 3072, seed=2)
    whole, cut = o.linear(x, w), o.linear(x, w, sums_ok=True)
    assert isinstance(cut, PartialSums) and cut.sums.shape[0] == o.f32_slices_for(100, 1024, 3072) > 1
    check(whole, x, w)
    check(cut.total(), x, w)
    assert o.f32_slices_for(100, 1022, 3072) == 1 and o.f32_slices_for(100, 1 << 17, 4096) == 1


@pytest.mark.parametrize("tiles", TILES)
@pytest.mark.parametrize("M,N,K", [(1, 1, 4), (65, 64, 32), (64, 129, 36), (257, 127, 100), (128, 256, 28), (300, 2049, 64), (96, 1024, 4100)])
def test_halves_at_their_edges(tiles, M, N, K):
    o = ops()
    x, w = operands(M, N, K, seed=6)
    check(o.linear_f32_halves(x, w, exponent(w), tiles=tiles)[0], x, w)


def test_a_model_learns_its_weights_exponents():
    """Projections of a float32 model know them once all weights are bound; their products are the halves' from 96 rows on."""
    from litellmengine_amd.models import make_context
    from litellmengine_amd.parts import Linear

    ctx = make_context("float32")
    part = Linear(["a", "b"], 2048, [2048, 2048])
    weights = {n: torch.randn(2048, 2048, device="cuda") * 0.02 for n in ("a", "b")}
    part.bind(weights, ctx)
    assert part.known == {}
    ctx.settle()
    assert part.known == {"exponent": exponent(part.weight)} and ctx.looked_over == []
    x, w = operands(96, 4096, 2048, seed=8)
    part.weight.copy_(w)
    check(part.forward(x), x, w)
    assert torch.equal(part.forward(x), ctx.ops.linear_f32_halves(x, w, part.known["exponent"])[0])


@pytest.mark.parametrize("slices,K", [(2, 128), (3, 260), (8, 96)])
def test_halves_in_slices(slices, K):
    o = ops()
    x, w = operands(130, 192, K, seed=7)
    check(o.linear_f32_halves(x, w, exponent(w), slices).double().sum(0), x, w)


@pytest.mark.parametrize("far", [0, 12, 24, 60])
def test_halves_of_numbers_far_apart(far):
    """Numbers of a row up to 2^far apart, rows and weights of any size: off by float32's own roundings of the products, or by
    2^-37 of a row's largest number (what its halves hold no more of) times the other row's, whichever is more."""
    o = ops()
    g = torch.Generator(device="cuda").manual_seed(far)
    M, N, K = 100, 136, 512
    powers = lambda rows, most: torch.exp2(-torch.randint(0, most + 1, (rows, K), generator=g, device="cuda").float())
    x = torch.randn(M, K, generator=g, device="cuda") * powers(M, far) * torch.exp2(torch.randint(-60, 61, (M, 1), generator=g, device="cuda").float())
    w = torch.randn(N, K, generator=g, device="cuda") * powers(N, far) * torch.exp2(torch.randint(-8, 1, (N, 1), generator=g, device="cuda").float()) * 2.0 ** 20
    x[7], w[9] = 0.0, 0.0
    got, (a, b) = o.linear_f32_halves(x, w, exponent(w))[0].double(), (x.double(), w.double())
    off = (got - a @ b.T).abs()
    most = lambda t: t.abs().amax(1)
    rest = 2.0 ** -37 * (most(a)[:, None] * b.abs().sum(1)[None] + a.abs().sum(1)[:, None] * b.abs().max())
    assert bool((off <= 2.0 ** -24 * (K + 16) * (a.abs() @ b.abs().T) + rest).all())


def test_which_weights_have_an_exponent():
    o = ops()
    w = torch.randn(1029, 4100, device="cuda") * 0.02
    assert o.weight_bounds(w.bfloat16()) is None and o.weight_bounds(w[:, :4099].contiguous()) is None and o.weight_bounds(w[:1000]) is None
    bounds, want = [o.weight_bounds(w)], [exponent(w)]
    for change in (lambda t: t[3].mul_(2.0 ** -20), lambda t: t.mul_(2.0 ** 110), lambda t: t[0, 0].fill_(math.inf), lambda t: t[1028, 4099].fill_(math.nan),
                   lambda t: t[1028, 4099].fill_(-2.0 ** 12), lambda t: t.zero_()):
        t = w.clone()
        change(t)
        bounds.append(o.weight_bounds(t))
        want.append(None)
    t = w.clone()
    t[3] = 0.0  # (a row of zeros has nothing to lose)
    t[700, 5] = -4.0
    assert o.product_exponents(bounds + [o.weight_bounds(t)]) == want + [2] and o.product_exponents([]) == []


@pytest.mark.parametrize("M", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("N,K,slices", [(64, 128, 1), (100, 260, 2), (1024, 3072, 16), (72, 1028, 7), (64, 4, 1)])
def test_few_rows_in_slices(M, N, K, slices):
    """One step for a wavefront, an odd number, a last step that is not whole, rows of the weight that fill no group."""
    x, w = operands(M, N, K, seed=4)
    check(ops().linear_f32_slices(x, w, slices).double().sum(0), x, w)


@pytest.mark.parametrize("M", [1, 8, 16, 17, 32])
@pytest.mark.parametrize("K", [512, 1024, 1536, 2560, 3072, 4096, 520])
def test_few_rows_streamed(M, K):
    """More rows of the weight than sixteen for every CU: a row of x in the registers (and K that is not held), plain and gated."""
    o = ops()
    N = 2 * (17 * o.compute_units() + 5)
    x, w = operands(M, N, K, seed=5)
    check(o.linear(x, w), x, w)
    x = x / x.abs().max()
    gate, up = (x.double() @ w.double().T).chunk(2, dim=1)
    want = torch.nn.functional.silu(gate) * up
    assert float((o.gate_up_silu(x, w).double() - want).norm() / want.norm()) < 2.0 ** -24 * 6 * max(1.0, math.sqrt(K) / 8)


@pytest.mark.parametrize("halves", [False, True])
@pytest.mark.parametrize("tiles", TILES)
def test_values_at_the_ends_of_the_range(tiles, halves):
    """Infinities and NaN where plain float32 has them, numbers that round to infinity in bfloat16, and small ones."""
    x, w = operands(70, 72, 40, seed=3)
    x[3, 5], x[9, 0], x[11, 39] = math.inf, -math.inf, math.nan
    x[20] = 0.0
    x[21], x[22] = x[21] * 2.0 ** -100, x[22] * 2.0 ** 80
    exp = 20
    if halves:
        w *= 2.0 ** 20
        w[8] *= 2.0 ** 12  # (a weight that has grown since it was looked over: infinities among its halves, made again)
        x[20, 8] = 2.0 ** 90
    else:
        x[20, 8], w[:, 8] = 3.4e38, 2.0 ** -30 * w[:, 8].sign()
    w[7, 2] = math.inf
    o = ops()
    got = (o.linear_f32_halves(x, w, exp, tiles=tiles) if halves else o.linear_f32_tiles(x, w, tiles=tiles))[0].cpu()
    want = (x.double().cpu() @ w.double().cpu().T)  # (an infinity's sign follows the weights' signs in both)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[want.isinf()].double(), want[want.isinf()])
    fine = want.isfinite()
    a, b = torch.nan_to_num(x.double().cpu(), posinf=0, neginf=0).abs(), torch.nan_to_num(w.double().cpu(), posinf=0).abs()
    rest = 2.0 ** -37 * (a.amax(1)[:, None] * b.sum(1)[None] + a.sum(1)[:, None] * 2.0 ** (exp + 1)) if halves else 0.0
    assert bool(((got.double() - want).abs() <= 2.0 ** -24 * 56 * (a @ b.T) + rest + 2.0 ** -126)[fine].all())
