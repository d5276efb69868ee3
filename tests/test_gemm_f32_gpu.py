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


@pytest.mark.parametrize("tiles", TILES)
def test_values_at_the_ends_of_the_range(tiles):
    """Infinities and NaN where plain float32 has them, numbers that round to infinity in bfloat16, and small ones."""
    x, w = operands(70, 72, 40, seed=3)
    x[3, 5], x[9, 0], x[11, 39] = math.inf, -math.inf, math.nan
    w[7, 2] = math.inf
    x[20] = 0.0
    x[20, 8], w[:, 8] = 3.4e38, 2.0 ** -30 * w[:, 8].sign()
    x[21], x[22] = x[21] * 2.0 ** -100, x[22] * 2.0 ** 90
    got = ops().linear_f32_tiles(x, w, tiles=tiles)[0].cpu()
    want = (x.double().cpu() @ w.double().cpu().T)  # (an infinity's sign follows the weights' signs in both)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[want.isinf()].double(), want[want.isinf()])
    fine = want.isfinite()
    size = torch.nan_to_num(x.double().cpu(), posinf=0, neginf=0).abs() @ torch.nan_to_num(w.double().cpu(), posinf=0).abs().T
    assert bool(((got.double() - want).abs()[fine] <= (2.0 ** -24 * 56 * size)[fine] + 2.0 ** -126).all())


def projection(weight):
    """A model's projection of one weight, bound as a model binds it."""
    from litellmengine_amd.models import make_context
    from litellmengine_amd.parts import Linear

    part = Linear(["w"], weight.shape[1], [weight.shape[0]])
    part.bind({"w": weight}, make_context("float32"))
    return part


@pytest.mark.parametrize("M", [65, 96, 300])
def test_all_bits_of_an_operand_count(M):
    """Numbers with bits at both ends of a float32 significand, and beside the largest number of a row others 2^23 below it
    whose weights are all that is not zero.  Four products of the first kind: at most a rounding each and one for each of
    three additions, or what the parts leave out, 2^-24 of each."""
    N = K = 2048
    x, w = torch.zeros(M, K, device="cuda"), torch.zeros(N, K, device="cuda")
    x[:, 512:516] = w[:, 512:516] = 1.0 + 2.0 ** -11 + 2.0 ** -23
    got = projection(w).forward(x).double()
    want = x.double() @ w.double().T
    assert float(((got - want).abs() / want).max()) <= 7 * 2.0 ** -24
    x, w = operands(M, N, K, seed=9)
    x = x / x.abs().amax(1, keepdim=True) * 1e-3
    x[:, 7], w[:, 7] = 1e4, 0.0
    check(projection(w).forward(x), x, w)


@pytest.mark.parametrize("N,K", [(1024, 3072), (4096, 4096), (2048, 1028), (1000, 512)])
def test_a_row_does_not_depend_on_its_step(N, K):
    """Beyond the few rows that the weight-streaming kernels take, a row's sums are the same to the last bit however many rows
    there are, also where slices of K are left to the reader."""
    o = ops()
    x, w = operands(1100, N, K, seed=10)
    whole, cut = o.linear(x, w), o.linear(x, w, sums_ok=True)
    sums = lambda t: t.sums if hasattr(t, "sums") else t[None]
    for M in (65, 100, 209, 513):
        part = x[-M:].contiguous()
        assert torch.equal(o.linear(part, w), whole[-M:]), M
        assert torch.equal(sums(o.linear(part, w, sums_ok=True)), sums(cut)[:, -M:]), M


@pytest.mark.parametrize("value", [math.nan, math.inf])
def test_rows_that_are_no_numbers_are_not_waited_for(value):
    """One request whose stream is no number any more shares every product with the others: one such row, or all of them, cost
    no more than the float32 instruction takes for the tiles they are in (measured 2.5 and 2.9 times the product without them;
    a loop over K for every element took a hundred times as long for 64 such rows)."""
    o = ops()
    x, w = operands(512, 4096, 4096, seed=11)

    def seconds(x):
        best = math.inf
        for _ in range(5):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            o.linear(x, w)
            end.record()
            end.synchronize()
            best = min(best, start.elapsed_time(end))
        return best

    clean = seconds(x)
    one, all_ = x.clone(), x.clone()
    one[77, 5], all_[:, 5] = value, value
    assert seconds(one) < 4 * clean and seconds(all_) < 12 * clean
    got, plain = o.linear(one, w), o.linear(x, w)
    others = torch.arange(512, device="cuda") != 77
    assert not bool(torch.isfinite(got[77]).any())
    check(got[others], x[others], w)
    assert torch.equal(got[:64], plain[:64])  # (rows of other tiles: to the last bit)


@pytest.mark.parametrize("tiles", TILES)
@pytest.mark.parametrize("slices", [1, 2])
def test_rows_beside_one_that_is_no_number_keep_their_bits(tiles, slices):
    """Also those of the same matrix tile, which is made again."""
    x, w = operands(300, 192, 260, seed=13)
    odd = x.clone()
    odd[77, 5], odd[200, 100], odd[299, 259] = math.nan, math.inf, -math.inf
    got, plain = (ops().linear_f32_tiles(t, w, slices=slices, tiles=tiles) for t in (odd, x))
    fine = got.isfinite()
    assert int((~fine).sum()) == 3 * 192 and not bool(fine[:, [77, 200, 299]].all(0).any())
    assert torch.equal(got[fine], plain[fine])


@pytest.mark.parametrize("few", [False, True])
@pytest.mark.parametrize("K", [20, 512, 520, 1024, 1300, 2560, 3072, 4096])
def test_a_decoded_row_does_not_depend_on_the_batch(K, few):
    """Up to 64 rows: streamed or not, gated in one launch or in two, a row's sums are the same to the last bit."""
    o = ops()
    N = 500 if few else 2 * (17 * o.compute_units() + 5)
    x, w = operands(64, N, K, seed=12)
    x = x / x.abs().max()
    want = o.linear(x, w)
    check(want, x, w)
    gated = o.silu_mul(want)
    for M in (1, 4, 5, 16, 17, 32, 33, 63):
        assert torch.equal(o.linear(x[:M].contiguous(), w), want[:M]), M
        assert torch.equal(o.gate_up_silu(x[:M].contiguous(), w), gated[:M]), M


def test_short_products_are_not_cut():
    """Where the sums' way to the norm costs what the slices gain (512 x 512 at 32 rows, with its norm, 7.0 us whole and 10.0 cut)."""
    o = ops()
    for N, K in ((128, 512), (512, 1024), (1024, 1024)):
        assert o.f32_slices_for(32, N, K) == 1, (N, K)
    if o.compute_units() == 256:
        assert o.f32_slices_for(1, 1024, 2048) == 10 and o.f32_slices_for(64, 1024, 3072) == 16 and o.f32_slices_for(8, 4096, 12288) == 4


@pytest.mark.parametrize("M,N2,K,one", [(1, 2048, 1024, True), (32, 4096, 1024, True), (8, 4096, 1028, False), (9, 4096, 1028, True),
                                        (16, 2048, 2560, True), (17, 2048, 2560, False), (1, 2048, 2560, False), (17, 4096, 4096, False),
                                        (1, 4104, 2048, True), (17, 4104, 4096, True), (8, 8192, 4096, False), (33, 4104, 512, False)])
def test_gate_and_up_in_one_launch_or_two(monkeypatch, M, N2, K, one):
    """One where that is faster (4096 x 2048 at 17 rows took 14.8 us in two, 17.2 in one), and the same bits."""
    o = ops()
    if o.compute_units() != 256:
        pytest.skip("the choice follows the number of CUs")
    x, w = operands(M, N2, K, seed=14)
    x = x / x.abs().max()
    launched, run = [], o._run
    monkeypatch.setattr(o, "_run", lambda lib, name, *a: (launched.append(name), run(lib, name, *a))[1])
    got = o.gate_up_silu(x, w)
    assert len(launched) == (1 if one else 2), launched
    assert torch.equal(got, o.silu_mul(o.linear(x, w)))
