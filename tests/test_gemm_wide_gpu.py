"""Tiled bfloat16 products of many rows, gate and up with the activation between them (csrc/gemm_wide.hip): silu, the clamped one."""
import pytest
import torch

from tests.test_kernels_gpu import ops, rnd

pytestmark = pytest.mark.gpu
LIMIT = 3.0


def bounds(x, w, bias, activation):
    """(the result in 64 bits, how far a correct one may be from it): products and sums in 32 bits (K roundings of the sum of the
    magnitudes at most, half of them used up by a margin), the activation's slope (1.1 for silu, 1.7 for the clamped one, whose other
    factor is at most LIMIT + 1), the hardware's exponential and reciprocal, the result rounded to 8 bits."""
    x, w = x.double(), w.double()
    z, size = x @ w.T, (x.abs() @ w.abs().T) * x.shape[1] * 2.0 ** -24
    if bias is not None:
        z = z + bias.double()
    half = w.shape[0] // 2
    (g, u), (eg, eu) = z.split(half, 1), size.split(half, 1)
    if activation == "silu":
        want = g * torch.sigmoid(g) * u
        off = 1.1 * eg * u.abs() + g.abs() * eu
    else:
        g, u = g.clamp(max=LIMIT), u.clamp(-LIMIT, LIMIT)
        want = g * torch.sigmoid(1.702 * g) * (u + 1.0)
        off = 1.7 * eg * (LIMIT + 1) + g.abs() * eu
    return want, off + (2.0 ** -8 + 2.0 ** -18) * want.abs() + 1e-30


# one stage, two, odd and even numbers of them; rows and columns that end inside a tile, a half, a fragment; one row, more tiles
# than CUs (dies with unequal shares), bands of unequal height
@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (129, 264, 128), (128, 256, 192), (257, 520, 256), (191, 1000, 320), (193, 1032, 1024),
                                   (383, 512, 64), (2111, 776, 128), (700, 8200, 192), (2500, 4104, 64), (289, 520, 384)])
@pytest.mark.parametrize("activation,form", [(a, f) for a in ("silu", "clamp") for f in range(11)])
def test_wide_product(M, N, K, activation, form):
    x, w = rnd((M, K), torch.bfloat16, 1), rnd((N, K), torch.bfloat16, 2, 2.0 * K ** -0.5)
    for bias in ((None, rnd((N,), torch.bfloat16, 3)) if activation == "clamp" else (None,)):
        got = ops().gated_wide(x, w, form, activation, bias, LIMIT).double()
        want, off = bounds(x, w, bias, activation)
        assert got.shape == want.shape and ((got - want).abs() <= off).all()


def test_wide_product_keeps_what_is_not_finite_in_its_row_and_column():
    x, w = rnd((300, 128), torch.bfloat16, 1), rnd((512, 128), torch.bfloat16, 2)
    clean = ops().gated_wide(x, w, 4, "silu")
    x[77, 5], w[300, 9] = float("inf"), float("nan")  # (row 300: the up row of column 44)
    got = ops().gated_wide(x, w, 4, "silu")
    g, u = (x.double() @ w.double().t()).split(256, 1)
    assert torch.equal(got[77].isnan(), (g * torch.sigmoid(g) * u)[77].isnan()) and got[:, 44].isnan().all()
    keep = torch.ones_like(clean, dtype=torch.bool)
    keep[77], keep[:, 44] = False, False
    assert torch.equal(got[keep], clean[keep])


def test_which_products_are_taken_in_wide_tiles():
    o = ops()
    if o.compute_units() != 256:
        pytest.skip("measured with 256 CUs")
    shape = lambda M, K: torch.empty((M, K), dtype=torch.bfloat16, device="cuda")
    x, w = shape(2048, 4096), shape(24576, 4096)
    assert o.wide_form(x, w) == 0 and o.wide_form(x[:128], w) == -1
    assert o.wide_form(x[:, :4090].contiguous(), w[:, :4090].contiguous()) == -1
    assert o.wide_form(x[:262], w) >= 0 and o.wide_form(shape(129, 1024), shape(6144, 1024)) == -1
    o.force_library_gemm = True
    try:
        assert o.wide_form(x, w) == -1
    finally:
        o.force_library_gemm = False


@pytest.mark.parametrize("activation", ["silu", "clamp"])
def test_operands_that_do_not_begin_at_16_bytes_are_the_librarys(activation):
    o = ops()
    M, N, K = 2048, 8192, 1024
    x, w, bias = rnd((M * K + 1,), torch.bfloat16, 1), rnd((N, K), torch.bfloat16, 2, 0.06), rnd((N + 1,), torch.bfloat16, 3)
    run = {"silu": lambda x, b: o.gate_up_silu(x, w), "clamp": lambda x, b: o.gate_up_clamped(x, w, b, LIMIT)}[activation]
    odd, odd_bias = x[1:].view(M, K), bias[1:]
    assert odd.data_ptr() % 16 and o.wide_form(odd, w) == -1
    # (the library's way rounds gate and up to 16 bits before the activation)
    want = run(odd.clone(), odd_bias.clone()).double()
    assert (run(odd, odd_bias).double() - want).norm() <= 1e-2 * want.norm()
    assert (run(odd.clone(), odd_bias).double() - want).norm() <= 1e-2 * want.norm()
