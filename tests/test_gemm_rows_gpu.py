"""bfloat16 products of 33 to 256 rows that take the weight in one round of the CUs (csrc/gemm_rows.hip): whole ones, silu, the clamped one."""
import pytest
import torch

from tests.test_gemm_wide_gpu import LIMIT, bounds
from tests.test_kernels_gpu import ops, rnd

pytestmark = pytest.mark.gpu


# one to four tiles of 64 rows of X at their edges (four only gated); one stage, two, more than LDS holds; weights that end inside a workgroup's rows, its
# sixteen and its eight
@pytest.mark.parametrize("M", [1, 33, 64, 65, 128, 129, 192, 193, 256])
@pytest.mark.parametrize("N,K,tile", [(8, 256, 8), (520, 512, 8), (1000, 1024, 16), (1336, 2816, 24), (1032, 4096, 32), (2104, 768, 40), (1640, 1280, 48)])
def test_rows_product(M, N, K, tile):
    x, w = rnd((M, K), torch.bfloat16, 1), rnd((N, K), torch.bfloat16, 2, 2.0 * K ** -0.5)
    if M <= 192:
        got = ops().linear_rows(x, w, tile).double()
        want = x.double() @ w.double().T
        # sums of K products in 32 bits, half of their roundings a margin, and the result's to 8 bits
        off = (x.double().abs() @ w.double().abs().T) * K * 2.0 ** -24 + 2.0 ** -8 * want.abs() + 1e-30
        assert got.shape == want.shape and ((got - want).abs() <= off).all()
    for activation, bias in (("silu", None), ("clamp", None), ("clamp", rnd((N,), torch.bfloat16, 3))):
        got = ops().linear_rows(x, w, tile, activation, bias, LIMIT).double()
        want, off = bounds(x, w, bias, activation)
        assert got.shape == want.shape and ((got - want).abs() <= off).all()


def test_what_is_not_finite_stays_in_its_row_and_column():
    x, w = rnd((100, 512), torch.bfloat16, 1), rnd((512, 512), torch.bfloat16, 2)
    clean = ops().linear_rows(x, w, 16)
    x[77, 5], w[300, 9] = float("inf"), float("nan")
    got = ops().linear_rows(x, w, 16)
    assert not got[77].isfinite().any() and got[:, 300].isnan().all()
    keep = torch.ones_like(clean, dtype=torch.bool)
    keep[77], keep[:, 300] = False, False
    assert torch.equal(got[keep], clean[keep])


def test_which_products_are_taken(monkeypatch):
    """By the sizes: the rows of X, one round of the CUs, X not many times the CU's share of W; and operands that begin at 16 bytes."""
    o = ops()
    if o.compute_units() != 256:
        pytest.skip("measured with 256 CUs")
    shape = lambda M, K: torch.empty((M, K), dtype=torch.bfloat16, device="cuda")
    tile = lambda M, N, K, gated: o.rows_tile(shape(M, K), shape(N, K), gated)
    assert [tile(M, 24576, 4096, True) for M in (32, 33, 256, 257)] == [0, 48, 48, 0]
    assert [tile(M, 6144, 4096, False) for M in (32, 33, 128, 129)] == [0, 24, 24, 0]
    assert [tile(M, N, K, True) for M, N, K in ((193, 16384, 2048), (192, 16384, 2048), (256, 8192, 1024), (256, 8192, 2048))] == [0, 32, 16, 0]
    assert tile(64, 51200, 5120, True) == 0 and tile(64, 12296, 1024, False) == 0 and tile(64, 12288, 1024, False) == 48
    assert tile(64, 2048, 4096, False) == 8 and tile(65, 2048, 4096, False) == 0 and tile(64, 4096, 8192, False) == 0
    assert tile(64, 6144, 960, True) == 0 and tile(64, 6144, 1152, True) == 0 and tile(64, 6148, 1024, True) == 0
    odd = shape(65, 1024).view(-1)[4: 4 + 64 * 1024].view(64, 1024)
    assert o.rows_tile(odd, shape(4096, 1024), False) == 0 and o.linear(odd, shape(4096, 1024)).shape == (64, 4096)
    launched, run = [], o._run
    monkeypatch.setattr(o, "_run", lambda lib, name, *a: (launched.append(name), run(lib, name, *a))[1])
    x, w = rnd((40, 1024), torch.bfloat16, 4), rnd((6144, 1024), torch.bfloat16, 5, 0.05)
    for call in (lambda: o.linear(x, w), lambda: o.gate_up_silu(x, w), lambda: o.gate_up_clamped(x, w, None, LIMIT)):
        launched.clear()
        call()
        assert launched == ["lle_gemm_rows_bf16"]
    assert o.linear(x, w, out_dtype=torch.float32).dtype == torch.float32
