"""Float32 products of gate and up of many rows that take the activation with them (csrc/gemm_f32.hip): to the last bit what the product and
the activation's pass give, at the edges of the tiles and beside rows that are no numbers."""
import math

import pytest
import torch

from tests.test_gemm_f32_gpu import operands, ops

pytestmark = pytest.mark.gpu

LIMIT = 7.0


def both(x, w, tiles, activation, bias=None):
    o = ops()
    z = o.linear_f32_tiles(x, w, tiles=tiles)[0]
    return (o.gated_f32(x, w, tiles, activation, bias, LIMIT),
            o.silu_mul(z) if activation == "silu" else o.bias_act(z, "clamp", True, bias=bias, limit=LIMIT))


def same(got, want):
    return torch.equal(torch.nan_to_num(got, nan=12345.0), torch.nan_to_num(want, nan=12345.0)) and torch.equal(got.isnan(), want.isnan())


@pytest.mark.parametrize("tiles", [0, 1])
@pytest.mark.parametrize("M,N,K", [(1, 2, 4), (65, 62, 32), (128, 64, 36), (129, 66, 100), (256, 130, 28), (257, 254, 64), (300, 4098, 260)])
def test_tiles_at_their_edges(tiles, M, N, K):
    x, w = operands(M, N, K)
    bias = torch.linspace(-3.0, 3.0, N, device="cuda")
    for activation, b in (("silu", None), ("clamp", None), ("clamp", bias)):
        got, want = both(x, w, tiles, activation, b)
        assert got.shape == (M, N // 2) and same(got, want)


@pytest.mark.parametrize("tiles", [0, 1])
def test_what_is_no_number(tiles):
    """Infinities of gate, of up and of both, and NaN; the other rows of their tiles keep their bits."""
    x, w = operands(300, 192, 260, seed=13)
    clean, _ = both(x, w, tiles, "silu")
    odd = x.clone()
    odd[77, 5], odd[200, 100], odd[299, 259], odd[20, 8] = math.nan, math.inf, -math.inf, 3.4e38
    for activation in ("silu", "clamp"):
        got, want = both(odd, w, tiles, activation)
        assert same(got, want)
        if activation == "silu":
            keep = [r for r in range(300) if r not in (20, 77, 200, 299)]
            assert torch.equal(got[keep], clean[keep])
    w[7, 2], w[150, 9] = math.inf, math.nan
    assert same(*both(x, w, tiles, "silu")) and same(*both(x, w, tiles, "clamp"))


def test_which_products_are_taken(monkeypatch):
    """More rows than stream the weight, where the tiles of 128 rows of the weight are more than one for a CU; the rest is in two launches."""
    o = ops()
    if o.compute_units() != 256:
        pytest.skip("measured with 256 CUs")
    launched, run = [], o._run
    monkeypatch.setattr(o, "_run", lambda lib, name, *a: (launched.append(name), run(lib, name, *a))[1])
    for M, N, K, one in ((1024, 6144, 1024, True), (700, 8192, 1024, True), (400, 8192, 1024, False), (2048, 24576, 1024, True), (66, 192, 1024, False), (64, 6144, 1024, False), (512, 8192, 1022, False)):
        x, w = operands(M, N, K)
        x = x / x.abs().max()
        for call in (lambda: o.gate_up_silu(x, w), lambda: o.gate_up_clamped(x, w, None, LIMIT)):
            launched.clear()
            got = call()
            assert ("lle_gemm_nt_gated_f32" in launched) == one and (len(launched) == 1 or not one), (M, N, K, launched)
            assert got.shape == (M, N // 2)
        if M > 64 and K % 4 == 0:
            assert torch.equal(o.gate_up_silu(x, w), o.silu_mul(o.linear(x, w)))
