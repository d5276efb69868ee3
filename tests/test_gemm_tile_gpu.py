"""The bfloat16 product in tiles and slices of K against float64: every tile shape at its edges, slices without work, and which
products take it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def ops():
    from litellmengine_amd.csrc.ops import default_ops

    return default_ops()


@pytest.mark.parametrize("tiles", [-1, 0, 1, 2])
@pytest.mark.parametrize("M,N,K,slices", [(1, 4, 64, 1), (64, 128, 64, 1), (65, 132, 128, 2), (257, 124, 192, 2), (255, 256, 448, 3),
                                          (130, 1028, 1088, 16), (300, 640, 320, 5), (40, 2048, 640, 4)])
def test_partial_sums(tiles, M, N, K, slices):
    """Products of bfloat16 numbers are exact in float32, so a sum of K of them is off by K roundings at most (slices that are
    left without a stage are zeros).  Rows that tell their number show a tile in the wrong place."""
    g = torch.Generator(device="cuda").manual_seed(M + 3 * N + 5 * K)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = torch.randn(N, K, generator=g, device="cuda").bfloat16()
    x[:, 0], w[:, 1] = torch.arange(M, device="cuda") % 128, torch.arange(N, device="cuda") % 128
    got = ops().linear_tile_sums(x, w, slices, tiles)
    assert got.shape == (slices, M, N)
    each = -(-(K // 64) // slices) * 64
    for s in range(slices):
        xs, ws = x[:, s * each : (s + 1) * each].double(), w[:, s * each : (s + 1) * each].double()
        off = (got[s].double() - xs @ ws.T).abs()
        assert bool((off <= 2.0 ** -24 * (each + 16) * (xs.abs() @ ws.abs().T)).all()), s


def test_which_products_take_it():
    from litellmengine_amd.parts import PartialSums

    o = ops()
    if o.compute_units() != 256:
        pytest.skip("the choice follows the number of CUs")
    took = lambda m, n, k: o.tile_slices_for(m, n, k) > 0
    assert took(96, 4096, 12288) and not took(209, 4096, 12288) and not took(16, 4096, 12288) and not took(32, 4096, 12288)
    assert not took(96, 4096, 4096) and took(129, 4096, 4096) and took(512, 4096, 4096) and not took(513, 4096, 4096)
    assert took(17, 5120, 25600) and took(17, 5120, 8192) and took(2048, 1024, 2048) and not took(2049, 1024, 2048)
    assert not took(96, 4096, 12288 + 32) and not took(96, 8196, 32768) and not took(96, 64, 128)
    # the library's tiles fill the CUs, or its slices of K are better (measured 6 to 24 % faster)
    for m, n, k in ((400, 6144, 4096), (330, 8192, 8192), (512, 5120, 2048), (1536, 1024, 4096), (2048, 768, 4096)):
        assert not took(m, n, k), (m, n, k)
    assert took(512, 5120, 8192) and took(330, 4096, 4096) and took(1536, 512, 2048) and took(2048, 1024, 3072)
    # in 3 slices and tiles of 64 rows a die would get 33 workgroups for its 32 CUs
    assert o.tile_slices_for(129, 3584, 3584) != 3
    x, w = torch.randn(200, 4096, device="cuda").bfloat16(), torch.randn(4096, 4096, device="cuda").bfloat16()
    cut = o.linear(x, w, sums_ok=True)
    assert isinstance(cut, PartialSums) and o.linear(x, w).shape == (200, 4096)
    want = x.double() @ w.double().T
    assert float((cut.total().double() - want).norm() / want.norm()) < 2.0 ** -24 * 64  # (sqrt(K) roundings)


def test_other_numbers_choose_anew(monkeypatch):
    """The form that was chosen for a product's sizes is chosen again when the numbers behind the choice change."""
    import dataclasses

    from litellmengine_amd.csrc.ops import HipOps

    o = ops()
    sizes = [(m, n, k) for m in (17, 64, 100, 512) for n, k in ((4096, 4096), (4096, 12288), (1024, 3072))]
    before = [o._form_of_delta(torch.bfloat16, *s) for s in sizes]
    other = dataclasses.replace(o.tuning, sliced_min_fill=0.0, partial_sums_bytes_per_s=1e15, library_max_slices=1)
    monkeypatch.setattr(o, "tuning", other)
    assert [o._form_of_delta(torch.bfloat16, *s) for s in sizes] == [HipOps(tuning=other)._form_of_delta(torch.bfloat16, *s) for s in sizes]
    monkeypatch.undo()
    assert [o._form_of_delta(torch.bfloat16, *s) for s in sizes] == before
