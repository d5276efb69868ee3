"""The weight-streaming product by way of LDS (bfloat16, up to 32 rows of X, K a multiple of 64 from 1024 on) against the same
product with operands in registers, which operands that do not begin at 16 bytes still take: the same products and sums in the
same order, so the same bits.  (test_gemm_f32_gpu.py has the float32 twins at these edges.)"""
import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

_PLAIN = [ctypes.c_void_p] * 3 + [ctypes.c_int] * 4 + [ctypes.c_void_p]
_GATED = [ctypes.c_void_p] * 3 + [ctypes.c_int] * 3 + [ctypes.c_void_p]

# few rows of X in one load of eight (1, 7, 8), two (9, 16), two tiles (17, 31, 32)
ROWS = [1, 7, 8, 9, 16, 17, 31, 32]
# tiles of four rows and of eight, of sixteen and a last one of a few; steps: one for every wavefront, two for some, more than LDS holds
SIZES = [(1024, 1024), (1030, 1088), (2048, 1600), (1024, 3072), (1500, 4160), (528, 8192)]
# more than a tile of sixteen rows for every CU (of 256), of the plain product or of the gated one too: as a stream; shares of 17, 33 and 51
# rows, the last workgroup's of one row
SIZES += [(4100, 2048), (4098, 3072), (4200, 6144), (4354, 8192), (8450, 1024), (12802, 1024), (8196, 4096), (8710, 5120)]


def ops():
    from litellmengine_amd.csrc.ops import default_ops

    return default_ops()


def operands(M, N, K, seed=0):
    g = torch.Generator(device="cuda").manual_seed(1000 * seed + M + 7 * N + 13 * K)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    return x, (torch.randn(N, K, generator=g, device="cuda") * 0.05).bfloat16()


def off_lines(x):
    """The same rows, at an address that no load into LDS takes."""
    t = torch.empty(x.numel() + 8, dtype=x.dtype, device=x.device)
    view = t[8 // x.element_size():][: x.numel()].view(x.shape)
    assert view.data_ptr() % 16 == 8
    return view.copy_(x)


def close(got, want, K):
    """Sums of exact products in 32 bits, a rounding to 16 at the end."""
    scale = want.abs().max()
    assert float((got.double() - want).abs().max() / scale) <= 2.0 ** -8 + K * 2.0 ** -24


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("N,K", SIZES)
def test_plain(M, N, K):
    o = ops()
    x, w = operands(M, N, K)
    run = lambda t, out: o._run("gemm", "lle_gemm_skinny_bf16", _PLAIN, t.data_ptr(), w.data_ptr(), out.data_ptr(), M, N, K,
                                0 if out.dtype == torch.float32 else 1)
    for dtype in (torch.bfloat16, torch.float32):
        a, b = (torch.full((M, N), math.nan, dtype=dtype, device="cuda") for _ in range(2))
        run(x, a)
        run(off_lines(x), b)
        close(a, x.double() @ w.double().T, K)
        assert torch.equal(a, b)


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("N,K", SIZES)
def test_gated(M, N, K):
    """Also gate rows that are odd in number (515)."""
    o = ops()
    x, w = operands(M, N, K, seed=1)
    gate, up = (x.double() @ w.double().T).chunk(2, dim=1)
    outs = []
    for t in (x, off_lines(x)):
        out = torch.full((M, N // 2), math.nan, dtype=torch.bfloat16, device="cuda")
        o._run("gemm", "lle_gemm_skinny_gated_bf16", _GATED, t.data_ptr(), w.data_ptr(), out.data_ptr(), M, N, K)
        outs.append(out)
    close(outs[0], torch.nn.functional.silu(gate) * up, K)
    assert torch.equal(*outs)


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("N,K", SIZES)
def test_around_a_folded_norm(M, N, K):
    """A product into the residual stream (its rows, the norm's input and sums), and products that apply the row factors."""
    from litellmengine_amd.parts import Prenormed
    from litellmengine_amd.parts.base import NormFold

    o = ops()
    x, w = operands(M, N, K, seed=2)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    hidden = torch.randn(M, N, generator=g, device="cuda")
    norm = torch.randn(N, generator=g, device="cuda").bfloat16()
    got = []
    for t in (x, off_lines(x)):
        h = hidden.clone()
        if o.can_fold_norm(M, N, x.dtype):
            pre = o.linear(t, w, fold=NormFold(h, norm, 1e-6))
            got.append((h, pre.xw, pre.sums[:M]))
    if got:
        want = hidden.double() + x.double() @ w.double().T
        close(got[0][0], want, K)
        close(got[0][1], got[0][0].double() * norm.double(), 1)
        assert torch.allclose(got[0][2].double().sum(1), (got[0][0].double() ** 2).sum(1), rtol=1e-5)
        for a, b in zip(*got):
            assert torch.equal(a, b)
    if not o.can_fold_norm(M, K, x.dtype):
        return
    sums = torch.rand(16 if M <= 16 else 32, o.norm_sum_parts(K), generator=g, device="cuda")
    factors = torch.rsqrt(sums[:M].double().sum(1) / K + 1e-6)[:, None]
    product = x.double() @ w.double().T * factors
    plain = [o.linear(Prenormed(t, sums, 1e-6), w) for t in (x, off_lines(x))]
    close(plain[0], product, K)
    assert torch.equal(*plain)
    gated = [o.gate_up_silu(Prenormed(t, sums, 1e-6), w) for t in (x, off_lines(x))]
    gate, up = product.chunk(2, dim=1)
    close(gated[0], torch.nn.functional.silu(gate) * up, K)
    assert torch.equal(*gated)


def test_replayed_in_a_graph():
    """One launch and nothing kept between them: every replay gives the eager bits."""
    o = ops()
    x, w = operands(5, 1024, 2048, seed=3)
    want = o.linear(x, w)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = o.linear(x, w)
    for _ in range(3):
        out.fill_(math.nan)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        o.linear(x, w)


@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 33, 48, 49, 64])
@pytest.mark.parametrize("N,K", [(1024, 512), (1030, 544), (2000, 1600), (4100, 2048), (4354, 4096), (8450, 1024), (12802, 512)])
def test_float32(M, N, K):
    """Tiles and steps as above, three and four tiles of X's rows; sums of K float32 products: 2^-24 (K + 16) of their sizes at most.
    The last row alone gives the bits that it has among the others."""
    o = ops()
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device="cuda")
    w = torch.randn(N, K, generator=g, device="cuda")
    out = torch.full((M, N), math.nan, device="cuda")
    run = lambda t, y: o._run("gemm", "lle_gemm_skinny_f32", _GATED, t.data_ptr(), w.data_ptr(), y.data_ptr(), t.shape[0], N, K)
    run(x, out)
    size = x.double().abs() @ w.double().abs().T
    assert bool(((out.double() - x.double() @ w.double().T).abs() <= 2.0 ** -24 * (K + 16) * size).all())
    last = torch.full((1, N), math.nan, device="cuda")
    run(x[-1:].contiguous(), last)
    assert torch.equal(last, out[-1:])


@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33, 48, 64])
@pytest.mark.parametrize("N,K,slices", [(64, 32, 1), (100, 96, 3), (1024, 2048, 10), (72, 2080, 5), (130, 3072, 4), (64, 4160, 2)])
def test_float32_slices(M, N, K, slices):
    """One step for one of four wavefronts and none for the others, slices of 16 steps and of 17, the last one shorter, columns that fill no
    group of 64: the bits of operand-shaped loads, which an address that is no multiple of 16 still takes."""
    o = ops()
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda")
    got = o.linear_f32_slices(x, w, slices)
    size = x.double().abs() @ w.double().abs().T
    assert bool(((got.double().sum(0) - x.double() @ w.double().T).abs() <= 2.0 ** -24 * (K + 16) * size).all())
    assert torch.equal(got, o.linear_f32_slices(off_lines(x), w, slices))


@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("N,K,N2", [(1024, 2048, 1000), (1536, 512, 4100), (520, 1300, 700), (2048, 72, 8450), (4096, 4160, 516)])
def test_a_float32_norm_folded_into_products(M, N, K, N2):
    """The residual rows, the norm's input and sums behind a product, and the products after the norm, plain and gated, in float64; the last
    row alone has the bits that it has among the others (also where a tile holds two parts of the sums); operands at odd
    addresses are taken."""
    from litellmengine_amd.parts import NormFold

    o = ops()
    if not o.can_fold_norm_f32(M, N):
        assert N % 32 != 0
        return
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda") * 0.05
    hidden, norm = torch.randn(M, N, generator=g, device="cuda"), 1 + 0.3 * torch.randn(N, generator=g, device="cuda")
    hidden[:, N - 3] += 20.0
    w2 = torch.randn(N2, N, generator=g, device="cuda") * 0.1
    want = hidden.double() + x.double() @ w.double().T
    normed = want * torch.rsqrt((want ** 2).mean(1, keepdim=True) + 1e-6) * norm.double()
    y = normed @ w2.double().T
    gate, up = y.chunk(2, dim=1)

    def run(x, hidden, w, w2):
        h = hidden.clone()
        pre = o.linear(x, w, fold=NormFold(h, norm, 1e-6))
        return h, pre.xw, pre.sums[: x.shape[0]], o.linear(pre, w2), o.gate_up_silu(pre, w2)

    got = run(x, hidden, w, w2)
    # a row's products of K and N float32 numbers: a rounding for each, and for their sums', of their sizes; the gate's slope is below 1.1
    size = (x.double().abs() @ w.double().abs().T + hidden.double().abs()) * 2.0 ** -24 * (K + 16)
    assert bool(((got[0].double() - want).abs() <= size).all())
    assert torch.allclose(got[1].double(), got[0].double() * norm.double(), rtol=2.0 ** -23, atol=0)
    assert torch.allclose(got[2].double().sum(1), (got[0].double() ** 2).sum(1), rtol=1e-5)
    for mine, exact in ((got[3], y), (got[4], torch.nn.functional.silu(gate) * up)):
        assert float((mine.double() - exact).norm() / exact.norm()) <= 2.0 ** -24 * 40
    for a, b in zip(got, run(x[-1:].contiguous(), hidden[-1:].contiguous(), w, w2)):
        assert torch.equal(a[-1:], b)
    odd = run(off_lines(x), hidden, off_lines(w), off_lines(w2))
    assert float((odd[4].double() - got[4].double()).norm() / got[4].double().norm()) <= 2.0 ** -24 * 40


@pytest.mark.parametrize("M", [1, 7, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(12290, 4096), (12800, 3072), (24576, 4096), (20996, 3072)])
def test_float32_gated_streams_of_long_rows(M, N, K):
    """Shares of 25, 25, 48 and 42 gate rows, the last workgroup's whole or of a few: one launch, plain and behind a folded norm, to the last bit what
    the product and silu_mul give."""
    from litellmengine_amd.parts import Prenormed

    o = ops()
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda") * 0.05
    sums = torch.rand(16, o.norm_sum_parts(K), generator=g, device="cuda") * K
    if o.compute_units() == 256:
        assert o._gated_f32_in_one(M, N, K) and not any(o._gated_f32_in_one(M, n, K) for n in (8192, 8704, 16896))
    gate, up = (x.double() @ w.double().T).chunk(2, dim=1)
    got, want = o.gate_up_silu(x, w), torch.nn.functional.silu(gate) * up
    assert float((got.double() - want).norm() / want.norm()) <= 2.0 ** -24 * 40
    assert torch.equal(got, o.silu_mul(o.linear(x, w)))
    assert torch.equal(o.gate_up_silu(Prenormed(x, sums, 1e-6), w), o.silu_mul(o.linear(Prenormed(x, sums, 1e-6), w)))
