"""Products into the residual stream of 17 to 32 rows, whose workgroups take sixteen rows of X each: the edges of the row halves, of
tiles of W and of the parts of the norm's sums."""
import pytest
import torch

from tests.test_kernels_gpu import ops, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [16, 17, 31, 32])
@pytest.mark.parametrize("H,K", [(64, 64), (72, 40), (1024, 3072), (1032, 520), (2048, 2048), (2040, 128)])
def test_residual_product_and_sums_of_squares(M, H, K):
    from litellmengine_amd.parts import NormFold

    o = ops()
    a, w = rnd((M, K), torch.bfloat16, 1), rnd((H, K), torch.bfloat16, 2, 0.2)
    hidden, nw = rnd((M, H), torch.float32, 3), 1 + 0.3 * rnd((H,), torch.float32, 4)
    hidden[M - 1, H - 1] += 30.0  # the last row and column count
    want = hidden.double() + a.double() @ w.double().t()
    pre = o.linear(a, w, fold=NormFold(hidden, nw, 1e-3))
    # sums of up to 3072 products in 32 bits, spread over sixteen wavefronts: 200 x 2^-24 of sums of terms of size |x| |w| sqrt(K)
    assert (hidden.double() - want).abs().max() < 2e-5 * float(want.abs().max())
    assert pre.sums.shape[1] == o.norm_sum_parts(H)
    assert torch.allclose(pre.sums.double().sum(1)[:M], (want ** 2).sum(1), rtol=1e-5)
