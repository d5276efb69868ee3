"""The norms that add into the residual stream, where few rows take more threads each: at the widths and numbers of rows where that changes."""
import pytest
import torch

from tests.test_kernels_gpu import ops, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [1, 256, 257, 512, 513])
@pytest.mark.parametrize("H", [1024, 1028, 2048, 2052, 4096, 4100, 8192])
def test_few_rows_and_many(R, H):
    o = ops()
    hidden, w = rnd((R, H), torch.float32, 1), (1 + 0.3 * rnd((H,), torch.float32, 2)).bfloat16()
    a, b, vec = rnd((R, H), torch.bfloat16, 3), rnd((R, H), torch.bfloat16, 4), rnd((H,), torch.float32, 5)
    sums = rnd((3, R, H), torch.float32, 6)
    hidden[:, H - 1] += 20.0  # (the last element dominates the mean)
    x = hidden.double()
    for new, call in ((x + a.double(), lambda h: o.add_rmsnorm(h, a, w, 1e-3, torch.bfloat16)),
                      (x + sums.double().sum(0), lambda h: o.add_rmsnorm(h, sums, w, 1e-3, torch.bfloat16)),
                      (x + 0.5 * a.double() + 0.25 * b.double(), lambda h: o.scaled_add_rmsnorm(h, a, b, 0.5, w, 1e-3, torch.bfloat16, mult_b=0.25)),
                      (x + a.double() + vec.double(), lambda h: o.inject_rmsnorm(h, a, vec, None, w, 1e-3, torch.bfloat16))):
        h = hidden.clone()
        got = call(h).double()
        want = new * torch.rsqrt((new ** 2).mean(1, keepdim=True) + 1e-3) * w.double()
        # a few roundings of numbers up to 24 in 32 bits; the result's rounding to 8 bits and the norm's factor
        assert float((h.double() - new).abs().max()) <= 8 * 24 * 2.0 ** -24
        assert bool(((got - want).abs() <= (2.0 ** -8 + 2.0 ** -18) * want.abs() + 1e-5).all())
