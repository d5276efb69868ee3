"""The walks of the delta rule and of the state-space heads at the edges of their lanes' channel layout: heads of whole and of broken fours, of one and of two
stretches of channels, of more than 128; chunks of tokens that are just whole, one short and one over; state rows that
16-byte loads can and cannot reach."""
import pytest
import torch

from .torch_ops import TorchOps

pytestmark = pytest.mark.gpu
REF = TorchOps()


@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("pad", [0, 1, 4])
@pytest.mark.parametrize("dim,vdim", [(64, 64), (63, 17), (65, 8), (128, 20), (129, 9), (256, 24), (32, 16), (16, 33)])
def test_walk_over_whole_and_broken_layouts(dim, vdim, pad, channel):
    from litellmengine_amd.csrc.ops import HipOps

    H, G, lens = 2, 1, [16, 1, 15, 33]
    N, rand = sum(lens), torch.Generator().manual_seed(dim * 8 + pad)
    f = lambda *shape: torch.randn(shape, generator=rand).cuda()
    unit = lambda t: torch.nn.functional.normalize(t.view(N, G, dim), dim=-1).reshape(N, G * dim).contiguous()
    q, k, v, ba = unit(f(N, G * dim)), unit(f(N, G * dim)), f(N, H * vdim), f(N, 2 * H)
    a_log, dt_bias = (None, None) if channel else (f(H), f(H))
    decay = torch.sigmoid(3.0 * f(N, H * dim)) if channel else None
    ints = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    cu, slots = ints([0, 16, 17, 32, 65]), ints([3, 0, 4, 1])
    start = 0.3 * f(6, H * vdim * dim + pad)
    a, b = start.clone(), start.clone()
    want = REF.delta_scan(q, k, v, ba, a_log, dt_bias, a, H, G, dim, vdim, slots, cu, decay=decay)
    got = HipOps().delta_scan(q, k, v, ba, a_log, dt_bias, b, H, G, dim, vdim, slots, cu, decay=decay)
    # |S| stays of the order of |v| + |S_0| (unit keys, decays and betas up to one): 33 tokens of sums of up to 256 products in
    # 32 bits, 33 x 16 x 2^-24 = 3e-5 of values up to about 3
    assert (got.double() - want.double()).abs().max() < 1e-4
    assert (a.double() - b.double()).abs().max() < 1e-4
    assert torch.equal(b[:, H * vdim * dim:], start[:, H * vdim * dim:]) and torch.equal(b[2], start[2]) and torch.equal(b[5], start[5])


@pytest.mark.parametrize("pad", [0, 3, 8])
@pytest.mark.parametrize("n,vdim", [(128, 64), (127, 16), (64, 17), (65, 4), (256, 20), (200, 3), (16, 33), (30, 8)])
def test_state_space_walk_over_whole_and_broken_layouts(n, vdim, pad):
    from litellmengine_amd.csrc.ops import HipOps

    H, G, lens = 4, 2, [1, 9, 8, 32]
    N, rand = sum(lens), torch.Generator().manual_seed(n * 8 + pad)
    f = lambda *shape: torch.randn(shape, generator=rand).cuda()
    c, dt_in, dt_bias, a_log, D = f(N, H * vdim + 2 * G * n), f(N, H), f(H), f(H), f(H)
    ints = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    cu, slots = ints([0, 1, 10, 18, 50]), ints([3, 0, 4, 1])
    start = 0.3 * f(6, H * vdim * n + pad)
    a, b = start.clone(), start.clone()
    want = REF.ssd_scan(c, dt_in, dt_bias, a_log, D, a, H, G, vdim, n, slots, cu, 1, 32)
    got = HipOps().ssd_scan(c, dt_in, dt_bias, a_log, D, b, H, G, vdim, n, slots, cu, 1, 32)
    # sums of up to 256 products and 32 steps in 32 bits beside terms of that size: (256 + 32) x 2^-24 = 2e-5 of the largest
    assert (got.double() - want.double()).abs().max() < 2e-5 * max(1.0, float(want.abs().max()))
    assert (a.double() - b.double()).abs().max() < 2e-5 * max(1.0, float(a.abs().max()))
    assert torch.equal(b[:, H * vdim * n:], start[:, H * vdim * n:]) and torch.equal(b[2], start[2]) and torch.equal(b[5], start[5])
