"""The delta rule's walk at the edges of its lanes' channel layout: heads of whole and of broken fours, of one and of two
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
