"""The state-space recurrence's chunks, whose workgroups take several heads of a group one after the
other: every number of value tiles (odd ones hand the next head's entry rows over), widths of LDS rows,
states of one and of two register sets, sizes that 16-byte loads do not fit, and more heads a group than
a workgroup holds step sizes of."""

import pytest
import torch

from tests.test_kezasun_kernels_gpu import ops
from tests.test_rorevik_kernels_gpu import REF, close, ssd_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("together,H,G,vdim,n", [
    (3, 6, 2, 48, 132), (4, 4, 1, 80, 128), (2, 4, 2, 16, 20), (5, 5, 1, 20, 6), (4, 4, 1, 6, 33), (2, 2, 1, 144, 64), (2, 2, 1, 208, 100),
    (40, 40, 1, 16, 16), (34, 68, 2, 32, 24), (37, 37, 1, 12, 8)])
def test_heads_of_a_workgroup(together, H, G, vdim, n, monkeypatch):
    """The rows and states are those of a workgroup a head to the last bit, and the oracle's."""
    o = ops()
    q_lens = [130, 33, 1, 64]
    c, dt_in, dt_bias, a_log, D, wide, seq_slots, cu = ssd_case(H, G, vdim, n, q_lens)
    args = (c, dt_in, dt_bias, a_log, D)
    got = {}
    for k in (1, together):
        monkeypatch.setattr(o, "ssd_heads_a_group", lambda *a, k=k: k)
        state = wide.clone()
        got[k] = o.ssd_scan(*args, state, H, G, vdim, n, seq_slots, cu, 1, 130), state
    assert torch.equal(got[1][0], got[together][0]) and torch.equal(got[1][1], got[together][1])
    state = wide.clone()
    want = REF.ssd_scan(*args, state, H, G, vdim, n, seq_slots, cu)
    # sums of at most 64 tokens and n <= 132 channels, in 32 bits: under 64 roundings of the largest result
    close(got[together][0], want, 64 * 2**-24 * max(1.0, float(want.abs().max())))
    close(got[together][1], state, 64 * 2**-24 * max(1.0, float(state.abs().max())))
